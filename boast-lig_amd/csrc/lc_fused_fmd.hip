// lc_fused_fmd.hip -- fused 3D kernel variants for the FMD filter.
#include "lc_fused_impl.hpp"

namespace lc {
LC_FUSED_INSTANTIATE(double, FMD)
LC_FUSED_INSTANTIATE(float, FMD)
template hipError_t launch_sepq_pot<double>(const Box3&, const double*, double*, double, hipStream_t,
                                            const double*, double*);
template hipError_t launch_sepq_pot<float>(const Box3&, const float*, float*, float, hipStream_t, const float*,
                                           float*);
}  // namespace lc
