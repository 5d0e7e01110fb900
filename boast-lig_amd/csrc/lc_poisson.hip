// lc_poisson.hip -- the Poisson nabla operators (BigDFT/Poisson2.rb) on the GPU.
//
// First derivatives of order nord in {2, 4, 6, 8, 16} along the dims of a 3D
// grid, with the border rows of GenericConvolution2.rb:237-294 (PoissonFilter):
// on a periodic dim every output uses the centred row with wrap-around; on a
// non-periodic dim (bc -2) output i < m uses row i - m on inputs 0 .. 2m and
// output i >= n - m row i - n + m + 1 on inputs n - 1 - 2m .. n - 1.  The
// weights are the exact Lagrange weights of lc_taps.h.
//
// These stencils are short (nord + 1 taps) and carry ~2 flop per byte, so the
// kernels are HBM / L2 bound: one lane per output point, x fastest across the
// lanes of a wave (coalesced loads and stores); the taps of one output along
// a strided dim are loads of the same lanes at a fixed offset, which the L2
// serves: each XCD works through its own slab of every plane in z order
// (pblock), so the planes a z stencil needs are in its L2.  Each operator is
// one pass:
//   poisson_1d:          du = a D_idim u (+ a_y du)          (Poisson_broker)
//   div_u_i:             du = sum_k D_k u_k / h_k, optional cc
//   nabla_u:             du_k = D_k u / h_k
//   nabla_u_and_square:  the same and du2 = |du|^2
//   nabla_u_square:      du2 only
//   nabla_u_epsilon:     du_k = eps D_k u / h_k
//   update_rhopol:       res = eta ((dlogeps . du) / (4 pi) - rhopol),
//                        rhopol += res, rhores2 = sum res^2
// The derivative sums run in increasing tap order, as the reference loops;
// the 1 / h_k factors are products with the rounded reciprocals (within an
// ulp of the quotients: a division is a dozen FP64 instructions).
#include <hip/hip_runtime.h>

#include <algorithm>

#include <stdlib.h>

#include "lc_common.hpp"
#include "lc_fused.hpp"
#include "lc_kernels.hpp"
#include "lc_taps.h"

namespace lc {

namespace {

#define LC_PQD(p, q) ((double)(p) / (double)(q)),
#define LC_PQF(p, q) (float)((double)(p) / (double)(q)),
__constant__ double kPoiD2[] = {LC_POISSON_2(LC_PQD)};
__constant__ double kPoiD4[] = {LC_POISSON_4(LC_PQD)};
__constant__ double kPoiD6[] = {LC_POISSON_6(LC_PQD)};
__constant__ double kPoiD8[] = {LC_POISSON_8(LC_PQD)};
__constant__ double kPoiD16[] = {LC_POISSON_16(LC_PQD)};
__constant__ float kPoiF2[] = {LC_POISSON_2(LC_PQF)};
__constant__ float kPoiF4[] = {LC_POISSON_4(LC_PQF)};
__constant__ float kPoiF6[] = {LC_POISSON_6(LC_PQF)};
__constant__ float kPoiF8[] = {LC_POISSON_8(LC_PQF)};
__constant__ float kPoiF16[] = {LC_POISSON_16(LC_PQF)};
// the same rows as compile-time constants: the z-marching kernels' centred
// taps then become instruction operands, not loads
template <int NORD>
struct PoiRows;
#define LC_POI_ROWS(NO)                                       \
  template <>                                                 \
  struct PoiRows<NO> {                                        \
    static constexpr double d[] = {LC_POISSON_##NO(LC_PQD)};  \
    static constexpr float f[] = {LC_POISSON_##NO(LC_PQF)};   \
  };
LC_POI_ROWS(2)
LC_POI_ROWS(4)
LC_POI_ROWS(6)
LC_POI_ROWS(8)
LC_POI_ROWS(16)
#undef LC_POI_ROWS
#undef LC_PQD
#undef LC_PQF

template <typename R, int NORD>
__device__ __forceinline__ constexpr R prow(int k) {
  if constexpr (sizeof(R) == 8) return PoiRows<NORD>::d[k]; else return PoiRows<NORD>::f[k];
}

template <typename R, int NORD>
__device__ __forceinline__ const R* ptab() {
  if constexpr (sizeof(R) == 8) {
    if constexpr (NORD == 2) return kPoiD2;
    else if constexpr (NORD == 4) return kPoiD4;
    else if constexpr (NORD == 6) return kPoiD6;
    else if constexpr (NORD == 8) return kPoiD8;
    else return kPoiD16;
  } else {
    if constexpr (NORD == 2) return kPoiF2;
    else if constexpr (NORD == 4) return kPoiF4;
    else if constexpr (NORD == 6) return kPoiF6;
    else if constexpr (NORD == 8) return kPoiF8;
    else return kPoiF16;
  }
}

// unscaled derivative at point i of a line of n points (stride s) starting at
// `line`; per: periodic
template <typename R, int NORD>
__device__ __forceinline__ R pderiv(const R* __restrict__ line, long s, int n, int i, bool per) {
  constexpr int M = NORD / 2, W = NORD + 1;
  const R* c = ptab<R, NORD>();
  R t = R(0);
  if (i >= M && i < n - M) {  // interior: centred row, no wrap
    const R* row = c + M * W;
#pragma unroll
    for (int j = -M; j <= M; ++j) t = fmar(row[j + M], line[(long)(i + j) * s], t);
  } else if (per) {
    const R* row = c + M * W;
#pragma unroll
    for (int j = -M; j <= M; ++j) t = fmar(row[j + M], line[(long)pmod(i + j, n) * s], t);
  } else if (i < M) {
    const R* row = c + i * W;  // row i - m
#pragma unroll
    for (int j = -M; j <= M; ++j) t = fmar(row[j + M], line[(long)(j + M) * s], t);
  } else {
    const R* row = c + (i - n + 2 * M + 1) * W;  // row i - n + m + 1
#pragma unroll
    for (int j = -M; j <= M; ++j) t = fmar(row[j + M], line[(long)(n - 1 - M + j) * s], t);
  }
  return t;
}

struct PGeom {
  int n0, n1, n2;
  long np;
  bool per0, per1, per2;
  int z0, nz;  // planes the one-point kernels compute: z0 .. z0 + nz - 1
};

__device__ __forceinline__ void pcoords(const PGeom& g, long p, int& i0, int& i1, int& i2) {
  i0 = (int)(p % g.n0);
  const long q = p / g.n0;
  i1 = (int)(q % g.n1);
  i2 = (int)(q / g.n1);
}

template <typename R, int NORD>
__device__ __forceinline__ R dk(const PGeom& g, const R* __restrict__ f, long p, int k, int i0, int i1,
                                int i2) {
  const long s1 = g.n0, s2 = (long)g.n0 * g.n1;
  if (k == 0) return pderiv<R, NORD>(f + (p - i0), 1, g.n0, i0, g.per0);
  if (k == 1) return pderiv<R, NORD>(f + (p - (long)i1 * s1), s1, g.n1, i1, g.per1);
  return pderiv<R, NORD>(f + (p - (long)i2 * s2), s2, g.n2, i2, g.per2);
}

constexpr int kPThreads = 256;

// Block -> (plane z, 256-point segment of the plane).  The dispatcher hands
// consecutive block ids to the 8 XCDs in turn; XCD k serves the segments
// [k S / 8, (k + 1) S / 8) of every plane, plane after plane, so the 2m + 1
// planes a z stencil reads were loaded into that XCD's L2 by its own recent
// blocks.  Blocks beyond their XCD's share exit at once.
__device__ __forceinline__ bool pblock(const PGeom& g, int segs, long& p0, int& count) {
  const int b = blockIdx.x, x = b & 7;
  const long l = b >> 3;
  const int lo = (int)((long)segs * x / 8), hi = (int)((long)segs * (x + 1) / 8);
  const int c = hi - lo;
  if (c <= 0 || l >= (long)c * g.nz) return false;
  const long plane = (long)g.n0 * g.n1;
  const int z = g.z0 + (int)(l / c), seg = lo + (int)(l % c);
  p0 = (long)z * plane + (long)seg * kPThreads;
  count = (int)std::min<long>(kPThreads, plane - (long)seg * kPThreads);
  return true;
}

template <typename R, int NORD>
__global__ __launch_bounds__(kPThreads) void poisson_1d_kernel(PGeom g, int segs, int idim, const R* __restrict__ u,
                                                               R* __restrict__ du, R a, R a_y) {
  long p0;
  int count;
  if (!pblock(g, segs, p0, count) || (int)threadIdx.x >= count) return;
  const long p = p0 + threadIdx.x;
  int i0, i1, i2;
  pcoords(g, p, i0, i1, i2);
  R t = dk<R, NORD>(g, u, p, idim, i0, i1, i2) * a;
  if (a_y != R(0)) t = fmar(a_y, du[p], t);
  du[p] = t;
}

template <typename R, int NORD>
__global__ __launch_bounds__(kPThreads) void div_u_i_kernel(PGeom g, int segs, const R* __restrict__ u,
                                                            R* __restrict__ du, R* __restrict__ cc, R rh0, R rh1, R rh2) {
  long p0;
  int count;
  if (!pblock(g, segs, p0, count) || (int)threadIdx.x >= count) return;
  const long p = p0 + threadIdx.x;
  const R* u0 = u;
  const R* u1 = u + g.np;
  const R* u2 = u + 2 * g.np;
  int i0, i1, i2;
  pcoords(g, p, i0, i1, i2);
  const R dx = dk<R, NORD>(g, u0, p, 0, i0, i1, i2) * rh0;
  const R dy = dk<R, NORD>(g, u1, p, 1, i0, i1, i2) * rh1;
  const R dz = dk<R, NORD>(g, u2, p, 2, i0, i1, i2) * rh2;
  du[p] = (dx + dy) + dz;
  if (cc) {  // uniform
    const R x = u0[p], y = u1[p], z = u2[p];
    const R xy = dk<R, NORD>(g, u1, p, 0, i0, i1, i2) * rh0;
    const R xz = dk<R, NORD>(g, u2, p, 0, i0, i1, i2) * rh0;
    const R yz = dk<R, NORD>(g, u2, p, 1, i0, i1, i2) * rh1;
    cc[p] = (((x * x) * dx + (y * y) * dy) + (z * z) * dz) + R(2) * ((x * y * xy + x * z * xz) + y * z * yz);
  }
}

// What the gradient kernels do with the scaled derivatives (dx, dy, dz) of
// point p: MODE 2 (nabla_u) du_k = d_k, and du2 = (dx^2 + dy^2) + dz^2 when
// du2 is given; 3 (nabla_u_square) du2 only; 4 (nabla_u_epsilon) du_k =
// d_k eps; 5 (update_rhopol) res = ((e1 dx + e2 dy) + e3 dz) / (4 pi) with
// (e1, e2, e3) = dlogeps(:, p), res = (res - rhopol) eta, rhopol = res +
// rhopol, and res^2 returned for the block's partial sum.  The products and
// sums follow the reference's order (Poisson2.rb:2278-2550).
enum { GE_GRAD = 2, GE_SQUARE = 3, GE_EPS = 4, GE_RHOPOL = 5 };
template <typename R>
struct GradEpi {
  R* du;
  R* du2;
  const R* eps;
  const R* dlogeps;  // (3, n0, n1, n2), the component fastest
  R* rhopol;
  double* part;      // update_rhopol: one partial sum of res^2 per block
  R eta;
};

template <typename R, int MODE>
__device__ __forceinline__ double grad_epilogue(const GradEpi<R>& e, long np, long p, R dx, R dy, R dz) {
  if constexpr (MODE == GE_GRAD) {
    e.du[p] = dx;
    e.du[np + p] = dy;
    e.du[2 * np + p] = dz;
    if (e.du2) e.du2[p] = (dx * dx + dy * dy) + dz * dz;  // uniform branch
  } else if constexpr (MODE == GE_SQUARE) {
    e.du2[p] = (dx * dx + dy * dy) + dz * dz;
  } else if constexpr (MODE == GE_EPS) {
    const R ep = e.eps[p];
    e.du[p] = dx * ep;
    e.du[np + p] = dy * ep;
    e.du[2 * np + p] = dz * ep;
  } else {
    const R* d = e.dlogeps + 3 * p;
    const R oneo4pi = (R)0.07957747154594766788444188168625718101722982287022822437383367203;  // 1 / (4 pi)
    R res = (d[0] * dx + d[1] * dy) + d[2] * dz;
    res = res * oneo4pi;
    const R rho = e.rhopol[p];
    res = (res - rho) * e.eta;
    e.rhopol[p] = res + rho;
    return (double)(res * res);
  }
  return 0.0;
}

// sum of v over a block of NT threads in a fixed order (shuffle tree in each
// wave, then the waves in order); the result in thread 0
template <int NT>
__device__ __forceinline__ double pblock_sum(double v, double* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) s += red[w];
  return s;
}

template <typename R, int NORD, int MODE>
__global__ __launch_bounds__(kPThreads) void grad_point_kernel(PGeom g, int segs, const R* __restrict__ u,
                                                               GradEpi<R> ep, R rh0, R rh1, R rh2) {
  long p0;
  int count;
  const bool blk = pblock(g, segs, p0, count);
  if constexpr (MODE != GE_RHOPOL) {
    if (!blk || (int)threadIdx.x >= count) return;
  } else if (!blk) {  // uniform: the block's partial is 0
    if (threadIdx.x == 0) ep.part[blockIdx.x] = 0.0;
    return;
  }
  double sq = 0.0;
  if ((int)threadIdx.x < count) {
    const long p = p0 + threadIdx.x;
    int i0, i1, i2;
    pcoords(g, p, i0, i1, i2);
    const R dx = dk<R, NORD>(g, u, p, 0, i0, i1, i2) * rh0;
    const R dy = dk<R, NORD>(g, u, p, 1, i0, i1, i2) * rh1;
    const R dz = dk<R, NORD>(g, u, p, 2, i0, i1, i2) * rh2;
    sq = grad_epilogue<R, MODE>(ep, g.np, p, dx, dy, dz);
  }
  if constexpr (MODE == GE_RHOPOL) {
    __shared__ double red[kPThreads / 64];
    const double s = pblock_sum<kPThreads>(sq, red);
    if (threadIdx.x == 0) ep.part[blockIdx.x] = s;
  }
}

// ------------------------------------------------------------ z-marching form
// Every operator as one z march per tile of 32 x TY output columns.  Per plane
// z the tiles of the inputs (the tile plus an M-point halo along x, and along y
// where a y-derivative is taken) go to LDS from registers loaded one plane
// ahead; every lane owns two neighbouring columns (i0, i0 + 1): their x- and
// y-stencils read the LDS a pair at a time, their z-stencil of the last input
// comes from a register window of both columns along z.
//
// What bounds it (256^3, order 16, FP64): LDS reads.  With one column per lane
// and 8-byte reads, div_u_i with cc read 85 values per output (five stencils of
// 17 taps) and the LDS was busy 62% of the kernel: 282 us.  A pair of columns
// takes 9 reads of 16 bytes for both x-stencils and 17 for both y-stencils,
// 30.5 per output, at twice the bytes per clock: 240 us.  What is left is the
// overlap: order 16 in FP64 keeps 2 x 17 window values and asks for two waves
// per SIMD (at four it spills: 585 us).
//
// Non-periodic borders: an output within M points of the border uses the
// shifted row on inputs 0 .. 2m or n - 1 - 2m .. n - 1.  A tile holding such
// outputs along x or y shifts its LDS window to [0, T + 2m) or
// [n - T - 2m, n), which holds every input its outputs use, and its border
// lanes read their row from LDS too (the rows are copied to LDS once).  On a
// non-periodic z the window of the column stays on planes 0 .. 2m (the last
// 2m + 1 planes) for the border planes, which take their rows from LDS.  Taps,
// order and operations equal pderiv's, so all forms give identical bits.
constexpr int kZTX = 32;

// MODE 0: div_u_i, 1: div_u_i with cc, 2..5: the gradient family (GE_*).
// Derivatives taken of input k (X, Y in LDS; Z in the register window).
template <int MODE, int K>
struct PNeed {
  static constexpr bool X = MODE == 0 ? K == 0 : true;
  static constexpr bool Y = MODE == 0 ? K == 1 : (MODE == 1 ? K >= 1 : true);
  static constexpr bool TILE = X || Y || MODE == 1;  // cc also needs the centre values
};

template <typename R, int NORD, int TY>
struct PzGeo {
  static constexpr int M = NORD / 2, W = NORD + 1;
  static constexpr int NT = kZTX / 2 * TY;  // lanes: two output columns each
  // even row stride (a pair never straddles 16 bytes), with a spare column for
  // tiles whose window starts at an odd distance from their first output
  static constexpr int TWP = (kZTX + 2 * M + 2) & ~1, TH = TY + 2 * M;
  static constexpr int TSZ = TH * TWP + 2;  // one tile plus a spare slot
  static constexpr int nload(bool x, bool y) { return (TY + (y ? 2 * M : 0)) * (kZTX + (x ? 2 * M : 0)); }
  static constexpr int nlane(bool x, bool y) { return (nload(x, y) + NT - 1) / NT; }
};

// first index of a tile's LDS window along one dim: the centred halo, or on
// a non-periodic dim the window [0, T + 2m) / [n - T - 2m, n) of a tile that
// holds border outputs (the low rule wins when both apply)
__device__ __forceinline__ int pz_window(int o0, int t, int m, int n, bool per) {
  if (per) return o0 - m;
  if (o0 < m) return 0;
  if (o0 + t > n - m) return n - t - 2 * m;
  return o0 - m;
}

// a lane's entries of a tile that holds an x and / or a y halo: LDS slot and
// byte offset in a plane (the inputs with the same halos share them)
template <typename R, int NORD, int TY, bool X, bool Y>
struct PzMap {
  using G = PzGeo<R, NORD, TY>;
  static constexpr int NL = G::nlane(X, Y);
  int slot[NL], boff[NL];
  __device__ __forceinline__ void init(const PGeom& g, int X0, int Y0, int wx0, int wy0, int sh, int t) {
    constexpr int M = G::M;
    constexpr int NC = kZTX + (X ? 2 * M : 0), NLD = G::nload(X, Y);
    const int rx0 = X ? wx0 : X0, ry0 = Y ? wy0 : Y0;  // region origin
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      const int e = t + j * G::NT;
      const int gx = rx0 + e % NC, gy = ry0 + e / NC;
      const int sx = g.per0 ? pmod(gx, g.n0) : gx, sy = g.per1 ? pmod(gy, g.n1) : gy;
      // on a non-periodic dim only [0, n) is ever read
      const bool in = e < NLD && sx >= 0 && sx < g.n0 && sy >= 0 && sy < g.n1;
      slot[j] = in ? (gy - wy0) * G::TWP + (gx - wx0) + sh : G::TSZ - 1;
      boff[j] = plane_boff<R>(in ? sx + g.n0 * sy : -1);
    }
  }
};
// input k's tile values of one plane in flight
template <typename R, class Map>
struct PzTile {
  R val[Map::NL];
  __device__ __forceinline__ void load(const Map& m, const R* u, long plane, int s2) {
    const __amdgpu_buffer_rsrc_t rs = plane_rsrc(u, plane, s2);
#pragma unroll
    for (int j = 0; j < Map::NL; ++j) val[j] = plane_ld<R>(rs, m.boff[j]);
  }
  __device__ __forceinline__ void store(const Map& m, R* T) const {
#pragma unroll
    for (int j = 0; j < Map::NL; ++j) T[m.slot[j]] = val[j];
  }
};

// two neighbouring values in LDS (aligned to the pair, where M is even), and
// of a global array (aligned like one)
template <typename R>
struct Pz2;
template <> struct Pz2<double> { using T = double2; };
template <> struct Pz2<float> { using T = float2; };
template <typename R>
__device__ __forceinline__ typename Pz2<R>::T pz_ld2(__amdgpu_buffer_rsrc_t rs, int boff) {
  using T = typename Pz2<R>::T;
  if constexpr (sizeof(R) == 8)
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(rs, boff, 0, 0));
  else
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(rs, boff, 0, 0));
}
template <typename R>
struct PzMem;
template <> struct PzMem<double> { typedef double T __attribute__((ext_vector_type(2), aligned(8))); };
template <> struct PzMem<float> { typedef float T __attribute__((ext_vector_type(2), aligned(4))); };
template <typename R>
__device__ __forceinline__ void pz_put(R* base, long p, const R* v, bool both) {
  if (both) {
    typename PzMem<R>::T q;
    q.x = v[0];
    q.y = v[1];
    *reinterpret_cast<typename PzMem<R>::T*>(base + p) = q;
  } else {
    base[p] = v[0];
  }
}
template <typename R>
__device__ __forceinline__ void pz_get(const R* base, long p, R* v, bool both) {
  if (both) {
    const typename PzMem<R>::T q = *reinterpret_cast<const typename PzMem<R>::T*>(base + p);
    v[0] = q.x;
    v[1] = q.y;
  } else {
    v[0] = base[p];
    v[1] = R(0);
  }
}

// update_rhopol's other inputs at the points p and (both) p + 1, loaded before
// the stencils (loads and a store per point after them are two chained round
// trips: order 16 at 256^3 FP64 203 us against 168)
template <typename R>
struct RhoIn {
  R d[6], rho[2];
  __device__ __forceinline__ void load(const GradEpi<R>& e, long p, bool both) {
    pz_get(e.dlogeps, 3 * p, d, true);
    if (both) {
      pz_get(e.dlogeps, 3 * p + 2, d + 2, true);
      pz_get(e.dlogeps, 3 * p + 4, d + 4, true);
    } else {
      d[2] = e.dlogeps[3 * p + 2];
      d[3] = d[4] = d[5] = R(0);
    }
    pz_get(e.rhopol, p, rho, both);
  }
};

// grad_epilogue for the points p and (both) p + 1
template <typename R, int MODE>
__device__ __forceinline__ double grad_epilogue2(const GradEpi<R>& e, const RhoIn<R>& in, long np, long p, bool both,
                                                 R (*d)[2]) {
  if constexpr (MODE == GE_GRAD || MODE == GE_SQUARE) {
    R q[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) q[k] = (d[0][k] * d[0][k] + d[1][k] * d[1][k]) + d[2][k] * d[2][k];
    if constexpr (MODE == GE_GRAD) {
#pragma unroll
      for (int c = 0; c < 3; ++c) pz_put(e.du + c * np, p, d[c], both);
      if (e.du2) pz_put(e.du2, p, q, both);  // uniform branch
    } else {
      pz_put(e.du2, p, q, both);
    }
    return 0.0;
  } else if constexpr (MODE == GE_EPS) {
    R ep[2];
    pz_get(e.eps, p, ep, both);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const R o[2] = {d[c][0] * ep[0], d[c][1] * ep[1]};
      pz_put(e.du + c * np, p, o, both);
    }
    return 0.0;
  } else {
    const R oneo4pi = (R)0.07957747154594766788444188168625718101722982287022822437383367203;  // 1 / (4 pi)
    R o[2];
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      R res = (in.d[3 * k] * d[0][k] + in.d[3 * k + 1] * d[1][k]) + in.d[3 * k + 2] * d[2][k];
      res = res * oneo4pi;
      res = (res - in.rho[k]) * e.eta;
      o[k] = res + in.rho[k];
      if (k == 0 || both) s += (double)(res * res);
    }
    pz_put(e.rhopol, p, o, both);
    return s;
  }
}

// waves per SIMD asked of the compiler
template <typename R, int NORD, int MODE>
constexpr int pz_waves() { return sizeof(R) == 8 && NORD == 16 ? (MODE == GE_SQUARE || MODE == GE_EPS ? 3 : 2) : 4; }

template <typename R, int NORD, int MODE, int TY>
__global__ __launch_bounds__((PzGeo<R, NORD, TY>::NT))
__attribute__((amdgpu_waves_per_eu(pz_waves<R, NORD, MODE>()))) void poisson_zm_kernel(
    PGeom g, int tiles_x, int tiles, int zchunk, const R* __restrict__ u, R* __restrict__ o0, R* __restrict__ o1,
    GradEpi<R> ep, R rh0, R rh1, R rh2) {
  using G = PzGeo<R, NORD, TY>;
  constexpr int NT = G::NT, M = G::M, W = G::W, TWP = G::TWP, TSZ = G::TSZ;
  constexpr int NI = MODE >= GE_GRAD ? 1 : 3;
  using T2 = typename Pz2<R>::T;
  __shared__ __align__(16) R lds[NI * TSZ];
  __shared__ R rows[W * W];  // every coefficient row (border lanes index it)
  for (int k = threadIdx.x; k < W * W; k += NT) rows[k] = prow<R, NORD>(k);
  const int lin = xcd_linear();
  const int tile = lin % tiles, zc = lin / tiles;
  const int X0 = (tile % tiles_x) * kZTX, Y0 = (tile / tiles_x) * TY;
  const int zb = zc * zchunk, ze = min(zb + zchunk, g.n2);
  const int t = threadIdx.x, tx = 2 * (t % (kZTX / 2)), ty = t / (kZTX / 2);
  const int i0 = X0 + tx, i1 = Y0 + ty;
  const bool out_ok = i0 < g.n0 && i1 < g.n1, both = i0 + 1 < g.n0;
  const long plane = (long)g.n0 * g.n1;
  const R* uz = u + (NI - 1) * g.np;  // the input taken along z
  const int wx0 = pz_window(X0, kZTX, M, g.n0, g.per0), wy0 = pz_window(Y0, TY, M, g.n1, g.per1);
  const int sh = (X0 - M - wx0) & 1;  // the centred stencils of a pair start on an even LDS column

  // the lane's stencils in the LDS window: row of its y, centred first columns;
  // border lanes of non-periodic dims take the shifted rows
  const int lr = i1 - wy0, lc = i0 - wx0 + sh;
  const bool byl = !g.per1 && i1 < M, byh = !g.per1 && i1 >= g.n1 - M, by = byl || byh;
  const int ys = (byl ? 0 : byh ? g.n1 - 1 - 2 * M : i1 - M) - wy0;
  const int yrow = (byl ? i1 : byh ? i1 - g.n1 + 2 * M + 1 : M) * W;  // first tap of the row
  const bool bx = !g.per0 && (i0 < M || i0 + 1 >= g.n0 - M);
  int xs[2], xrow[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int i = i0 + e;
    const bool l = !g.per0 && i < M, h = !g.per0 && i >= g.n0 - M;
    // (the second column of a pair may lie past the grid: any row in the tile)
    xs[e] = (l ? 0 : h ? g.n0 - 1 - 2 * M : i - M) - wx0 + sh;
    xrow[e] = (l ? i : h ? min(i - g.n0 + 2 * M + 1, 2 * M) : M) * W;
  }

  PzMap<R, NORD, TY, PNeed<MODE, 0>::X, PNeed<MODE, 0>::Y> m0;
  PzMap<R, NORD, TY, PNeed<MODE, 1>::X, PNeed<MODE, 1>::Y> m1;  // inputs 1 and 2 (with cc the same halos)
  m0.init(g, X0, Y0, wx0, wy0, sh, t);
  if constexpr (NI == 3) m1.init(g, X0, Y0, wx0, wy0, sh, t);
  PzTile<R, decltype(m0)> t0;
  PzTile<R, decltype(m1)> t1, t2;
  FDim dz{};
  dz.n = g.n2; dz.nx = g.n2; dz.bc = g.per2 ? PER : FREE;
  ZCursor zc_tile(dz, zb);
  auto load_tiles = [&]() {
    const int s2 = zc_tile.src();
    t0.load(m0, u, plane, s2);
    if constexpr (NI == 3) t1.load(m1, u + g.np, plane, s2);
    if constexpr (PNeed<MODE, 2>::TILE && NI == 3) t2.load(m1, u + 2 * g.np, plane, s2);
    zc_tile.next();
  };
  // (a pair whose second column lies past the grid is loaded one column
  // earlier, so that no load runs past the plane)
  const int cboff = plane_boff<R>(out_ok ? i0 + g.n0 * i1 - (both ? 0 : 1) : -1);
  auto col_at = [&](const ZCursor& c) -> T2 { return pz_ld2<R>(plane_rsrc(uz, plane, c.src()), cboff); };
  // the window: planes c, c + 1, .. of both columns (c moves past them)
  auto load_window = [&](ZCursor& c, R (&win)[W][2]) {
    T2 first[W];
#pragma unroll
    for (int k = 0; k < W; ++k) {
      first[k] = col_at(c);
      c.next();
    }
#pragma unroll
    for (int k = 0; k < W; ++k) {
      win[k][0] = both ? first[k].x : first[k].y;
      win[k][1] = first[k].y;
    }
  };
  load_tiles();

  // order 16: six taps' LDS reads in flight at a time (all of them take more
  // registers than there are)
  auto fence = [&]() {
    if constexpr (NORD == 16) __builtin_amdgcn_sched_barrier(0);
  };
  auto fence_at = [&](int j) {
    if (j % 6 == 5) fence();
  };
  // x- / y-stencils of both columns from a tile (centred taps are constants;
  // the shifted border rows come per lane)
  auto sx = [&](const R* T, R* d) {
    d[0] = d[1] = R(0);
    if (!bx) {
      const T2* v = reinterpret_cast<const T2*>(T + lr * TWP + (lc - M));
#pragma unroll
      for (int k = 0; k < W + 1; k += 2) {
        const T2 q = v[k / 2];
        const R e0 = q.x, e1 = q.y;
        if (k < W) d[0] = fmar(prow<R, NORD>(M * W + k), e0, d[0]);
        if (k > 0) d[1] = fmar(prow<R, NORD>(M * W + k - 1), e0, d[1]);
        if (k + 1 < W) d[0] = fmar(prow<R, NORD>(M * W + k + 1), e1, d[0]);
        d[1] = fmar(prow<R, NORD>(M * W + k), e1, d[1]);
        if (k % 8 == 6) fence();
      }
    } else {
      const R* v = T + lr * TWP;
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int j = 0; j < W; ++j) {
          d[e] = fmar(rows[xrow[e] + j], v[xs[e] + j], d[e]);
          fence_at(j);
        }
    }
    d[0] *= rh0;
    d[1] *= rh0;
    fence();
  };
  auto pair = [&](const R* v) -> T2 {  // columns lc, lc + 1 of a tile row
    if constexpr (M % 2 == 0) {
      return *reinterpret_cast<const T2*>(v);
    } else {
      T2 q;
      q.x = v[0];
      q.y = v[1];
      return q;
    }
  };
  auto sy = [&](const R* T, R* d) {
    const R* v = T + ys * TWP + lc;
    d[0] = d[1] = R(0);
    if (!by) {
#pragma unroll
      for (int j = 0; j < W; ++j) {
        const T2 q = pair(v + j * TWP);
        d[0] = fmar(prow<R, NORD>(M * W + j), q.x, d[0]);
        d[1] = fmar(prow<R, NORD>(M * W + j), q.y, d[1]);
        fence_at(j);
      }
    } else {
#pragma unroll
      for (int j = 0; j < W; ++j) {
        const T2 q = pair(v + j * TWP);
        d[0] = fmar(rows[yrow + j], q.x, d[0]);
        d[1] = fmar(rows[yrow + j], q.y, d[1]);
        fence_at(j);
      }
    }
    d[0] *= rh1;
    d[1] *= rh1;
    fence();
  };

  double sq = 0.0;  // update_rhopol: this lane's sum of res^2, z in order
  // output plane z with the z-stencil zdot
  auto step = [&](int z, auto zdot) {
    t0.store(m0, lds);
    if constexpr (NI == 3) t1.store(m1, lds + TSZ);
    if constexpr (PNeed<MODE, 2>::TILE && NI == 3) t2.store(m1, lds + 2 * TSZ);
    load_tiles();
    __syncthreads();
    if (out_ok) {
      const long p = (long)z * plane + i0 + (long)g.n0 * i1;
      R dzv[2];
      zdot(dzv);
      dzv[0] *= rh2;
      dzv[1] *= rh2;
      fence();
      if constexpr (MODE >= GE_GRAD) {
        RhoIn<R> in;
        if constexpr (MODE == GE_RHOPOL) in.load(ep, p, both);
        R d[3][2];
        sx(lds, d[0]);
        sy(lds, d[1]);
        d[2][0] = dzv[0];
        d[2][1] = dzv[1];
        sq += grad_epilogue2<R, MODE>(ep, in, g.np, p, both, d);
      } else {
        R dx[2], dy[2], o[2];
        sx(lds, dx);
        sy(lds + TSZ, dy);
#pragma unroll
        for (int e = 0; e < 2; ++e) o[e] = (dx[e] + dy[e]) + dzv[e];
        pz_put(o0, p, o, both);
        if constexpr (MODE == 1) {
          R xy[2], xz[2], yz[2];
          sx(lds + TSZ, xy);
          sx(lds + 2 * TSZ, xz);
          sy(lds + 2 * TSZ, yz);
          const T2 cx = pair(lds + lr * TWP + lc);
          const T2 cy = pair(lds + TSZ + lr * TWP + lc);
          const T2 cz = pair(lds + 2 * TSZ + lr * TWP + lc);
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const R x = e ? cx.y : cx.x, y = e ? cy.y : cy.x, zv = e ? cz.y : cz.x;
            o[e] = (((x * x) * dx[e] + (y * y) * dy[e]) + (zv * zv) * dzv[e]) +
                   R(2) * ((x * y * xy[e] + x * zv * xz[e]) + y * zv * yz[e]);
          }
          pz_put(o1, p, o, both);
        }
      }
    }
    __syncthreads();
  };
  // a border plane of a non-periodic z: row `row` on the window's planes
  auto border = [&](int z, const R (&win)[W][2], int row) {
    step(z, [&](R* d) {
      d[0] = d[1] = R(0);
#pragma unroll
      for (int j = 0; j < W; ++j) {
        d[0] = fmar(rows[row * W + j], win[j][0], d[0]);
        d[1] = fmar(rows[row * W + j], win[j][1], d[1]);
        fence_at(j);
      }
    });
  };
  int z = zb;  // (the rows are read after the first step's barrier)
  const int zl = g.per2 ? zb : min(ze, M), zh = g.per2 ? ze : min(ze, g.n2 - M);
  if (z < zl) {  // the first M planes, on planes 0 .. 2M
    ZCursor c(dz, 0);
    R win[W][2];
    load_window(c, win);
    for (; z < zl; ++z) border(z, win, z);
  }
  if (z < zh) {
    ZCursor c(dz, z - M);
    R win[W][2];
    load_window(c, win);
    T2 nxt = col_at(c);
    c.next();
    for (;;) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {  // four steps per trip: the window moves by renaming
        step(z, [&](R* d) {
          d[0] = d[1] = R(0);
#pragma unroll
          for (int j = 0; j < W; ++j) {
            d[0] = fmar(prow<R, NORD>(M * W + j), win[j][0], d[0]);
            d[1] = fmar(prow<R, NORD>(M * W + j), win[j][1], d[1]);
          }
        });
        if (++z >= zh) goto high;
#pragma unroll
        for (int j = 0; j < W - 1; ++j) {
          win[j][0] = win[j + 1][0];
          win[j][1] = win[j + 1][1];
        }
        win[W - 1][0] = both ? nxt.x : nxt.y;
        win[W - 1][1] = nxt.y;
        nxt = col_at(c);
        c.next();
      }
    }
  }
high:
  if (z < ze) {  // the last M planes, on planes n - 1 - 2M .. n - 1
    ZCursor c(dz, g.n2 - W);
    R win[W][2];
    load_window(c, win);
    for (; z < ze; ++z) border(z, win, z - g.n2 + W);
  }
  if constexpr (MODE == GE_RHOPOL) {
    __shared__ double red[NT / 64];
    const double s = pblock_sum<NT>(sq, red);
    if (threadIdx.x == 0) ep.part[blockIdx.x] = s;
  }
}

PGeom pgeom(const int* n, int geocode, int bc_idim, int idim) {
  PGeom g;
  g.n0 = n[0]; g.n1 = n[1]; g.n2 = n[2];
  g.np = (long)n[0] * n[1] * n[2];
  g.z0 = 0;
  g.nz = n[2];
  if (idim >= 0) {  // one dim, its own bc
    g.per0 = g.per1 = g.per2 = bc_idim == 0;
  } else {          // div_u_i_ref's perx / pery / perz
    g.per0 = geocode != 1;
    g.per1 = geocode == 2;
    g.per2 = geocode != 1;
  }
  return g;
}

int psegs(const PGeom& g) { return (int)(((long)g.n0 * g.n1 + kPThreads - 1) / kPThreads); }

// 8 XCD shares of ceil(S / 8) segments times nz planes
unsigned pgrid(const PGeom& g) { return (unsigned)(8L * ((psegs(g) + 7) / 8) * g.nz); }

}  // namespace

bool poisson_order_ok(int nord) { return nord == 2 || nord == 4 || nord == 6 || nord == 8 || nord == 16; }

#define LC_POISSON_DISPATCH(NORD_VAR, CALL) \
  switch (NORD_VAR) {                       \
    case 2: { constexpr int NO = 2; CALL; } break;   \
    case 4: { constexpr int NO = 4; CALL; } break;   \
    case 6: { constexpr int NO = 6; CALL; } break;   \
    case 8: { constexpr int NO = 8; CALL; } break;   \
    case 16: { constexpr int NO = 16; CALL; } break; \
    default: return hipErrorInvalidValue;            \
  }

template <typename R>
hipError_t poisson_1d(int nord, int idim, const int* n, int bc, const R* u, R* du, R a, R a_y, hipStream_t st) {
  const PGeom g = pgeom(n, 0, bc, idim);
  if (g.np == 0) return hipSuccess;
  LC_POISSON_DISPATCH(nord, (poisson_1d_kernel<R, NO><<<pgrid(g), kPThreads, 0, st>>>(g, psegs(g), idim, u, du, a, a_y)))
  return hipGetLastError();
}

// z-march launch shape: tiles x z chunks.  Chunks of at least 6 planes by the
// expected time of the busiest CU, in planes of a block alone on its CU: k
// blocks on a CU, in rounds of at most `resident` (what it holds), take max(1,
// add + mul k) of that per plane, or bw k where the arrays are beyond the
// last-level cache; a chunk costs its plane count, `pre` planes for the loads of
// its window and `blk` to start.  What the rule avoids is a CU
// with one block more than the others: 190 tiles of 300^3 points in FP64, order
// 8, nabla_u with square: 2 chunks (1.5 blocks per CU) 425 us, 4 (3.0) 357, 7
// (5.2) 377.  Below 6 planes, down to 2, only when the grid would leave CUs
// without a block (order 4 on 100 x 60 x 40: 11.6 us against 13.8 with 4).
struct PzCost {
  double blk, pre, add, mul, bw;
};
// fitted to 1 .. 40 chunks of every operator on 128^3 to 350^3 points
constexpr double kPzCached = 128e6;  // bytes of four arrays: half the cache
template <typename R, int NO, int MODE>
static PzCost pz_cost(const PGeom& g, const GradEpi<R>& ep) {
  if (sizeof(R) == 8) return PzCost{1.3, 0.2 * NO, 0, NO == 16 ? 0.44 : 0.4, 0};
  // few arrays: several blocks overlap better
  if (NO < 16 && (MODE == 0 || (MODE == GE_GRAD && !ep.du2))) return PzCost{0.3, 0.3 * NO, 0, 0.4, 0};
  return PzCost{0.3, 0.3 * NO, 0.75, 0.31, 4.0 * sizeof(R) * g.np > kPzCached ? 0.5 : 0};
}
static int pz_zchunk(const PzCost& m, long tiles, int nz, int resident) {
  int best = nz;
  double bt = 1e300;
  for (int c = 1; c <= std::max(1, nz / 6); ++c) {
    const int zc = (nz + c - 1) / c;
    const long k = (tiles * ((nz + zc - 1) / zc) + num_cu() - 1) / num_cu(), kr = std::min<long>(k, resident);
    const long rounds = (k + resident - 1) / resident;
    if (c > 1 && rounds > 3) break;
    const double t = rounds * ((zc + m.pre) * std::max({1.0, m.add + m.mul * kr, m.bw * kr}) + m.blk * kr);
    if (t < bt) bt = t, best = zc;
  }
  return best;
}
// False when the one-point kernels must do all (LIBCONV_POISSON_POINT set,
// planes beyond the buffer-record limit).
struct PzLaunch {
  int tiles_x, tiles, zchunk;
  unsigned blocks;
};
static bool pz_launch(const PGeom& g, int ty, int resident, const PzCost& cost, bool thin, PzLaunch& L) {
  if (getenv("LIBCONV_POISSON_POINT")) return false;
  if ((long)g.n0 * g.n1 * 8 > kPlaneMax) return false;
  L.tiles_x = (g.n0 + kZTX - 1) / kZTX;
  const long tiles = (long)L.tiles_x * ((g.n1 + ty - 1) / ty);
  if (tiles * (g.n2 / 6) >= num_cu()) {
    L.zchunk = thin ? std::min(g.n2, 9) : pz_zchunk(cost, tiles, g.n2, resident);
  } else {
    const long chunks = std::max(1L, std::min<long>((num_cu() + tiles - 1) / tiles, g.n2 / 2));
    L.zchunk = (int)((g.n2 + chunks - 1) / chunks);
  }
  const long nb = tiles * ((g.n2 + L.zchunk - 1) / L.zchunk);
  if (nb > 0x7fffffffL) return false;
  L.tiles = (int)tiles;
  L.blocks = (unsigned)nb;
  return true;
}
// tile rows: 16; 32 for the gradient operators of order 16, whose y halo is as
// high as the tile (nabla_u_and_square at 256^3: FP64 151 us against 179, FP32
// 68 against 93), where that still gives a CU two chunks of 16 planes.  In FP64
// the others' tall tiles are no faster (nabla_u_square 106 against 100 us).
// div_u_i holds three tiles and gains nothing (FP64 257 against 240 us).
template <typename R, int NO, int MODE>
static constexpr bool pz_tall() { return NO == 16 && (MODE == GE_GRAD || (sizeof(R) == 4 && MODE > GE_GRAD)); }
static bool pz_fills(const PGeom& g) {
  const long tiles = (long)((g.n0 + kZTX - 1) / kZTX) * ((g.n1 + 31) / 32);
  return tiles * (g.n2 / 16) >= 2L * num_cu();
}

// blocks of one z-march kernel that a CU holds (registers, LDS), cached
template <auto KER, int NT>
static int pz_resident() {
  static int nb = 0;
  if (!nb) {
    int v = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&v, KER, NT, 0) != hipSuccess || v < 1) v = 1;
    nb = v;
  }
  return nb;
}

// Chunks of 9 planes, in order along z, on arrays well beyond the cache whose
// rows are of odd length, so that a lane's pairs straddle lines: the lines that
// tiles share are then read close together.  283^3 points, order 4: update_rhopol
// FP64 248 us against 265 with chunks by expected time, FP32 136 against 146,
// nabla_u with square FP64 285 against 315; 257 x 255 x 129 108 against 125.
// With rows of even length or fewer arrays the expected time is the better rule
// (update_rhopol 300^3 FP64 286 against 279, nabla_u_square 283^3 118 against 114,
// nabla_u 257 x 255 x 129 70 against 62).
template <typename R, int NO, int MODE>
static bool pz_thin(const PGeom& g, const GradEpi<R>& ep) {
  if (g.n0 % 2 == 0) return false;
  const double bytes = (double)sizeof(R) * g.np;
  if (MODE == GE_RHOPOL && (NO < 16 || sizeof(R) == 8)) return 4 * bytes > kPzCached;
  if (MODE == GE_EPS && NO < 16) return 4 * bytes > kPzCached;
  if (MODE == GE_GRAD && NO < 16 && sizeof(R) == 8) return bytes > (ep.du2 ? 0.5 : 1.0) * kPzCached;
  return false;
}

// one z-march launch; its blocks, or 0 when the one-point kernels must run;
// dry: count only
template <typename R, int NO, int MODE, int TY>
static long pz_run_rows(const PGeom& g, const R* u, R* o0, R* o1, const GradEpi<R>& ep, R r0, R r1, R r2,
                        hipStream_t st, bool dry) {
  constexpr int NT = PzGeo<R, NO, TY>::NT;
  PzLaunch L;
  const int resident = pz_resident<poisson_zm_kernel<R, NO, MODE, TY>, NT>();
  if (!pz_launch(g, TY, resident, pz_cost<R, NO, MODE>(g, ep), pz_thin<R, NO, MODE>(g, ep), L)) return 0;
  if (!dry)
    poisson_zm_kernel<R, NO, MODE, TY><<<L.blocks, NT, 0, st>>>(g, L.tiles_x, L.tiles, L.zchunk, u, o0, o1, ep, r0,
                                                                r1, r2);
  return L.blocks;
}
template <typename R, int NO, int MODE>
static long pz_run(const PGeom& g, const R* u, R* o0, R* o1, const GradEpi<R>& ep, R r0, R r1, R r2, hipStream_t st,
                   bool dry) {
  if constexpr (pz_tall<R, NO, MODE>()) {
    if (pz_fills(g)) return pz_run_rows<R, NO, MODE, 32>(g, u, o0, o1, ep, r0, r1, r2, st, dry);
  }
  return pz_run_rows<R, NO, MODE, 16>(g, u, o0, o1, ep, r0, r1, r2, st, dry);
}

template <typename R>
hipError_t div_u_i(int geocode, const int* n, const R* u, R* du, R* cc, int nord, const double* h, hipStream_t st) {
  const PGeom g = pgeom(n, geocode, 0, -1);
  if (g.np == 0) return hipSuccess;
  const R r0 = (R)(1.0 / h[0]), r1 = (R)(1.0 / h[1]), r2 = (R)(1.0 / h[2]);
  auto point = [&](const PGeom& q) -> hipError_t {
    LC_POISSON_DISPATCH(nord, (div_u_i_kernel<R, NO><<<pgrid(q), kPThreads, 0, st>>>(q, psegs(q), u, du, cc, r0, r1, r2)))
    return hipGetLastError();
  };
  long done = 0;
  if (cc) {
    LC_POISSON_DISPATCH(nord, (done = pz_run<R, NO, 1>(g, u, du, cc, GradEpi<R>{}, r0, r1, r2, st, false)))
  } else {
    LC_POISSON_DISPATCH(nord, (done = pz_run<R, NO, 0>(g, u, du, cc, GradEpi<R>{}, r0, r1, r2, st, false)))
  }
  return done ? hipGetLastError() : point(g);
}

// The launch of one gradient-family operator: the z march, or the one-point
// kernel.  Returns its block count, which is the number of partial sums
// update_rhopol writes (ep.part[0 .. count)); dry: count only.
template <typename R, int NO, int MODE>
static long grad_launch(const PGeom& g, const R* u, const GradEpi<R>& ep, R r0, R r1, R r2, hipStream_t st,
                        bool dry) {
  const long nb = pz_run<R, NO, MODE>(g, u, nullptr, nullptr, ep, r0, r1, r2, st, dry);
  if (nb) return nb;
  const unsigned np = pgrid(g);
  if (!dry) grad_point_kernel<R, NO, MODE><<<np, kPThreads, 0, st>>>(g, psegs(g), u, ep, r0, r1, r2);
  return np;
}

template <typename R, int MODE>
static hipError_t grad_op(int geocode, const int* n, const R* u, const GradEpi<R>& ep, int nord, const double* h,
                          hipStream_t st, long* blocks, bool dry) {
  const PGeom g = pgeom(n, geocode, 0, -1);
  *blocks = 0;
  if (g.np == 0) return hipSuccess;
  const R r0 = h ? (R)(1.0 / h[0]) : R(1), r1 = h ? (R)(1.0 / h[1]) : R(1), r2 = h ? (R)(1.0 / h[2]) : R(1);
  LC_POISSON_DISPATCH(nord, (*blocks = grad_launch<R, NO, MODE>(g, u, ep, r0, r1, r2, st, dry)))
  return dry ? hipSuccess : hipGetLastError();
}

template <typename R>
hipError_t nabla_u(int geocode, const int* n, const R* u, R* du, R* du2, int nord, const double* h, hipStream_t st) {
  GradEpi<R> ep{};
  ep.du = du;
  ep.du2 = du2;
  long nb;
  return grad_op<R, GE_GRAD>(geocode, n, u, ep, nord, h, st, &nb, false);
}

template <typename R>
hipError_t nabla_u_square(int geocode, const int* n, const R* u, R* ddu, int nord, const double* h, hipStream_t st) {
  GradEpi<R> ep{};
  ep.du2 = ddu;
  long nb;
  return grad_op<R, GE_SQUARE>(geocode, n, u, ep, nord, h, st, &nb, false);
}

template <typename R>
hipError_t nabla_u_epsilon(int geocode, const int* n, const R* u, R* du, const R* eps, int nord, const double* h,
                           hipStream_t st) {
  GradEpi<R> ep{};
  ep.du = du;
  ep.eps = eps;
  long nb;
  return grad_op<R, GE_EPS>(geocode, n, u, ep, nord, h, st, &nb, false);
}

template <typename R>
long update_rhopol_partials(int geocode, const int* n, int nord) {
  if (!poisson_order_ok(nord)) return -1;
  long nb = 0;
  (void)grad_op<R, GE_RHOPOL>(geocode, n, nullptr, GradEpi<R>{}, nord, nullptr, nullptr, &nb, true);
  return nb;
}

template <typename R>
hipError_t update_rhopol(int geocode, const int* n, const R* u, int nord, const double* h, R eta, const R* dlogeps,
                         R* rhopol, double* part, long nparts, double* rhores2, hipStream_t st) {
  GradEpi<R> ep{};
  ep.dlogeps = dlogeps;
  ep.rhopol = rhopol;
  ep.part = part;
  ep.eta = eta;
  long nb = 0;
  hipError_t e = grad_op<R, GE_RHOPOL>(geocode, n, u, ep, nord, h, st, &nb, true);
  if (e != hipSuccess) return e;
  if (nb > nparts) return hipErrorInvalidValue;  // the caller sized part by update_rhopol_partials
  e = grad_op<R, GE_RHOPOL>(geocode, n, u, ep, nord, h, st, &nb, false);
  if (e != hipSuccess) return e;
  return sum_partial_sets(part, nb, rhores2, 1, 0, st);
}

#undef LC_POISSON_DISPATCH

template hipError_t poisson_1d<double>(int, int, const int*, int, const double*, double*, double, double,
                                       hipStream_t);
template hipError_t poisson_1d<float>(int, int, const int*, int, const float*, float*, float, float, hipStream_t);
template hipError_t div_u_i<double>(int, const int*, const double*, double*, double*, int, const double*,
                                    hipStream_t);
template hipError_t div_u_i<float>(int, const int*, const float*, float*, float*, int, const double*, hipStream_t);
template hipError_t nabla_u<double>(int, const int*, const double*, double*, double*, int, const double*,
                                    hipStream_t);
template hipError_t nabla_u<float>(int, const int*, const float*, float*, float*, int, const double*, hipStream_t);
template hipError_t nabla_u_square<double>(int, const int*, const double*, double*, int, const double*, hipStream_t);
template hipError_t nabla_u_square<float>(int, const int*, const float*, float*, int, const double*, hipStream_t);
template hipError_t nabla_u_epsilon<double>(int, const int*, const double*, double*, const double*, int,
                                            const double*, hipStream_t);
template hipError_t nabla_u_epsilon<float>(int, const int*, const float*, float*, const float*, int, const double*,
                                           hipStream_t);
template long update_rhopol_partials<double>(int, const int*, int);
template long update_rhopol_partials<float>(int, const int*, int);
template hipError_t update_rhopol<double>(int, const int*, const double*, int, const double*, double, const double*,
                                          double*, double*, long, double*, hipStream_t);
template hipError_t update_rhopol<float>(int, const int*, const float*, int, const double*, float, const float*,
                                         float*, double*, long, double*, hipStream_t);

}  // namespace lc
