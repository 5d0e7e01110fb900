// lc_fused_wav.hip -- single-pass 3D wavelet transforms on gfx950.
//
// One level of the separable 3D DWT (analysis) or IDWT (synthesis): along
// every dim the transform maps input steps j (two values each: a sample
// pair for the DWT, the L and H bands for the IDWT) to output steps i (two
// values each) with a W-step window,
//   out[i][c'] = sum_{s<W} sum_{c<2} C[c'][c](s) * in[i + LO + s][c],
// the split filters of WaveletFilterDecompose / WaveletFilterRecompose
// (BigDFT/GenericConvolution2.rb:386-410, :453-462, :505-671).  The three
// per-dim sweeps of the libconv composition (:2160-2240) become one pass, in
// two forms of equal bits: the pair-wise one (lc_body_wavq.hpp), and the
// step-at-a-time one, which takes planes beyond 32-bit buffer records: per input z-step the two z-planes of the (TX+W-1) x (TY+W-1)-step tile go
// to LDS, x-tasks filter rows into LDS, every lane filters one column along
// y for both bands and feeds its register window along z, which emits both
// z bands of the output step.  Data layout per dim (storage extents 2 nx and
// 2 ny values):
//   DWT   input  sample c of step j at c + 2 (j - ox),  output band b of
//         step i at (i - oy) + ny b
//   IDWT  input  band b of step j at (j - ox) + nx b,   output sample c of
//         step i at c + 2 (i - oy)
// Periodic dims wrap, free dims read zero outside the stored input, exactly
// as the 1D sweeps.  Epilogue: y = a * t + a_y * y.
#include <math.h>
#include <stdio.h>
#include <stdlib.h>

#include <string>

#include "lc_body_wav.hpp"
#include "lc_body_wavq.hpp"

namespace lc {

template <typename R, class Op, int TX, int TY, int QX, int BZ, int AD, int WPE>
__global__ __launch_bounds__(2 * TX * TY) __attribute__((amdgpu_waves_per_eu(WPE))) void sepw3d_fused(
    FusedArgs<R> p) {
  __shared__ __align__(16) unsigned char lds[sepw3d_lds_bytes<R, Op, TX, TY, QX, BZ, AD>()];
  int bx, by, zc, arr;
  block_coords(p.tiles_x, bx, by, zc, arr);
  sepw3d_body<R, Op, TX, TY, QX, BZ, AD>(p, bx, by, zc, arr, lds);
}

template <typename R, class Op, int TX, int TY, int QX, int BZ, int AD, int WPE>
__global__ __launch_bounds__(2 * TX * TY) __attribute__((amdgpu_waves_per_eu(WPE))) void sepw3d_batch(
    const FusedArgs<R>* __restrict__ tab, BatchOrder ord) {
  int o, local;
  if (!batch_block(ord, o, local)) return;
  const FusedArgs<R> p = tab[o];
  const int tiles = p.tiles_x * p.tiles_y;
  const int tile = local % tiles, zc = local / tiles;
  __shared__ __align__(16) unsigned char lds[sepw3d_lds_bytes<R, Op, TX, TY, QX, BZ, AD>()];
  sepw3d_body<R, Op, TX, TY, QX, BZ, AD>(p, tile % p.tiles_x, tile / p.tiles_x, zc, 0, lds);
}

// the pair-wise form (lc_body_wavq.hpp): blocks for NG groups of TX x TY output
// steps, QX outputs per x-task, PD planes of prefetch, 4 WPE waves per EU, KB + 1
// lanes per y-task.  *_acc: with the a_y y term (ME), apart because the union
// of both bodies spills.
#define LC_WAVQ_ATTR                                                                         \
  template <typename R, class Op, int NG, int TX, int TY, int QX, int PD, int WPE, int KB>   \
  __global__ __launch_bounds__((WavqBlock{NG * TX * TY, QX, KB + 1}.nt()))                   \
  __attribute__((amdgpu_waves_per_eu(4 * WPE)))
#define LC_WAVQ_KERNELS(SINGLE, BATCH, ME)                                                                  \
  LC_WAVQ_ATTR void SINGLE(FusedArgs<R> p) {                                                                \
    constexpr WavqBlock kB{NG * TX * TY, QX, KB + 1};                                                       \
    __shared__ __align__(16) unsigned char lds[kB.lds(sizeof(R))];                                          \
    int bx, by, zc, arr;                                                                                    \
    block_coords(p.tiles_x, bx, by, zc, arr);                                                               \
    wavq_body<R, Op, kB.S, QX, kB.HB, PD / 2, ME>(p, bx, by, zc, arr, lds);                                 \
  }                                                                                                         \
  LC_WAVQ_ATTR void BATCH(const FusedArgs<R>* __restrict__ tab, BatchOrder ord) {                           \
    constexpr WavqBlock kB{NG * TX * TY, QX, KB + 1};                                                       \
    int o, local;                                                                                           \
    if (!batch_block(ord, o, local)) return;                                                                \
    const FusedArgs<R> p = tab[o];                                                                          \
    const int tiles = p.tiles_x * p.tiles_y;                                                                \
    const int tile = local % tiles, zc = local / tiles;                                                     \
    __shared__ __align__(16) unsigned char lds[kB.lds(sizeof(R))];                                          \
    wavq_body<R, Op, kB.S, QX, kB.HB, PD / 2, ME>(p, tile % p.tiles_x, tile / p.tiles_x, zc, 0, lds);       \
  }
LC_WAVQ_KERNELS(wavq_fused, wavq_batch, false)
LC_WAVQ_KERNELS(wavq_acc, wavq_batch_acc, true)
#undef LC_WAVQ_KERNELS
#undef LC_WAVQ_ATTR

// ====================================================================== host
// Compiled variants: tile TX x TY steps, QX outputs per x-task, BZ steps per
// window slide, AD prefetch depth (2 TX TY lanes per block), waves per EU,
// z chunks of a single call (0: ~2 blocks per CU, chunks >= 2 W steps;
// ZC < 0: at most -ZC blocks on any CU, chunks >= W steps)
#define LC_WAV_VARIANTS(X)                                                                            \
  X(0, 16, 8, 4, 2, 2, 1, 0) X(1, 8, 8, 4, 2, 2, 1, 0) X(2, 32, 4, 4, 2, 2, 1, 0) X(3, 16, 8, 4, 1, 1, 1, 0) \
  X(4, 16, 8, 4, 1, 1, 2, 0) X(5, 16, 8, 4, 1, 1, 1, -2) X(6, 16, 8, 4, 2, 2, 1, -2)

// pair-wise variants: NG groups of TX x TY output steps per block (the tile is
// any shape of up to NG TX TY steps, picked per grid by wav_pick), QX outputs
// per x-task, PD planes of prefetch, WPE times four waves per EU (at most 128
// VGPRs), KB = 1: two lanes per y-task
#define LC_WAVQ_VARIANTS(X)                                                                      \
  X(7, 1, 16, 8, 4, 2, 1, 0) X(8, 2, 16, 8, 4, 2, 1, 0) X(9, 4, 16, 8, 4, 2, 1, 0)                  \
  X(10, 4, 8, 8, 2, 2, 1, 0) X(11, 1, 8, 8, 2, 2, 1, 1) X(12, 2, 8, 8, 2, 2, 1, 1)                   \
  X(13, 8, 8, 8, 2, 2, 1, 0) X(14, 1, 8, 8, 2, 2, 1, 0) X(15, 1, 16, 8, 4, 2, 1, 1)                  \
  X(16, 2, 8, 8, 2, 2, 1, 0) X(17, 1, 8, 4, 2, 2, 1, 1)

int wav_variant_count() { return 18; }

// entries 16 and 17 exist in FP64 only (they were shapes of FP64's 16-byte
// pieces; tables tuned for FP32 never hold them)
template <typename R>
constexpr bool wavq_takes(int v) { return sizeof(R) == 8 || v < 16; }

static bool wavq_block(int v, WavqBlock* b) {
  switch (v) {
#define X(I, NG, TX, TY, QX, PD, WPE, KB) \
  case I: *b = WavqBlock{NG * TX * TY, QX, KB + 1}; return true;
    LC_WAVQ_VARIANTS(X)
#undef X
  }
  return false;
}

// output planes reached through 32-bit buffer records (the pair-wise
// variants store with buffer stores)
static bool wavq_fits(const Box3& b, int prec) {
  return wav_plane_fits(b, prec) && 4L * b.ny[0] * b.ny[1] * prec <= kPlaneMax;
}

std::string wav_kernel_name(int prec, int form, int id, int v, bool batch) {
  (void)id;
  const char* r = prec == 4 ? "float" : "double";
  const char* op = form == FORM_IDWT ? "Idwt<lc::WSplit<lc::FLP, lc::FHP, 8, true> >"
                                     : "Dwt<lc::WSplit<lc::FLP, lc::FHP, 8, false> >";
  char buf[200];
  buf[0] = 0;
  switch (v) {
#define X(I, TX, TY, QX, BZ, AD, WPE, ZC)                                                                   \
  case I:                                                                                         \
    snprintf(buf, sizeof buf, "%s<%s, lc::%s, %d, %d, %d, %d, %d, %d>", batch ? "sepw3d_batch" : "sepw3d_fused", \
             r, op, TX, TY, QX, BZ, AD, WPE);                                                        \
    break;
    LC_WAV_VARIANTS(X)
#undef X
#define X(I, NG, TX, TY, QX, PD, WPE, KB)                                                                   \
  case I:                                                                                                   \
    snprintf(buf, sizeof buf, "%s<%s, lc::%s, %d, %d, %d, %d, %d, %d, %d>", batch ? "wavq_batch" : "wavq_fused", r, \
             op, NG, TX, TY, QX, PD, WPE, KB);                                                              \
    break;
    LC_WAVQ_VARIANTS(X)
#undef X
  }
  return buf;
}

template <typename R, class Op, int TX, int TY, int QX, int BZ, int AD>
static FusedArgs<R> wav_args(const Box3& b, int narr, const R* x, R* y, R a, R a_y) {
  FusedArgs<R> p{};
  p.x = x; p.y = y;
  p.d0 = fdim(b.n[0], b.bc[0], b.nx[0], b.ny[0], Op::LO, Op::UP);
  p.d1 = fdim(b.n[1], b.bc[1], b.nx[1], b.ny[1], Op::LO, Op::UP);
  p.d2 = fdim(b.n[2], b.bc[2], b.nx[2], b.ny[2], Op::LO, Op::UP);
  p.nti = 8L * b.nx[0] * b.nx[1] * b.nx[2];
  p.nto = 8L * b.ny[0] * b.ny[1] * b.ny[2];
  p.narr = narr;
  p.tiles_x = (p.d0.nout + TX - 1) / TX;
  p.tiles_y = (p.d1.nout + TY - 1) / TY;
  p.a0 = a; p.a_y = a_y;
  p.flags = (a != R(1) ? F_A : 0) | (a_y != R(0) ? F_AY : 0);
  return p;
}

template <typename R, class Op, int TX, int TY, int QX, int BZ, int AD, int WPE, int ZC>
static hipError_t launch_sepw3d(const Box3& b, int narr, const R* x, R* y, R a, R a_y, hipStream_t st) {
  if (!wav_plane_fits(b, sizeof(R))) return hipErrorInvalidValue;
  FusedArgs<R> p = wav_args<R, Op, TX, TY, QX, BZ, AD>(b, narr, x, y, a, a_y);
  const long tiles = (long)p.tiles_x * p.tiles_y;
  if (ZC < 0) {
    // at most -ZC blocks on any CU, at least one where the grid allows
    const long per = tiles * std::max(narr, 1);
    long chunks = (long)(-ZC) * num_cu() / per;
    if (chunks * per < num_cu()) chunks = (num_cu() + per - 1) / per;
    chunks = std::max(1L, std::min<long>(chunks, std::max(1, p.d2.nout / Op::W)));
    p.zchunk = (int)((p.d2.nout + chunks - 1) / chunks);
  } else {
    // z chunks no shorter than 2 W steps (W steps when the grid is too
    // small to give every CU a block)
    p.zchunk = pick_zchunk(tiles, p.d2.nout, std::max(narr, 1), std::max(1, Op::W / 2), num_cu());
  }
  const int zch = (p.d2.nout + p.zchunk - 1) / p.zchunk;
  if (narr == 0) return hipSuccess;
  dim3 grid((unsigned)tiles, (unsigned)zch, (unsigned)narr);
  sepw3d_fused<R, Op, TX, TY, QX, BZ, AD, WPE><<<grid, 2 * TX * TY, 0, st>>>(p);
  return hipGetLastError();
}

// ---- tile and z chunk of the pair-wise kernels
// Work of one block-step: the issue of its FMAs in cycles (x-tasks 32 QX,
// y-tasks 128 / HB per wave of four cycles, over four SIMDs), its bytes and its
// runs of adjacent bytes.  A DWT row holds its pairs side by side and each band
// of the output is a run of its own; an IDWT row lies in two bands and the
// output's pairs side by side.
struct WavWork {
  double fma, rd, rd_runs, wr, wr_runs;
};
static WavWork wav_work(const WavqBlock& k, const WavqShape& g, int rs, bool inverse) {
  WavWork w;
  w.fma = 32.0 * k.QX * ((g.xtasks(k.QX) + 63) / 64) + 128.0 * ((2 * g.tx * g.ty + 63) / 64);
  w.rd = 4.0 * g.nr * (g.tx + 7) * rs;
  w.rd_runs = 2.0 * g.nr * (inverse ? 2 : 1);
  w.wr = 8.0 * g.tx * g.ty * rs;
  w.wr_runs = (inverse ? 4.0 : 8.0) * g.ty;
  return w;
}
// Time of one step of a single call, in us, with n blocks on the CU: the serial
// chain of a block (tile write, x, y, z with a barrier between), hardly longer
// with a second one beside it, or what the blocks' FMAs and bytes take together.
//   step(n) = max(lat (1 + 0.05 n), add + n (fma + mem bytes))
// Fitted to 5 to 6000 launches (tile x chunk) of each of 70 calls: cubes of 32
// to 160 pairs and flat and long boxes, all boundary conditions, with and
// without a_y; the picked launch is 3 - 5% behind the best of them on average.
// half: the chain of the two-lane block; halo: weight of the bytes read; run:
// bytes that a run costs beside those it holds.
struct WavFit {
  double lat, half, halo, fma, mem, add, run;
};
constexpr WavFit kWavFit[2][2] = {  // [FP64, FP32][DWT, IDWT]
    {{1.14, 0.83, 3.76, 0.096e-3, 0.671e-5, 0.451, 14}, {1.19, 0.776, 4.25, 0.355e-3, 0.235e-5, 0.481, 79}},
    {{0.942, 0.70, 6.41, 0.288e-3, 0.07e-5, 0.367, 175}, {1.16, 0.693, 2.28, 0.121e-3, 0.735e-5, 0.418, 39}}};
struct WavStep {
  double lat, add, per;
  double operator()(double n) const { return std::max(lat * (1.0 + 0.05 * n), add + n * per); }
};
// acc: with the a_y y term, whose loads of y end the step
static WavStep wav_step(const WavqBlock& k, const WavqShape& g, int rs, bool inverse, bool acc) {
  const WavFit& f = kWavFit[rs == 4][inverse];
  const WavWork w = wav_work(k, g, rs, inverse);
  // FP64 synthesis with two outputs per x-task takes narrow tiles better: 96^3
  // pairs 49.1 us with tiles of 8 x 16 steps, 50.9 with 16 x 8
  const double run = k.QX == 2 && k.HB == 1 && rs == 8 && inverse ? 55 : f.run;
  const double bytes = f.halo * (w.rd + run * w.rd_runs) + (acc ? 2 : 1) * (w.wr + run * w.wr_runs);
  WavStep s;
  s.lat = f.lat * (k.HB == 2 ? f.half : k.S > 128 ? 1.35 : 1.0) * (acc ? 1.8 : 1.0);
  s.add = acc ? 0.9 : f.add;
  s.per = (f.fma * w.fma + f.mem * bytes) * (acc ? 1.1 : 1.0);
  return s;
}
// Cycles and bytes of a step where blocks fill the chip for many rounds (batch
// stages): half of the halo reads hit L2, rows and runs cost most of a line more
// than they hold, 9.3 bytes per cycle are the CU's share of the copy rate.
struct WavCost {
  double fma, mem;
};
static WavCost wav_cost(const WavqBlock& k, const WavqShape& g, int rs) {
  const double rd = 2.0 * g.nr * (2 * (g.tx + 7) * rs + 96), own = 8.0 * g.tx * g.ty * rs;
  const double wr = 8.0 * g.ty * (g.tx * rs + 48);
  return WavCost{wav_work(k, g, rs, false).fma, (0.5 * (rd + own) + wr) / 9.3};
}
struct WavPick {
  int tx = 0, ty = 0, zchunk = 0;
  double t = 1e300;
};
// candidate tiles of a w0 x w1 grid: the extents split into equal parts
template <typename F>
static void wav_tiles(const WavqBlock& k, int w0, int w1, int rs, F&& f) {
  for (int ny = 1, ty = 0; ny <= w1; ++ny) {
    const int y = (w1 + ny - 1) / ny;
    if (y == ty || y > k.S) continue;
    ty = y;
    for (int nx = (w0 * ty + k.S - 1) / k.S, tx = 0; nx <= w0; ++nx) {
      const int x = (w0 + nx - 1) / nx;
      if (x == tx) continue;
      tx = x;
      const WavqShape g(tx, ty, k.QX);
      if (k.fits(g, rs)) f(g, (long)nx * ny);
      if (tx <= 4) break;
    }
    if (ty <= 4) break;
  }
}
// Single calls: the tile and z chunk with the least expected time.  A chunk of c
// output steps takes c + 7 input steps; every CU is as late as the busiest.
static WavPick wav_pick(const WavqBlock& k, int w0, int w1, int nz, int narr, int rs, bool inverse, bool acc) {
  WavPick best;
  const long ncu = num_cu();
  const int occ = std::max(1, 1024 / k.nt());  // blocks per CU: 128 VGPRs, four waves per SIMD
  wav_tiles(k, w0, w1, rs, [&](const WavqShape& g, long tiles) {
    const WavStep step = wav_step(k, g, rs, inverse, acc);
    auto consider = [&](long chunks) {
      if (chunks < 1 || chunks > nz) return;
      const int zc = (int)((nz + chunks - 1) / chunks);
      const long blocks = tiles * narr * ((nz + zc - 1) / zc);
      const double t = (zc + 7) * step((double)((blocks + ncu - 1) / ncu));
      if (t < best.t) best = WavPick{g.tx, g.ty, zc, t};
    };
    for (int q = 1; q <= 2 * occ; ++q) consider(q * ncu / (tiles * narr));
    consider(1);
    consider(nz);
  });
  return best;
}
// The picks of recent shapes (the search takes some 10 us), per host thread.
static WavPick wav_pick_cached(int v, const WavqBlock& k, int w0, int w1, int nz, int narr, int rs, bool inverse,
                               bool acc) {
  struct Entry {
    int key[6];
    WavPick p;
  };
  constexpr int kEntries = 64;
  static thread_local Entry cache[kEntries];  // zero-initialised: no variant 0 here
  const int key[6] = {4 * v + 2 * inverse + acc, w0, w1, nz, narr, rs};
  unsigned h = 0;
  for (int q : key) h = h * 31u + (unsigned)q;
  Entry& e = cache[h % kEntries];
  if (!std::equal(key, key + 6, e.key)) {
    e.p = wav_pick(k, w0, w1, nz, narr, rs, inverse, acc);
    std::copy(key, key + 6, e.key);
  }
  return e.p;
}

// The variant a call takes by default: of the block for 128 output steps (four
// outputs per x-task) and the two-lane block for 64 the one expected to be
// faster.  The best launches of larger blocks and of two outputs per x-task are
// within 1.5% of the best of these on average, 5% up to 112^3 pairs (144^3 FP64
// 115 us in 256 steps against 117).  Except FP64 synthesis of some 95^3 to 119^3
// pairs, where two outputs per x-task take less: 2% on average of periodic, grown
// and accumulated calls of 96^3 to 116^3 (96^3 48.4 us against 49.0, 100^3 55.6
// against 58.1, 112^3 grown 75.2 against 81.3, with a_y 82.8 against 90.2); 88^3
// and 128^3 and more take 1% to 9% longer.
int wav_default_variant(int prec, int form, const Box3& b, int narr, bool acc) {
  const int lo = form == FORM_IDWT ? Idwt<Sym8Rec>::LO : Dwt<Sym8Dec>::LO;
  const FDim d0 = fdim(b.n[0], b.bc[0], b.nx[0], b.ny[0], lo, lo + 7), d1 = fdim(b.n[1], b.bc[1], b.nx[1], b.ny[1], lo, lo + 7),
             d2 = fdim(b.n[2], b.bc[2], b.nx[2], b.ny[2], lo, lo + 7);
  int best = 5;
  double t = 1e300;
  const double points = (double)d0.nout * d1.nout * d2.nout * std::max(narr, 1);
  const bool two = prec == 8 && form == FORM_IDWT && points >= 8.5e5 && points <= 1.7e6;
  // on equal tiles the two-lane block: 40^3 pairs FP64, five arrays, synthesis on 8
  // x 8 steps 30.8 us against 35.8
  for (int v : {11, two ? 16 : 7}) {
    WavqBlock k;
    if (!wavq_block(v, &k)) continue;
    const WavPick p = wav_pick_cached(v, k, d0.nout, d1.nout, d2.nout, std::max(narr, 1), prec,
                                      form == FORM_IDWT, acc);
    if (p.t < t) { t = p.t; best = v; }
  }
  return best;
}

// How many items of this one's size the items of a stage make together: the
// stage is laid out as a call with that many arrays.
static double wav_points(const Box3& b) { return (double)b.ny[0] * b.ny[1] * b.ny[2]; }
static int wav_copies(double total, const Box3& b) {
  return (int)std::min(1e6, std::max(1.0, std::ceil(total / wav_points(b))));
}

// The default of a batch stage: one that fills every CU is bound by bytes, so it
// takes the block with the widest tiles, in FP64 512 output steps, in FP32 (more
// blocks per CU) 256.  128 orbitals of 24..96 pairs, DWT stage: FP64 1.55 / 1.34
// / 1.25 ms for 128 / 256 / 512 steps, FP32 0.90 / 0.78 / 0.83.  A smaller one
// takes what a call with as many arrays of its largest item would.
int wav_batch_variant(int prec, int form, const Box3* b, int count, bool acc) {
  long steps = 0;
  double total = 0;
  int big = 0;
  for (int i = 0; i < count; ++i) {
    if (!wavq_fits(b[i], prec)) return 5;  // the step-at-a-time form: planes beyond the buffer records
    steps += (long)b[i].ny[0] * b[i].ny[1];
    total += wav_points(b[i]);
    if (wav_points(b[i]) > wav_points(b[big])) big = i;
  }
  const int v = prec == 4 ? 10 : 9;
  WavqBlock k;
  if (wavq_block(v, &k) && steps >= (long)k.S * num_cu() * std::max(1, 1024 / k.nt())) return v;
  return wav_default_variant(prec, form, b[big], wav_copies(total, b[big]), acc);
}

template <int V, typename R, class Op, int NG, int TX, int TY, int QX, int PD, int WPE, int KB>
static hipError_t launch_wavq(const Box3& b, int narr, const R* x, R* y, R a, R a_y, hipStream_t st) {
  if constexpr (!wavq_takes<R>(V)) {
    return hipErrorInvalidValue;
  } else {
  if (!wavq_fits(b, sizeof(R))) return hipErrorInvalidValue;
  if (narr == 0) return hipSuccess;
  constexpr WavqBlock kB{NG * TX * TY, QX, KB + 1};
  FusedArgs<R> p = wav_args<R, Op, TX, TY, QX, 1, 1>(b, narr, x, y, a, a_y);
  const WavPick k = wav_pick_cached(V, kB, p.d0.nout, p.d1.nout, p.d2.nout, narr, sizeof(R), WavCoef<Op>::K == KIDWT,
                                    (p.flags & F_AY) != 0);
  p.tile_x = k.tx;
  p.tile_y = k.ty;
  p.tiles_x = (p.d0.nout + k.tx - 1) / k.tx;
  p.tiles_y = (p.d1.nout + k.ty - 1) / k.ty;
  p.zchunk = k.zchunk;
  const int zch = (p.d2.nout + p.zchunk - 1) / p.zchunk;
  dim3 grid((unsigned)(p.tiles_x * p.tiles_y), (unsigned)zch, (unsigned)narr);
  if (p.flags & F_AY)
    wavq_acc<R, Op, NG, TX, TY, QX, PD, WPE, KB><<<grid, kB.nt(), 0, st>>>(p);
  else
    wavq_fused<R, Op, NG, TX, TY, QX, PD, WPE, KB><<<grid, kB.nt(), 0, st>>>(p);
  return hipGetLastError();
  }
}

template <typename R, class Op>
static hipError_t sepw3d_variant(int v, const Box3& b, int narr, const R* x, R* y, R a, R a_y,
                                 hipStream_t st) {
  switch (v) {
#define X(I, TX, TY, QX, BZ, AD, WPE, ZC) \
  case I: return launch_sepw3d<R, Op, TX, TY, QX, BZ, AD, WPE, ZC>(b, narr, x, y, a, a_y, st);
    LC_WAV_VARIANTS(X)
#undef X
#define X(I, NG, TX, TY, QX, PD, WPE, KB) \
  case I: return launch_wavq<I, R, Op, NG, TX, TY, QX, PD, WPE, KB>(b, narr, x, y, a, a_y, st);
    LC_WAVQ_VARIANTS(X)
#undef X
  }
  return hipErrorInvalidValue;
}

// The symicomb8 family is not instantiated: its single-pass kernel (420
// VGPRs, spilling to AGPRs) returned wrong high bands on the GPU and then
// faulted, while a CPU emulation of its exact address arithmetic stays in
// bounds and matches the oracle.  symicomb8 3D transforms run as three 1D
// sweeps instead (lc_api.cpp).
template <typename R>
hipError_t sepw3d_v(int v, int kind, int id, const Box3& b, int narr, const R* x, R* y, R a, R a_y,
                    hipStream_t st) {
  if (id != WAV_SYM8) return hipErrorNotSupported;
  if (kind == KDWT) return sepw3d_variant<R, Dwt<Sym8Dec>>(v, b, narr, x, y, a, a_y, st);
  if (kind == KIDWT) return sepw3d_variant<R, Idwt<Sym8Rec>>(v, b, narr, x, y, a, a_y, st);
  return hipErrorInvalidValue;
}

template <typename R>
hipError_t sepw3d(int kind, int id, const Box3& b, int narr, const R* x, R* y, R a, R a_y,
                  hipStream_t st) {
  const int form = kind == KIDWT ? FORM_IDWT : FORM_DWT;
  int v = chosen_variant(sizeof(R), form, id, b);
  if (v < 0) v = default_variant(sizeof(R), form, b, narr, a_y != R(0));
  return sepw3d_v<R>(v, kind, id, b, narr, x, y, a, a_y, st);
}

// ---- batches of independent 3D sym8 wavelet transforms
// Tiles and z chunks of a pair-wise stage that leaves CUs without a full load and
// whose arrays the last-level cache holds.  Items of one shape: as one call with
// that many arrays.  Others: the tiles with the least work, and marches of one
// length, the one with the least expected time of the busiest CU.
constexpr double kWavCached = 256e6;  // bytes read and written
template <typename R, class Op>
static void wav_batch_layout(const WavqBlock& k, const BatchItem<R>* it, int count, bool acc, FusedArgs<R>* tab) {
  constexpr bool inverse = WavCoef<Op>::K == KIDWT;
  bool same = true;
  for (int o = 1; o < count; ++o)
    same = same && tab[o].d0.nout == tab[0].d0.nout && tab[o].d1.nout == tab[0].d1.nout && tab[o].d2.nout == tab[0].d2.nout;
  if (same) {
    const WavPick w = wav_pick(k, tab[0].d0.nout, tab[0].d1.nout, tab[0].d2.nout, count, sizeof(R), inverse, acc);
    for (int o = 0; o < count; ++o) {
      tab[o].tile_x = w.tx;
      tab[o].tile_y = w.ty;
      tab[o].zchunk = w.zchunk;
    }
  } else {
    double lat = 0, add = 0, per = 0, tiles_all = 0;
    int nz = 1;
    for (int o = 0; o < count; ++o) {
      FusedArgs<R>& p = tab[o];
      double best = 1e300;
      WavStep bs{};
      wav_tiles(k, p.d0.nout, p.d1.nout, sizeof(R), [&](const WavqShape& g, long tiles) {
        const WavStep st = wav_step(k, g, sizeof(R), inverse, acc);
        if (tiles * st.per < best) { best = tiles * st.per; bs = st; p.tile_x = g.tx; p.tile_y = g.ty; }
      });
      const double t = (double)((p.d0.nout + p.tile_x - 1) / p.tile_x) * ((p.d1.nout + p.tile_y - 1) / p.tile_y);
      lat = bs.lat;
      add = bs.add;
      per += t * bs.per;
      tiles_all += t;
      nz = std::max(nz, p.d2.nout);
    }
    const WavStep mean{lat, add, per / tiles_all};
    int march = nz;
    double bt = 1e300;
    for (int z = std::min(4, nz); z <= nz; ++z) {
      long n = 0;
      int most = 0;
      for (int o = 0; o < count; ++o) {
        const FusedArgs<R>& p = tab[o];
        const int c = (p.d2.nout + z - 1) / z, zc = (p.d2.nout + c - 1) / c;
        n += (long)((p.d0.nout + p.tile_x - 1) / p.tile_x) * ((p.d1.nout + p.tile_y - 1) / p.tile_y) *
             ((p.d2.nout + zc - 1) / zc);
        most = std::max(most, zc);
      }
      const double t = (most + 7) * mean((double)((n + num_cu() - 1) / num_cu()));
      if (t < bt) { bt = t; march = z; }
    }
    for (int o = 0; o < count; ++o) {
      const int c = (tab[o].d2.nout + march - 1) / march;
      tab[o].zchunk = (tab[o].d2.nout + c - 1) / c;
    }
  }
  for (int o = 0; o < count; ++o) {
    FusedArgs<R>& p = tab[o];
    p.tiles_x = (p.d0.nout + p.tile_x - 1) / p.tile_x;
    p.tiles_y = (p.d1.nout + p.tile_y - 1) / p.tile_y;
  }
}

template <typename R, class Op, int TX, int TY, int QX, int BZ, int AD, int WPE>
static hipError_t wav_stage_build(const BatchItem<R>* it, int count, BatchStage* s) {
  std::vector<FusedArgs<R>> tab(count);
  long tiles_all = 0;
  double total = 0;
  WavqBlock k{};
  const bool pairwise = wavq_block(s->variant, &k);
  for (int o = 0; o < count; ++o)
    if (!wav_plane_fits(it[o].b, sizeof(R))) return hipErrorInvalidValue;
  for (int o = 0; o < count; ++o) {
    FusedArgs<R>& p = tab[o];
    p = wav_args<R, Op, TX, TY, QX, BZ, AD>(it[o].b, 1, it[o].x, it[o].y, (R)it[o].a[0], (R)it[o].a_y);
    if (p.flags & F_AY) s->any_acc = true;
    total += wav_points(it[o].b);
    if (pairwise) {
      // a full chip: the tile with the least bytes and (half hidden) FMAs
      double best = 1e300;
      wav_tiles(k, p.d0.nout, p.d1.nout, sizeof(R), [&](const WavqShape& g, long tiles) {
        const WavCost c = wav_cost(k, g, sizeof(R));
        const double t = tiles * (c.mem + 0.5 * c.fma);
        if (t < best) { best = t; p.tile_x = g.tx; p.tile_y = g.ty; }
      });
      p.tiles_x = (p.d0.nout + p.tile_x - 1) / p.tile_x;
      p.tiles_y = (p.d1.nout + p.tile_y - 1) / p.tile_y;
    }
    tiles_all += (long)tab[o].tiles_x * tab[o].tiles_y;
  }
  // two blocks per CU (pair-wise: what fills four waves per SIMD)
  const long want = (pairwise ? std::max(1, 1024 / k.nt()) : 2) * (long)num_cu();
  const long chunks = std::max(1L, (want + tiles_all - 1) / std::max(1L, tiles_all));
  std::vector<long> blocks(count), steps(count);
  const bool fitted = pairwise && chunks > 1 && 16.0 * sizeof(R) * total <= kWavCached;
  if (fitted) wav_batch_layout<R, Op>(k, it, count, s->any_acc, tab.data());
  for (int o = 0; o < count; ++o) {
    FusedArgs<R>& p = tab[o];
    if (!fitted) {
      const long c = std::max(1L, std::min<long>(chunks, std::max(1, p.d2.nout / (2 * Op::W))));
      p.zchunk = (int)((p.d2.nout + c - 1) / c);
    }
    blocks[o] = (long)p.tiles_x * p.tiles_y * ((p.d2.nout + p.zchunk - 1) / p.zchunk);
    steps[o] = p.zchunk + Op::W - 1;
  }
  std::vector<int> order, first;
  const hipError_t e = batch_order(blocks, steps, &order, &first, s);
  if (e != hipSuccess) return e;
  std::vector<FusedArgs<R>> sorted;
  for (int i : order) sorted.push_back(tab[i]);
  return batch_upload(sorted.data(), sizeof(FusedArgs<R>) * count, first, s);
}

template <typename R, class Op>
static hipError_t wav_stage_t(bool build, const BatchItem<R>* it, int count, BatchStage* s, hipStream_t st) {
  if (build) {
    switch (s->variant) {
#define X(I, TX, TY, QX, BZ, AD, WPE, ZC) \
  case I: return wav_stage_build<R, Op, TX, TY, QX, BZ, AD, WPE>(it, count, s);
      LC_WAV_VARIANTS(X)
#undef X
#define X(I, NG, TX, TY, QX, PD, WPE, KB)                                  \
  case I:                                                                  \
    if (!wavq_takes<R>(I)) return hipErrorInvalidValue;                    \
    for (int o = 0; o < count; ++o)                                        \
      if (!wavq_fits(it[o].b, sizeof(R))) return hipErrorInvalidValue;     \
    return wav_stage_build<R, Op, TX, TY, QX, 1, 1, WPE>(it, count, s);
      LC_WAVQ_VARIANTS(X)
#undef X
    }
    return hipErrorInvalidValue;
  }
  if (s->blocks == 0) return hipSuccess;
  const FusedArgs<R>* tab = static_cast<const FusedArgs<R>*>(s->tab);
  switch (s->variant) {
#define X(I, TX, TY, QX, BZ, AD, WPE, ZC)                                                                     \
  case I:                                                                                           \
    sepw3d_batch<R, Op, TX, TY, QX, BZ, AD, WPE><<<s->grid, 2 * TX * TY, 0, st>>>(tab, batch_order_of(s)); \
    break;
    LC_WAV_VARIANTS(X)
#undef X
#define X(I, NG, TX, TY, QX, PD, WPE, KB)                                                                 \
  case I:                                                                                                 \
    if constexpr (wavq_takes<R>(I)) {                                                                     \
      constexpr int nt = WavqBlock{NG * TX * TY, QX, KB + 1}.nt();                                        \
      if (s->any_acc)                                                                                     \
        wavq_batch_acc<R, Op, NG, TX, TY, QX, PD, WPE, KB><<<s->grid, nt, 0, st>>>(tab, batch_order_of(s)); \
      else                                                                                                \
        wavq_batch<R, Op, NG, TX, TY, QX, PD, WPE, KB><<<s->grid, nt, 0, st>>>(tab, batch_order_of(s)); \
    } else {                                                                                              \
      return hipErrorInvalidValue;                                                                        \
    }                                                                                                     \
    break;
    LC_WAVQ_VARIANTS(X)
#undef X
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <typename R>
hipError_t wav_stage(bool build, int kind, int id, int bc, const BatchItem<R>* it, int count,
                     BatchStage* s, hipStream_t st) {
  (void)bc;
  if (id != WAV_SYM8) return hipErrorNotSupported;
  if (kind == KDWT) return wav_stage_t<R, Dwt<Sym8Dec>>(build, it, count, s, st);
  if (kind == KIDWT) return wav_stage_t<R, Idwt<Sym8Rec>>(build, it, count, s, st);
  return hipErrorInvalidValue;
}

template hipError_t sepw3d<double>(int, int, const Box3&, int, const double*, double*, double, double,
                                   hipStream_t);
template hipError_t sepw3d<float>(int, int, const Box3&, int, const float*, float*, float, float,
                                  hipStream_t);
template hipError_t sepw3d_v<double>(int, int, int, const Box3&, int, const double*, double*, double, double,
                                     hipStream_t);
template hipError_t sepw3d_v<float>(int, int, int, const Box3&, int, const float*, float*, float, float,
                                    hipStream_t);
template hipError_t wav_stage<double>(bool, int, int, int, const BatchItem<double>*, int, BatchStage*,
                                      hipStream_t);
template hipError_t wav_stage<float>(bool, int, int, int, const BatchItem<float>*, int, BatchStage*,
                                     hipStream_t);

}  // namespace lc
