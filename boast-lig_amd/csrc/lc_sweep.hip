// lc_sweep.hip -- one-dimensional libconv sweeps on gfx950.
//
// A sweep applies one operator (convolution filter, wavelet analysis or
// synthesis) along one dimension of an array seen as (L, line, R) with L
// the product of the faster dims and R the product of the slower dims
// (the libconv 1D dispatcher's ndat_left / ndat_right,
// BigDFT/GenericConvolution2.rb:1701-1766).  Two tiled kernels: a block
// stages a tile of lines -- every line's input steps for a chunk of outputs,
// halo included -- in LDS with all of its loads in flight at once, and every
// lane then computes Q consecutive outputs of one line, each LDS value feeding
// all of its outputs.
//
//   sweep_strided  L > 1: the tile is [step][column], consecutive lanes on
//                  consecutive columns in every phase, so loads and stores
//                  are coalesced and the LDS is free of bank conflicts;
//   sweep_contig   L == 1 (the processed dim is the contiguous one): the tile
//                  is [line][step] with an odd row stride, filled along the
//                  lines and read with consecutive lanes on consecutive lines;
//                  the outputs go back through the LDS to be stored along the
//                  lines.
//
// And two without a tile of fixed size, for lines that would leave most of one
// empty (ring_pays, seg_pays):
//
//   sweep_ring     L > 1: one lane per column, which walks a chunk of the line
//                  with a register ring of W input steps;
//   sweep_seg      L == 1: 4 to 64 lanes share a segment of one line.
//
// All sum in the same order, so an output's bits do not depend on the form.
//
// What bounds them: latency.  A sweep moves two values per output and the
// arrays of one orbital are 2..130 MB, so a launch lasts a few memory round
// trips; what counts is how many loads are in flight (a block's whole tile: 4
// loads per lane for the magic filter with Q = 2, 20 for the second derivative
// with Q = 16) and that every CU has its blocks in the first wave.  The ring
// keeps one load per lane in flight per step: 27 us for a 128^3 FP64
// second-derivative sweep with its energy along a strided dim, 12 with tiles;
// the segments' LDS has bank conflicts on a third of its cycles: 19 us along
// the contiguous dim, 13 with tiles.
//
// Epilogue per output (ConvolutionFilter#post_process_and_store_values,
// GenericConvolution2.rb:173-203): t *= a; dot += x_i t; t += a_x x_i;
// t += a_y y_i; y_i = t -- the dot and a_x steps only where the output
// carries an input value (grow borders skip them).  dot is accumulated in
// FP64 whatever the storage precision, per block, then summed in a fixed
// order by a one-block kernel (deterministic).
#include <type_traits>

#include "lc_fused.hpp"
#include "lc_kernels.hpp"

namespace lc {

// ---------------------------------------------------------------- helpers
template <typename R>
__device__ __forceinline__ double block_sum(double v, double* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) red[wid] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0) {
    const int nw = (blockDim.x + 63) >> 6;
    for (int w = 0; w < nw; ++w) s += red[w];
  }
  return s;
}

// The input steps of a block's chunk: element offset (in line strides) of
// component c of step j, or -1 where x is zero; steps past jmax are never used
// and may lie outside x (shrink).  near: a periodic chunk within one wrap of
// the line, where a compare replaces the modulo.
template <int K, int BC, typename R>
struct SweepSrc {
  int n, nx, ox, jmax;
  bool near;
  __device__ __forceinline__ SweepSrc(const SweepArgs<R>& p, int jmin, int jmax_)
      : n(p.n), nx(p.nx), ox(p.ox), jmax(jmax_), near(jmin >= -p.n && jmax_ < 2 * p.n) {}
  __device__ __forceinline__ long at(int j, int c) const {
    if (j > jmax) return -1;
    if (BC == PER) {
      int w = j;
      if (near) {
        w += w < 0 ? n : 0;
        w -= w >= n ? n : 0;
      } else {
        w = pmod(j, n);
      }
      return in_elem<K>(w, c, nx);
    }
    if (BC == GROW) return (j >= 0) & (j < n) ? in_elem<K>(j, c, nx) : -1;
    return in_elem<K>(j - ox, c, nx);
  }
};

// one input value of a line (the forms without a tile)
template <int K, int BC, typename R>
__device__ __forceinline__ R load_step(const R* __restrict__ xb, long L, int j, int c, int n, int nx, int ox) {
  if (BC == PER) return xb[in_elem<K>(pmod(j, n), c, nx) * L];
  if (BC == GROW) {
    const bool ok = (j >= 0) & (j < n);
    const R v = xb[in_elem<K>(ok ? j : 0, c, nx) * L];
    return ok ? v : R(0);
  }
  return xb[in_elem<K>(j - ox, c, nx) * L];
}

// the epilogue of output step i up to the a_y term; xc: x at step i
template <class Op, int BC, typename R>
__device__ __forceinline__ void sweep_post(const SweepArgs<R>& p, int i, R xc, bool want_dot, double& dot, R* o) {
  if (p.flags & F_A) {
#pragma unroll
    for (int c = 0; c < Op::OUT; ++c) o[c] = o[c] * p.a;
  }
  if (Op::DOT) {
    const bool has_x = BC != GROW || (i >= 0 && i < p.n);
    if (has_x) {
      if (want_dot) dot = fmar((double)xc, (double)o[0], dot);
      if (p.flags & F_AX) o[0] = fmar(xc, p.a_x, o[0]);
    }
  }
}

// Q consecutive outputs from the LDS values v(c, s), s = 0 .. Q + W - 2 (the
// input steps of the first output's window onwards): every accumulator takes
// its terms in the order of Op::step.  xc[q]: the value at the output's own
// step (operators with the dot / a_x terms).
template <typename R, class Op, int Q>
struct SweepTask {
  R o[Q][Op::OUT];
  R xc[Q];
  template <class V>
  __device__ __forceinline__ void run(const V& v) {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      xc[q] = R(0);
#pragma unroll
      for (int c = 0; c < Op::OUT; ++c) o[q][c] = R(0);
    }
#pragma unroll
    for (int k = 0; k < Q + Op::W - 1; ++k) {
      R w[Op::IN];
#pragma unroll
      for (int c = 0; c < Op::IN; ++c) w[c] = v(c, k);
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int s = k - q;
        if (s >= 0 && s < Op::W) {
          Op::step(s, w, o[q]);
          if (Op::DOT && s == -Op::LO) xc[q] = w[0];
        }
      }
    }
  }
};

// Tile of both kernels: 256 lanes, C columns (or lines) of 256 / C lanes that
// take Q outputs each, so a chunk of up to CH outputs and NS input steps.
// 32 columns: a row of the tile is 256 bytes in FP64 and a full line in FP32,
// whose chunk would halve (and its halo reads double) with 64.
constexpr int kSweepCols = 32;
constexpr int kSweepRun = 8;
template <typename R, class Op, int Q>
struct SweepGeo {
  static constexpr int C = kSweepCols, G = 256 / C, CH = G * Q, NS = CH + Op::W - 1;
  static constexpr int NL = (Op::IN * NS + G - 1) / G;  // strided: loads per lane
  // contiguous: a row holds IN runs of NS steps (or OUT runs of CH outputs)
  static constexpr int ROW = (Op::IN * NS > Op::OUT * CH ? Op::IN * NS : Op::OUT * CH) | 1;
};

// t / n and t % n, inv = min(2^32 / n, 2^32 - 1): the product is at most one short
__device__ __forceinline__ unsigned div_inv(unsigned t, unsigned n, unsigned inv, unsigned& r) {
  unsigned q = __umulhi(t, inv);
  r = t - q * n;
  if (r >= n) {
    ++q;
    r -= n;
  }
  return q;
}

// The tile of a block, chunks of a line fastest.  Consecutive blocks go to the 8
// XCDs in turn; here each XCD takes runs of p.run neighbouring tiles, so what
// those share -- the halo of a chunk, the memory lines that a tile's edge splits
// -- is in one L2: the chunks of one column of tiles, of kSweepRun of them where
// L is not a multiple of the tile's columns and its rows end within lines.
// Against tiles dealt out one by one: strided 0.85 to 0.91 of the time with such
// L, 0.96 to 1.02 with others (second derivative FP64 of 192^3 30.2 -> 25.3 us).
// One run per XCD, an eighth of the array, is 0 to 3% behind in FP64.  The blocks
// past the last full round of runs take the tiles in order.
template <typename R>
__device__ __forceinline__ long tile_of(const SweepArgs<R>& p, int& bk) {
  const unsigned b = blockIdx.x;
  unsigned t = b, w;
  if (b < p.run_end) {
    const unsigned g = div_inv(b >> 3, (unsigned)p.run, p.run_inv, w);
    t = (g * 8 + (b & 7)) * (unsigned)p.run + w;
  }
  const unsigned bc = div_inv(t, (unsigned)p.nchunk, p.nchunk_inv, w);
  bk = (int)w;
  return bc;
}

// ---------------------------------------------------------------- strided
template <typename R, class Op, int BC, int Q>
__global__ __launch_bounds__(256) void sweep_strided(SweepArgs<R> p) {
  using G = SweepGeo<R, Op, Q>;
  constexpr int K = KindOf<Op>::v, C = G::C;
  __shared__ R tile[Op::IN * G::NS * C];
  __shared__ double red[4];
  const int tc = threadIdx.x % C, tg = threadIdx.x / C;
  // arrays of a call lie line_in * nr (line_out * nr) apart, so a line's place
  // follows from its number in the whole call
  int bk;
  const long bc = tile_of(p, bk);
  const long col = bc * C + tc;
  const bool active = col < p.ncols;
  const long line = !active ? 0 : p.ncols <= 0x7fffffffL ? (int)col / (int)p.L : col / p.L;
  const long l = active ? col - line * p.L : 0;
  const R* __restrict__ xb = p.x + line * p.line_in + l;
  R* __restrict__ yb = p.y + line * p.line_out + l;
  const int i0 = p.i_first + bk * p.chunk;
  const int i1 = min(i0 + p.chunk, p.i_first + p.nout);
  const SweepSrc<K, BC, R> src(p, i0 + Op::LO, i1 - 1 + Op::UP);
  // row e of the tile: component e / NS of step i0 + LO + e % NS
  R val[G::NL];
#pragma unroll
  for (int k = 0; k < G::NL; ++k) {
    const int e = tg + k * G::G, c = e / G::NS;
    const long at = c < Op::IN && active ? src.at(i0 + Op::LO + (e - c * G::NS), c) : -1;
    val[k] = at >= 0 ? xb[at * p.L] : R(0);
  }
  // the lane's outputs, and the y values its a_y term needs
  const int ib = i0 + tg * Q;
  R yv[Q][Op::OUT];
  if (p.flags & F_AY) {
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int c = 0; c < Op::OUT; ++c)
        yv[q][c] = active && ib + q < i1 ? yb[out_elem<K>(ib + q - p.oy, c, p.ny) * p.L] : R(0);
  }
#pragma unroll
  for (int k = 0; k < G::NL; ++k) {
    const int e = tg + k * G::G;
    if ((k + 1) * G::G <= Op::IN * G::NS || e < Op::IN * G::NS) tile[e * C + tc] = val[k];
  }
  __syncthreads();
  double dot = 0.0;
  if (active && ib < i1) {
    const bool want_dot = Op::DOT && (p.flags & F_DOT) && line >= (p.narr - 1) * p.nr;
    SweepTask<R, Op, Q> t;
    const R* base = tile + tg * Q * C + tc;
    t.run([&](int c, int k) { return base[(c * G::NS + k) * C]; });
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int i = ib + q;
      if (i < i1) {
        sweep_post<Op, BC>(p, i, t.xc[q], want_dot, dot, t.o[q]);
#pragma unroll
        for (int c = 0; c < Op::OUT; ++c) {
          R o = t.o[q][c];
          if (p.flags & F_AY) o = fmar(p.a_y, yv[q][c], o);
          yb[out_elem<K>(i - p.oy, c, p.ny) * p.L] = o;
        }
      }
    }
  }
  if (p.dot_part) {
    const double s = block_sum<R>(dot, red);
    if (threadIdx.x == 0) p.dot_part[blockIdx.x] = s;
  }
}

// ---------------------------------------------------------------- contiguous
template <typename R, class Op, int BC, int Q, bool AY>
__global__ __launch_bounds__(256) void sweep_contig(SweepArgs<R> p) {
  using G = SweepGeo<R, Op, Q>;
  constexpr int K = KindOf<Op>::v, C = G::C;
  __shared__ R tile[C * G::ROW];
  __shared__ double red[4];
  int bk;
  const long bc = tile_of(p, bk);
  const int i0 = p.i_first + bk * p.chunk;
  const int i1 = min(i0 + p.chunk, p.i_first + p.nout);
  const SweepSrc<K, BC, R> src(p, i0 + Op::LO, i1 - 1 + Op::UP);
  const long line0 = bc * C;
  // filled 64 lanes along a line: 4 lines per pass
  constexpr int NX = (Op::IN * G::NS + 63) / 64, NY = C / 4;
  const int lx = threadIdx.x & 63, ly = threadIdx.x >> 6;
  R val[NX * NY];
#pragma unroll
  for (int b = 0; b < NY; ++b) {
    const long line = line0 + ly + 4 * b;
    const bool act = line < p.ncols;
    const R* __restrict__ xb = p.x + (act ? line * p.line_in : 0);
#pragma unroll
    for (int a = 0; a < NX; ++a) {
      const int e = lx + 64 * a;  // memory order: pairs (DWT), bands (IDWT)
      const int c = K == KDWT ? e & 1 : e / G::NS, s = K == KDWT ? e >> 1 : e - c * G::NS;
      const long at = act && e < Op::IN * G::NS ? src.at(i0 + Op::LO + s, c) : -1;
      val[b * NX + a] = at >= 0 ? xb[at] : R(0);
    }
  }
  // The outputs of the tile in memory order along its lines: a wave's lanes take
  // 64 of one line, or all of several lines with short chunks.  The y values of
  // the a_y term come with the loads of x; they are a kernel of their own, for
  // their registers cost the others a wave per SIMD (second derivative FP64 of
  // 160^3 without a_y: 23.1 us in one kernel, 20.9 in its own).  Magic filter FP64
  // of 107 x 118 x 64 points with a_y: 11.4 us with 64 lanes per line, y read last
  // and the chunks of a line on different XCDs, now 6.5.
  constexpr int OC = Op::OUT * G::CH, LW = OC < 64 ? OC : 64, OX = OC / LW, LP = 256 / LW, OY = C / LP;
  const int of = threadIdx.x % LW, ol = threadIdx.x / LW;
  R* __restrict__ yb = p.y + (line0 + ol) * p.line_out;
  // output a of a line: element in the line (or -1), f its place in the tile's row
  auto out_at = [&](int a, int& f) {
    f = of + LW * a;
    const int c = K == KIDWT ? f & 1 : f / G::CH, i = i0 + (K == KIDWT ? f >> 1 : f - c * G::CH);
    return i < i1 ? out_elem<K>(i - p.oy, c, p.ny) : -1;
  };
  R yv[AY ? OX * OY : 1];
  if (AY) {
#pragma unroll
    for (int a = 0; a < OX; ++a) {
      int f;
      const long at = out_at(a, f);
#pragma unroll
      for (int b = 0; b < OY; ++b)
        yv[a * OY + b] = at >= 0 && line0 + ol + LP * b < p.ncols ? yb[LP * b * p.line_out + at] : R(0);
    }
  }
#pragma unroll
  for (int b = 0; b < NY; ++b)
#pragma unroll
    for (int a = 0; a < NX; ++a) {
      const int e = lx + 64 * a;
      const int c = K == KDWT ? e & 1 : e / G::NS, s = K == KDWT ? e >> 1 : e - c * G::NS;
      if (64 * (a + 1) <= Op::IN * G::NS || e < Op::IN * G::NS)
        tile[(ly + 4 * b) * G::ROW + c * G::NS + s] = val[b * NX + a];
    }
  __syncthreads();
  // lane -> line tc, outputs ib .. ib + Q - 1
  const int tc = threadIdx.x % C, tg = threadIdx.x / C;
  const long line = line0 + tc;
  const int ib = i0 + tg * Q;
  double dot = 0.0;
  SweepTask<R, Op, Q> t;
  {
    const R* base = tile + tc * G::ROW + tg * Q;
    t.run([&](int c, int k) { return base[c * G::NS + k]; });
    const bool want_dot = Op::DOT && (p.flags & F_DOT) && line < p.ncols && line >= (p.narr - 1) * p.nr;
#pragma unroll
    for (int q = 0; q < Q; ++q)
      if (ib + q < i1) sweep_post<Op, BC>(p, ib + q, t.xc[q], want_dot, dot, t.o[q]);
  }
  __syncthreads();
  // outputs back through the tile, in memory order along the line
#pragma unroll
  for (int q = 0; q < Q; ++q)
#pragma unroll
    for (int c = 0; c < Op::OUT; ++c)
      tile[tc * G::ROW + (K == KIDWT ? 2 * (tg * Q + q) + c : c * G::CH + tg * Q + q)] = t.o[q][c];
  __syncthreads();
#pragma unroll
  for (int b = 0; b < OY; ++b) {
    if (line0 + ol + LP * b >= p.ncols) break;
#pragma unroll
    for (int a = 0; a < OX; ++a) {
      int f;
      const long at = out_at(a, f);
      if (at < 0) continue;
      R o = tile[(ol + LP * b) * G::ROW + f];
      if (AY) o = fmar(p.a_y, yv[a * OY + b], o);
      yb[LP * b * p.line_out + at] = o;
    }
  }
  if (p.dot_part) {
    const double s = block_sum<R>(dot, red);
    if (threadIdx.x == 0) p.dot_part[blockIdx.x] = s;
  }
}

// ------------------------------------------------- strided, a column per lane
template <typename R, class Op, int BC>
__global__ __launch_bounds__(256) void sweep_ring(SweepArgs<R> p) {
  constexpr int K = KindOf<Op>::v;
  constexpr int W = Op::W, IN = Op::IN, OUT = Op::OUT;
  __shared__ double red[4];
  const long col = (long)(blockIdx.x % (unsigned)p.cblocks) * 256 + threadIdx.x;
  double dot = 0.0;
  if (col < p.ncols) {
    const long line = p.ncols <= 0x7fffffffL ? (int)col / (int)p.L : col / p.L, l = col - line * p.L;
    const R* __restrict__ xb = p.x + line * p.line_in + l;
    R* __restrict__ yb = p.y + line * p.line_out + l;
    const bool want_dot = Op::DOT && (p.flags & F_DOT) && line >= (p.narr - 1) * p.nr;
    const int i0 = p.i_first + (int)(blockIdx.x / (unsigned)p.cblocks) * p.chunk;
    const int i1 = min(i0 + p.chunk, p.i_first + p.nout);
    R win[W][IN];  // step j is in slot (j - (i0 + LO)) mod W
    int jp = BC == PER ? pmod(i0 + Op::LO, p.n) : 0;
    auto load = [&](R* w, int j) {
#pragma unroll
      for (int c = 0; c < IN; ++c)
        w[c] = BC == PER ? xb[in_elem<K>(jp, c, p.nx) * p.L] : load_step<K, BC>(xb, p.L, j, c, p.n, p.nx, p.ox);
      if (BC == PER) jp = jp + 1 == p.n ? 0 : jp + 1;
    };
#pragma unroll
    for (int s = 0; s < W - 1; ++s) load(win[s], i0 + Op::LO + s);
    for (int base = i0; base < i1; base += W) {
#pragma unroll
      for (int u = 0; u < W; ++u) {
        const int i = base + u;
        if (i < i1) {
          load(win[(u + W - 1) % W], i + Op::UP);
          R o[OUT];
#pragma unroll
          for (int c = 0; c < OUT; ++c) o[c] = R(0);
#pragma unroll
          for (int s = 0; s < W; ++s) Op::step(s, win[(u + s) % W], o);
          sweep_post<Op, BC>(p, i, win[(u - Op::LO) % W][0], want_dot, dot, o);
#pragma unroll
          for (int c = 0; c < OUT; ++c) {
            R* yp = yb + out_elem<K>(i - p.oy, c, p.ny) * p.L;
            if (p.flags & F_AY) o[c] = fmar(p.a_y, *yp, o[c]);
            *yp = o[c];
          }
        }
      }
    }
  }
  if (p.dot_part) {
    const double s = block_sum<R>(dot, red);
    if (threadIdx.x == 0) p.dot_part[blockIdx.x] = s;
  }
}

// ------------------------------------------------- contiguous, a segment per group
// 2^lg lanes of Q outputs share a line's segment: 256 >> lg lines per block,
// the input steps of each in LDS, one run per component.
constexpr int kSegQ = 4;
template <typename R, class Op, int BC>
__global__ __launch_bounds__(256) void sweep_seg(SweepArgs<R> p, int lg) {
  constexpr int K = KindOf<Op>::v, Q = kSegQ;
  constexpr int W = Op::W, IN = Op::IN, OUT = Op::OUT;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  R* sm = reinterpret_cast<R*>(smem_raw);
  __shared__ double red[4];
  const int TPL = 1 << lg, LPB = 256 >> lg, NS = p.chunk + W - 1;  // chunk = TPL Q
  const int tl = threadIdx.x & (TPL - 1), lnb = threadIdx.x >> lg;
  const long line = (long)(blockIdx.x % (unsigned)p.cblocks) * LPB + lnb;
  const bool active = line < p.ncols;
  const int i0 = p.i_first + (int)(blockIdx.x / (unsigned)p.cblocks) * p.chunk;
  const int iend = p.i_first + p.nout;
  const R* __restrict__ xb = p.x + (active ? line * p.line_in : 0);
  R* __restrict__ yb = p.y + (active ? line * p.line_out : 0);
  if (active) {
    // steps beyond iend - 1 + UP are never used and may lie outside x (shrink)
    const int jmax = iend - 1 + Op::UP;
    for (int e = tl; e < NS * IN; e += TPL) {  // memory order: pairs (DWT), bands (IDWT)
      const int c = K == KDWT ? e & 1 : K == KIDWT ? e / NS : 0, s = K == KDWT ? e >> 1 : e - c * NS;
      const int j = i0 + Op::LO + s;
      sm[(c * LPB + lnb) * NS + s] = j <= jmax ? load_step<K, BC>(xb, 1, j, c, p.n, p.nx, p.ox) : R(0);
    }
  }
  __syncthreads();
  double dot = 0.0;
  if (active) {
    const bool want_dot = Op::DOT && (p.flags & F_DOT) && line >= (p.narr - 1) * p.nr;
    const int ib = i0 + tl * Q;
    SweepTask<R, Op, Q> t;
    const R* base = sm + lnb * NS + tl * Q;
    t.run([&](int c, int k) { return base[c * LPB * NS + k]; });
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int i = ib + q;
      if (i < iend) {
        sweep_post<Op, BC>(p, i, t.xc[q], want_dot, dot, t.o[q]);
#pragma unroll
        for (int c = 0; c < OUT; ++c) {
          R* yp = yb + out_elem<K>(i - p.oy, c, p.ny);
          R o = t.o[q][c];
          if (p.flags & F_AY) o = fmar(p.a_y, *yp, o);
          *yp = o;
        }
      }
    }
  }
  if (p.dot_part) {
    const double s = block_sum<R>(dot, red);
    if (threadIdx.x == 0) p.dot_part[blockIdx.x] = s;
  }
}

// Sums of NS (<= 4) sets of nparts partials, in a fixed order (one block of
// whole waves): out[k] = sum of set k.  The launch is latency only: every
// thread has kPartUnroll partials of every set in flight before it adds them
// (in index order), the waves sum by shuffles and the first wave adds their
// sums by shuffles again, 16 lanes per set.  Sizes as they come: a few hundred
// to some ten thousand partials; blocks of 256 threads up to 1024 partials.
// 4.9 us for three sets of 4000 partials with the tail's loads one after the
// other and the waves' sums added by one lane; now 3.8 - 4.1, an empty launch 2.
constexpr int kPartUnroll = 4, kPartThreads = 1024, kPartThreadsFew = 256, kPartFew = 1024;
template <int NS>
__global__ __launch_bounds__(kPartThreads) void sum_partials(const double* __restrict__ part, long nparts,
                                                              double* __restrict__ out, long stride) {
  __shared__ double red[NS][16];
  const int nt = blockDim.x, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  double v[NS];
#pragma unroll
  for (int k = 0; k < NS; ++k) v[k] = 0.0;
  for (long i0 = threadIdx.x; i0 < nparts; i0 += (long)kPartUnroll * nt) {
    double a[NS][kPartUnroll];
#pragma unroll
    for (int u = 0; u < kPartUnroll; ++u) {
      const long i = i0 + (long)u * nt;
#pragma unroll
      for (int k = 0; k < NS; ++k) a[k][u] = i < nparts ? part[k * stride + i] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < kPartUnroll; ++u)
#pragma unroll
      for (int k = 0; k < NS; ++k) v[k] += a[k][u];
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
#pragma unroll
    for (int k = 0; k < NS; ++k) v[k] += __shfl_xor(v[k], o, 64);
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < NS; ++k) red[k][wid] = v[k];
  __syncthreads();
  if (wid == 0) {
    const int k = lane >> 4, w = lane & 15;
    double s = k < NS && w < nt / 64 ? red[k < NS ? k : 0][w] : 0.0;
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (w == 0 && k < NS) out[k] = s;
  }
}

// ---------------------------------------------------------------- launcher
// Which form.  The tiles hold 32 columns and at least 16 outputs of each and
// are latency-lean; the forms without a tile need no column or output that is
// not there.  They win where the tile would be mostly padding -- a few outputs
// per line, or a few long lines -- once there are enough lines to fill the chip
// by themselves, and for the wavelets, whose tile re-reads W - 1 pairs per
// chunk, on ranges of longer lines too (up to 1.4 times as fast; over the rest
// of those ranges the tiles are).  The bounds are where the two measured
// times cross (periodic sweeps, device time): second derivative FP64, strided,
// 131072 columns: 6 outputs 7.0 us without a tile against 11.0 with one, 32
// outputs 19 against 15; a contiguous line of 2^20 points 11.4 against 57, of
// 28000 points 3.8 against 5.7, 8 of 57000 points 6.2 against 7.3, 16 of them
// 8.8 against 8.1; symicomb8 FP64 along the second of 100^3 pairs 28 against
// 37; sym8 FP64 on 32768 columns of 8 pairs 5.6 against 5.4, of 80 pairs 17
// against 20.8.  Over 15000 calls tried (boxes, and grids of 1 .. 2^19 lines
// by 1 .. 2^20 outputs, L odd and even) the choice is 0.4% behind the faster
// form on average, and more than 15% behind it in 70.
static bool ring_pays(long ncols, long L, int nout, int in, int W, int rs) {
  const double total = (double)ncols * nout;
  if (in == 1)
    return (ncols >= 49152 && nout <= (rs == 4 && ncols >= 196608 ? 16 : W > 16 ? 12 : 8)) ||
           (ncols >= 32768 && nout <= 4);
  if (ncols >= 16384 && nout <= 4) return true;
  if (L < 8 && nout > 12) return false;  // lanes of a wave on several lines, far apart
  if (W <= 8) {
    if (rs == 8)
      return (ncols >= 32768 && nout <= 12) || (ncols >= 196608 && nout >= 32 && nout <= 64) ||
             (ncols >= 100 && nout >= 40 && total >= (ncols >= 24576 ? 1.9e6 : 2.3e6) && total <= 8.5e6);
    return (ncols >= 49152 && nout <= 40) || (ncols >= 2048 && nout >= 40 && total >= 1.2e6 && total <= 2.7e6);
  }
  if (rs == 8)
    return (ncols >= 65536 && nout <= 160) || (ncols >= 49152 && nout <= 20) ||
           (ncols >= 64 && total >= 2.6e6 && total <= 8.5e6);
  return (ncols >= 24576 && nout <= 6) || (ncols >= 49152 && nout <= 12) || (ncols >= 65536 && nout <= 28) ||
         (ncols >= 131072 && nout <= 160) || (ncols >= 98304 && nout >= 64 && nout <= 160) ||
         (ncols >= 16384 && nout >= 80 && nout <= 512 && total >= 5e6);
}
static bool seg_pays(long ncols, int nout, int in, int W, int rs) {
  if ((ncols <= 8 && nout >= 50000) || (ncols <= 12 && nout >= 80000)) return true;
  if (ncols <= 4 && nout >= (in == 2 ? 34000 : ncols > 2 ? 25000 : rs == 8 ? 17000 : 22000)) return true;
  if (in == 1) return ncols >= 24576 && nout <= 12;
  if (W <= 8) return (ncols >= 16384 && nout <= 2) || (ncols >= 262144 && nout <= 4);
  return ncols >= 24576 && nout <= (rs == 8 ? 4 : 6);
}

// Launch shape.  Tiles: the largest chunk (outputs per lane Q in 2, 4, 8, 16)
// whose blocks still number four per CU -- halo rows cost reads, few blocks
// leave CUs idle in a launch that lasts one round of blocks --, not more than
// twice the line (32 outputs of 65536 FP64 magic-filter columns: 15 us with
// chunks for 128, 9 with chunks for 32), and chunks of equal length.  The
// wavelets' tiles are twice as deep per output step: Q up to 8 (sym8) and 4
// (windows of 16 pairs).  Ring: chunks of two windows and more, until eight
// waves per CU.  Segments: the lanes that a line's outputs fill, 4 to 64.
enum SweepForm { SWEEP_TILE, SWEEP_RING, SWEEP_SEG };
struct SweepPlan {
  SweepForm form;
  int q, lg;  // outputs per lane of a tile; lanes per segment (log2)
  int chunk;
  long cblocks, blocks;
};
template <typename R>
static SweepPlan sweep_plan(const SweepArgs<R>& p, int in, int W) {
  constexpr int C = kSweepCols, G = 256 / C;
  SweepPlan s{};
  int n;
  if (p.L == 1 && seg_pays(p.ncols, p.nout, in, W, sizeof(R))) {
    s.form = SWEEP_SEG;
    s.lg = 2;
    while (s.lg < 6 && (kSegQ << s.lg) < p.nout) ++s.lg;
    s.chunk = kSegQ << s.lg;
    s.cblocks = (p.ncols + (256 >> s.lg) - 1) / (256 >> s.lg);
    n = (p.nout + s.chunk - 1) / s.chunk;
  } else if (p.L > 1 && ring_pays(p.ncols, p.L, p.nout, in, W, sizeof(R))) {
    s.form = SWEEP_RING;
    const long waves = (p.ncols + 63) / 64;
    n = (int)std::max(1L, std::min<long>((8L * num_cu() + waves - 1) / waves, p.nout / (2 * W)));
    s.chunk = (p.nout + n - 1) / n;
    s.cblocks = (p.ncols + 255) / 256;
    n = (p.nout + s.chunk - 1) / s.chunk;
  } else {
    s.form = SWEEP_TILE;
    s.cblocks = (p.ncols + C - 1) / C;
    s.q = in == 1 ? 16 : W > 8 ? 4 : 8;
    while (s.q > 2 && (s.cblocks * ((p.nout + G * s.q - 1) / (G * s.q)) < 4L * num_cu() || p.nout <= G * s.q / 2))
      s.q /= 2;
    n = (p.nout + G * s.q - 1) / (G * s.q);
    s.chunk = (p.nout + n - 1) / n;
  }
  s.blocks = s.cblocks * n;
  return s;
}

// for div_inv
static unsigned inv32(int n) { return (unsigned)std::min<unsigned long>((1ul << 32) / (unsigned)n, 0xfffffffful); }

template <typename R, class Op, int BC>
static hipError_t run_sweep(const SweepArgs<R>& a0, hipStream_t st, double* dot_out) {
  SweepArgs<R> p = a0;
  if (p.ncols == 0 || p.nout == 0) {
    if (dot_out) return hipMemsetAsync(dot_out, 0, sizeof(double), st);
    return hipSuccess;
  }
  const SweepPlan s = sweep_plan(p, Op::IN, Op::W);
  if (s.blocks > 0x7fffffffL) return hipErrorInvalidValue;
  p.chunk = s.chunk;
  p.cblocks = (int)s.cblocks;
  if (s.form == SWEEP_RING) {
    sweep_ring<R, Op, BC><<<(unsigned)s.blocks, 256, 0, st>>>(p);
  } else if (s.form == SWEEP_SEG) {
    const size_t lds = (size_t)(256 >> s.lg) * (s.chunk + Op::W - 1) * Op::IN * sizeof(R);
    sweep_seg<R, Op, BC><<<(unsigned)s.blocks, 256, lds, st>>>(p, s.lg);
  }
  p.nchunk = (int)(s.blocks / s.cblocks);
  // whole rounds of 8 runs, of about as many columns of tiles as said at tile_of
  const long col = (long)p.nchunk * (p.L > 1 && p.L % kSweepCols ? kSweepRun : 1);
  p.run = (int)std::max(1L, s.blocks / (8 * std::max(1L, s.blocks / (8 * col))));
  p.nchunk_inv = inv32(p.nchunk);
  p.run_inv = inv32(p.run);
  p.run_end = (unsigned)(s.blocks - s.blocks % (8L * p.run));
  auto launch = [&](auto q) {
    constexpr int Q = decltype(q)::value;
    if (p.L == 1 && (p.flags & F_AY))
      sweep_contig<R, Op, BC, Q, true><<<(unsigned)s.blocks, 256, 0, st>>>(p);
    else if (p.L == 1)
      sweep_contig<R, Op, BC, Q, false><<<(unsigned)s.blocks, 256, 0, st>>>(p);
    else
      sweep_strided<R, Op, BC, Q><<<(unsigned)s.blocks, 256, 0, st>>>(p);
  };
  constexpr int QM = Op::IN == 1 ? 16 : Op::W > 8 ? 4 : 8;
  if constexpr (QM >= 16) {
    if (s.q == 16) launch(std::integral_constant<int, 16>{});
  }
  if constexpr (QM >= 8) {
    if (s.q == 8) launch(std::integral_constant<int, 8>{});
  }
  if (s.q == 4) launch(std::integral_constant<int, 4>{});
  if (s.q == 2) launch(std::integral_constant<int, 2>{});
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (p.dot_part && dot_out) {
    e = sum_partial_sets(p.dot_part, s.blocks, dot_out, 1, 0, st);
  }
  return e;
}

template <typename R>
long sweep_partials_needed(const SweepArgs<R>& p, int W) {
  return sweep_plan(p, 1, W).blocks;  // only the filters form partials
}

template <typename R, class Op>
static hipError_t run_bc(int bc, const SweepArgs<R>& p, hipStream_t st, double* dot_out) {
  switch (bc) {
    case PER: return run_sweep<R, Op, PER>(p, st, dot_out);
    case GROW: return run_sweep<R, Op, GROW>(p, st, dot_out);
    case SHRINK: return run_sweep<R, Op, SHRINK>(p, st, dot_out);
  }
  return hipErrorInvalidValue;
}

template <typename R>
hipError_t sweep(int kind, int id, int bc, const SweepArgs<R>& p, hipStream_t st, double* dot_out) {
  if (kind == KCONV) {
    switch (id) {
      case OP_MD: return run_bc<R, Conv<FMD>>(bc, p, st, dot_out);
      case OP_IMD: return run_bc<R, Conv<FIMD>>(bc, p, st, dot_out);
      case OP_D2: return run_bc<R, Conv<FD2>>(bc, p, st, dot_out);
      case OP_D1: return run_bc<R, Conv<FD1>>(bc, p, st, dot_out);
    }
  } else if (kind == KDWT) {
    if (id == WAV_SYM8) return run_bc<R, Dwt<Sym8Dec>>(bc, p, st, nullptr);
    if (id == WAV_SYMICOMB8)
      return bc == PER ? run_bc<R, Dwt<CombPDec>>(bc, p, st, nullptr)
                       : run_bc<R, Dwt<CombGDec>>(bc, p, st, nullptr);
  } else if (kind == KIDWT) {
    if (id == WAV_SYM8) return run_bc<R, Idwt<Sym8Rec>>(bc, p, st, nullptr);
    if (id == WAV_SYMICOMB8)
      return bc == PER ? run_bc<R, Idwt<CombPRec>>(bc, p, st, nullptr)
                       : run_bc<R, Idwt<CombGRec>>(bc, p, st, nullptr);
  }
  return hipErrorInvalidValue;
}

template hipError_t sweep<double>(int, int, int, const SweepArgs<double>&, hipStream_t, double*);
template hipError_t sweep<float>(int, int, int, const SweepArgs<float>&, hipStream_t, double*);
template long sweep_partials_needed<double>(const SweepArgs<double>&, int);
template long sweep_partials_needed<float>(const SweepArgs<float>&, int);

hipError_t sum_partial_sets(const double* part, long nparts, double* out, int nsets, long stride,
                            hipStream_t st) {
  const int nt = nparts <= kPartFew ? kPartThreadsFew : kPartThreads;
  switch (nsets) {
    case 1: sum_partials<1><<<1, nt, 0, st>>>(part, nparts, out, stride); break;
    case 2: sum_partials<2><<<1, nt, 0, st>>>(part, nparts, out, stride); break;
    case 3: sum_partials<3><<<1, nt, 0, st>>>(part, nparts, out, stride); break;
    case 4: sum_partials<4><<<1, nt, 0, st>>>(part, nparts, out, stride); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace lc
