// lc_body_wavq.hpp -- device body of the pair-wise 3D sym8 wavelet kernel
// (internal).  Same arithmetic and summation order as sepw3d_body (x, then y,
// then z; within a pass the window steps in increasing order, value 0 before
// value 1), so both give identical bits.
//
// The two values of a step lie next to each other in LDS, so that every filter
// read takes a whole step (16 bytes in FP64) at any step offset, and a block
// works one input z-step (two planes) per pair of barriers:
//
//   * the tile A[plane][row][step] holds pairs (value 0, value 1 along x);
//     row 2 s1 + v1 is value v1 of y-step s1;
//   * x-tasks filter QX output steps of a row (both x-bands) from QX + 7 pair
//     reads and write them transposed into B[plane][col][s1] as the v1 half of
//     a pair;
//   * y-tasks (one column, one output step per lane) read 8 pairs per plane
//     and push the y-bands into a ring of 8 z-steps in registers; the lane
//     emits the output z-step whose window is complete (both z-bands).  With
//     HB = 2 the two y-bands go to two lanes: half the ring per lane and half
//     the serial work per step, for grids that leave the chip idle.
//
// All waves run x-tasks, then y-tasks: one tile and one x-filtered copy in
// LDS, so that several blocks fit on a CU and fill each other's barriers.
// Strides of A and B are odd numbers of pairs, and consecutive lanes take
// consecutive rows (x) or columns (y): no bank conflicts.
//
// What bounds it (FP64).  A batch that fills the chip (128 orbitals): bytes.
// Without its FMAs it takes as long as with them (1.45 ms on fixed 16 x 16 tiles;
// the FMAs and LDS reads alone 0.87), and it moves 3.9 GB, halo lines that miss
// L2 included, at 3.6 TB/s (a copy: 5.1).  Hence tiles of any shape, chosen per
// grid (WavqShape): no lanes on padding and the widest tile the block holds,
// since a halo read that misses L2 costs as much as an input value.  A single
// call (96^3 pairs): the serial chain of a step with two barriers, 504 blocks
// or two waves per SIMD to hide it -- 3.0 TB/s, VALU busy 35% and LDS 24 - 31%
// of the time, none of them at its limit; hence the choice of tile and z chunk
// by expected time.  The form with a plane per barrier on 8 x 8 tiles and 8-byte
// y reads (LDS busy 52% of its cycles, a fifth of that bank conflicts) takes
// 1.65 ms for the batch.
//
// ME: the epilogue reads y (F_AY).  Without (ME false) every wave issues the
// same memory operations in every step, the outputs as buffer stores that drop
// invalid lanes (offset out of range) and the steps that emit nothing (record
// count 0), so the compiler's wait counts are exact and a step waits only for
// the tile loads it uses.
#pragma once

#include <type_traits>

#include "lc_body_wav.hpp"

namespace lc {

template <typename R>
struct Pair2;
template <> struct Pair2<double> { using T = double2; };
template <> struct Pair2<float> { using T = float2; };

// A block's tile is tx x ty output steps, chosen per grid: any shape whose
// y-tasks, x-tasks and tile pairs fit the block's lanes (WavqBlock::fits).
// The strides and task maps follow from it once per block.
struct WavqShape {
  int tx, ty;
  int txr;     // columns per x-band in B: whole x-tasks
  int as, bs;  // row stride of A, column stride of B (odd numbers of pairs)
  int nr;      // tile rows per plane
  __host__ __device__ WavqShape(int tx_, int ty_, int qx) : tx(tx_), ty(ty_) {
    txr = (tx + qx - 1) / qx * qx;
    as = (txr + 7) | 1;
    bs = (ty + 7) | 1;
    nr = 2 * (ty + 7);
  }
  __host__ __device__ int pa() const { return nr * as; }          // pairs per plane of A
  __host__ __device__ int pb() const { return 2 * txr * bs; }     // and of B
  __host__ __device__ int pairs() const { return nr * (tx + 7); } // tile pairs per plane
  __host__ __device__ int xtasks(int qx) const { return 2 * nr * (txr / qx); }
};
// A block for S output steps per plane: its lanes, the tile pairs per lane and
// plane, the rounds of x-tasks, its LDS bytes (rs = sizeof(R)), and the tiles
// it takes.
struct WavqBlock {
  int S, QX, HB;
  constexpr int nt() const { return 2 * HB * S; }
  constexpr int nul() const { return HB == 2 || S >= 512 ? 2 : 3; }
  constexpr int nxl() const { return QX == 2 && HB == 1 ? 2 : 1; }
  // four blocks of 256 lanes (FP64) or eight (FP32) fill the 160 KB of a CU
  constexpr size_t lds(int rs) const { return (size_t)nt() * 20 * rs; }
  bool fits(const WavqShape& g, int rs) const {
    return g.tx * g.ty <= S && g.xtasks(QX) <= nxl() * nt() && g.pairs() <= nul() * nt() &&
           4 * (size_t)rs * (g.pa() + g.pb()) <= lds(rs);
  }
};

// The high-pass taps are the low-pass taps reversed with alternating signs, so
// 16 values serve all 32 coefficients of a pass.  FP64: kept in scalar
// registers behind an empty asm, the sign an operand modifier (32 separate
// constants are more scalar registers than a wave has left, and spill to VGPR
// lanes: 53 spills against none).  FP32: instruction literals (128-orbital
// batch 0.80 ms, 0.94 with the taps in scalar registers).
template <typename R>
struct WavTaps {
  R v[FLP::N];
  __device__ __forceinline__ WavTaps() {
#pragma unroll
    for (int k = 0; k < FLP::N; ++k) {
      v[k] = tap<R, FLP>(k);
      if constexpr (sizeof(R) == 8) asm("" : "+s"(v[k]));
    }
  }
  // index of the tap of this magnitude, and its sign
  static constexpr int idx(R c) {
    for (int k = 0; k < FLP::N; ++k)
      if (tap<R, FLP>(k) == c || tap<R, FLP>(k) == -c) return k;
    return -1;
  }
  template <class C, int CO, int CI, int S>
  __device__ __forceinline__ R get() const {
    constexpr R c = C::template c<R>(CO, CI, S);
    constexpr int k = idx(c);
    static_assert(k >= 0, "a low-pass tap up to its sign");
    return tap<R, FLP>(k) == c ? v[k] : -v[k];
  }
};
// f(integral_constant<0>) .. f(integral_constant<N - 1>)
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (N > 0) {
    static_for<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

// one pair of adjacent values at byte offset `boff` (kOffNone reads zeros)
template <typename R>
__device__ __forceinline__ typename Pair2<R>::T plane_ld2(__amdgpu_buffer_rsrc_t rs, int boff) {
  using T = typename Pair2<R>::T;
  if constexpr (sizeof(R) == 8)
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(rs, boff, 0, 0));
  else
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(rs, boff, 0, 0));
}

template <typename R, class Op, int S, int QX, int HB, int PD, bool ME>
__device__ __forceinline__ void wavq_body(const FusedArgs<R>& p, int bx, int by, int zc, int arr,
                                          unsigned char* lds) {
  using P2 = typename Pair2<R>::T;
  using C = WavCoef<Op>;
  constexpr WavqBlock kB{S, QX, HB};
  constexpr int K = C::K, W = Op::W, LO = Op::LO, NT = kB.nt(), NUL = kB.nul(), NXL = kB.nxl();
  static_assert(W == 8 && NT % (64 * HB) == 0, "sym8 split filters, whole waves per band");
  const WavqShape g(p.tile_x, p.tile_y, QX);
  const int PA = g.pa(), PB = g.pb(), tws = g.tx + W - 1;
  P2* const A = reinterpret_cast<P2*>(lds);  // [2][nr][as]
  P2* const B = A + 2 * PA;                  // [2][2 txr][bs]

  const int t = threadIdx.x;
  const R* __restrict__ xa = p.x + arr * p.nti;
  R* __restrict__ ya = p.y + arr * p.nto;
  const int X0 = p.d0.olo + bx * g.tx, Y0 = p.d1.olo + by * g.ty;
  const int zb = p.d2.olo + zc * p.zchunk;
  const int ze = min(zb + p.zchunk, p.d2.olo + p.d2.nout);
  const long rs_in = 2L * p.d0.nx, ps_in = 4L * p.d0.nx * p.d1.nx;
  const long rs_out = 2L * p.d0.ny, ps_out = 4L * p.d0.ny * p.d1.ny;
  const int nsteps = (ze - zb) + W - 1;  // input z-steps of this chunk

  // ---- tile pairs of this lane: pair t + j NT of a plane (the same places in
  // both planes).  Along x the DWT finds its pair adjacent in memory, the
  // IDWT its two values nx apart (one per band).
  int aoff[NUL], aslot[NUL];
#pragma unroll
  for (int j = 0; j < NUL; ++j) {
    const int u = t + j * NT;
    const int rr = u / tws, s0 = u - rr * tws;
    const int s1 = rr >> 1, v1 = rr & 1;
    const int j0 = fsrc(p.d0, X0 + LO + s0), j1 = fsrc(p.d1, Y0 + LO + s1);
    const bool ok = rr < g.nr && j0 >= 0 && j1 >= 0;
    aoff[j] = plane_boff<R>(ok ? (int)(in_elem<K>(j0, 0, p.d0.nx) + rs_in * in_elem<K>(j1, v1, p.d1.nx)) : -1);
    aslot[j] = rr < g.nr ? rr * g.as + s0 : -1;
  }
  const int hoff = p.d0.nx * (int)sizeof(R);  // IDWT: L to H
  ZCursor zcur(p.d2, zb + LO);
  P2 bufs[PD][2][NUL];
  auto load_step = [&](P2 (&buf)[2][NUL]) {
    const int s2 = zcur.src();
    zcur.next();
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const long pl = s2 >= 0 ? in_elem<K>(s2, c, p.d2.nx) : 0;
      const __amdgpu_buffer_rsrc_t rs = span_rsrc(xa + ps_in * pl, s2 >= 0 ? ps_in : 0);
#pragma unroll
      for (int j = 0; j < NUL; ++j) {
        if constexpr (K == KDWT) {
          buf[c][j] = plane_ld2<R>(rs, aoff[j]);
        } else {
          buf[c][j].x = plane_ld<R>(rs, aoff[j]);
          buf[c][j].y = plane_ld<R>(rs, aoff[j], hoff);
        }
      }
    }
  };

  // ---- y-task: output column yl (memory order along x), output step yi and,
  // with HB = 2, one y-band
  constexpr int NB = 2 / HB;
  const int band = HB == 2 ? __builtin_amdgcn_readfirstlane(t / (NT / 2)) : 0;
  const int yt = HB == 2 ? t - band * (NT / 2) : t;
  const bool ylane = yt < 2 * g.tx * g.ty;
  const int yi = ylane ? yt / (2 * g.tx) : 0, yl = ylane ? yt - yi * 2 * g.tx : 0;
  const int c0 = K == KIDWT ? (yl & 1) : (yl >= g.tx ? 1 : 0);
  const int i0l = K == KIDWT ? (yl >> 1) : yl - c0 * g.tx;
  const P2* const ycol = B + (K == KIDWT ? yl : c0 * g.txr + i0l) * g.bs + yi;
  const bool out_ok = ylane && (X0 + i0l < p.d0.olo + p.d0.nout) && (Y0 + yi < p.d1.olo + p.d1.nout);
  const long oyb = rs_out * (out_elem<K>(0, 1, p.d1.ny) - out_elem<K>(0, 0, p.d1.ny));  // y-band 1 - y-band 0
  const long oxy = out_elem<K>(X0 + i0l - p.d0.oy, c0, p.d0.ny) +
                   rs_out * out_elem<K>(Y0 + yi - p.d1.oy, 0, p.d1.ny) + band * oyb;
  const long ozb = ps_out * (out_elem<K>(0, 1, p.d2.ny) - out_elem<K>(0, 0, p.d2.ny));  // z-band 1 - z-band 0
  const long zstep = ps_out * (out_elem<K>(1, 0, p.d2.ny) - out_elem<K>(0, 0, p.d2.ny));
  long zo = ps_out * out_elem<K>(zb - p.d2.oy, 0, p.d2.ny);

  // ---- x-tasks: consecutive lanes take consecutive rows of both planes
  // (offsets of the row in A, of the first output value in B)
  const P2* xsrc[NXL];
  R* xdst[NXL];
  bool xlane[NXL];
#pragma unroll
  for (int r = 0; r < NXL; ++r) {
    const int xt = t + r * NT;
    const int xg = xt / (2 * g.nr), row = xt - xg * 2 * g.nr, c = row >= g.nr ? 1 : 0;
    xlane[r] = xt < g.xtasks(QX);
    xsrc[r] = A + (xlane[r] ? row * g.as + xg * QX : 0);
    // row 2 s1 + v1 of the plane: half v1 of pair s1
    xdst[r] = reinterpret_cast<R*>(B + c * PB + (K == KIDWT ? 2 : 1) * xg * QX * g.bs) + (row - c * g.nr);
  }
  const int dq = (K == KIDWT ? 4 : 2) * g.bs;               // next step's column
  const int d1 = (K == KIDWT ? 2 : 2 * g.txr) * g.bs;       // x-band 1 - x-band 0

  const WavTaps<R> taps;
  R ring[NB][W][2];  // [y-band][z-step mod 8][plane]
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int k = 0; k < W; ++k) ring[b][k][0] = ring[b][k][1] = R(0);
#pragma unroll
  for (int k = 0; k < PD; ++k) load_step(bufs[k]);

  for (int sb = 0;; sb += W) {
#pragma unroll
    for (int u = 0; u < W; ++u) {
      const int s = sb + u;
      // ---- tile of step s, then the loads of step s + PD
      P2 (&buf)[2][NUL] = bufs[u % PD];
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int j = 0; j < NUL; ++j)
          if (aslot[j] >= 0) A[c * PA + aslot[j]] = buf[c][j];
      load_step(buf);
      __syncthreads();
#pragma unroll
      for (int r = 0; r < NXL; ++r) {
        if (xlane[r]) {
          R t0[QX], t1[QX];
#pragma unroll
          for (int q = 0; q < QX; ++q) t0[q] = t1[q] = R(0);
          static_for<QX + W - 1>([&](auto kk) {
            constexpr int k = decltype(kk)::value;
            const P2 v = xsrc[r][k];
            static_for<QX>([&](auto qq) {
              constexpr int q = decltype(qq)::value, ss = k - q;
              if constexpr (ss >= 0 && ss < W) {
                t0[q] = fmar(v.x, taps.template get<C, 0, 0, ss>(), t0[q]);
                t1[q] = fmar(v.x, taps.template get<C, 1, 0, ss>(), t1[q]);
                t0[q] = fmar(v.y, taps.template get<C, 0, 1, ss>(), t0[q]);
                t1[q] = fmar(v.y, taps.template get<C, 1, 1, ss>(), t1[q]);
              }
            });
          });
#pragma unroll
          for (int q = 0; q < QX; ++q) {
            xdst[r][q * dq] = t0[q];
            xdst[r][q * dq + d1] = t1[q];
          }
        }
      }
      __syncthreads();
      // ---- y-tasks on both planes, into the ring
      auto ytask = [&](auto b0) {  // y-bands b0 .. b0 + NB - 1
        constexpr int B0 = decltype(b0)::value;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          R y[NB];
#pragma unroll
          for (int b = 0; b < NB; ++b) y[b] = R(0);
          static_for<W>([&](auto sv) {
            constexpr int ss = decltype(sv)::value;
            const P2 v = ycol[c * PB + ss];
            static_for<NB>([&](auto bb) {
              constexpr int b = decltype(bb)::value;
              y[b] = fmar(v.x, taps.template get<C, B0 + b, 0, ss>(), y[b]);
              y[b] = fmar(v.y, taps.template get<C, B0 + b, 1, ss>(), y[b]);
            });
          });
#pragma unroll
          for (int b = 0; b < NB; ++b) ring[b][u][c] = y[b];
        }
      };
      if (HB == 1 || band == 0)
        ytask(std::integral_constant<int, 0>{});
      else if constexpr (HB == 2)
        ytask(std::integral_constant<int, 1>{});
      // ---- z: the output step whose window is input steps s - 7 .. s
      const bool em = s >= W - 1;  // uniform
      R outv[NB][2];
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        R o0 = R(0), o1 = R(0);
        static_for<W>([&](auto sv) {
          constexpr int ss = decltype(sv)::value;
          const R v0 = ring[b][(u + 1 + ss) % W][0], v1 = ring[b][(u + 1 + ss) % W][1];
          o0 = fmar(v0, taps.template get<C, 0, 0, ss>(), o0);
          o1 = fmar(v0, taps.template get<C, 1, 0, ss>(), o1);
          o0 = fmar(v1, taps.template get<C, 0, 1, ss>(), o0);
          o1 = fmar(v1, taps.template get<C, 1, 1, ss>(), o1);
        });
        if (p.flags & F_A) {
          o0 = o0 * p.a0;
          o1 = o1 * p.a0;
        }
        outv[b][0] = o0;
        outv[b][1] = o1;
      }
      if constexpr (ME) {
        if (em && out_ok) {
#pragma unroll
          for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int zbd = 0; zbd < 2; ++zbd) {
              R* yp = ya + zo + zbd * ozb + oxy + b * oyb;
              R v = outv[b][zbd];
              if (p.flags & F_AY) v = fmar(p.a_y, *yp, v);
              *yp = v;
            }
        }
      } else {
        const __amdgpu_buffer_rsrc_t r0 = span_rsrc(ya + zo, em ? ps_out : 0);
        const __amdgpu_buffer_rsrc_t r1 = span_rsrc(ya + zo + ozb, em ? ps_out : 0);
        const int boff = out_ok ? (int)(oxy * (long)sizeof(R)) : kOffNone;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const int sb_off = (int)(b * oyb * (long)sizeof(R));
          plane_st<R>(r0, boff, outv[b][0], sb_off);
          plane_st<R>(r1, boff, outv[b][1], sb_off);
        }
      }
      zo += em ? zstep : 0;
      if (s + 1 == nsteps) return;
    }
  }
}

}  // namespace lc
