// The dense Newton factor stage above 32 dofs on one wavefront per world, its matrices in the
// wavefront's matrix-core tiles (nv_pad = 16 NB = 48, 64 or 80): the incremental update of H's upper
// triangle over the changed rows, the augmented blocked Cholesky U'U = H (16 x 16 blocks, the gradient
// as the last column) or, without changed rows, the solve with the stored factor, the backward solve,
// search = -x and the two sums.
// Reference: src/instantmimic/utils/mjw_kernels/newton_stages.py:614-742 (stage), :473-611 (augmented
// blocked factor), :451-470 and :651-701 (update over the dof union).
//
// The upper block triangle is NB (NB + 1) / 2 accumulator tiles of v_mfma_f32_16x16x4_f32 (four
// registers each): register v of lane (g, c) = (lane / 16, lane % 16) holds row 4 g + v, column c.
//   * a sum of the blocked order (sixteen fused multiply-adds from zero over an earlier block row, then
//     one subtraction) is four chained instructions and a subtraction;
//   * inside a block row the elements lose the rows above one multiply-add after the other: four rows
//     at a time (a panel: the four registers of lane group p) the 4 x 4 diagonal block is worked out
//     from scalars, every tile's four rows follow by multiply-adds within their lanes, and one
//     instruction with the tile itself as its addend takes the four rows out of all rows below --
//     the instruction adds its four products one after the other, so the chain is the scalar one;
//   * a finished panel is turned into one register per tile (lane group g: row 4 p + g) with three
//     lane swaps, which is the operand layout of both factors of every later product and the layout in
//     which U is stored.
// The backward solve takes its products with U's rows the same way, the tiles turned round through LDS.
// About 2400 vector instructions and 125 matrix instructions per factor at 80 columns.  What bounds it: the
// chain of pivots (four per panel, a square root and a reciprocal each) with two to four wavefronts per
// SIMD to hide it.  Whole solves of the resident loop on this stage, before (a lane per column with
// broadcasts up to 64 columns, stage launches with a workgroup per world at 80) and after: 35 dofs x 8192
// worlds 1167 -> 717 us, 56 dofs x 4096 1459 -> 780 us, 70 dofs x 2048 2177 -> 970 us.
// Same operations in the same order as the workgroup-per-world kernel of blocked_kernels.hip and the CPU
// restatement both are tested against.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <utility>

#include "jtdj_wave.h"
#include "newton_wave.h"
#include "pivot.h"

namespace im {
namespace {

using resident::wave_sync;

template <int NB>
constexpr int kTiles = NB * (NB + 1) / 2;
// tile (i, j), i <= j, of NB block rows
template <int NB>
__host__ __device__ constexpr int tile_at(int i, int j) {
  return i * NB - i * (i - 1) / 2 + j - i;
}

// LDS words of one world's stage: the solution (16 NB), a 16 x 16 tile turned round (rows 17 words apart)
template <int NB>
__host__ __device__ constexpr int wave_stage_words() {
  return 16 * NB + 16 * 17;
}

__device__ __forceinline__ float lane_value(float v, int lane) {  // `lane` the same for the whole wavefront
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}
__device__ __forceinline__ float4v mfma16(float a, float b, float4v c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// Lane group g's value of the result: f_g of lane group P, column by column (P a constant).  The first swap
// exchanges odd groups of one register with even groups of its partner, which brings (f0, f1) and
// (f2, f3) of group P side by side; the second exchanges the wavefront's halves.  Written out with their
// wait states: the compiler's builtins return one result twice when both operands hold the same value.
template <int P>
__device__ __forceinline__ float panel_gather(float f0, float f1, float f2, float f3) {
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3\n\ts_nop 1" : "+v"(f0), "+v"(f1), "+v"(f2), "+v"(f3));
  float x = P & 1 ? f1 : f0, z = P & 1 ? f3 : f2;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(x), "+v"(z));
  return P < 2 ? x : z;
}

// The upper triangle of a 4 x 4 block's factor, the same in every lane: u[a][b] (a < b), the diagonal d[a]
// and its reciprocals i[a].
struct Panel {
  float u01, u02, u03, u12, u13, u23, d[4], inv[4];
};
template <bool FAST>
__device__ __forceinline__ unsigned panel_pivots(Panel &k, float a00, float a01, float a02, float a03, float a11, float a12, float a13,
                                                 float a22, float a23, float a33) {
  auto root = [](float x, float &d, float &inv) __attribute__((always_inline)) {
    if constexpr (FAST) {
      pivot_sqrt_rcp_fast(x, d, inv);
    } else {
      pivot_sqrt_rcp_any(x, d, inv);
    }
  };
  // distance of the pivots' bit patterns from 2^-96: negative, tiny, infinite and NaN ones lie far out
  constexpr unsigned kLow = 0x0f800000u;
  root(a00, k.d[0], k.inv[0]);
  k.u01 = a01 * k.inv[0], k.u02 = a02 * k.inv[0], k.u03 = a03 * k.inv[0];
  a11 = fma_(-k.u01, k.u01, a11);
  root(a11, k.d[1], k.inv[1]);
  a12 = fma_(-k.u01, k.u02, a12), a13 = fma_(-k.u01, k.u03, a13);
  k.u12 = a12 * k.inv[1], k.u13 = a13 * k.inv[1];
  a22 = fma_(-k.u12, k.u12, fma_(-k.u02, k.u02, a22));
  root(a22, k.d[2], k.inv[2]);
  a23 = fma_(-k.u12, k.u13, fma_(-k.u02, k.u03, a23));
  k.u23 = a23 * k.inv[2];
  a33 = fma_(-k.u23, k.u23, fma_(-k.u13, k.u13, fma_(-k.u03, k.u03, a33)));
  root(a33, k.d[3], k.inv[3]);
  auto far = [&](float x) { return __builtin_bit_cast(unsigned, x) - kLow; };
  const unsigned m01 = far(a00) > far(a11) ? far(a00) : far(a11), m23 = far(a22) > far(a33) ? far(a22) : far(a33);
  return m01 > m23 ? m01 : m23;
}

// f(0) .. f(N - 1) with the index as a constant, whatever the size of the body: an index into the tiles that
// is left to the compiler's unrolling would put them into scratch memory where it declines.
template <int... I, class F>
__device__ __forceinline__ void each_of(std::integer_sequence<int, I...>, F &&f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void each(F &&f) {
  each_of(std::make_integer_sequence<int, N>{}, f);
}

// The products of panels P0 .. P1 - 1 of two tiles, one after the other from zero.
template <int P0, int P1, class A, class C>
__device__ __forceinline__ float4v block_sum(const A &a, const C &b) {
  float4v s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int p = P0; p < P1; ++p) s = mfma16(a[p], b[p], s);
  return s;
}

// on ? a : b, by one instruction
__device__ __forceinline__ float pick(bool on, float a, float b) {
  const float v = on ? a : b;
  asm("" : : "v"(v));
  return v;
}

// The rows of a panel from its pivots: r's rows 4 g + v of lane group p, in panel layout.
__device__ __forceinline__ float panel_rows(const Panel &q, const float4v &r, int p) {
  const float f0 = r[0] * q.inv[0];
  const float f1 = fma_(-q.u01, f0, r[1]) * q.inv[1];
  const float f2 = fma_(-q.u12, f1, fma_(-q.u02, f0, r[2])) * q.inv[2];
  const float f3 = fma_(-q.u23, f2, fma_(-q.u13, f1, fma_(-q.u03, f0, r[3]))) * q.inv[3];
  return p == 0 ? panel_gather<0>(f0, f1, f2, f3) : p == 1 ? panel_gather<1>(f0, f1, f2, f3)
         : p == 2 ? panel_gather<2>(f0, f1, f2, f3) : panel_gather<3>(f0, f1, f2, f3);
}

// r -= the sums of the N block rows above, whose solution is in xl; above(k): the tile of block row k in this column
template <int N, int B, class Above>
__device__ __forceinline__ void less_sums(float4v &r, const float *xl, int g, Above &&above) {
  each<N>([&](auto k) __attribute__((always_inline)) {
    float z[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) z[p] = xl[16 * k + 4 * p + g];
    if constexpr (B == 8) {
      r = r - block_sum<0, 2>(above(k), z);
      r = r - block_sum<2, 4>(above(k), z);
    } else {
      r = r - block_sum<0, 4>(above(k), z);
    }
  });
}

// Factor of the tiles in place: U in panel layout (register p of lane (g, c): row 4 p + g, column c), its
// diagonal in the diagonal tiles, its reciprocals in rd[k] (lane r and 16 + r, ..: row 16 k + r).
// `last`: whether the last row's pivot counts as 1 (the corner of an augmented matrix).  Rows at and past nv
// are rows of the identity (but for the corner), and panels of such rows are not computed.  B: rows of a block of
// the blocked order, 16 or 8 (then two to a tile row, and a tile row's upper block leaves the lower one by a
// sum of its own).
// RHS: also z = U'^-1 rhs, for matrices without a spare column: rhs in xl (16 NB words, zero at and past nv), z in
// its place.
template <int NB, int B = 16, bool RHS = false>
__device__ __forceinline__ void factor_tiles(float4v (&t)[kTiles<NB>], float (&rd)[NB], bool last, float *xl, int nv, int lane) {
  const int g = lane >> 4, c = lane & 15;
  each<NB>([&](auto block_row) __attribute__((always_inline)) {
    constexpr int k = block_row;
    float uk[NB][4];  // the finished panels of block row k, tile k + j at [j]
    float rk = 1.0f;
    float4v r = {0.0f, 0.0f, 0.0f, 0.0f};
    float zk[4];
    if constexpr (RHS) {
      r = *(const float4v *)(xl + 16 * k + 4 * g);
      less_sums<k, B>(r, xl, g, [&](auto above) __attribute__((always_inline)) { return t[tile_at<NB>(above, k)]; });
    }
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      if (k == NB - 1 && p > 0 && 16 * k + 4 * p >= nv && !(last && p == 3)) {
        const bool one = c - 4 * p == g;
        uk[0][p] = one ? 1.0f : 0.0f;
        rk = c >> 2 == p ? 1.0f : rk;
        if constexpr (RHS) zk[p] = 0.0f;
        continue;
      }
      const float4v dg = t[tile_at<NB>(k, k)];
      const int l0 = 20 * p;  // lane (p, 4 p)
      Panel q;
      const float a00 = lane_value(dg[0], l0), a01 = lane_value(dg[0], l0 + 1), a02 = lane_value(dg[0], l0 + 2), a03 = lane_value(dg[0], l0 + 3);
      const float a11 = lane_value(dg[1], l0 + 1), a12 = lane_value(dg[1], l0 + 2), a13 = lane_value(dg[1], l0 + 3);
      const float a22 = lane_value(dg[2], l0 + 2), a23 = lane_value(dg[2], l0 + 3);
      float a33 = lane_value(dg[3], l0 + 3);
      // the corner: the gradient column's own row, whose pivot nothing below reads
      const bool corner = last && k == NB - 1 && p == 3;
      // (a branch per panel costs the larger matrices registers, the largest a hundred spilled ones: they take the
      // forms for every number, which are a twentieth of their work)
      constexpr bool kBranch = NB < 5;
      const unsigned far = panel_pivots<kBranch>(q, a00, a01, a02, a03, a11, a12, a13, a22, a23, corner ? 0x1p60f : a33);
      if constexpr (kBranch)
        if (__builtin_expect(__builtin_amdgcn_readfirstlane((int)(far >= 0x7f800000u - 0x0f800000u)), 0))
          (void)panel_pivots<false>(q, a00, a01, a02, a03, a11, a12, a13, a22, a23, corner ? 0x1p60f : a33);
      if (corner) q.d[3] = q.inv[3] = 1.0f;
      // (one select after another: as a choice among four the compiler makes branches of them)
      float dsel = pick(g == 0, q.d[0], q.d[3]);
      dsel = pick(g == 1, q.d[1], dsel);
      dsel = pick(g == 2, q.d[2], dsel);
      const int at = c - 4 * p;
#pragma unroll
      for (int a = 0; a < 4; ++a) rk = pick(at == a, q.inv[a], rk);
#pragma unroll
      for (int j = k; j < NB; ++j) {
        if constexpr (NB >= 6)
          if ((j - k) % 2 == 0) __builtin_amdgcn_sched_barrier(0);
        float u = panel_rows(q, t[tile_at<NB>(k, j)], p);
        if (j == k) u = at == g ? dsel : u;
        uk[j - k][p] = u;
      }
      if constexpr (RHS) {
        zk[p] = panel_rows(q, r, p);
        xl[16 * k + 4 * p + g] = zk[p];  // sixteen lanes the same word: cheaper than a branch
        if (B == 8 && p == 1) {
          r = r - block_sum<0, 2>(uk[0], zk);
        } else if (p < 3) {
          const float4v n = mfma16(-uk[0][p], zk[p], r);
#pragma unroll
          for (int v = 0; v < 4; ++v) r[v] = B == 8 && p == 0 && g != 1 ? r[v] : n[v];
        }
      }
      // the rows below, in this block: groups p + 1 .. (what lands in the finished groups is not read again)
      if (p < 3 && !(B == 8 && p == 1)) {
        const float minus = -uk[0][p];
#pragma unroll
        for (int j = k; j < NB; ++j) {
          const float4v n = mfma16(minus, uk[j - k][p], t[tile_at<NB>(k, j)]);
          if (B == 8 && p == 0) {  // the lower block's groups wait for the upper block's whole sum
#pragma unroll
            for (int v = 0; v < 4; ++v) t[tile_at<NB>(k, j)][v] = g == 1 ? n[v] : t[tile_at<NB>(k, j)][v];
          } else {
            t[tile_at<NB>(k, j)] = n;
          }
        }
      }
      if (B == 8 && p == 1) {
#pragma unroll
        for (int j = k; j < NB; ++j) t[tile_at<NB>(k, j)] = t[tile_at<NB>(k, j)] - block_sum<0, 2>(uk[0], uk[j - k]);
      }
    }
    // the block rows below lose this one's sums
#pragma unroll
    for (int i = k + 1; i < NB; ++i) {
      // (with many tiles the scheduler would start every one of these sums at once and spill)
      if constexpr (NB >= 6) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = i; j < NB; ++j) {
        float4v &m = t[tile_at<NB>(i, j)];
        if constexpr (B == 8) {
          m = m - block_sum<0, 2>(uk[i - k], uk[j - k]);
          m = m - block_sum<2, 4>(uk[i - k], uk[j - k]);
        } else {
          m = m - block_sum<0, 4>(uk[i - k], uk[j - k]);
        }
      }
    }
#pragma unroll
    for (int j = k; j < NB; ++j) t[tile_at<NB>(k, j)] = float4v{uk[j - k][0], uk[j - k][1], uk[j - k][2], uk[j - k][3]};
    rd[k] = rk;
    if constexpr (RHS) wave_sync();
  });
}

// z = U'^-1 rhs with a finished factor in panel layout: rhs(row) for the 16 NB rows, z into xl.
template <int NB, class Rhs>
__device__ __forceinline__ void forward_tiles(const float4v (&t)[kTiles<NB>], const float (&rd)[NB], Rhs &&rhs, float *xl, int nv, int lane) {
  const int g = lane >> 4, c = lane & 15;
  each<NB>([&](auto tile_row) __attribute__((always_inline)) {
    constexpr int i = tile_row;
    float4v r;
#pragma unroll
    for (int v = 0; v < 4; ++v) r[v] = rhs(16 * i + 4 * g + v);
    less_sums<i, 16>(r, xl, g, [&](auto above) __attribute__((always_inline)) { return t[tile_at<NB>(above, i)]; });
    const float4v dg = t[tile_at<NB>(i, i)];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      if (i == NB - 1 && p > 0 && 16 * i + 4 * p >= nv) {  // beyond the dofs
        if (c == 0) xl[16 * i + 4 * p + g] = 0.0f;
        continue;
      }
      auto u = [&](int a, int col) { return lane_value(dg[p], 16 * a + 4 * p + col); };
      Panel q;
      q.u01 = u(0, 1), q.u02 = u(0, 2), q.u03 = u(0, 3), q.u12 = u(1, 2), q.u13 = u(1, 3), q.u23 = u(2, 3);
#pragma unroll
      for (int a = 0; a < 4; ++a) q.inv[a] = lane_value(rd[i], 4 * p + a);
      const float z = panel_rows(q, r, p);
      if (p < 3) r = mfma16(-dg[p], z, r);
      if (c == 0) xl[16 * i + 4 * p + g] = z;
    }
    wave_sync();
  });
}

// U x = z: z in xl (16 NB words, zero at and past nv), x in its place.  tt: 16 x 17 words.
template <int NB, int B = 16>
__device__ __forceinline__ void backward_tiles(const float4v (&t)[kTiles<NB>], const float (&rd)[NB], float *xl, float *tt, int nv, int lane) {
  const int g = lane >> 4, c = lane & 15;
  float *put = tt + g * 17 + c;          // row 4 p + g: 68 p words on
  const float *take = tt + c * 17 + g;   // row c, column 4 q + g
  const float *last = tt + c * 17 + 3 - g;  // row c, column 4 p + 3 - g
  each<NB>([&](auto from_below) __attribute__((always_inline)) {
    constexpr int ib = NB - 1 - from_below;
    float4v r = *(const float4v *)(xl + 16 * ib + 4 * g);
    // (blocks of 8: the upper block loses the lower one's sum before these, so they are kept)
    float4v later[B == 8 ? 2 * NB : 1];
    const float4v z = r;
    each<NB - 1 - ib>([&](auto right) __attribute__((always_inline)) {
      constexpr int j = ib + 1 + right;
      const float4v u = t[tile_at<NB>(ib, j)];
#pragma unroll
      for (int p = 0; p < 4; ++p) put[68 * p] = u[p];
      wave_sync();
      float a[4], x[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) a[q] = take[4 * q], x[q] = xl[16 * j + 4 * q + g];
      if constexpr (B == 8) {
        later[2 * (j - ib - 1)] = block_sum<0, 2>(a, x), later[2 * (j - ib - 1) + 1] = block_sum<2, 4>(a, x);
        r = r - later[2 * (j - ib - 1)];
        r = r - later[2 * (j - ib - 1) + 1];
      } else {
        r = r - block_sum<0, 4>(a, x);
      }
      wave_sync();
    });
    const float4v dg = t[tile_at<NB>(ib, ib)];
#pragma unroll
    for (int p = 0; p < 4; ++p) put[68 * p] = dg[p];
    wave_sync();
    float ad[4], own[4];
#pragma unroll
    for (int p = 1; p < 4; ++p) ad[p] = -last[4 * p];
    if constexpr (B == 8) own[2] = take[8], own[3] = take[12];
#pragma unroll
    for (int p = 3; p >= 0; --p) {
      if (B == 8 && p == 1) {  // the upper block: less the lower one's sum, then the later blocks'
        float x[4];
        x[2] = xl[16 * ib + 8 + g], x[3] = xl[16 * ib + 12 + g];
        r = z - block_sum<2, 4>(own, x);
#pragma unroll
        for (int j = 0; j < 2 * (NB - 1 - ib); ++j) r = r - later[j];
      }
      if (ib == NB - 1 && p > 0 && 16 * ib + 4 * p >= nv) continue;
      auto u = [&](int a, int col) { return lane_value(dg[p], 16 * a + 4 * p + col); };
      auto inv = [&](int a) { return lane_value(rd[ib], 4 * p + a); };
      const float x3 = r[3] * inv(3);
      const float x2 = fma_(-u(2, 3), x3, r[2]) * inv(2);
      const float x1 = fma_(-u(1, 2), x2, fma_(-u(1, 3), x3, r[1])) * inv(1);
      const float x0 = fma_(-u(0, 1), x1, fma_(-u(0, 2), x2, fma_(-u(0, 3), x3, r[0]))) * inv(0);
      if (lane == 16 * p) *(float4v *)(xl + 16 * ib + 4 * p) = float4v{x0, x1, x2, x3};
      if (p > 0 && !(B == 8 && p == 2)) {  // the rows above in this block lose rows 4 p + 3 .. 4 p in that order
        const float b = p == 1 ? panel_gather<1>(x3, x2, x1, x0) : p == 2 ? panel_gather<2>(x3, x2, x1, x0) : panel_gather<3>(x3, x2, x1, x0);
        r = mfma16(ad[p], b, r);
      }
      if (B == 8) wave_sync();
    }
    wave_sync();
  });
}

// The sums over the changed rows of every pair of dofs, from zero in the list's order, as tiles; the dofs
// that some row touches into `hit` (bit c of hit[b]: dof 16 b + c).
template <int NB>
__device__ __forceinline__ void changed_pairs(float4v (&t)[kTiles<NB>], unsigned (&hit)[NB], const float *Jw, const float *Dw,
                                              const int32_t *sw, const int32_t *idw, int count, int quad, int nv, int lane) {
  const int g = lane >> 4, c = lane & 15;
#pragma unroll
  for (int m = 0; m < kTiles<NB>; ++m) t[m] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
  unsigned long long seen[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) seen[b] = 0ull;
  for (int base = 0; base < count; base += 64) {
    // the rows' numbers and signed weights, a row per lane; a step's four reach their lane groups by a shuffle
    const int n = count - base < 64 ? count - base : 64;
    const int rq = idw[base + (lane < n ? lane : n - 1)];
    const float dq = Dw[rq];
    const float sd = lane < n ? (sw[rq] == quad ? dq : -dq) : 0.0f;
    const int nstep = (n + 3) >> 2;
    float u[NB], un[NB], w, wn;
    auto fetch = [&](int q, float (&uu)[NB], float &ww) __attribute__((always_inline)) {
      const int from = 4 * q + g;
      const int r = __shfl(rq, from);
      ww = __shfl(sd, from);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int col = 16 * b + c;
        const float v = Jw[(size_t)r * nv + (b < NB - 1 || col < nv ? col : nv - 1)];
        uu[b] = from < n && (b < NB - 1 || col < nv) ? v : 0.0f;
      }
    };
    fetch(0, u, w);
    for (int q = 0; q < nstep; ++q) {
      if (q + 1 < nstep) fetch(q + 1, un, wn);
      float a[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        a[b] = w * u[b];
        seen[b] |= __ballot(u[b] != 0.0f);
      }
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = i; j < NB; ++j) t[tile_at<NB>(i, j)] = mfma16(a[i], u[j], t[tile_at<NB>(i, j)]);
      w = wn;
#pragma unroll
      for (int b = 0; b < NB; ++b) u[b] = un[b];
    }
  }
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const unsigned both = (unsigned)seen[b] | (unsigned)(seen[b] >> 32);
    hit[b] = (both | both >> 16) & 0xffffu;
  }
}

// Ascending list of the dofs in `hit` and their count (uni[nv]).
template <int NB>
__device__ __forceinline__ void write_union(int32_t *uni, const unsigned (&hit)[NB], int nv, int lane) {
  unsigned long long lo = hit[0] | (unsigned long long)hit[1] << 16 | (unsigned long long)hit[2] << 32;
  if constexpr (NB > 3) lo |= (unsigned long long)hit[3] << 48;
  if ((lo >> lane) & 1ull) uni[__popcll(lo & ((1ull << lane) - 1ull))] = lane;
  int total = __popcll(lo);
  if constexpr (NB > 4) {
    if (lane < 16 && ((hit[4] >> lane) & 1u)) uni[total + __popc(hit[4] & ((1u << lane) - 1u))] = 64 + lane;
    total += __popc(hit[4]);
  }
  if (lane == 0) uni[nv] = total;
}


// The stage for one world; `changes_raw`: the count of changed rows as the stage receives it (negative: factor
// H as it lies there; zero: solve with the stored factor).  READY: t holds H's upper tiles already.
template <int NB, bool READY>
__device__ __forceinline__ void dense_wave_world(float4v (&t)[kTiles<NB>], float *scr, float *Hw, float *Uw, const float *Jw,
                                                 const float *Dw, const float *gw, const int32_t *sw, const int32_t *idw,
                                                 int changes_raw, int ld_ids, int quad, int32_t *uni, float *search_w,
                                                 float *search_dot_w, float *decrement_w, int nv, int lane) {
  constexpr int PAD = 16 * NB;
  float *xl = scr, *tt = scr + PAD;
  const int g = lane >> 4, c = lane & 15;
  const bool refactor = READY || changes_raw != 0;
  const int count = changes_raw < 0 ? 0 : (changes_raw < ld_ids ? changes_raw : ld_ids);
  float rd[NB];
  if (refactor) {
    // H (with its update), the identity beyond the dofs, the gradient in the last column.  The gradient passes through
    // xl; H's tiles are asked for kAhead at a time ahead of the pairs and of one another, and what the update changed is stored
    // behind the last of them: a store under a condition between two tiles had every tile wait for its own trip to memory
    // (a stage of 29.2 -> 23.4 us in the slowest worlds at 70 dofs, the solve of 2048 of them 741 -> 711 us, of 8192 at 43
    // dofs 621 -> 605; 4 and 6 tiles ahead were no faster up to 48 dofs and beyond them took registers kept in memory).
#pragma unroll
    for (int i0 = 0; i0 < PAD; i0 += 64) {
      const int i = i0 + lane;
      if (i < PAD) xl[i] = gw[i < nv ? i : nv - 1];
    }
    auto beyond = [&](int row, int col, float e, float grad) __attribute__((always_inline)) {
      const bool in = col < nv && row < nv;
      return in ? e : (c == 15 && row < nv) ? grad : row == col ? 1.0f : 0.0f;
    };
    // element (16 i + first, c) of a matrix: what is beyond a tile row is in the instruction's own offset (as constants of
    // one base the rows' offsets took a pair of scalar registers each)
    auto row_at = [&](float *base, int first, int i) __attribute__((always_inline)) {
      unsigned at = 4u * (unsigned)(first * PAD + c);
      asm volatile("" : "+v"(at));
      return (char *)base + (at + 64u * PAD * i);
    };
    if constexpr (!READY) {
      constexpr int kAhead = 2;
      float4v h[kAhead];
      auto fetch = [&](auto tile_row, auto tile_col) __attribute__((always_inline)) {
        constexpr int i = tile_row, j = tile_col, at = tile_at<NB>(i, j) % kAhead;
#pragma unroll
        for (int v = 0; v < 4; ++v) h[at][v] = *(const float *)(row_at(Hw, 4 * g, i) + 4 * (v * PAD + 16 * j));
      };
      auto each_tile = [&](auto &&f) __attribute__((always_inline)) {
        each<NB>([&](auto i) __attribute__((always_inline)) {
          each<NB - i>([&](auto right) __attribute__((always_inline)) { f(i, std::integral_constant<int, i + right>{}); });
        });
      };
      each_tile([&](auto i, auto j) __attribute__((always_inline)) {
        if constexpr (tile_at<NB>(i, j) < kAhead) fetch(i, j);
      });
      unsigned hit[NB];
      changed_pairs<NB>(t, hit, Jw, Dw, sw, idw, count, quad, nv, lane);
      write_union<NB>(uni, hit, nv, lane);
      unsigned changed = 0u;  // tiles
      each_tile([&](auto tile_row, auto tile_col) __attribute__((always_inline)) {
        constexpr int i = tile_row, j = tile_col, m = tile_at<NB>(i, j);
        bool any = false;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float d = t[m][v], e = h[m % kAhead][v];
          any |= d != 0.0f;
          t[m][v] = d != 0.0f ? e + d : e;
        }
        changed |= (__ballot(any) != 0ull ? 1u : 0u) << m;
        // (the tile kAhead further on into its place)
        each_tile([&](auto i2, auto j2) __attribute__((always_inline)) {
          if constexpr (tile_at<NB>(i2, j2) == m + kAhead) fetch(i2, j2);
        });
      });
      each_tile([&](auto tile_row, auto tile_col) __attribute__((always_inline)) {
        constexpr int i = tile_row, j = tile_col, m = tile_at<NB>(i, j);
        if (!(changed >> m & 1u)) return;
        const int col = 16 * j + c;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = 16 * i + 4 * g + v;
          const bool in = j < NB - 1 || (col < nv && (i < NB - 1 || row < nv));
          if (in && (i < j || row <= col)) *(float *)(row_at(Hw, 4 * g, i) + 4 * (v * PAD + 16 * j)) = t[m][v];  // (elements without a change: as they are)
        }
      });
    } else if (lane == 0) {
      uni[nv] = 0;
    }
    wave_sync();
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      float4v &m = t[tile_at<NB>(i, NB - 1)];
      const float4v grad = *(const float4v *)(xl + 16 * i + 4 * g);
#pragma unroll
      for (int v = 0; v < 4; ++v) m[v] = beyond(16 * i + 4 * g + v, 16 * (NB - 1) + c, m[v], grad[v]);
    }
    wave_sync();
    factor_tiles<NB>(t, rd, true, xl, nv, lane);
    // the forward-solved gradient, and the corner of the augmented column: 1e30 less its squares in order,
    // which leaves 1e30 as it is unless one of them comes near half an ulp of it (3.7e22)
    bool large = false;
    if (c == 15) {
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const int row = 16 * i + 4 * p + g;
          const float z = row < nv ? t[tile_at<NB>(i, NB - 1)][p] : 0.0f;
          large = large || !(z * z < 1.0e22f);
          xl[row] = z;
        }
    }
    wave_sync();
    float corner = 1.0e30f;
    if (__builtin_expect(__any(large), 0))
      for (int i = 0; i < nv; ++i) corner = fma_(-xl[i], xl[i], corner);
    corner = sqrtf(corner);
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = i; j < NB; ++j) {
        const int col = 16 * j + c;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const int row = 16 * i + 4 * p + g;
          float v = t[tile_at<NB>(i, j)][p];
          if (i == j) v = row <= col ? v : 0.0f;
          if (j == NB - 1 && c == 15) v = row < nv ? v : row == PAD - 1 ? corner : 0.0f;
          *(float *)(row_at(Uw, g, i) + 4 * (4 * p * PAD + 16 * j)) = v;
        }
      }
  } else {
    // the stored factor, the identity in place of its augmented column; forward solve
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const float dgv = Uw[(size_t)(16 * i + c) * (PAD + 1)];
      rd[i] = i == NB - 1 && c == 15 ? 1.0f : 1.0f / dgv;
#pragma unroll
      for (int j = i; j < NB; ++j)
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const float v = Uw[(size_t)(16 * i + 4 * p + g) * PAD + 16 * j + c];
          t[tile_at<NB>(i, j)][p] = j == NB - 1 && c == 15 ? (i == j && 4 * p + g == 15 ? 1.0f : 0.0f) : v;
        }
    }
    forward_tiles<NB>(t, rd, [&](int row) { return row < nv ? gw[row < nv ? row : 0] : 0.0f; }, xl, nv, lane);
  }
  backward_tiles<NB>(t, rd, xl, tt, nv, lane);
  // search = -x, x . x and grad . x as 64 lanes striding the dofs sum them
  float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
  for (int i0 = 0; i0 < PAD; i0 += 64) {
    const int i = i0 + lane;
    const float x = i < nv ? xl[i < PAD ? i : 0] : 0.0f;
    if (i < nv) {
      search_w[i] = -x;
      s0 = fma_(x, x, s0);
      s1 = fma_(gw[i], x, s1);
    }
  }
  // the shuffle-down tree of 64 lanes: the halves, then as for 32 lanes (both sums at once, newton_search.h)
  float h0 = s0, h1 = s1;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\tv_permlane32_swap_b32 %2, %3\n\ts_nop 1" : "+v"(s0), "+v"(h0), "+v"(s1), "+v"(h1));
  s0 = s0 + h0, s1 = s1 + h1;
  search::swap_rows(s0, s1);
  const float s = search::row_sum(s0 + s1);
  const float dot = search::lane_of(s, 0), descent = search::lane_of(s, 16);
  if (lane == 0) {
    *search_dot_w = dot;
    *decrement_w = descent;
  }
}

}  // namespace
}  // namespace im
