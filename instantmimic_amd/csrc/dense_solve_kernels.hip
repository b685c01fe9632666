// Factor and solve of whole dense matrices on one wavefront per world, in the wavefront's matrix-core tiles
// (dense_wave.h): the blocked Cholesky of an indexed mass matrix (blocks of 8 or 16) and H = M + J'DJ with
// the same factor and solve behind it.
// Reference: src/instantmimic/utils/mjw_kernels/indexed_factor.py:15-215, mjw_step_optimized.py:893-993;
// the assembly at newton_fusion.py:470.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.h"
#include "dense_solve.h"
#include "dense_wave.h"
#include "jtdj_wave.h"

namespace im {
namespace {

// An index of which the compiler does not know that a test later on goes with it (it would make branches of the loads)
__device__ __forceinline__ int opaque(int i) {
  asm("" : "+v"(i));
  return i;
}

// n words as a buffer: a load at or past its end gives zero, a store there is dropped
__device__ __forceinline__ __amdgpu_buffer_rsrc_t words_of(const void *p, int n) {
  return __builtin_amdgcn_make_buffer_rsrc((void *)p, (short)0, 4 * n, 0x00020000);
}
// the word `lane_bytes` + `bytes` from the buffer's start, the second the same for the whole wavefront
__device__ __forceinline__ unsigned load_word(__amdgpu_buffer_rsrc_t words, int lane_bytes, int bytes) {
  return __builtin_amdgcn_raw_buffer_load_b32(words, lane_bytes, bytes, 0);
}

// A world's right-hand side, a word or two a lane, zero where there is none; asked for ahead of the matrix, whose
// words would otherwise be waited for first.
template <int NB>
constexpr int kRhs = (16 * NB + 63) / 64;
template <int NB>
__device__ __forceinline__ void load_rhs(float (&to)[kRhs<NB>], const float *yw, int nv, int lane) {
#pragma unroll
  for (int k = 0; k < kRhs<NB>; ++k) to[k] = yw && lane + 64 * k < nv ? yw[lane + 64 * k] : 0.0f;
}

// The factor, its store (rows and columns below `pad`, the tiles on and right of the block diagonal) and the
// solution, which both kernels end with.  The tiles hold the matrix and the identity beyond
// the dofs.  The right-hand side takes a spare last column
// where there is one (nv < 16 NB: SPARE), and is forward-solved with the factor in either case.
template <int NB, int B, bool SPARE>
__device__ __forceinline__ void factor_solve_store(float4v (&t)[kTiles<NB>], float *xl, float *tt, const float (&y)[kRhs<NB>],
                                                   float *xw, float *Uw, int nv, int pad, int lane) {
  const int g = lane >> 4, c = lane & 15;
  float rd[NB];
#pragma unroll
  for (int k = 0; k < kRhs<NB>; ++k)
    if (lane + 64 * k < 16 * NB) xl[lane + 64 * k] = y[k];
  wave_sync();
  if constexpr (SPARE) {
    if (c == 15) {
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const float4v r = *(const float4v *)(xl + 16 * i + 4 * g);
        if (i < NB - 1 || g < 3) t[tile_at<NB>(i, NB - 1)] = r;
        else t[tile_at<NB>(i, NB - 1)] = float4v{r[0], r[1], r[2], 1.0f};
      }
    }
    factor_tiles<NB, B>(t, rd, true, xl, nv, lane);
  } else {
    factor_tiles<NB, B, true>(t, rd, false, xl, nv, lane);
  }
  if constexpr (SPARE) {
    if (c == 15) {
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const int row = 16 * i + 4 * p + g;
          float4v &m = t[tile_at<NB>(i, NB - 1)];
          xl[row] = row < nv ? m[p] : 0.0f;
          m[p] = row == 16 * NB - 1 ? 1.0f : 0.0f;
        }
    }
    wave_sync();
  }
  if (Uw) {
    const __amdgpu_buffer_rsrc_t words = words_of(Uw, pad * pad);
    const int at = 4 * (g * pad + c);
    auto tile = [&](int i, int j, int rows) __attribute__((always_inline)) {
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        if (4 * p >= rows) break;
        const float v = t[tile_at<NB>(i, j)][p];
        // (blocks of 8: a diagonal tile's lower left block lies below the block diagonal)
        if (!(B == 8 && i == j && p > 1) || c >= 8)
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, i == j && 4 * p + g > c ? 0.0f : v), words, at, 4 * ((16 * i + 4 * p) * pad + 16 * j), 0);
      }
    };
    each<NB>([&](auto tile_row) __attribute__((always_inline)) {
      constexpr int i = tile_row;
      each<NB - 1 - i>([&](auto right) __attribute__((always_inline)) {
        constexpr int j = NB - 2 - right;  // the full columns
        tile(i, j, 16);
      });
    });
    const int edge = pad - 16 * (NB - 1);  // 16, or 8 with blocks of 8
    if (B == 16 || c < edge)
      each<NB>([&](auto tile_row) __attribute__((always_inline)) {
        constexpr int i = tile_row;
        tile(i, NB - 1, B == 8 && i == NB - 1 ? edge : 16);
      });
  }
  if (!xw) return;
  backward_tiles<NB, B>(t, rd, xl, tt, nv, lane);
  for (int i = lane; i < nv; i += 64) xw[i] = xl[i];
}

// The blocked factor and solve, a wavefront per world: the matrix cores do the sums, the vector unit the pivots and
// the panels' rows, about a third of the instructions each chain on the one before, and up to eight wavefronts per
// SIMD fill the gaps.  Before, a workgroup had a world (nv 48 .. 128, in LDS, at its barriers most of the time) or a
// wavefront four (below, with B = 8 up to 40, in LDS): 8192 worlds of 35 / 64 dofs took 39.5 / 159 us with B = 8 and
// 78 / 129 us with B = 16, 2048 of 128 dofs 225 and 127; here 37.7 / 77, 36.8 / 71, 107 and 92.  500 worlds of 35 dofs, one
// wavefront each instead of a quarter: 24.3 -> 9.4 us.
// The matrix, the table and the factor go through buffer descriptors: what lies past a world's words reads as zero without a
// test, and a tile's place is a scalar, so that an element takes its two loads and three vector instructions where it took
// twelve, and a store none beside its value.  The right-hand side, which the first panel needs, is asked for ahead of the
// matrix.  B = 8 / B = 16, before and after: 35 dofs x 100 worlds 9.15 / 8.72 -> 8.88 / 8.62 us, x 8192 38.0 / 36.6 -> 36.0 / 34.2;
// 64 x 1000 16.7 / 15.8 -> 15.9 / 15.0; 101 x 8192 233 / 220 -> 204 / 172 (registers that addresses held); 128 x 8192
// 328 / 293 -> 281 / 256.  Priorities by a workgroup's place in the grid made no difference.
// Element (r, c) of tile (i, j) is M[block_idx[tile][r][c]], zero at or past nM, with 1 on the padded diagonal;
// of a diagonal block the lower triangle counts, as in the workgroup-per-world kernel.
template <int NB, int B, bool SPARE>
__global__ __launch_bounds__(256, NB <= 4 ? 4 : NB <= 6 ? 3 : 2) void blocked_solve_wave_kernel(
    const float *__restrict__ M, int64_t ldM, int nM, const int32_t *__restrict__ block_idx, const float *__restrict__ y, int64_t ldy,
    float *__restrict__ U, float *__restrict__ x, int64_t ldx, int nv, int pad, int nworld, const int32_t *__restrict__ active) {
  __shared__ __align__(16) float lds[4 * wave_stage_words<NB>()];
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t w = (int64_t)blockIdx.x * 4 + wv;
  if (w >= nworld || (active && active[w] == 0)) return;
  float *xl = lds + wv * wave_stage_words<NB>(), *tt = xl + 16 * NB;
  const bool solve = y && x;
  float rhs[kRhs<NB>];
  load_rhs<NB>(rhs, solve ? y + w * ldy : nullptr, nv, lane);
  const int nblk = pad / B, edge = pad - 16 * (NB - 1);
  const __amdgpu_buffer_rsrc_t Mw = words_of(M + w * ldM, nM), table = words_of(block_idx, pad * pad);
  // the lane's first element in the table, and where a diagonal block's upper triangle is found below it, in bytes; with blocks
  // of 8 the last tile row and column may hold one block, whose place the lanes beyond it read instead
  const int brow = 4 * g / B, bcol = c / B, here = 4 * (brow * nblk + bcol) * B * B;
  const int at = here + 4 * ((4 * g % B) * B + c % B), across = here + 4 * ((c % B) * B + 4 * g % B);
  const bool in_last = B == 16 || c < edge, in_corner = B == 16 || (c < edge && 4 * g < edge);
  const int back = in_last ? 0 : 4 * bcol * B * B, corner_back = in_corner ? 0 : 4 * ((4 * g < edge ? 0 : brow * nblk) + (in_last ? 0 : bcol)) * B * B;
  int upper[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) upper[v] = brow == bcol && 4 * g + v < c ? across + 4 * v : at + 4 * v * B;
  float4v t[kTiles<NB>];
  unsigned idx[kTiles<NB>][4];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = i; j < NB; ++j) {
      const int tile = 4 * (16 / B) * B * B * (i * nblk + j);
      const int less = j < NB - 1 ? 0 : i < NB - 1 ? back : corner_back;
#pragma unroll
      for (int v = 0; v < 4; ++v) idx[tile_at<NB>(i, j)][v] = load_word(table, (i == j ? upper[v] : at + 4 * v * B) - less, tile);
    }
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = i; j < NB; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        unsigned e = idx[tile_at<NB>(i, j)][v];
        e = e < (unsigned)nM ? e : (unsigned)nM;
        if (B == 8 && j == NB - 1) e = (i == NB - 1 ? in_corner : in_last) ? e : (unsigned)nM;
        float m = __builtin_bit_cast(float, load_word(Mw, (int)(4 * e), 0));
        if (i == NB - 1) m += 4 * g + v == c && 16 * i + c >= nv ? 1.0f : 0.0f;
        t[tile_at<NB>(i, j)][v] = m;
      }
  factor_solve_store<NB, B, SPARE>(t, xl, tt, rhs, solve ? x + w * ldx : nullptr, U ? U + w * (int64_t)pad * pad : nullptr, nv,
                                   pad, lane);
}

// H's upper tiles into both triangles (a diagonal tile's upper half counts); ld a multiple of four and Hw on 16
// bytes.  Rows below the last block row go out without a test.
template <int NB>
__device__ __forceinline__ void store_upper_tiles(float *Hw, const float4v (&t)[kTiles<NB>], int nv, int ld, int lane) {
  const int g = lane >> 4, c = lane & 15;
  float *up = Hw + 4 * g * ld + c, *low = Hw + c * ld + 4 * g;
  each<NB>([&](auto tile_col) __attribute__((always_inline)) {
    constexpr int j = tile_col;
    if (j < NB - 1 || 16 * j + c < nv)
      each<j>([&](auto above) __attribute__((always_inline)) {
        constexpr int i = above;
        const float4v &h = t[tile_at<NB>(i, j)];
#pragma unroll
        for (int v = 0; v < 4; ++v) up[(16 * i + v) * ld + 16 * j] = h[v];
        *(float4v *)(low + 16 * j * ld + 16 * i) = h;
      });
  });
#pragma unroll
  for (int v = 0; v < 4; ++v)
    if (4 * g + v <= c) {
#pragma unroll
      for (int i = 0; i < NB; ++i)
        if (i < NB - 1 || 16 * i + c < nv) {
          const float h = t[tile_at<NB>(i, i)][v];
          up[(16 * i + v) * ld + 16 * i] = h;
          low[16 * i * ld + 16 * i + v] = h;
        }
    }
}

// H = M + J' D_act J (dense M) and its factor and solve, a wavefront per world: no barrier, no staging, the matrix in
// registers from the first product to the solution.  Two wavefronts per SIMD at 128 dofs, where the bound is
// the memory traffic (233 KB per world, 3.6 TB/s of the 4.85 that a copy reaches; a workgroup per world, with rows
// and factor in LDS: 2.9), eight at 16.  16384 worlds of 128 dofs, 256 rows: 1312 -> 1050 us; 4096 worlds with 96 rows: 33 dofs
// 140 -> 38 us, 64: 182 -> 80, 112: 345 -> 198; 8192 of 9: 147 -> 18.  The rows that contribute are listed first (their numbers and weights in LDS, ascending: a row with weight zero leaves every chain
// as it is), then every element of theirs is read once, straight into the operand registers, two steps of four
// rows ahead of the products.
template <int NB, bool SPARE>
__global__ __launch_bounds__(256, NB <= 4 ? 4 : NB <= 6 ? 3 : 2) void jtdj_solve_wave_kernel(
    const float *__restrict__ Mdense, const float *__restrict__ J, int njmax, const float *__restrict__ D,
    const int32_t *__restrict__ state, const int32_t *__restrict__ nefc_p, int quad, float *__restrict__ H, int nv, int nv_pad,
    const float *__restrict__ y, int64_t ldy, float *__restrict__ U, float *__restrict__ x, int64_t ldx, int pad, int nworld) {
  extern __shared__ __align__(16) float lds[];
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t w = (int64_t)blockIdx.x * (blockDim.x >> 6) + wv;
  if (w >= nworld) return;
  const int list_words = (njmax + 3 + 16) & ~3;  // (three rows' room behind the last for a step's remainder)
  float *xl = lds + (size_t)wv * (wave_stage_words<NB>() + 2 * list_words), *tt = xl + 16 * NB;
  float *lw = xl + wave_stage_words<NB>();
  int *lr = (int *)(lw + list_words);
  const float *Mw = Mdense + w * (int64_t)nv * nv, *Jw = J + w * (int64_t)njmax * nv, *Dw = D + w * (int64_t)njmax;
  const int32_t *sw = state + w * (int64_t)njmax;
  int nefc = nefc_p ? nefc_p[w] : njmax;
  nefc = __builtin_amdgcn_readfirstlane(nefc < njmax ? nefc : njmax);
  const bool solve = y && x;
  float rhs[kRhs<NB>];
  load_rhs<NB>(rhs, solve ? y + w * ldy : nullptr, nv, lane);
  float4v t[kTiles<NB>];
  // M first: its trips to memory pass under the listing
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = i; j < NB; ++j) {
      const float *Mt = Mw + (16 * i) * nv + 16 * j;
      const bool in = j < NB - 1 || c < nv - 16 * (NB - 1);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const bool here = in && (i < NB - 1 || 4 * g + v < nv - 16 * (NB - 1));
        const float m = Mt[opaque(here ? (4 * g + v) * nv + c : 0)];
        t[tile_at<NB>(i, j)][v] = here ? m : 0.0f;
      }
    }
  int cnt = 0;
  for (int base = 0; base < nefc; base += 64) {
    const int r = base + lane, rc = r < nefc ? r : nefc - 1;
    const float d = Dw[rc];
    const bool on = r < nefc && sw[rc] == quad;
    const unsigned long long m = __ballot(on);
    if (on) {
      const int at = cnt + __popcll(m & ((1ull << lane) - 1ull));
      lw[at] = d;
      lr[at] = r * nv;
    }
    cnt += __popcll(m);
  }
  wave_sync();
  if (lane < 16) {  // what a step's remainder reads: the last row again, with a weight of zero
    const int r = cnt > 0 ? lr[cnt - 1] : 0;
    lw[cnt + lane] = 0.0f;
    lr[cnt + lane] = r;
  }
  wave_sync();
  const int nstep = (cnt + 3) >> 2, tail = nv - 16 * (NB - 1);
  const bool in_last = c < tail;
  const int c_last = in_last ? c : tail - 1;
  float u0[NB], u1[NB], w0 = 0.0f, w1 = 0.0f;
  auto fetch = [&](int q, float (&uu)[NB], float &ww) __attribute__((always_inline)) {
    const float *at = Jw + lr[4 * q + g];
    ww = lw[4 * q + g];
#pragma unroll
    for (int b = 0; b < NB - 1; ++b) uu[b] = at[16 * b + c];
    uu[NB - 1] = at[16 * (NB - 1) + c_last];
  };
  auto product = [&](float (&uu)[NB], float ww) __attribute__((always_inline)) {
    float a[NB];
    uu[NB - 1] = in_last ? uu[NB - 1] : 0.0f;
#pragma unroll
    for (int b = 0; b < NB; ++b) a[b] = ww * uu[b];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = i; j < NB; ++j) t[tile_at<NB>(i, j)] = mfma16(a[i], uu[j], t[tile_at<NB>(i, j)]);
  };
  // (steps at and past the last change nothing)
  if (nstep > 0) {
    fetch(0, u0, w0);
    fetch(1, u1, w1);
    for (int q = 0; q < nstep; q += 2) {
      product(u0, w0);
      if (q + 2 < nstep) fetch(q + 2, u0, w0);
      product(u1, w1);
      if (q + 2 < nstep) fetch(q + 3, u1, w1);
    }
  }
  if (H) {
    float *Hw = H + w * (int64_t)nv_pad * nv_pad;
    if ((nv_pad & 3) == 0 && ((uintptr_t)H & 15) == 0) {
      store_upper_tiles<NB>(Hw, t, nv, nv_pad, lane);
    } else {
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = i; j < NB; ++j) store_h_mirrored(Hw, nv, nv_pad, false, 16 * i + 4 * g, 16 * j + c, t[tile_at<NB>(i, j)], i != j);
    }
  }
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) {  // the identity beyond the dofs
      const bool out = c >= tail || (i == NB - 1 && 4 * g + v >= tail);
      if (out) t[tile_at<NB>(i, NB - 1)][v] = i == NB - 1 && 4 * g + v == c ? 1.0f : 0.0f;
    }
  factor_solve_store<NB, 16, SPARE>(t, xl, tt, rhs, solve ? x + w * ldx : nullptr, U ? U + w * (int64_t)pad * pad : nullptr, nv,
                                    pad, lane);
}

template <int NB, int B>
int launch_blocked(const float *M, int64_t ldM, int nM, const int32_t *block_idx, int nv, int pad, const float *y, int64_t ldy,
                   float *U, float *x, int64_t ldx, const int32_t *active, int nworld, hipStream_t stream) {
  auto fn = nv < 16 * NB ? blocked_solve_wave_kernel<NB, B, true> : blocked_solve_wave_kernel<NB, B, false>;
  hipLaunchKernelGGL(fn, dim3((unsigned)((nworld + 3) / 4)), dim3(256), 0, stream, M, ldM, nM, block_idx, y,
                     ldy, U, x, ldx, nv, pad, nworld, active);
  IM_HIP_CHECK(hipGetLastError());
  return IM_OK;
}

}  // namespace

int blocked_solve_wave(const float *M, int64_t ldM, int nM, const int32_t *block_idx, int block_size, int nv, int pad, const float *y,
                       int64_t ldy, float *U, float *x, int64_t ldx, const int32_t *active, int nworld, hipStream_t stream) {
#define IM_BLOCKED_CASE(NB)                                                                                                     \
  if (nv <= 16 * NB)                                                                                                            \
    return block_size == 8                                                                                                      \
               ? launch_blocked<NB, 8>(M, ldM, nM, block_idx, nv, pad, y, ldy, U, x, ldx, active, nworld, stream)               \
               : launch_blocked<NB, 16>(M, ldM, nM, block_idx, nv, pad, y, ldy, U, x, ldx, active, nworld, stream);
  IM_BLOCKED_CASE(1) IM_BLOCKED_CASE(2) IM_BLOCKED_CASE(3) IM_BLOCKED_CASE(4) IM_BLOCKED_CASE(5) IM_BLOCKED_CASE(6) IM_BLOCKED_CASE(7) IM_BLOCKED_CASE(8)
#undef IM_BLOCKED_CASE
  return IM_ERR_UNSUPPORTED;
}

int jtdj_solve_wave(const float *Mdense, const float *J, int njmax, const float *D, const int32_t *state, const int32_t *nefc, int quad,
                    float *H, int nv, int nv_pad, const float *y, int64_t ldy, float *U, int pad, float *x, int64_t ldx, int nworld,
                    hipStream_t stream) {
  const int list_words = 2 * ((njmax + 3 + 16) & ~3);
#define IM_JTDJ_CASE(NB)                                                                                                        \
  if (nv <= 16 * NB) {                                                                                                          \
    const size_t world = 4 * ((size_t)wave_stage_words<NB>() + list_words);                                                     \
    const int waves = 4 * world <= 160 * 1024 ? 4 : 1;  /* a list too long for four worlds' workgroups */                       \
    const size_t lds = waves * world;                                                                                           \
    if (lds > 160 * 1024) return IM_ERR_UNSUPPORTED;                                                                            \
    auto fn = nv < 16 * NB ? jtdj_solve_wave_kernel<NB, true> : jtdj_solve_wave_kernel<NB, false>;                              \
    if (lds > 64 * 1024) IM_HIP_CHECK(hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)); \
    hipLaunchKernelGGL(fn, dim3((unsigned)((nworld + waves - 1) / waves)), dim3(64 * waves), lds, stream, Mdense, J, njmax, D, state, \
                       nefc, quad, H, nv, nv_pad, y, ldy, U, x, ldx, pad, nworld);                                              \
    IM_HIP_CHECK(hipGetLastError());                                                                                            \
    return IM_OK;                                                                                                               \
  }
  IM_JTDJ_CASE(1) IM_JTDJ_CASE(2) IM_JTDJ_CASE(3) IM_JTDJ_CASE(4) IM_JTDJ_CASE(5) IM_JTDJ_CASE(6) IM_JTDJ_CASE(7) IM_JTDJ_CASE(8)
#undef IM_JTDJ_CASE
  return IM_ERR_UNSUPPORTED;
}

}  // namespace im
