// The kernels of the dense Newton stage above 32 dofs on one wavefront per world (dense_wave.h), for
// nv_pad = 48, 64 or 80 with its last block row in use: the stage as a launch of its own, the first Hessian with its
// factor, and the resident Newton loop.
// Reference: src/instantmimic/utils/mjw_kernels/newton_stages.py:473-742, newton_fusion.py:57-298, :470.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "common.h"
#include "dense_wave.h"
#include "jtdj_wave.h"
#include "newton_solve.h"
#include "newton_wave.h"

namespace im {
namespace {

// A wavefront per world, four worlds per workgroup.
template <int NB>
__global__ __launch_bounds__(256, NB == 5 ? 3 : 4) void dense_update_wave_kernel(
    const uint8_t *__restrict__ done, const int32_t *__restrict__ state_changes, const int32_t *__restrict__ changes,
    const int32_t *__restrict__ ids, int ld_ids, const float *__restrict__ J, int njmax, const float *__restrict__ D,
    const int32_t *__restrict__ state, int quad, const float *__restrict__ grad, int64_t ldg, float *H_, float *U_,
    int32_t *__restrict__ uni_, float *__restrict__ search, int64_t ld_search, float *__restrict__ search_dot,
    float *__restrict__ decrement, int nv, int nworld) {
  extern __shared__ float lds[];
  constexpr int PAD = 16 * NB;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t w = (int64_t)blockIdx.x * 4 + wv;
  if (w >= nworld) return;
  if ((done && done[w]) || state_changes[w] == 0) return;
  float4v t[kTiles<NB>];
  dense_wave_world<NB, false>(t, lds + wv * wave_stage_words<NB>(), H_ + w * (int64_t)PAD * PAD, U_ + w * (int64_t)PAD * PAD,
                              J + w * (int64_t)njmax * nv, D + w * njmax, grad + w * ldg, state + w * njmax, ids + w * ld_ids,
                              changes[w], ld_ids, quad, uni_ + w * (nv + 1), search + w * ld_search, search_dot + w,
                              decrement + w, nv, lane);
}

// H = M + J' D_act J of one world, as jtdj_wave (jtdj_wave.h) forms it, over the rows that contribute: their numbers
// are listed in LDS (ascending, by ballot, kListedRows rows of J at a time) while nothing else uses the area, and only
// they are read.  A row with weight zero leaves every chain as it is, but costs its trip to memory: with two wavefronts
// per SIMD (2048 worlds) the launch is a chain of such trips, a fetch of STEPS steps of four rows each.
// Whole solves, all rows read (and at 80 columns two steps in flight) -> now: 70 dofs x 2048 with 192 rows 873 -> 840 us, 56 x
// 4096 with 128 rows 705 -> 691, 35 x 8192 with 96 rows 694 -> 676, 62 x 2000 521 -> 511.
constexpr int kListedRows = 256;

template <int NB, int STEPS>
__device__ __forceinline__ void jtdj_listed(const float *__restrict__ Mw, const int32_t *__restrict__ elemid,
                                            const float *__restrict__ Jw, const float *__restrict__ Dw,
                                            const int32_t *__restrict__ sw, int nefc, int quad, int nv,
                                            float *__restrict__ Hw, int *list, int lane, float4v (&acc)[kTiles<NB>]) {
  static_assert(kListedRows <= wave_stage_words<NB>(), "the list lies in the stage's area");
  const int c = lane & 15, kq = lane >> 4;
  float u[STEPS][NB], dk[STEPS], un[STEPS][NB], dn[STEPS];
  int cnt = 0;
  auto list_rows = [&](int r0) __attribute__((always_inline)) {
    const int end = nefc - r0 < kListedRows ? nefc : r0 + kListedRows;
    cnt = 0;
    for (int base = r0; base < end; base += 64) {
      const int r = base + lane;
      const bool on = r < end && sw[r < end ? r : end - 1] == quad;
      const unsigned long long m = __ballot(on);
      if (on) list[cnt + __popcll(m & ((1ull << lane) - 1ull))] = r;
      cnt += __popcll(m);
    }
    wave_sync();
  };
  // the operands of STEPS steps (four rows each): asked for a group ahead of the products that use them
  auto fetch = [&](int q0, float (&uu)[STEPS][NB], float (&dd)[STEPS]) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const int at = 4 * (q0 + s) + kq;
      const bool in = at < cnt;
      const int row = list[in ? at : cnt - 1];
      const float dv = Dw[row];
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int col = 16 * b + c;
        const float jv = Jw[(int64_t)row * nv + (col < nv ? col : nv - 1)];
        uu[s][b] = (in && col < nv) ? jv : 0.0f;
      }
      dd[s] = in ? dv : 0.0f;
    }
  };
  if (nefc > 0) list_rows(0);
  if (cnt > 0) fetch(0, u, dk);  // on their way while M is gathered
  int m = 0;
  // the accumulators start from M (a lane holds column j = l % 16 and rows 4 (l / 16) + v of a tile)
#pragma unroll
  for (int bi = 0; bi < NB; ++bi)
#pragma unroll
    for (int bj = bi; bj < NB; ++bj, ++m) {
      const int j = 16 * bj + c, jc = j < nv ? j : nv - 1;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = 16 * bi + 4 * kq + v, ic = i < nv ? i : nv - 1;
        const int id = elemid[ic * nv + jc];
        const float mv = Mw[id < 0 ? 0 : id];
        acc[m][v] = (i < nv && j < nv && id >= 0) ? mv : 0.0f;
      }
    }
  for (int r0 = 0; r0 < nefc;) {
    const int nstep = (cnt + 3) >> 2;
    for (int q0 = 0; q0 < nstep; q0 += STEPS) {
      if (q0 + STEPS < nstep) fetch(q0 + STEPS, un, dn);
#pragma unroll
      for (int s = 0; s < STEPS; ++s) {
        float wt[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) wt[b] = u[s][b] * dk[s];
        int t = 0;
#pragma unroll
        for (int bi = 0; bi < NB; ++bi)
#pragma unroll
          for (int bj = bi; bj < NB; ++bj, ++t)
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wt[bi], u[s][bj], acc[t], 0, 0, 0);
      }
#pragma unroll
      for (int s = 0; s < STEPS; ++s) {
        dk[s] = dn[s];
#pragma unroll
        for (int b = 0; b < NB; ++b) u[s][b] = un[s][b];
      }
    }
    r0 += kListedRows;
    if (r0 < nefc) {
      wave_sync();
      list_rows(r0);
      if (cnt > 0) fetch(0, u, dk);
    }
  }
  wave_sync();  // the stage takes the list's area
  m = 0;
#pragma unroll
  for (int bi = 0; bi < NB; ++bi)
#pragma unroll
    for (int bj = bi; bj < NB; ++bj, ++m)
      store_h_mirrored(Hw, nv, 16 * NB, true, 16 * bi + 4 * kq, 16 * bj + c, acc[m], bi != bj);
}

// The first Hessian and its factor in one launch: H = M + J' D_act J of every world on the matrix
// cores of its wavefront (jtdj_listed), stored, and for the worlds that are not done factored where it lies: in
// the accumulators.
// STEPS 2 (with 80 columns): four wavefronts per SIMD of 128 registers, where four steps take 162 and leave three.  The
// batches that three hold gain nothing by it and have fewer loads on their way; beyond, a fourth spares them a second turn
// on the chip.  70 dofs with 157 rows, four steps / two, us: x 300 47.7 / 48.5, x 1024 54.1 / 56.7, x 2048 71.8 / 73.4, x
// 3072 86.7 / 87.0, x 4096 139.4 / 107.4, x 6144 185.2 / 183.6, x 8192 266.6 / 235.4 (all rows read, two steps, x 4096:
// 132.7).
template <int NB, int STEPS>
__global__ __launch_bounds__(256, NB == 3 ? 3 : STEPS == 2 ? 4 : 2) void dense_init_wave_kernel(
    const uint8_t *__restrict__ done, const int32_t *__restrict__ nefc_p, const float *__restrict__ J, int njmax,
    const float *__restrict__ D, const int32_t *__restrict__ state, int quad, const float *__restrict__ M, int64_t ldM,
    const int32_t *__restrict__ elemid, const float *__restrict__ grad, int64_t ldg, float *H_, float *U_,
    int32_t *__restrict__ uni_, float *__restrict__ search, int64_t ld_search, float *__restrict__ search_dot,
    float *__restrict__ decrement, int nv, int nworld) {
  extern __shared__ float lds[];
  constexpr int PAD = 16 * NB;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t w = (int64_t)blockIdx.x * 4 + wv;
  if (w >= nworld) return;
  int nefc = nefc_p ? nefc_p[w] : njmax;
  nefc = nefc < njmax ? nefc : njmax;
  float *Hw = H_ + w * (int64_t)PAD * PAD;
  const float *Jw = J + w * (int64_t)njmax * nv;
  float4v t[kTiles<NB>];
  nefc = __builtin_amdgcn_readfirstlane(nefc);
  float *area = lds + wv * wave_stage_words<NB>();
  jtdj_listed<NB, STEPS>(M + w * ldM, elemid, Jw, D + w * njmax, state + w * njmax, nefc, quad, nv, Hw, (int *)area, lane, t);
  if (done && done[w]) return;
  dense_wave_world<NB, true>(t, area, Hw, U_ + w * (int64_t)PAD * PAD, Jw, D + w * njmax,
                             grad + w * ldg, state + w * njmax, nullptr, -1, 0, quad, uni_ + w * (nv + 1),
                             search + w * ld_search, search_dot + w, decrement + w, nv, lane);
}

// The resident Newton loop (newton_wave.h) with this stage: a wavefront per world from the first
// line search to convergence, WAVES worlds per workgroup.  Per wavefront in LDS: what the loop
// keeps from round to round and one area that the staged tile of J, the gradient's row list and
// the stage use one after the other.
template <int NB>
__host__ __device__ inline int wave_resident_area_words(int nv, int njmax) {
  int words = wave_stage_words<NB>();
  const int tile = 64 * 17, grad = 2 * njmax + nv;
  words = words > tile ? words : tile;
  words = words > grad ? words : grad;
  return (words + 3) & ~3;
}
__host__ __device__ inline int wave_resident_shared_words(int nterm, int nv) { return (nterm + nv + 1 + 3) & ~3; }

template <int NB, int WAVES, int HELD>
__global__ __launch_bounds__(64 * WAVES, NB == 5 ? 3 : 4) void newton_dense_wave_resident_kernel(
    resident::NewtonArgs a, float *__restrict__ H_, float *__restrict__ U_, int32_t *__restrict__ uni_,
    int *__restrict__ next_world) {
  extern __shared__ float lds[];
  constexpr int PAD = 16 * NB;
  const int tid = threadIdx.x;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nv = a.nv, njmax = a.njmax, nworld = a.nworld;
  uint32_t *term = (uint32_t *)lds;
  int *radr = (int *)(term + a.nterm);
  const int area = wave_resident_area_words<NB>(nv, njmax);
  float *mine = lds + wave_resident_shared_words(a.nterm, nv) + wv * (area + resident::kept_words(nv, njmax, 0));
  resident::LoopLds L;
  L.votes = nullptr;
  L.worlds = nullptr;
  L.term = term, L.radr = radr;
  L.rows = mine;  // the shared area: M's row, the tile of J, then the gradient's lists, then the stage
  L.f = mine;
  L.rowl = (int *)(mine + njmax);
  L.gl = mine + 2 * njmax;
  L.m_lds = nullptr;  // M is read from memory by the round's one product with it
  L.sv = mine + area;
  L.Ma = L.sv + nv;
  L.mv = L.Ma + nv;
  L.qacc = L.mv + nv;
  L.Jaref = L.qacc + nv;
  L.jv = L.Jaref + njmax;
  L.D = L.jv + njmax;
  L.fl = L.D + njmax;
  for (int k = tid; k < a.nterm; k += 64 * WAVES) term[k] = (uint32_t)a.mulm_col[k] | (uint32_t)a.mulm_madr[k] << 16;
  for (int k = tid; k <= nv; k += 64 * WAVES) radr[k] = a.mulm_rowadr[k];
  __syncthreads();  // the only workgroup barrier
  int64_t w = resident::first_world(a, wv);
  auto stage = [&]() __attribute__((always_inline)) {
    const resident::NewtonArgs &b = resident::kernel_args(0);  // the kernel's first parameter
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));  // (nothing formed from it is kept in registers from round to round)
    float4v t[kTiles<NB>];
    dense_wave_world<NB, false>(t, mine, H_ + w * (int64_t)PAD * PAD, U_ + w * (int64_t)PAD * PAD, b.J + w * (int64_t)b.njmax * b.nv,
                                b.D + w * b.njmax, b.grad + w * b.ld_grad, b.state + w * b.njmax, b.ids + w * (int64_t)b.ld_ids,
                                b.quad_count[w], b.ld_ids, b.quad, uni_ + w * (b.nv + 1), b.search + w * b.nv, b.search_dot + w,
                                b.decrement + w, b.nv, lane);
  };
  // as many wavefronts as the chip keeps resident; one whose world is done takes the next world
  // nobody has started (a counter in memory that only grows: every wavefront reaches the end)
  while (w < nworld) {
    if (NB == 5) {
      const resident::NewtonArgs &b = resident::kernel_args(0);
      resident::row_priority(__builtin_amdgcn_readfirstlane(b.nefc ? b.nefc[w] : b.njmax), b.njmax);
    }
    resident::newton_loop<HELD, NB == 5 ? 2 : 1, NB != 3, false, false>(0, L, w, stage);
    int next = 0;
    if ((threadIdx.x & 63) == 0) next = atomicAdd(next_world, 1);
    w = __builtin_amdgcn_readfirstlane(next);
  }
}


// the sizes the wavefront's tiles take: the last of 3, 4 or 5 block rows in use
bool wave_shape(int nv, int nv_pad) { return nv > 32 && nv_pad > nv && nv_pad <= 80 && nv_pad % 16 == 0 && nv >= nv_pad - 16; }

}  // namespace
}  // namespace im

extern "C" int im_newton_solve_dense_column(const im_newton_args *p, float *H, float *U, int32_t *dof_union, int nv,
                                            int nv_pad, int nM, int32_t *next_world, void *stream) {
  return im::newton_solve_dense_column(p, H, U, dof_union, nv, nv_pad, nM, next_world, (hipStream_t)stream, nullptr);
}

extern "C" int im_dense_update_column(const uint8_t *done, const int32_t *state_changes, const int32_t *changes,
                                      const int32_t *ids, int ld_ids, const float *J, int njmax, const float *D,
                                      const int32_t *state, int quad, const float *grad, int64_t ldg, float *H, float *U,
                                      int nv, int nv_pad, int32_t *dof_union, float *search, int64_t ld_search,
                                      float *search_dot, float *decrement, int nworld, void *stream) {
  if (nworld < 0 || nv <= 0 || nv_pad <= nv || ld_ids < 0 || njmax <= 0) return IM_ERR_ARG;
  if (nworld == 0) return IM_OK;
  if (!state_changes || !changes || !ids || !J || !D || !state || !grad || !H || !U || !dof_union || !search ||
      !search_dot || !decrement)
    return IM_ERR_ARG;
  if (ldg < nv || ld_search < nv) return IM_ERR_STRIDE;
  if (!im::wave_shape(nv, nv_pad)) return IM_ERR_UNSUPPORTED;
  const dim3 grid((unsigned)((nworld + 3) / 4)), wg(256);
#define IM_UPDATE_WAVE(NB)                                                                                                    \
  hipLaunchKernelGGL(im::dense_update_wave_kernel<NB>, grid, wg, 16 * im::wave_stage_words<NB>(), (hipStream_t)stream, done,  \
                     state_changes, changes, ids, ld_ids, J, njmax, D, state, quad, grad, ldg, H, U, dof_union, search,      \
                     ld_search, search_dot, decrement, nv, nworld)
  if (nv_pad == 48) IM_UPDATE_WAVE(3);
  else if (nv_pad == 64) IM_UPDATE_WAVE(4);
  else IM_UPDATE_WAVE(5);
#undef IM_UPDATE_WAVE
  IM_HIP_CHECK(hipGetLastError());
  return IM_OK;
}

extern "C" int im_dense_init_tile(const uint8_t *done, const int32_t *nefc, const float *J, int njmax, const float *D,
                                  const int32_t *state, int quad, const float *M, int64_t ldM, const int32_t *elemid,
                                  const float *grad, int64_t ldg, float *H, int nv, int nv_pad, int32_t *dof_union,
                                  float *search, int64_t ld_search, float *search_dot, float *decrement, int nworld,
                                  void *stream);

static int init_factor(int most, const uint8_t *done, const int32_t *nefc, const float *J, int njmax, const float *D,
                       const int32_t *state, int quad, const float *M, int64_t ldM, const int32_t *elemid, const float
                       *grad, int64_t ldg, float *H, float *U, int nv, int nv_pad, int32_t *dof_union, float *search,
                       int64_t ld_search, float *search_dot, float *decrement, int nworld, void *stream) {
  if (nworld < 0 || nv <= 0 || nv_pad < nv || njmax <= 0) return IM_ERR_ARG;
  if (nworld == 0) return IM_OK;
  if (!J || !D || !state || !M || !elemid || !grad || !H || !dof_union || !search || !search_dot || !decrement)
    return IM_ERR_ARG;
  if (ldg < nv || ld_search < nv || ((uintptr_t)H & 15) != 0 || (nv_pad & 3) != 0) return IM_ERR_STRIDE;
  if (nv <= 32)
    return im_dense_init_tile(done, nefc, J, njmax, D, state, quad, M, ldM, elemid, grad, ldg, H, nv, nv_pad, dof_union,
                              search, ld_search, search_dot, decrement, nworld, stream);
  if (!U) return IM_ERR_ARG;
  if (!im::wave_shape(nv, nv_pad) || nv_pad > most) return IM_ERR_UNSUPPORTED;
  const dim3 grid((unsigned)((nworld + 3) / 4)), wg(256);
#define IM_INIT_WAVE(NB, STEPS)                                                                                               \
  hipLaunchKernelGGL((im::dense_init_wave_kernel<NB, STEPS>), grid, wg, 16 * im::wave_stage_words<NB>(), (hipStream_t)stream, \
                     done, nefc, J, njmax, D, state, quad, M, ldM, elemid, grad, ldg, H, U, dof_union, search, ld_search,     \
                     search_dot, decrement, nv, nworld)
  if (nv_pad == 48) {
    IM_INIT_WAVE(3, 4);
  } else if (nv_pad == 64) {
    IM_INIT_WAVE(4, 4);
  } else {
    int ncu = 0;
    if (const int st = im::compute_units(&ncu)) return st;
    if (nworld <= 12 * ncu) IM_INIT_WAVE(5, 4);
    else IM_INIT_WAVE(5, 2);
  }
#undef IM_INIT_WAVE
  IM_HIP_CHECK(hipGetLastError());
  return IM_OK;
}

extern "C" int im_dense_init_factor(const uint8_t *done, const int32_t *nefc, const float *J, int njmax, const float
                                    *D, const int32_t *state, int quad, const float *M, int64_t ldM, const int32_t
                                    *elemid, const float *grad, int64_t ldg, float *H, float *U, int nv, int nv_pad,
                                    int32_t *dof_union, float *search, int64_t ld_search, float *search_dot, float
                                    *decrement, int nworld, void *stream) {
  return init_factor(64, done, nefc, J, njmax, D, state, quad, M, ldM, elemid, grad, ldg, H, U, nv, nv_pad, dof_union,
                     search, ld_search, search_dot, decrement, nworld, stream);
}

namespace im {

int dense_init_factor(const uint8_t *done, const int32_t *nefc, const float *J, int njmax, const float *D, const
                      int32_t *state, int quad, const float *M, int64_t ldM, const int32_t *elemid, const float *grad,
                      int64_t ldg, float *H, float *U, int nv, int nv_pad, int32_t *dof_union, float *search, int64_t
                      ld_search, float *search_dot, float *decrement, int nworld, void *stream) {
  return init_factor(80, done, nefc, J, njmax, D, state, quad, M, ldM, elemid, grad, ldg, H, U, nv, nv_pad, dof_union,
                     search, ld_search, search_dot, decrement, nworld, stream);
}

int newton_solve_dense_column(const im_newton_args *p, float *H, float *U, int32_t *dof_union, int nv, int nv_pad, int nM,
                              int32_t *next_world, hipStream_t stream, Before *before) {
  if (!p || !H || !U || !dof_union || !next_world || p->nworld < 0 || nv <= 0 || nv_pad <= nv || nM <= 0) return IM_ERR_ARG;
  if (!wave_shape(nv, nv_pad)) return IM_ERR_UNSUPPORTED;
  if (p->nworld == 0) return IM_OK;
  resident::NewtonArgs a{};
  const int bad = resident::convert_args(*p, nv, nM, a);
  if (bad != IM_OK) return bad;
  const int njmax = p->njmax;
  struct Variant {
    int nblk, waves, held;
    const void *fn;
  };
#define IM_WAVE_VARIANT(NB, WAVES, HELD) {NB, WAVES, HELD, (const void *)newton_dense_wave_resident_kernel<NB, WAVES, HELD>}
  // four worlds per workgroup (a CU takes as many as its LDS and registers hold); the line search keeps a lane's two
  // rows in registers up to 64 rows and reads them from LDS beyond
  static const Variant variants[] = {IM_WAVE_VARIANT(3, 4, 2), IM_WAVE_VARIANT(3, 4, 0), IM_WAVE_VARIANT(4, 4, 2),
                                     IM_WAVE_VARIANT(4, 4, 0), IM_WAVE_VARIANT(5, 4, 2), IM_WAVE_VARIANT(5, 4, 0)};
#undef IM_WAVE_VARIANT
  constexpr int kVariants = 6;
  static Kept<int, std::array<bool, kVariants>> probed;
  std::array<bool, kVariants> usable;
  if (const int st = usable_variants(probed, variants, &usable)) return st;
  const int nblk = nv_pad / 16;
  for (int i = 0; i < kVariants; ++i) {
    const Variant &v = variants[i];
    if (!usable[i] || v.nblk != nblk || v.held != (njmax <= 64 ? 2 : 0)) continue;
    const int area = nblk == 3 ? wave_resident_area_words<3>(nv, njmax) : nblk == 4 ? wave_resident_area_words<4>(nv, njmax) : wave_resident_area_words<5>(nv, njmax);
    const size_t per_wave = (size_t)area + resident::kept_words(nv, njmax, 0);
    const size_t lds = 4 * ((size_t)wave_resident_shared_words(p->nterm, nv) + v.waves * per_wave);
    if (lds > 158 * 1024) continue;
    int ncu = 0;
    if (const int st = compute_units(&ncu)) return st;
    // as many workgroups as stay resident at once: by LDS and by registers
    int per_cu = 0;
    if (const int st = resident_per_cu(v.fn, nullptr, 64 * v.waves, lds, &per_cu)) return st;
    per_cu = std::max(1, per_cu);
    const int grid = resident_worlds_grid(p->nworld, v.waves, ncu, per_cu, false, &a.group_worlds);
    if (before) {
      a.final_force = 1;
      if (const int st = (*before)(next_world, grid * v.waves)) return st;
    } else {
      set_counter(next_world, grid * v.waves, stream);
    }
    void *args[] = {&a, &H, &U, &dof_union, &next_world};
    IM_HIP_CHECK(hipLaunchKernel(v.fn, dim3((unsigned)grid), dim3(64 * v.waves), args, lds, stream));
    return IM_OK;
  }
  return IM_ERR_UNSUPPORTED;
}

}  // namespace im
