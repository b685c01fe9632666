// The resident Newton loop: one wavefront per world from the first line search to convergence,
// four worlds per workgroup, as the reference keeps a world in one block for the whole loop
// (src/instantmimic/utils/mjw_kernels/newton_fusion.py:57-298).  Per iteration and world, in the
// reference kernel's order (:170-296): M search, J search, the scalar line search with the step
// and the constraints' new forces and states (newton_stages.py:79-444), the gradient (:745-798),
// the factor stage, the convergence test.  Every stage performs the operations of the per-stage
// kernels of this library in their order, so a solve gives the same bits whichever way it runs.
//
// The factor stage is handed in by the kernel that includes this file (a generated kernel for the
// model's tree: four wavefronts work on the workgroup's four worlds together), which is why the
// loop keeps the four wavefronts in step at two workgroup barriers per iteration; a world that is
// done idles through them until the workgroup's last world finishes.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/imhip.h"
#include "newton_search.h"

namespace im {
namespace resident {

struct NewtonArgs {
  // options (arrays indexed by world modulo their length)
  const float *tolerance, *ls_tolerance, *meaninertia;
  int ntolerance, nls_tolerance, nmeaninertia;
  int nv, njmax, nworld, ls_iterations, maxiter, block, quad, ls_overflow_bit, iter_overflow_bit;
  // row tables of M v: nv + 1 offsets, then per term the column and the element of M
  const int32_t *mulm_rowadr, *mulm_col, *mulm_madr;
  int nterm, nM;
  // the step's inputs
  const int32_t *ne, *nf, *nefc;
  const float *M;
  int64_t ldM;
  const float *J, *D, *frictionloss, *smooth;  // J (nworld, njmax, nv); D, frictionloss (nworld, njmax); smooth (nworld, nv)
  // solver state, rows of nv or njmax floats per world unless a stride is given
  float *qacc, *Ma, *force, *Jaref, *search, *search_dot, *mv, *jv, *alpha, *improvement, *grad, *grad_dot,
      *grad_scale, *decrement, *qfrc_constraint;
  int64_t ld_grad;
  int32_t *state, *ids, *quad_count, *state_count, *niter, *overflow, *nsolving;
  int ld_ids;
  uint8_t *done, *exhausted, *unchanged;
  int stage_lds_floats;  // dynamic LDS the factor stage uses from offset 0; the loop's own arrays follow
  // cooperative loop: a counter in memory, set to four times the grid's workgroups before the launch,
  // from which a wavefront whose world is done takes the next world nobody has started (null: a
  // workgroup keeps to its own four worlds)
  int *next_world;
  // cooperative loop: whether a wavefront keeps its world's row of M in LDS (1) or reads it from
  // memory in the round's one product with it (0: the LDS saved admits another workgroup per CU)
  int m_lds;
  // one call for the whole solve: a world that finishes writes its constraint force from the last
  // gradient (newton_fusion.py:537-555) itself ...
  int final_force;
  // ... and (cooperative loop) forms the two sums of the first search direction as it enters, which
  // a launch of their own would leave in memory
  int sums_at_enter;
  // the worlds that a workgroup starts with, its first wavefronts' (resident_worlds_grid)
  int group_worlds;
};

// The public argument block checked and turned into the kernels' (host side).
inline int convert_args(const im_newton_args &p, int nv, int nM, NewtonArgs &a) {
  const int njmax = p.njmax;
  if (njmax <= 0 || p.iterations < 0 || p.ls_iterations < 0 || (p.block != 32 && p.block != 64) || p.ntolerance <= 0 ||
      p.nls_tolerance <= 0 || p.nmeaninertia <= 0 || p.nterm <= 0)
    return IM_ERR_ARG;
  if (!p.opt_tolerance || !p.opt_ls_tolerance || !p.stat_meaninertia || !p.M_mulm_rowadr || !p.M_mulm_col ||
      !p.M_mulm_madr || !p.M || !p.efc_J || !p.efc_D || !p.qfrc_smooth || !p.qacc || !p.efc_Ma || !p.efc_force ||
      !p.efc_state || !p.Jaref || !p.search || !p.search_dot || !p.mv || !p.jv || !p.alpha || !p.improvement || !p.grad ||
      !p.grad_dot || !p.grad_scale || !p.newton_decrement || !p.qfrc_constraint || !p.quad_changed_ids ||
      !p.quad_changed_count || !p.state_changed_count || !p.solver_niter || !p.done || !p.ls_exhausted ||
      !p.search_unchanged || (p.nf && !p.efc_frictionloss))
    return IM_ERR_ARG;
  if (p.ldM < nM || p.ld_grad < nv || p.ld_ids < 0) return IM_ERR_STRIDE;
  if (p.nterm >= 65536 || nM >= 65536 || 64 * (int64_t)nv >= (1 << 20) || (int64_t)njmax * nv >= (1 << 29)) return IM_ERR_UNSUPPORTED;
  a.tolerance = p.opt_tolerance, a.ls_tolerance = p.opt_ls_tolerance, a.meaninertia = p.stat_meaninertia;
  a.ntolerance = p.ntolerance, a.nls_tolerance = p.nls_tolerance, a.nmeaninertia = p.nmeaninertia;
  a.nv = nv, a.njmax = njmax, a.nworld = p.nworld, a.ls_iterations = p.ls_iterations, a.maxiter = p.iterations;
  a.block = p.block, a.quad = p.quad, a.ls_overflow_bit = p.ls_overflow_bit;
  a.iter_overflow_bit = p.iterations_overflow_bit;
  a.mulm_rowadr = p.M_mulm_rowadr, a.mulm_col = p.M_mulm_col, a.mulm_madr = p.M_mulm_madr;
  a.nterm = p.nterm, a.nM = nM;
  a.ne = p.ne, a.nf = p.nf, a.nefc = p.nefc, a.M = p.M, a.ldM = p.ldM, a.J = p.efc_J, a.D = p.efc_D;
  a.frictionloss = p.efc_frictionloss, a.smooth = p.qfrc_smooth;
  a.qacc = p.qacc, a.Ma = p.efc_Ma, a.force = p.efc_force, a.Jaref = p.Jaref, a.search = p.search;
  a.search_dot = p.search_dot, a.mv = p.mv, a.jv = p.jv, a.alpha = p.alpha, a.improvement = p.improvement;
  a.grad = p.grad, a.grad_dot = p.grad_dot, a.grad_scale = p.grad_scale, a.decrement = p.newton_decrement;
  a.qfrc_constraint = p.qfrc_constraint, a.ld_grad = p.ld_grad;
  a.state = p.efc_state, a.ids = p.quad_changed_ids, a.quad_count = p.quad_changed_count;
  a.state_count = p.state_changed_count, a.niter = p.solver_niter, a.overflow = p.overflow, a.nsolving = p.nsolving;
  a.ld_ids = p.ld_ids, a.done = p.done, a.exhausted = p.ls_exhausted, a.unchanged = p.search_unchanged;
  a.stage_lds_floats = 0;
  a.next_world = nullptr;
  a.m_lds = 1;
  a.final_force = 0;
  a.sums_at_enter = 0;
  a.group_worlds = 1;
  return IM_OK;
}

__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
// a value every lane holds alike, as a scalar (so that it occupies no vector register while it waits)
__device__ __forceinline__ float uniform(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}

// the world that a workgroup's wavefront `wv` starts with; nworld: none
__device__ __forceinline__ int64_t first_world(const NewtonArgs &a, int wv) {
  return wv < a.group_worlds ? (int64_t)blockIdx.x * a.group_worlds + wv : a.nworld;
}

// orders this wavefront's writes (LDS and memory) before its later reads: the stages hand their
// results on through memory, written by some lanes and read by others
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ void block_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// words of LDS of the loop's own arrays behind the factor stage's area: four flags, the row tables of M v
// (one word per term, nv + 1 offsets), then per wavefront the search direction, Ma, mv, qacc, Jaref, jv, D and the
// friction losses, the gradient's list of rows with a force (value and row number) and its copy of the gradient, the
// world's row of M.  The factor stage's area must also hold four wavefronts'
// rows of M where those are read from memory, and their tiles of J (kTileWords each).
// words a wavefront keeps from round to round: M, the search direction, Ma, mv, qacc; Jaref, jv, D, friction losses
__host__ __device__ inline size_t kept_words(int nv, int njmax, int nM) { return (size_t)nM + 4 * (size_t)nv + 4 * (size_t)njmax; }
// a wavefront's own words in a cooperative kernel, a multiple of four (the search direction first)
__host__ __device__ inline size_t coop_wave_words(int nv, int njmax, int nM) {
  return (kept_words(nv, njmax, nM) + 2 * (size_t)njmax + nv + 3) & ~(size_t)3;
}
__host__ __device__ inline size_t loop_lds_words(int nv, int njmax, int nM, int nterm) {
  return 8 + (size_t)nterm + nv + 1 + 6 + 4 * coop_wave_words(nv, njmax, nM);
}
constexpr int kTileWords = 64 * 17;  // (a tile of J takes 64 * 16 of them, a row of M up to all)
constexpr size_t kStagedWords = 4 * kTileWords;

// ---- M search (newton_fusion.py:171-176) -------------------------------------------------------
// WALK: more dofs than lanes.
template <bool WALK>
__device__ __forceinline__ void mul_m_world(const NewtonArgs &a, const uint32_t *term, const int *radr, const float *m,
                                            const float *v, float *out, float *out_lds, int lane) {
  const int nv = a.nv;
  if constexpr (!WALK) {
    for (int dof = lane; dof < nv; dof += 64) {
      float value = 0.0f;
      const int end = radr[dof + 1];
      for (int k = radr[dof]; k < end; k += 8) {  // eight terms' operands at a time, a term past the end dropped
        float x[8], y[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const uint32_t t = term[k + u < end ? k + u : end - 1];
          x[u] = m[t >> 16];
          y[u] = v[t & 0xffffu];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) value = k + u < end ? fma_(x[u], y[u], value) : value;
      }
      out[dof] = value;
      out_lds[dof] = value;
    }
    return;
  }
  // a lane takes dof `lane`, then 127 - lane, 128 + lane, ..: one after the other without waiting for the others, so
  // that the long rows (a free body's dofs, the first ones) have nothing behind them.  Eight terms' operands at a time,
  // a term past the end dropped; the next terms are read ahead of the current ones' operands.
  int dof = lane, base = 0;
  int k = 0, end = 0;
  if (dof < nv) k = radr[dof], end = radr[dof + 1];
  uint32_t t[8];
  auto read = [&](int k) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 8; ++u) t[u] = term[k + u < end ? k + u : end > 0 ? end - 1 : 0];
  };
  if (dof < nv) read(k);
  float value = 0.0f;
  while (dof < nv) {
    float x[8], y[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      x[u] = m[t[u] >> 16];
      y[u] = v[t[u] & 0xffffu];
    }
    const int k0 = k, last = end;
    k += 8;
    int done = -1;
    if (k >= end) {
      done = dof;
      base += 64;
      dof = base + (base & 64 ? 63 - lane : lane);
      if (dof < nv) k = radr[dof], end = radr[dof + 1];
    }
    if (dof < nv) read(k);
#pragma unroll
    for (int u = 0; u < 8; ++u) value = k0 + u < last ? fma_(x[u], y[u], value) : value;
    if (done >= 0) {
      out[done] = value;
      out_lds[done] = value;
      value = 0.0f;
    }
  }
}
// The same with the world's row of M in memory: it passes through `stage` (kTileWords of LDS) where it fits, the
// first LOADS words a lane asked for together, EARLY: by load() ahead of whatever else the round asks for (where the
// registers are not what bounds a kernel's wavefronts).  Read term by term a
// free body's dofs, whose rows are nv long, waited for memory once per four terms (70 dofs x 2048 worlds: 9 of the 22 us
// that a round's two products took).
template <bool WALK, int LOADS, bool EARLY>
struct StagedM {
  float x[LOADS];
  __device__ __forceinline__ void load(const float *m, int nM, int lane) {
    if constexpr (EARLY) fetch(m, nM, lane);
  }
  __device__ __forceinline__ void fetch(const float *m, int nM, int lane) {
    // (without a condition: what might be left as it was would be kept from round to round)
#pragma unroll
    for (int u = 0; u < LOADS; ++u) x[u] = m[(unsigned)(lane + 64 * u < nM ? lane + 64 * u : nM - 1)];
  }
  __device__ __forceinline__ void product(const NewtonArgs &a, const uint32_t *term, const int *radr, const float *m, int nM,
                                          const float *v, float *out, float *out_lds, float *stage, int lane) {
    if (nM > kTileWords) {
      wave_sync();
      return mul_m_world<WALK>(a, term, radr, m, v, out, out_lds, lane);
    }
    if constexpr (EARLY) {
#pragma unroll
      for (int u = 0; u < LOADS; ++u)
        if (lane + 64 * u < nM) stage[lane + 64 * u] = x[u];
      // a longer row's other words, four a lane at once (as many as the first took the start's kernel from 77 registers to 83,
      // past a wavefront)
      for (int k = lane + 64 * LOADS; k < nM; k += 64 * 4) {
        float y[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) y[u] = m[(unsigned)(k + 64 * u < nM ? k + 64 * u : nM - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (k + 64 * u < nM) stage[k + 64 * u] = y[u];
      }
    } else {
      // (a loop of its own behind the first words, though never run, cost 14 dofs x 64 worlds 0.8 of 93 us)
      for (int k0 = 0; k0 < nM; k0 += 64 * LOADS) {
        fetch(m + k0, nM - k0, lane);
#pragma unroll
        for (int u = 0; u < LOADS; ++u)
          if (k0 + lane + 64 * u < nM) stage[k0 + lane + 64 * u] = x[u];
      }
    }
    wave_sync();
    mul_m_world<WALK>(a, term, radr, stage, v, out, out_lds, lane);
  }
};

// ---- the gradient (newton_stages.py:745-798), a lane per dof ------------------------------------
// The world's scalars that the loop carries in registers (every lane the same values); they are
// written to memory as they change.
struct Scalars {
  float search_dot, grad_dot, decrement, grad_scale, alpha, improvement;
  int niter;
};
// For a world whose states changed: qfrc_constraint = J' force over the listed rows (`cnt` rows with
// a nonzero force, ascending, in f / rowl), grad = Ma - qfrc_smooth - qfrc_constraint, grad . grad.
// Otherwise the rescaling of the three scalars.  Returns whether the search direction stays.
// COLS: dofs of a lane (lane, lane + 64) whose sums run side by side; RING: batches of rows on their way at once.
// LAZY: a list of one batch asks for no second one.  (Otherwise rows past the list are the last one again: behind a branch
// every wait would count the youngest batch.)
template <int COLS, int RING, bool LAZY>
__device__ __forceinline__ void constraint_force(const float *Jw, int nv, int cnt, const float *f, const int *rowl, int d0, float (&sum)[COLS]) {
  constexpr int ROWS = 16 / COLS;
  float v[RING][ROWS][COLS];
  auto fetch = [&](int p0, float (&v)[ROWS][COLS]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < ROWS; ++u) {
      const uint32_t at = (uint32_t)(rowl[p0 + u < cnt ? p0 + u : cnt - 1] * nv);
#pragma unroll
      for (int k = 0; k < COLS; ++k) {
        const int dof = d0 + 64 * k;
        v[u][k] = *(const float *)((const char *)Jw + 4u * (at + (dof < nv ? dof : nv - 1)));
      }
    }
  };
  auto add = [&](int p0, float (&v)[ROWS][COLS]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < ROWS; ++u) {
      const float fu = f[p0 + u < cnt ? p0 + u : cnt - 1];
#pragma unroll
      for (int k = 0; k < COLS; ++k) sum[k] = p0 + u < cnt ? fma_(v[u][k], fu, sum[k]) : sum[k];
    }
  };
#pragma unroll
  for (int k = 0; k < COLS; ++k) sum[k] = 0.0f;
  if (cnt <= 0) return;
  fetch(0, v[0]);
  if (LAZY && cnt <= ROWS) return add(0, v[0]);
#pragma unroll
  for (int b = 1; b < RING; ++b) fetch(b * ROWS, v[b]);
  for (int p0 = 0; p0 < cnt; p0 += RING * ROWS) {
#pragma unroll
    for (int b = 0; b < RING; ++b) {
      if (p0 + b * ROWS >= cnt) return;
      add(p0 + b * ROWS, v[b]);
      fetch(p0 + (b + RING) * ROWS, v[b]);
    }
  }
}
template <int COLS, int RING, bool LAZY>
__device__ __forceinline__ bool gradient_world(const NewtonArgs &a, int64_t w, const float *Jw, bool changed, int cnt,
                                               const float *f, const int *rowl, const float *Ma_l, const float *smooth, float *gl,
                                               Scalars &sc, int lane) {
  if (!changed) {
    const float sigma = sc.grad_scale, new_sigma = sigma - sc.alpha;
    float ratio = 0.0f;
    if (sigma != 0.0f) ratio = new_sigma / sigma;
    const float ratio_sq = ratio * ratio;
    sc.grad_dot = uniform(sc.grad_dot * ratio_sq);
    sc.decrement = uniform(sc.decrement * ratio_sq);
    sc.grad_scale = uniform(new_sigma);
    if (lane == 0) {
      a.grad_dot[w] = sc.grad_dot;
      a.decrement[w] = sc.decrement;
      a.grad_scale[w] = sc.grad_scale;
      a.unchanged[w] = 1;
    }
    return true;
  }
  const int nv = a.nv;
  for (int d0 = lane; d0 - lane < nv; d0 += 64 * COLS) {
    float sum[COLS];
    constraint_force<COLS, RING, LAZY>(Jw, nv, cnt, f, rowl, d0, sum);
#pragma unroll
    for (int k = 0; k < COLS; ++k) {
      const int dof = d0 + 64 * k;
      if (dof < nv) {
        const float g = Ma_l[dof] - smooth[dof] - sum[k];
        a.qfrc_constraint[w * nv + dof] = sum[k];
        a.grad[w * a.ld_grad + dof] = g;
        gl[dof] = g;
      }
    }
  }
  wave_sync();
  // grad . grad as a block of `block` lanes sums it: lane `rank` its dofs rank, rank + block, ..,
  // 32 lanes in a shuffle-down tree, the trees in order
  float p = 0.0f;
  if (lane < a.block)
    for (int dof = lane; dof < nv; dof += a.block) p = fma_(gl[dof], gl[dof], p);
  float q = p;
  search::swap_rows(p, q);  // the even rows of p + q: a row and the one behind it
  p = search::row_sum(p + q);
  float total = 0.0f + search::lane_of(p, 0);
  if (a.block > 32) total = total + search::lane_of(p, 32);
  sc.grad_dot = uniform(total);
  sc.decrement = 0.0f;
  sc.grad_scale = 1.0f;
  if (lane == 0) {
    a.grad_dot[w] = total;
    a.decrement[w] = 0.0f;
    a.grad_scale[w] = 1.0f;
    a.unchanged[w] = 0;
  }
  return false;
}

// ---- search . search and grad . x of a factor stage that leaves only the search direction -----
// (and the direction itself, for the next round's products)
__device__ __forceinline__ void search_sums_world(const NewtonArgs &a, int64_t w, const float *gl, float *sv, Scalars &sc, int lane) {
  float s0 = 0.0f, s1 = 0.0f;
  for (int d = lane; d < a.nv && lane < a.block; d += a.block) {
    const float from = a.search[w * a.nv + d], v = -from;
    sv[d] = from;
    s0 = fma_(v, v, s0);
    s1 = fma_(gl[d], v, s1);
  }
  search::swap_rows(s0, s1);  // s0 + s1: the first sum's rows 16 apart in the even rows, the second's in the odd ones
  const float s = search::row_sum(s0 + s1);
  float ra = 0.0f + search::lane_of(s, 0), rb = 0.0f + search::lane_of(s, 16);
  if (a.block > 32) ra = ra + search::lane_of(s, 32), rb = rb + search::lane_of(s, 48);
  sc.search_dot = uniform(ra);
  sc.decrement = uniform(rb);
  if (lane == 0) {
    a.search_dot[w] = ra;
    a.decrement[w] = rb;
  }
}

// ---- J search (newton_stages.py:157-178) through a tile of 64 rows x 16 dofs in LDS -------------------
// A row's sum is a chain of multiply-adds over the dofs in order, beyond 50 dofs in parts of 20 that are added up: a lane
// per row, its operands by four 16-byte reads a tile, the direction's by four that every lane makes alike.  Lane (g, c) =
// (lane / 16, lane % 16) brings dofs 4 g .. 4 g + 3 of rows c, 16 + c, .. into the tile, whose rows lie 16 words apart
// with their quads changed round by the row (quad q of row r at q ^ (r / 4 % 4): neither the writes nor the reads meet in a
// bank).  DEPTH tiles are on their way at once.  What bounds the product is the trips to memory and the chain.  With the
// row of M asked for ahead (StagedM), the two products of a round of the slowest worlds: 70 dofs x 157 rows x 2048 worlds
// 19.2 -> 13.3 us, 43 x 96 x 8192 9.4 -> 7.2; the solves, three runs in turn within 0.3 %: 70 x 2048 797 -> 738 (the chains ran on the
// matrix cores there, sixteen equal columns to a result, their operands turned by lane swaps), 53 x 4096 715 -> 679, 43 x 8192
// 651 -> 621, 27 x 4096 249 -> 242, 14 x 64 106.8 -> 104.3 (a tile of single words, four times the LDS instructions).  1 tile ahead
// up to 64 dofs, where registers bound the wavefronts in flight, 3 beyond.
// `before` runs ahead of the first request, `between` while the first tiles are on their way; it leaves the direction in
// sv (16-byte aligned) and may use the tile.
typedef float v4 __attribute__((ext_vector_type(4)));
typedef v4 v4_words __attribute__((aligned(4)));
template <int DEPTH, class Before, class Between>
__device__ __forceinline__ void jv_world(const NewtonArgs &a, const float *Jw, int nefc, float *tile, const float *sv, float *jv,
                                         float *jv_lds, int lane, Before &&before, Between &&between) {
  const int nv = a.nv, g = lane >> 4, c = lane & 15;
  before();
  if (nefc <= 0 || nv < 4) {  // (rows shorter than a load: from memory)
    between();
    for (int r = lane; r < nefc; r += 64) {
      float p = 0.0f;
      for (int i = 0; i < nv; ++i) p = fma_(Jw[r * nv + i], sv[i], p);
      if (jv) jv[r] = p;
      jv_lds[r] = p;
    }
    return;
  }
  const bool split = nv > 50;
  struct Step {
    int r0, c0;
  };
  // (not behind a branch, the last row's again past the end: a wait for one tile's loads counts those of the next)
  auto fetch = [&](const Step &s, v4 (&v)[4]) __attribute__((always_inline)) {
    const int col = s.c0 + 4 * g, from = col < nv - 4 ? col : nv - 4;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int row = s.r0 + 16 * t + c;
      v[t] = *(const v4_words *)((const char *)Jw + 4u * (uint32_t)((row < nefc ? row : nefc - 1) * nv + from));
    }
  };
  auto advance = [&](Step &s) __attribute__((always_inline)) {
    s.c0 += 16;
    if (s.c0 >= nv) s.c0 = 0, s.r0 += 64;
  };
  Step now = {0, 0}, ahead = {0, 0};
  v4 v[DEPTH][4];
#pragma unroll
  for (int b = 0; b < DEPTH; ++b) fetch(ahead, v[b]), advance(ahead);
  between();
  wave_sync();
  float *put = tile + 16 * c + 4 * (g ^ (c >> 2));
  const float *take = tile + 16 * lane;
  const int turn = 4 * ((lane >> 2) & 3);
  float acc = 0.0f, p = 0.0f;
  auto work = [&](v4 (&v)[4]) __attribute__((always_inline)) {
    if (now.c0 + 16 > nv) {  // the row's last dofs were loaded from four before its end: moved down, zeros behind them
      const int by = now.c0 + 4 * g + 4 - nv;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        v4 m = v[t];
        m = by >= 1 ? v4{m[1], m[2], m[3], 0.0f} : m;
        m = by >= 2 ? v4{m[1], m[2], 0.0f, 0.0f} : m;
        m = by >= 3 ? v4{m[1], 0.0f, 0.0f, 0.0f} : m;
        v[t] = by >= 4 ? v4{0.0f, 0.0f, 0.0f, 0.0f} : m;
      }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) *(v4 *)(put + 256 * t) = v[t];
    wave_sync();
  };
  auto chain = [&]() __attribute__((always_inline)) {
    // (half a tile's operands at a time where a kernel has no registers to spare)
    constexpr int QUADS = DEPTH > 1 ? 4 : 2;
#pragma unroll
    for (int q0 = 0; q0 < 4; q0 += QUADS) {
      v4 x[QUADS], y[QUADS];
#pragma unroll
      for (int q = 0; q < QUADS; ++q) {
        const int col = now.c0 + 4 * (q0 + q);
        x[q] = y[q] = v4{0.0f, 0.0f, 0.0f, 0.0f};
        if (col >= nv) continue;
        x[q] = *(const v4 *)(take + ((4 * (q0 + q)) ^ turn));
        y[q] = *(const v4 *)(sv + col);
        if (col + 4 > nv) {  // (+0 of J times -0: what a sum takes without any change, its sign as a zero too)
          y[q][3] = -0.0f;
          y[q][2] = col + 2 < nv ? y[q][2] : -0.0f;
          y[q][1] = col + 1 < nv ? y[q][1] : -0.0f;
        }
      }
#pragma unroll
      for (int q = 0; q < QUADS; ++q) {
        const int col = now.c0 + 4 * (q0 + q);
        if (col >= nv) continue;
        if (split && col % 20 == 0) {  // (0 + 0 at the first)
          acc = acc + p;
          p = 0.0f;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) p = fma_(x[q][u], y[q][u], p);
      }
    }
    if (now.c0 + 16 >= nv) {
      const int row = now.r0 + lane;
      const float out = split ? acc + p : p;
      if (row < nefc) {
        if (jv) jv[row] = out;
        jv_lds[row] = out;
      }
      acc = p = 0.0f;
    }
    advance(now);
    wave_sync();  // the tile is read before the next one overwrites it
  };
  for (;;) {
#pragma unroll
    for (int b = 0; b < DEPTH; ++b) {
      work(v[b]);
      if (DEPTH > 1 || ahead.r0 < nefc) fetch(ahead, v[b]);
      advance(ahead);
      chain();
      if (now.r0 >= nefc) return;
    }
  }
}

// ---- the loop ------------------------------------------------------------------------------------
// Where the loop's arrays lie in LDS (set up by the kernel around it).
struct LoopLds {
  int *votes;            // [4] cooperative stage only
  int *worlds;           // [4] cooperative stage only: the world of each wavefront (nworld: none), read by the stage
  const uint32_t *term;  // [nterm] col | madr << 16, shared by the workgroup
  const int *radr;       // [nv + 1]
  // per wavefront, kept from round to round:
  float *m_lds;          // [nM] the world's row of M
  float *sv;             // [nv] the search direction; 16-byte aligned, as rows
  float *Ma, *mv, *qacc; // [nv] each
  float *Jaref, *jv;     // [njmax] each
  float *D, *fl;         // [njmax] each: the rows' weights and friction losses (read at every step of the line search)
  // per wavefront, used within a round (may share one area with the factor stage's own arrays):
  float *f;              // [njmax] forces of the listed rows
  int *rowl;             // [njmax] their numbers
  float *gl;             // [nv] qfrc_smooth, from the products to the gradient; then the gradient (a cooperative stage's loop
                         // reads it again after the stage)
  float *rows;           // kTileWords: the world's row of M on its way into the product, then the tile of J
};

// A world's vectors stay in LDS and its scalars in registers from round to round; memory receives
// every value as it is produced (the arrays end as after the stage launches) and is read again only
// for what another wavefront or the factor stage has written there.
// HELD: rows of a world a lane keeps in registers during the line search (0: read from LDS at every
// evaluation).  COLS: dofs of a lane in the gradient (2 beyond 64).  WIDE:
// registers to spare for operands read ahead.
// COOP: `stage()` works on the workgroup's four worlds together (every wavefront calls it in step,
// between two workgroup barriers; it takes the worlds' numbers from L.worlds and skips the worlds
// whose `unchanged` byte is set).  A wavefront whose world is done takes the next world from the
// counter a.next_world (or, without one, idles through the barriers); the workgroup leaves when all
// four are idle.  Otherwise
// `stage()` is the wavefront's own world's stage (it leaves search_dot and newton_decrement in
// memory itself), called only when that world needs it, and a wavefront leaves as soon as its world
// is done.  `w_raw`: the wavefront's world.
//
// `kernarg_offset`: where the kernel's NewtonArgs parameter lies in its kernel-argument segment.  The
// loop reads the arguments from there, through a pointer it launders once per round: about sixty
// pointers cannot stay in scalar registers across the stages (held, they are spilled to vector
// lanes and read back one by one), and from the segment each is one scalar load next to its use.
typedef const NewtonArgs __attribute__((address_space(4))) KernelNewtonArgs;
__device__ __forceinline__ const NewtonArgs &kernel_args(int kernarg_offset) {
  const char __attribute__((address_space(4))) *seg =
      (const char __attribute__((address_space(4))) *)__builtin_amdgcn_kernarg_segment_ptr();
  KernelNewtonArgs *ap = (KernelNewtonArgs *)(seg + kernarg_offset);
  asm volatile("" : "+s"(ap));
  return *(const NewtonArgs *)ap;
}

// The wavefront's priority among those of its SIMD: the quarter of the most rows that its world has.  A launch ends with
// its slowest world, and rows are what is known of that beforehand (a world's time goes with its rows by 0.4 at 27 dofs,
// 0.7 at 70).  Without / with it, us, medians of three runs in turn whose medians lie within 0.4 %: 27 dofs x 4096 worlds 241.9 / 239.3, 53 x 4096
// 676.6 / 670.2, 43 x 8192 618.3 / 616.6 (tree stages), 70 x 2048 688.5 / 681.8, 78 x 2048 722.2 / 710.3, 70 x 6000 1364 / 1340 (dense); 14 x 64,
// where a SIMD has one wavefront, 103.9 / 105.0.  The most rows of a workgroup's four worlds instead was worth half of that; on the
// sparse stage and the dense one up to 64 dofs it made no difference either way.
__device__ __forceinline__ void row_priority(int nefc, int njmax) {
  if (4 * nefc > 3 * njmax)
    __builtin_amdgcn_s_setprio(3);
  else if (2 * nefc > njmax)
    __builtin_amdgcn_s_setprio(2);
  else if (4 * nefc > njmax)
    __builtin_amdgcn_s_setprio(1);
  else
    __builtin_amdgcn_s_setprio(0);
}

// MLDS: the world's row of M is kept in LDS (where L.m_lds is not null); otherwise `M search` reads it from memory
// every round, which leaves the LDS to more worlds per CU.
template <int HELD, int COLS, bool WIDE, bool COOP, bool MLDS = true, class Stage>
__device__ __forceinline__ void newton_loop(int kernarg_offset, const LoopLds &L, int64_t w_raw, Stage &&stage) {
  const NewtonArgs &a0 = kernel_args(kernarg_offset);
  const NewtonArgs &a = a0;
  const int lane_fixed = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int nv = a.nv, njmax = a.njmax;
  // what belongs to the wavefront's current world
  int64_t w = 0;
  bool live = false, done = true, unchanged = false;
  int nefc = 0, ne = 0, nf = 0, budget = 0;
  const float *Jw = a.J;
  float tolerance = 0.0f, ls_tolerance = 0.0f, meaninertia = 1.0f;
  Scalars sc{};
  auto enter = [&](int64_t w_raw) __attribute__((always_inline)) {
    const NewtonArgs &a = kernel_args(kernarg_offset);
    // the world's number as a scalar: every address below is a scalar base plus a lane offset
    const int w_lo = __builtin_amdgcn_readfirstlane((int)(w_raw & 0xffffffff)), w_hi = __builtin_amdgcn_readfirstlane((int)(w_raw >> 32));
    const int64_t w_uniform = ((int64_t)w_hi << 32) | (uint32_t)w_lo;
    live = w_uniform < a.nworld;
    w = live ? w_uniform : (int64_t)a.nworld - 1;
    done = !live || a.done[w] != 0;
    if (live && done && lane_fixed == 0) a.unchanged[w] = 1;  // the factor stage leaves such a world alone
    unchanged = !done && a.unchanged[w] != 0;
    nefc = a.nefc ? a.nefc[w] : njmax;
    nefc = __builtin_amdgcn_readfirstlane(nefc < njmax ? nefc : njmax);
    ne = __builtin_amdgcn_readfirstlane(a.ne ? a.ne[w] : 0), nf = __builtin_amdgcn_readfirstlane(a.nf ? a.nf[w] : 0);
    Jw = a.J + w * (int64_t)njmax * nv;
    tolerance = a.tolerance[w % a.ntolerance], ls_tolerance = a.ls_tolerance[w % a.nls_tolerance];
    meaninertia = a.meaninertia[w % a.nmeaninertia];
    sc = Scalars{uniform(a.search_dot[w]), uniform(a.grad_dot[w]), uniform(a.decrement[w]), uniform(a.grad_scale[w]),
                 uniform(a.alpha[w]), uniform(a.improvement[w]), __builtin_amdgcn_readfirstlane(a.niter[w])};
    budget = a.maxiter;  // rounds this wavefront gives the world, whatever the data
    if (COOP) row_priority(nefc, njmax);
    if (done) return;
    // what the loop keeps: M, Ma, Jaref into LDS (mv and jv are formed before they are read: a world
    // enters with a new search direction unless it is done) and qacc
    if constexpr (MLDS)
      if (L.m_lds)
        for (int k = lane_fixed; k < a.nM; k += 64) L.m_lds[k] = a.M[w * a.ldM + k];
    for (int k = lane_fixed; k < nv; k += 64) {
      L.Ma[k] = a.Ma[w * nv + k];
      L.mv[k] = a.mv[w * nv + k];
      L.qacc[k] = a.qacc[w * nv + k];
      L.sv[k] = a.search[w * nv + k];
    }
    for (int r = lane_fixed; r < njmax; r += 64) {
      L.Jaref[r] = a.Jaref[w * njmax + r];
      L.jv[r] = a.jv[w * njmax + r];
      L.D[r] = a.D[w * njmax + r];
      L.fl[r] = a.frictionloss ? a.frictionloss[w * njmax + r] : 0.0f;
    }
    if (COOP && a.sums_at_enter) {
      for (int k = lane_fixed; k < nv; k += 64) L.gl[k] = a.grad[w * a.ld_grad + k];
      wave_sync();
      search_sums_world(a, w, L.gl, L.sv, sc, lane_fixed);
    }
    wave_sync();
  };
  enter(w_raw);
  bool queue_empty = !(COOP && a0.next_world);
#ifdef IM_NEWTON_STAMPS  // development aid: time per phase, summed over the rounds, left in the world's row of jv
  long long t_phase[8] = {0, 0, 0, 0, 0, 0, 0, 0}, t_last = wall_clock64();
#define IM_STAMP(k) do { const long long t_now = wall_clock64(); t_phase[k] += t_now - t_last; t_last = t_now; } while (0)
#else
#define IM_STAMP(k) do {} while (0)
#endif
  // Every world gets at most maxiter rounds of its wavefront, whatever the data, and the counter of
  // worlds only grows: every wavefront leaves the loop.
  for (;;) {
    const NewtonArgs &a = kernel_args(kernarg_offset);  // read afresh in every round
    if (COOP) {
      // a wavefront without a world to work on takes the next one nobody has started; the other
      // wavefronts' worlds go on with their own rounds beside it (the stage does not care which
      // iteration a world is in)
      while (done && !queue_empty) {
        int next = 0;
        if (lane_fixed == 0) next = atomicAdd(a.next_world, 1);
        next = __builtin_amdgcn_readfirstlane(next);
        if (next < a.nworld)
          enter(next);
        else
          queue_empty = true;
      }
      if (lane_fixed == 0) {
        L.votes[wv] = done ? 0 : 1;
        L.worlds[wv] = done ? a.nworld : (int)w;
      }
      block_sync();
      if (!(L.votes[0] | L.votes[1] | L.votes[2] | L.votes[3])) break;  // the workgroup's four worlds are done
    } else if (done) {
      break;
    }
    // the lane number as a value the compiler cannot see through, new in every round: nothing a
    // stage derives from it is kept in registers across the other stages
    int lane = lane_fixed;
    asm volatile("" : "+v"(lane));
    IM_STAMP(0);
    if (!done) {
      // qfrc_smooth on its way during the products, which may use its place in LDS
      float smooth[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) smooth[k] = a.smooth[w * nv + (lane + 64 * k < nv ? lane + 64 * k : 0)];
      if (!unchanged) {
        StagedM<COLS == 2, WIDE ? 12 : 8, !MLDS> row;
        const float *M = a.M + w * a.ldM;
        const bool staged = !(MLDS && L.m_lds);
        jv_world<COLS == 2 ? 3 : 1>(
            a, Jw, nefc, L.rows, L.sv, a.jv + w * njmax, L.jv, lane,
            [&]() __attribute__((always_inline)) {
              if constexpr (!MLDS) row.load(M, a.nM, lane);
            },
            [&]() __attribute__((always_inline)) {
              if (staged)
                row.product(a, L.term, L.radr, M, a.nM, L.sv, a.mv + w * nv, L.mv, L.rows, lane);
              else
                mul_m_world<COLS == 2>(a, L.term, L.radr, L.m_lds, L.sv, a.mv + w * nv, L.mv, lane);
            });
        wave_sync();
      }
#pragma unroll
      for (int k = 0; k < 2; ++k)
        if (lane + 64 * k < nv) L.gl[lane + 64 * k] = smooth[k];
      for (int k = lane + 128; k < nv; k += 64) L.gl[k] = a.smooth[w * nv + k];
      wave_sync();
      IM_STAMP(1);
      // the rows' states before the step, on their way during the line search
      constexpr int kBefore = HELD == 2 ? 1 : 2;  // (two held rows a lane: 64 rows)
      int before[kBefore];
#pragma unroll
      for (int k = 0; k < kBefore; ++k) before[k] = a.state[w * njmax + (lane + 64 * k < nefc ? lane + 64 * k : 0)];
      // (the force list and the row list of the gradient are free until the step is taken)
      const search::LsWorld lw{L.gl, L.D, L.fl, L.Jaref, L.sv, L.mv, L.jv, L.Ma, sc.search_dot, tolerance,
                               ls_tolerance, meaninertia, ne, nf, nefc, nv, a.ls_iterations, L.f, (float *)L.rowl};
      const search::LsResult ls = search::linesearch_rows<HELD, true>(lw, lane & 31);  // both halves on this world
      sc.alpha = uniform(ls.alpha), sc.improvement = uniform(ls.improvement);
      if (lane == 0) {
        a.alpha[w] = ls.alpha;
        a.improvement[w] = ls.improvement;
        a.exhausted[w] = ls.exhausted ? 1 : 0;
        if (!ls.converged && a.overflow) a.overflow[w] = a.overflow[w] | a.ls_overflow_bit;
      }
      IM_STAMP(2);
      // the step (newton_stages.py:373-381), then force and state of every row from the new Jaref, the
      // rows whose being quadratic flipped (ascending) and the two counts (:385-444); the rows with a
      // force are listed for the gradient as they are formed
      const float al = ls.alpha;
      for (int i = lane; i < nv; i += 64) {
        const float q = fma_(al, L.sv[i], L.qacc[i]), v = fma_(al, L.mv[i], L.Ma[i]);
        L.qacc[i] = q;
        L.Ma[i] = v;
        a.qacc[w * nv + i] = q;
        a.Ma[w * nv + i] = v;
      }
      int nquad = 0, nstate = 0, cnt = 0;
      for (int base = 0; base < nefc; base += 64) {
        const int r = base + lane;
        bool quad_flip = false, changed = false;
        float f = 0.0f;
        if (r < nefc) {
          const float x = L.Jaref[r] + al * L.jv[r], d = L.D[r];
          L.Jaref[r] = x;
          a.Jaref[w * njmax + r] = x;
          f = -d * x;
          int st = 1;
          if (r >= ne && r < ne + nf) {
            const float fr = L.fl[r], rf = search::safe_div(fr, d);
            if (x <= -rf) f = fr, st = 2;
            else if (x >= rf) f = -fr, st = 3;
          } else if (r >= ne && x >= 0.0f) {
            f = 0.0f, st = 0;
          }
          const int old = base == 0 ? before[0] : base < 64 * kBefore ? before[kBefore - 1] : a.state[w * njmax + r];
          a.force[w * njmax + r] = f;
          a.state[w * njmax + r] = st;
          quad_flip = (old == 1) != (st == 1);
          changed = old != st;
        }
        const unsigned long long below = (1ull << lane) - 1ull;
        const unsigned long long m = __ballot(quad_flip);
        if (quad_flip) {
          const int slot = nquad + __popcll(m & below);
          if (slot < a.ld_ids) a.ids[w * (int64_t)a.ld_ids + slot] = r;
        }
        nquad += __popcll(m);
        nstate += __popcll(__ballot(changed));
        const unsigned long long mf = __ballot(f != 0.0f);
        if (f != 0.0f) {
          const int pos = cnt + __popcll(mf & below);
          L.f[pos] = f;
          L.rowl[pos] = r;
        }
        cnt += __popcll(mf);
      }
      nstate += ls.exhausted ? 1 : 0;
      if (lane == 0) {
        a.quad_count[w] = nquad;
        a.state_count[w] = nstate;
      }
      wave_sync();
      IM_STAMP(3);
      unchanged = gradient_world<COLS, COLS == 2 ? 4 : 2, COOP>(a, w, Jw, nstate != 0, cnt, L.f, L.rowl, L.Ma, L.gl, L.gl, sc, lane);
      IM_STAMP(4);
    }
    if (COOP) {
      block_sync();  // gradients, states and the `unchanged` bytes of the four worlds are in place; the rows of J are done with
      IM_STAMP(5);
      stage();
      block_sync();  // the four search directions are complete
    } else {
      wave_sync();
      if (!done && !unchanged) stage();
      wave_sync();
    }
    IM_STAMP(6);
    lane = lane_fixed;
    asm volatile("" : "+v"(lane));  // no address from before the stage is kept through it
    if (!done) {
      const NewtonArgs &a = kernel_args(kernarg_offset);
      if (!unchanged) {
        if (COOP) {
          search_sums_world(a, w, L.gl, L.sv, sc, lane);
        } else {  // the stage has left the direction and the two sums in memory: one trip for all
          const float dot = a.search_dot[w], decrement = a.decrement[w];
          for (int k = lane; k < nv; k += 64) L.sv[k] = a.search[w * nv + k];
          sc.search_dot = uniform(dot);
          sc.decrement = uniform(decrement);
        }
      }
      // newton_fusion.py:265-296
      sc.niter += 1;
      const float scale = meaninertia * (float)nv;
      const bool converged = sc.alpha == 0.0f || (sc.improvement > 0.0f && sc.improvement / scale < tolerance) ||
                             sqrtf(sc.grad_dot) / scale < tolerance || 0.5f * sc.decrement / scale < tolerance;
      const bool finished = converged || sc.niter == a.maxiter;
      if (lane == 0) {
        a.niter[w] = sc.niter;
        if (finished) {
          if (!converged && a.overflow) a.overflow[w] = a.overflow[w] | a.iter_overflow_bit;
          a.done[w] = 1;
          a.unchanged[w] = 1;
          if (a.nsolving) atomicAdd(a.nsolving, -1);
        }
      }
      if (finished && a.final_force)
        for (int k = lane; k < nv; k += 64) {
          const float g = sc.grad_scale * a.grad[w * a.ld_grad + k];
          a.qfrc_constraint[w * nv + k] = L.Ma[k] - a.smooth[w * nv + k] - g;
        }
      budget -= 1;
      done = finished || budget <= 0;
    }
    IM_STAMP(7);
  }
#ifdef IM_NEWTON_STAMPS
  if (live && lane_fixed < 8) a0.jv[w * njmax + lane_fixed] = (float)t_phase[lane_fixed];
#endif
#undef IM_STAMP
}

// The layout behind a cooperative stage's area of `a.stage_lds_floats` words (the staged rows of J
// use that area between two stages): four flags, the row tables of M v, then each of the four
// wavefronts' own arrays.  Fills the tables; the caller synchronises the workgroup before the loop.
__device__ __forceinline__ LoopLds coop_layout(const NewtonArgs &a, float *lds) {
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int nv = a.nv, njmax = a.njmax, nM = a.m_lds ? a.nM : 0;
  LoopLds L;
  L.votes = (int *)(lds + a.stage_lds_floats);
  L.worlds = L.votes + 4;
  uint32_t *term = (uint32_t *)(L.worlds + 4);
  int *radr = (int *)(term + a.nterm);
  float *mine = lds + ((a.stage_lds_floats + 8 + a.nterm + nv + 1 + 3) & ~3) + wv * coop_wave_words(nv, njmax, nM);
  L.term = term, L.radr = radr;
  L.sv = mine;
  L.Ma = L.sv + nv;
  L.mv = L.Ma + nv;
  L.qacc = L.mv + nv;
  L.Jaref = L.qacc + nv;
  L.jv = L.Jaref + njmax;
  L.D = L.jv + njmax;
  L.fl = L.D + njmax;
  L.f = L.fl + njmax;
  L.rowl = (int *)(L.f + njmax);
  L.gl = (float *)(L.rowl + njmax);
  L.m_lds = a.m_lds ? L.gl + nv : nullptr;
  L.rows = lds + wv * kTileWords;
  for (int k = threadIdx.x; k < a.nterm; k += blockDim.x) term[k] = (uint32_t)a.mulm_col[k] | (uint32_t)a.mulm_madr[k] << 16;
  for (int k = threadIdx.x; k <= nv; k += blockDim.x) radr[k] = a.mulm_rowadr[k];
  return L;
}

}  // namespace resident
}  // namespace im
