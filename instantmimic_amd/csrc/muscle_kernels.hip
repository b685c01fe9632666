// Muscle moment-arm contractions for gfx950.
//
//   tau[w, root + j]  = sum over the entries e of torque dof j (torque-sorted order) of
//                       A[w, e] * f[w, muscle(e)]
//     reference: src/instantmimic/muscle/muscle_qfrc_projector.py:2941-2961
//   qDeriv[w, elem]  += h * sum over the element's chunks of 16 pairs, in order, of
//                       (s[w, muscle(i)] * A[w, i]) * A[w, j]
//     reference: muscle_qfrc_projector.py:736-774 (one block per world, no atomics)
//
// Both are bandwidth bound: a world's moment row (a few KB) is read once, staged in
// LDS, and gathered from there.  Summation order and fused multiply-adds follow the
// reference (Warp lowers `total += a * b` to one fma under NVRTC's default contraction).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "common.h"
#include "newton_solve.h"

namespace im {
namespace {

__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// One workgroup of NT threads per world.  A and the force of every term are first brought
// into LDS in the order the rows consume them (every lane busy, UN terms' look-ups in flight
// per lane); then lane j of the first wavefront runs row j's chain of fused multiply-adds over
// consecutive LDS words, the next eight terms on their way while these are added.  Same terms,
// same order per row as the reference kernel.
// What bounds it is the longest row's chain (hundreds of terms, one after the other) and the
// staging before it, not the 46 MB: the chain looked a term's muscle up and then its force, two
// LDS latencies per four terms, and rigs of more than 1536 entries gathered from memory.
// Two wavefronts with twelve terms a lane that looked a term's muscle up in the chain -> this, with the
// smallest NT x UN that takes the entries in one trip (places without an entry cost what the others do), x 8192
// worlds: 355 entries 11.1 -> 7.8 us (256 x 12: 14.1), 743 16.7 -> 14.3 (18.8), 1437 27.7 -> 24.8 (27.1),
// 2522 59.5 -> 39.3.
template <int NT, int UN>
__global__ __launch_bounds__(NT) void muscle_project_kernel(
    const float *__restrict__ moment, int64_t ldm, const float *__restrict__ force, int64_t ldf,
    const int32_t *__restrict__ offsets, const int32_t *__restrict__ entry_idx,
    const int32_t *__restrict__ entry_muscle, int nentry, int nmuscle, int ntorque, int root,
    float *__restrict__ qfrc, int64_t ldq, int nworld) {
  extern __shared__ float lds[];
  const int tid = threadIdx.x;
  const int64_t w = blockIdx.x;
  float *av = lds;           // [nentry] A[entry_idx[s]]
  float *fv = av + nentry;   // [nentry] the force of its muscle; in between its entry_muscle
  float *fs = fv + nentry;   // [nmuscle] the world's forces
  int *ms = (int *)fv;
  const float *mw = moment + w * ldm, *fw = force + w * ldf;
  // Every array is read from memory in its own order (coalesced); the permutation into the
  // rows' order goes through LDS, in place: gather into registers, barrier, write back.
  for (int i = tid; i < nmuscle; i += NT) fs[i] = fw[i];
  if (nentry <= UN * NT) {
    int e[UN], m[UN];
    float x[UN], f[UN];
#pragma unroll
    for (int k = 0; k < UN; ++k) {
      const int i = tid + NT * k < nentry ? tid + NT * k : nentry - 1;
      e[k] = entry_idx[i];
      m[k] = entry_muscle[i];
      x[k] = mw[i];
    }
#pragma unroll
    for (int k = 0; k < UN; ++k)
      if (tid + NT * k < nentry) {
        av[tid + NT * k] = x[k];
        ms[tid + NT * k] = m[k];
      }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < UN; ++k) {
      x[k] = av[e[k]];
      f[k] = fs[ms[e[k]]];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < UN; ++k)
      if (tid + NT * k < nentry) {
        av[tid + NT * k] = x[k];
        fv[tid + NT * k] = f[k];
      }
  } else {
    // more entries than one trip holds: gathered from memory, UN look-ups in flight per lane
    __syncthreads();
    for (int s0 = tid; s0 < nentry; s0 += UN * NT) {
      int e[UN], m[UN];
      float x[UN];
#pragma unroll
      for (int k = 0; k < UN; ++k) e[k] = entry_idx[s0 + NT * k < nentry ? s0 + NT * k : nentry - 1];
#pragma unroll
      for (int k = 0; k < UN; ++k) {
        m[k] = entry_muscle[e[k]];
        x[k] = mw[e[k]];
      }
#pragma unroll
      for (int k = 0; k < UN; ++k)
        if (s0 + NT * k < nentry) {
          av[s0 + NT * k] = x[k];
          fv[s0 + NT * k] = fs[m[k]];
        }
    }
  }
  __syncthreads();
  for (int j = tid; j < ntorque; j += NT) {
    float total = 0.0f;
    const int e1 = offsets[j + 1];
    int s = offsets[j];
    if (s + 8 <= e1) {
      float a[8], f[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) a[k] = av[s + k], f[k] = fv[s + k];
      for (s += 8; s + 8 <= e1; s += 8) {
        float an[8], fn[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) an[k] = av[s + k], fn[k] = fv[s + k];
#pragma unroll
        for (int k = 0; k < 8; ++k) total = fma_(a[k], f[k], total);
#pragma unroll
        for (int k = 0; k < 8; ++k) a[k] = an[k], f[k] = fn[k];
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) total = fma_(a[k], f[k], total);
    }
    for (; s < e1; ++s) total = fma_(av[s], fv[s], total);
    qfrc[w * ldq + root + j] = total;
  }
}

// One workgroup (of 256 threads, or 512 where its LDS is large) for W worlds side by side, a value of each next to one
// another in LDS: a chunk's sixteen packed pairs (64 KB of tables at 284 muscles, more than a CU's cache holds beside the
// worlds') are read and taken apart once for W products.
template <int W>
__global__ __launch_bounds__(512) void muscle_gather_kernel(
    const float *__restrict__ moment, int64_t ldm, const float *__restrict__ slope, int64_t lds_,
    const int32_t *__restrict__ entry_muscle, int nentry, const int32_t *__restrict__ elem_ids,
    int nelem, const int32_t *__restrict__ chunk_offsets, const int32_t *__restrict__ chunk_pairs,
    int chunk_count, float timestep, float *__restrict__ qderiv, int64_t ldq, int nworld) {
  typedef float vec __attribute__((ext_vector_type(W)));
  extern __shared__ __align__(16) float lds[];
  vec *m = (vec *)lds;                   // [nentry + 1]
  vec *weighted = m + nentry + 1;        // [nentry + 1]
  vec *partial = weighted + nentry + 1;  // [chunk_count]
  const int lane = threadIdx.x, width = blockDim.x;
  const int64_t w0 = (int64_t)blockIdx.x * W;
  int64_t w[W];  // (a batch's remainder: its last world again)
#pragma unroll
  for (int u = 0; u < W; ++u) w[u] = w0 + u < nworld ? w0 + u : nworld - 1;
  constexpr int N = 8 / W;
  for (int e0 = lane; e0 < nentry; e0 += N * width) {  // eight values' loads in flight per lane
    vec v[N], sl[N];
    int mu[N];
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const int e = e0 + k * width < nentry ? e0 + k * width : nentry - 1;
      mu[k] = entry_muscle[e];
#pragma unroll
      for (int u = 0; u < W; ++u) v[k][u] = moment[w[u] * ldm + e];
    }
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
      for (int u = 0; u < W; ++u) sl[k][u] = slope[w[u] * lds_ + mu[k]];
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const int e = e0 + k * width;
      if (e < nentry) {
        m[e] = v[k];
        weighted[e] = sl[k] * v[k];
      }
    }
  }
  if (lane == 0) m[nentry] = weighted[nentry] = vec(0.0f);
  __syncthreads();
  for (int c = lane; c < chunk_count; c += width) {
    vec total = vec(0.0f);
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int packed = chunk_pairs[(size_t)k * chunk_count + c];
      const vec a = weighted[packed & 0xFFFF], b = m[packed >> 16];
#pragma unroll
      for (int u = 0; u < W; ++u) total[u] = fma_(a[u], b[u], total[u]);
    }
    partial[c] = total;
  }
  __syncthreads();
  for (int slot = lane; slot < nelem; slot += width) {
    vec acc = vec(0.0f);
    const int c1 = chunk_offsets[slot + 1], at = elem_ids[slot];
    float q0[W];  // requested before the sum, used after it
#pragma unroll
    for (int u = 0; u < W; ++u) q0[u] = qderiv[w[u] * ldq + at];
    for (int c = chunk_offsets[slot]; c < c1; ++c) acc = acc + partial[c];
#pragma unroll
    for (int u = 0; u < W; ++u)
      if (u == 0 || w0 + u < nworld) qderiv[w[u] * ldq + at] = fma_(timestep, acc[u], q0[u]);
  }
}

}  // namespace
}  // namespace im

extern "C" {

int im_muscle_project(const float *moment, int64_t ld_moment, const float *force, int64_t ld_force,
                      const int32_t *torque_entry_offsets, const int32_t *torque_entry_idx,
                      const int32_t *entry_muscle, int nentry, int nmuscle, int ntorque,
                      int root_dof_count, float *qfrc, int64_t ld_qfrc, int nworld, void *stream) {
  if (nworld < 0 || nentry < 0 || ntorque < 0) return IM_ERR_ARG;
  if (nworld == 0 || ntorque == 0) return IM_OK;
  if (nentry == 0) return IM_ERR_ARG;  // entry indices are clamped to nentry - 1
  if (!moment || !force || !torque_entry_offsets || !torque_entry_idx || !entry_muscle || !qfrc) return IM_ERR_ARG;
  if (ld_moment < nentry || ld_force < nmuscle || ld_qfrc < root_dof_count + ntorque) return IM_ERR_STRIDE;
  if (nmuscle > 65535) return IM_ERR_UNSUPPORTED;  // muscle ids travel as 16 bits
  // the limit is that of a term in six bytes, which a caller has to reckon with; a term takes eight
  if (sizeof(float) * ((size_t)nentry + nmuscle) + 2 * (((size_t)nentry + 1) & ~(size_t)1) > 64 * 1024) return IM_ERR_UNSUPPORTED;
  const size_t lds_bytes = sizeof(float) * (2 * (size_t)nentry + nmuscle);
#define IM_PROJECT(NT, UN)                                                                                                        \
  do {                                                                                                                            \
    if (lds_bytes > 64 * 1024)                                                                                                    \
      IM_HIP_CHECK(hipFuncSetAttribute((const void *)im::muscle_project_kernel<NT, UN>, hipFuncAttributeMaxDynamicSharedMemorySize, \
                                       (int)lds_bytes));                                                                          \
    hipLaunchKernelGGL((im::muscle_project_kernel<NT, UN>), dim3(nworld), dim3(NT), lds_bytes, (hipStream_t)stream, moment,       \
                       ld_moment, force, ld_force, torque_entry_offsets, torque_entry_idx, entry_muscle, nentry, nmuscle,         \
                       ntorque, root_dof_count, qfrc, ld_qfrc, nworld);                                                           \
  } while (0)
  if (nentry <= 4 * 128) IM_PROJECT(128, 4);
  else if (nentry <= 8 * 128) IM_PROJECT(128, 8);
  else if (nentry <= 12 * 128) IM_PROJECT(128, 12);
  else if (nentry <= 8 * 256) IM_PROJECT(256, 8);
  else IM_PROJECT(256, 12);
#undef IM_PROJECT
  IM_HIP_CHECK(hipGetLastError());
  return IM_OK;
}

int im_muscle_gather_tables(const int32_t *pair_elem_id, const int32_t *pair_entry_i, const int32_t *pair_entry_j,
                            int npair, int nentry, int32_t *elem_ids, int32_t *chunk_offsets, int32_t *chunk_pairs,
                            int *nelem, int *chunk_count) {
  if (npair < 0 || nentry < 0 || !nelem || !chunk_count || (npair > 0 && !pair_elem_id)) return IM_ERR_ARG;
  if (nentry >= 0x7FFF) return IM_ERR_UNSUPPORTED;  // two entry indices share one int32
  // pairs in the order of their M element, ties in list order
  std::vector<int> order(npair);
  for (int q = 0; q < npair; ++q) order[q] = q;
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return pair_elem_id[a] < pair_elem_id[b]; });
  // first pass: elements and their chunks of 16 pairs
  int elems = 0, chunks = 0;
  for (int q = 0; q < npair;) {
    int end = q;
    while (end < npair && pair_elem_id[order[end]] == pair_elem_id[order[q]]) ++end;
    if (elem_ids) elem_ids[elems] = pair_elem_id[order[q]];
    if (chunk_offsets) chunk_offsets[elems] = chunks;
    chunks += (end - q + 15) / 16;
    ++elems;
    q = end;
  }
  if (chunk_offsets) chunk_offsets[elems] = chunks;
  *nelem = elems;
  *chunk_count = chunks;
  if (!chunk_pairs) return IM_OK;
  if (!pair_entry_i || !pair_entry_j || !chunk_offsets) return IM_ERR_ARG;
  // second pass: pair k of chunk c at k * chunk_count + c, the padding names entry `nentry` twice
  for (size_t v = 0; v < (size_t)16 * chunks; ++v) chunk_pairs[v] = nentry | (nentry << 16);
  int slot = 0, rank = 0;
  for (int q = 0; q < npair; ++q) {
    if (q > 0 && pair_elem_id[order[q]] != pair_elem_id[order[q - 1]]) {
      ++slot;
      rank = 0;
    }
    const int i = pair_entry_i[order[q]], j = pair_entry_j[order[q]];
    if (i < 0 || j < 0 || i >= nentry || j >= nentry) return IM_ERR_ARG;
    chunk_pairs[(size_t)(rank % 16) * chunks + chunk_offsets[slot] + rank / 16] = i | (j << 16);
    ++rank;
  }
  return IM_OK;
}

int im_muscle_implicit_gather(const float *moment, int64_t ld_moment, const float *slope, int64_t ld_slope,
                              const int32_t *entry_muscle, int nentry, const int32_t *elem_ids, int nelem,
                              const int32_t *chunk_offsets, const int32_t *chunk_pairs, int chunk_count,
                              float timestep, float *qderiv, int64_t ld_qderiv, int nworld, void *stream) {
  if (nworld < 0 || nentry < 0 || nelem < 0 || chunk_count < 0) return IM_ERR_ARG;
  if (nworld == 0 || nelem == 0) return IM_OK;
  if (!moment || !slope || !entry_muscle || !elem_ids || !chunk_offsets || !chunk_pairs || !qderiv) return IM_ERR_ARG;
  if (nentry >= 0x7FFF) return IM_ERR_UNSUPPORTED;  // two entry indices share one int32
  if (ld_moment < nentry) return IM_ERR_STRIDE;
  const size_t lds_bytes = sizeof(float) * (2 * ((size_t)nentry + 1) + chunk_count);
  if (lds_bytes > 64 * 1024) return IM_ERR_UNSUPPORTED;
  // Two worlds where a CU holds two such workgroups and the batch has two worlds for every CU; 512 threads where their LDS
  // leaves a CU three workgroups.  4096 worlds of 2522 entries, 1038 chunks: a world 34.2 us, two 32.0, two on 512 threads
  // 23.8.  A world / two by batch (256 CUs), us: 355 entries x 256 5.1 / 5.3, x 512 5.8 / 5.3, x 2047 9.1 / 7.5, x 8192
  // 26.4 / 17.1; 1077 entries x 256 5.6 / 6.2, x 512 6.5 / 6.5, x 1024 8.2 / 7.8; 2522 x 512 9.1 / 6.9, x 1024 12.2 / 8.7.
  // By LDS, x 4096: two of 61 KB 42.9 / 32.6, 72 KB 48.2 / 34.4, 78 KB 53.7 / 37.5; beyond, one to a CU, 85 KB 67.7 / 59.5
  // but 87 KB with fewer chunks 56.9 / 57.9.
  int ncu = 0;
  if (const int st = im::compute_units(&ncu)) return st;
  const bool two = nworld >= 2 * ncu && 2 * lds_bytes <= 80 * 1024;
  auto kernel = two ? im::muscle_gather_kernel<2> : im::muscle_gather_kernel<1>;
  const size_t bytes = two ? 2 * lds_bytes : lds_bytes;
  if (bytes > 64 * 1024) IM_HIP_CHECK(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
  hipLaunchKernelGGL(kernel, dim3(two ? (nworld + 1) / 2 : nworld), dim3(two && bytes > 27 * 1024 ? 512 : 256), bytes, (hipStream_t)stream, moment,
                     ld_moment, slope, ld_slope, entry_muscle, nentry, elem_ids, nelem, chunk_offsets, chunk_pairs,
                     chunk_count, timestep, qderiv, ld_qderiv, nworld);
  IM_HIP_CHECK(hipGetLastError());
  return IM_OK;
}

}  // extern "C"
