// Muscle path geometry and activation <-> joint-torque contractions for gfx950.
//
//   waypoints[w, i]   = xpos[w, body(i)] + rot(local(i), normalize(xquat[w, body(i)]))
//     reference: src/instantmimic/muscle/muscle_dynamics_kernels.py:73-86
//   unit/passive force magnitudes per (world, muscle) from the polyline length
//     reference: muscle_dynamics_kernels.py:644-705, curves muscle_qfrc_projector.py:103-277
//   torque[w, j]      = sum over the active (segment, muscle) entries of torque dof j of
//                       contribution(segment, dof j, unit * activation (+ passive))
//     reference: muscle_dynamics_kernels.py:1707-1793
//   grad_act[w, m]    = sum over muscle m's (segment, torque) entries of
//                       grad_out[w, j] * contribution(segment, dof j, unit)
//     reference: muscle_dynamics_kernels.py:1796-1859
//   moment[w, e]      = sum over entry e's segments of contribution(segment, dof(e), 1)
//     reference: muscle_qfrc_projector.py:2617-2662
//   contribution      = dot(a (lin + ang x (p0 - c0)) - b (lin + ang x (p1 - c1)), f dir)
//     reference: muscle_qfrc_projector.py:280-304
//
// All five are gathers over a world's row of poses (a few KB) and reuse nothing across worlds.  Their bytes would
// pass in a tenth of the time: what bounds each is instructions or the trips within a world, and stands at its
// kernel.  Threads are laid out output-major inside a world so that a wavefront's writes coalesce.  Arithmetic is written out operation by operation
// (this file is compiled without floating-point contraction) and the CPU oracle follows
// the same order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>

#include "../../include/imhip.h"
#include "common.h"
#include "newton_solve.h"

namespace im {
namespace {

// A workgroup per world up to what the chip keeps resident at once (the workgroups walk over worlds: one that
// does not get in starts when another has done all its worlds, and the launch takes up to twice as long).
// Less than the runtime's answer in two ways: a CU hands out its LDS in units of 1280 bytes, and the scalar registers
// (85 - 106) of most of these kernels leave 24 wavefronts to a CU (`waves`; 32 with up to 96).  Force-velocity state of 8192 worlds by workgroups per
// CU: 128 threads, 12: 20.1 us, 13: 23.3; 192 threads, 8: 25.6, 9: 32.5; 256 threads, 6: 47.1, 7: 61.1; 320
// threads, 4: 68.8, 5: 93.3.
int resident_grid(const void *fn, int threads, size_t lds, int nworld, unsigned *grid, int waves = 24) {
  int ncu = 0, per_cu = 0;
  if (const int st = compute_units(&ncu)) return st;
  if (const int st = resident_per_cu(fn, nullptr, threads, lds, &per_cu)) return st;
  const size_t unit = 1280, granted = (std::max<size_t>(lds, 1) + unit - 1) / unit * unit;
  per_cu = std::min({per_cu, (int)(160 * 1024 / granted), waves * 64 / threads});
  *grid = (unsigned)std::min(nworld, ncu * std::max(1, per_cu));
  return IM_OK;
}

struct V3 {
  float x, y, z;
};
__device__ __forceinline__ V3 ld3(const float *p) { return {p[0], p[1], p[2]}; }
__device__ __forceinline__ V3 sub(V3 a, V3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ V3 add(V3 a, V3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ V3 scale(float s, V3 a) { return {s * a.x, s * a.y, s * a.z}; }
__device__ __forceinline__ float dot(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ V3 cross(V3 a, V3 b) {
  return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ float length(V3 a) { return sqrtf(dot(a, a)); }

// muscle_qfrc_projector.py:280-304
__device__ __forceinline__ float contribution(V3 lin, V3 ang, V3 p0, V3 p1, V3 c0, V3 c1, float a,
                                              float b, float force) {
  const V3 seg = sub(p1, p0);
  const float len = length(seg);
  if (len < 1.0e-8f) return 0.0f;
  const V3 dir = {seg.x / len, seg.y / len, seg.z / len};
  const V3 f = scale(force, dir);
  const V3 st = add(lin, cross(ang, sub(p0, c0)));
  const V3 en = add(lin, cross(ang, sub(p1, c1)));
  return dot(sub(scale(a, st), scale(b, en)), f);
}

struct Geo {
  const float *wp, *com, *cdof;
  int64_t ldw, ldc, ldd;
};
struct Seg {
  const int32_t *p0, *p1, *b0, *b1;
};

__device__ __forceinline__ float seg_term(const Geo &g, const Seg &s, int64_t w, int seg, V3 lin,
                                          V3 ang, float a, float b, float force) {
  const float *wp = g.wp + w * g.ldw, *com = g.com + w * g.ldc;
  return contribution(lin, ang, ld3(wp + 3 * s.p0[seg]), ld3(wp + 3 * s.p1[seg]),
                      ld3(com + 3 * s.b0[seg]), ld3(com + 3 * s.b1[seg]), a, b, force);
}

// A body's renormalised quaternion as the rotation uses it: vector part u, s s - u.u and 2 s.
struct BodyTurn {
  V3 u;
  float k, s2;
};
__device__ __forceinline__ BodyTurn body_turn(const float *__restrict__ q) {
  const float q0 = q[0], q1 = q[1], q2 = q[2], q3 = q[3];
  // muscle_qfrc_projector.py:91-100
  const float inv = 1.0f / sqrtf(q0 * q0 + q1 * q1 + q2 * q2 + q3 * q3 + 1.0e-8f);
  const float s = q0 * inv;
  const V3 u = {q1 * inv, q2 * inv, q3 * inv};
  return {u, s * s - dot(u, u), 2.0f * s};
}
// mujoco_warp math.rot_vec_quat: 2 (u.v) u + (s s - u.u) v + 2 s (u x v)
__device__ __forceinline__ V3 turned(const BodyTurn &t, V3 v) {
  const V3 r = add(scale(2.0f, scale(dot(t.u, v), t.u)), scale(t.k, v));
  return add(r, scale(t.s2, cross(t.u, v)));
}
// One waypoint in the world frame: the body's position plus its local offset turned by the
// body's quaternion.  xpos and xquat are one world's rows.
__device__ __forceinline__ V3 world_waypoint(const float *__restrict__ xpos,
                                             const float *__restrict__ xquat,
                                             const int32_t *__restrict__ wp_body,
                                             const float *__restrict__ wp_local, int i) {
  const int b = wp_body[i];
  return add(ld3(xpos + 3 * b), turned(body_turn(xquat + 4 * b), ld3(wp_local + 3 * i)));
}

__global__ __launch_bounds__(256) void waypoints_kernel(
    const float *__restrict__ xpos, int64_t ldp, const float *__restrict__ xquat, int64_t ldq,
    const int32_t *__restrict__ wp_body, const float *__restrict__ wp_local, int nwp,
    float *__restrict__ out, int64_t ldo, int nworld) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t w = blockIdx.y;
  if (i >= nwp) return;
  const V3 p = world_waypoint(xpos + w * ldp, xquat + w * ldq, wp_body, wp_local, i);
  float *o = out + w * ldo + 3 * i;
  o[0] = p.x;
  o[1] = p.y;
  o[2] = p.z;
}

// muscle_qfrc_projector.py:103-187
__device__ __forceinline__ float active_fl(float l, const float *m) {
  if (m[0] < 0.5f) return expf(-((l - 1.0f) * (l - 1.0f)) / m[1]);
  const float lmin = m[1], lmax = m[2];
  if (l < lmin || l > lmax) return 0.0f;
  const float lo = 0.5f * (lmin + 1.0f), hi = 0.5f * (1.0f + lmax);
  if (l <= lo) {
    const float x = (l - lmin) / fmaxf(lo - lmin, 1.0e-8f);
    return 0.5f * x * x;
  }
  if (l <= 1.0f) {
    const float x = (1.0f - l) / fmaxf(1.0f - lo, 1.0e-8f);
    return 1.0f - 0.5f * x * x;
  }
  if (l <= hi) {
    const float x = (l - 1.0f) / fmaxf(hi - 1.0f, 1.0e-8f);
    return 1.0f - 0.5f * x * x;
  }
  const float x = (lmax - l) / fmaxf(lmax - hi, 1.0e-8f);
  return 0.5f * x * x;
}
// (scale: expf(m[1]) - 1, read for the exponential curve only)
__device__ __forceinline__ float passive_fl(float l, const float *m, float scale) {
  if (m[0] < 0.5f) {
    if (l < 1.0f) return 0.0f;
    float x = m[1] * (l - 1.0f) / m[2];
    x = fminf(fmaxf(x, -80.0f), 80.0f);
    return (expf(x) - 1.0f) / scale;
  }
  const float lmax = m[1], fpmax = m[2];
  if (l <= 1.0f) return 0.0f;
  const float mid = 0.5f * (1.0f + lmax), width = fmaxf(mid - 1.0f, 1.0e-8f);
  if (l <= mid) {
    const float st = (l - 1.0f) / width;
    return 0.5f * fpmax * st * st;
  }
  return fpmax * (0.5f + (l - mid) / width);
}

// Force magnitudes of a muscle of length len (par: f0, l_m0, l_t0, ..; c: its pennation's cosine).
__device__ __forceinline__ void force_of_length(float len, const float *__restrict__ par, float rest, float c, float passive_scale,
                                                const im_muscle_force_model &model, float *unit, float *passive) {
  const float f0 = par[0], lm0 = par[1], lt0 = par[2];
  // muscle_qfrc_projector.py:190-205
  const float lm = len / fmaxf(rest, 1.0e-6f) - lt0;
  const float ln =
      fminf(fmaxf(lm / fmaxf(lm0, 1.0e-6f), model.length_norm_min), model.length_norm_max);
  *unit = f0 * active_fl(ln, model.active) * c * model.force_scale;
  if (passive) {
    float pv = 0.0f;
    // muscle_qfrc_projector.py:249-277 with include_active 0, include_passive 1
    if (model.include_passive)
      pv = f0 * passive_fl(ln, model.passive, passive_scale) * c * model.force_scale;
    *passive = pv;
  }
}
// Length of muscle m along one world's waypoints and its force magnitudes.
__device__ __forceinline__ void muscle_force_magnitudes(
    const float *row, const int32_t *__restrict__ seg_start,
    const int32_t *__restrict__ seg_offsets, const float *__restrict__ params, int ldpar,
    const float *__restrict__ rest, const im_muscle_force_model &model, int m, float *unit,
    float *passive) {
  float len = 0.0f;  // muscle_dynamics_kernels.py:452-473
  for (int s = seg_offsets[m]; s < seg_offsets[m + 1]; ++s) {
    const int i = seg_start[s];
    len = len + length(sub(ld3(row + 3 * (i + 1)), ld3(row + 3 * i)));
  }
  force_of_length(len, params + m * ldpar, rest[m], cosf(params[m * ldpar + 3]),
                  passive && model.include_passive ? expf(model.passive[1]) - 1.0f : 1.0f, model, unit, passive);
}

// MuJoCo's force-velocity multiplier and its derivative in the normalised velocity
// (muscle_qfrc_projector.py:2505-2524)
__device__ __forceinline__ void force_velocity_curve(float v, float fvmax, float *mult, float *slope) {
  const float y = fvmax - 1.0f;
  if (v <= -1.0f) {
    *mult = 0.0f;
    *slope = 0.0f;
  } else if (v <= 0.0f) {
    const float shifted = v + 1.0f;
    *mult = shifted * shifted;
    *slope = 2.0f * shifted;
  } else if (v <= y) {
    const float remaining = y - v;
    *mult = fvmax - remaining * remaining / y;
    *slope = 2.0f * remaining / y;
  } else {
    *mult = fvmax;
    *slope = 0.0f;
  }
}

// eval_muscle_force_velocity_state_kernel (muscle_qfrc_projector.py:2816-2884): one muscle of
// one world -- its length over consecutive waypoints, its lengthening velocity -sum moment qvel
// over its (muscle, dof) entries, and the force-velocity response (:2528-2570).
__global__ __launch_bounds__(256) void force_velocity_state_kernel(
    const float *__restrict__ wp, int64_t ldw, const int32_t *__restrict__ waypoint_start,
    const float *__restrict__ params, int ldpar, const float *__restrict__ rest,
    const float *__restrict__ length_scale, const float *__restrict__ activation, int64_t lda,
    const float *__restrict__ qvel, int64_t ldq, const float *__restrict__ moment, int64_t ldm,
    const int32_t *__restrict__ dof_offsets, const int32_t *__restrict__ dof_torque_idx, int root,
    im_muscle_force_model model, im_muscle_force_velocity_model fv, int nmuscle, float *__restrict__ out_length,
    float *__restrict__ out_activation, float *__restrict__ out_velocity, float *__restrict__ out_multiplier,
    float *__restrict__ out_slope, int64_t ldo) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t w = blockIdx.y;
  if (m >= nmuscle) return;
  const float *row = wp + w * ldw;
  float len = 0.0f;
  for (int i = waypoint_start[m]; i < waypoint_start[m + 1] - 1; ++i)
    len = len + length(sub(ld3(row + 3 * (i + 1)), ld3(row + 3 * i)));
  float velocity = 0.0f;
  for (int e = dof_offsets[m]; e < dof_offsets[m + 1]; ++e)
    velocity = __builtin_fmaf(-moment[w * ldm + e], qvel[w * ldq + dof_torque_idx[e] + root], velocity);
  const float f0 = params[m * ldpar], lm0 = params[m * ldpar + 1], lt0 = params[m * ldpar + 2],
              pen = params[m * ldpar + 3];
  const float velocity_scale = fmaxf(length_scale[m] * fv.vmax, 1.0e-6f);
  float mult, dmult;
  force_velocity_curve(velocity / velocity_scale, fv.fvmax, &mult, &dmult);
  float active = activation[w * lda + m];
  if (fv.clamp_activation != 0.0f) active = fminf(fmaxf(active, 0.0f), 1.0f);
  const float lm = len / fmaxf(rest[m], 1.0e-6f) - lt0;
  const float ln = fminf(fmaxf(lm / fmaxf(lm0, 1.0e-6f), model.length_norm_min), model.length_norm_max);
  const float unit = f0 * active_fl(ln, model.active) * cosf(pen) * model.force_scale;
  out_length[w * ldo + m] = len;
  out_activation[w * ldo + m] = active * mult;
  out_velocity[w * ldo + m] = velocity;
  out_multiplier[w * ldo + m] = mult;
  out_slope[w * ldo + m] = fv.include_active * active * unit * dmult / velocity_scale;
}

// The same with a workgroup per world, resident over worlds.  What bounds it is latency, not
// traffic: a lane of the kernel above walks a few 12-byte waypoints and a few scattered entries
// of its own, a cache line per request, and its velocity is a chain of look-ups.  Here a world's
// waypoints, moment entries and velocities come into LDS with eight coalesced loads in flight
// per thread; the distances between neighbouring waypoints are taken by all threads side by side
// (a lane per muscle left the wavefront waiting for its longest muscle's roots); and what does
// not depend on the world (an entry's dof, a muscle's cos(pennation)) is left in LDS once.  Same
// operations in the same order, so the same bits.
// As many threads as it takes for a muscle each, 128 to 320: a workgroup's last phase is its muscles'
// chains, and threads beyond them only take a CU's places from other worlds (8192 worlds of 40 / 100 / 200
// muscles: 20.3 / 31.0 / 47.6 us, with 320 threads 50 / 59 / 68).  A launch per world with 256 threads,
// distances by the muscle's lane, took 23.1 / 39.2 / 59.1 us there, and 57.5 at 284 muscles x 4096 worlds, here 38.3;
// it is ahead where the whole batch is resident at once (2048 worlds of 40 / 100 / 200 muscles 6.7 / 9.5 / 17.8 us,
// here 7.6 / 11.2 / 19.2).
struct FvLds {
  int words_wp, nentry, nqvel, nmuscle;  // the longest rows that fit; what is read of them is what the tables name
  __host__ __device__ int bytes() const {
    return 4 * (words_wp + nentry + nqvel + words_wp / 3 + nmuscle + 1) + 2 * ((nentry + 1) & ~1);
  }
};

template <int nt>
__device__ __forceinline__ void stage_row(float *to, const float *__restrict__ from, int n, int tid) {
  int i = tid;
  for (; i + 7 * nt < n; i += 8 * nt) {
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = from[i + k * nt];
#pragma unroll
    for (int k = 0; k < 8; ++k) to[i + k * nt] = v[k];
  }
  if (i < n) {
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = from[min(i + k * nt, n - 1)];
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (i + k * nt < n) to[i + k * nt] = v[k];
  }
}

// What a muscle's sums and curves take that does not depend on the world: its distances i0 .. i1 - 1, its entries
// e0 .. e1 - 1, and its parameters with their lower bounds applied.
struct FvMuscle {
  int i0, i1, e0, e1;
  float f0, lt0, lm0, rest, velocity_scale;
};

// AHEAD: a thread holds its share of the next world's rows in registers while it works on this one's (rows of up to 14
// floats a thread of waypoints, nine of moments, one of velocities: every rig whose muscles have the threads they ask
// for; wider rows are fetched when the world before is done with).  A workgroup's trip to memory was in front of its
// two other phases: 4096 worlds of 284 muscles 48.5 -> 43.3 us, implicit terms of 300 muscles x 8192 worlds 315 -> 303.
// Its muscle's bounds and parameters stay in its registers and the next activation comes along with the rows, and both
// sums ask four terms ahead: implicit terms of 284 muscles x 4096 worlds 143.0 -> 140.2 us.
template <int nt, bool AHEAD>
__global__ __launch_bounds__(nt) void force_velocity_state_world_kernel(
    const float *__restrict__ wp, int64_t ldw, const int32_t *__restrict__ waypoint_start,
    const float *__restrict__ params, int ldpar, const float *__restrict__ rest,
    const float *__restrict__ length_scale, const float *__restrict__ activation, int64_t lda,
    const float *__restrict__ qvel, int64_t ldq, const float *__restrict__ moment, int64_t ldm,
    const int32_t *__restrict__ dof_offsets, const int32_t *__restrict__ dof_torque_idx, int root,
    im_muscle_force_model model, im_muscle_force_velocity_model fv, FvLds n, float *__restrict__ out_length,
    float *__restrict__ out_activation, float *__restrict__ out_velocity, float *__restrict__ out_multiplier,
    float *__restrict__ out_slope, int64_t ldo, int nworld) {
  extern __shared__ float fv_lds[];
  float *row = fv_lds;                  // the world's waypoints
  float *mom = row + n.words_wp;        // its moment entries
  float *qv = mom + n.nentry;           // its velocities
  float *dist = qv + n.nqvel;           // from every waypoint to the next one
  float *cosp = dist + n.words_wp / 3;  // [nmuscle]
  int *named = (int *)(cosp + n.nmuscle);  // the velocities up to the last dof that the tables name
  unsigned short *dof = (unsigned short *)(named + 1);  // [nentry]
  const int tid = threadIdx.x, nmuscle = n.nmuscle;
  // what the tables name of a row, which may be a part of a wider array's: the last world's row ends
  // with its last named value, wherever the stride would lead
  const int nwp = min(waypoint_start[nmuscle], n.words_wp / 3), ne = min(dof_offsets[nmuscle], n.nentry);
  if (tid == 0) *named = 0;
  __syncthreads();
  int most = 0;
  for (int e = tid; e < ne; e += nt) {
    const int d = dof_torque_idx[e] + root;
    dof[e] = (unsigned short)d;
    most = max(most, d + 1);
  }
  for (int o = 32; o; o >>= 1) most = max(most, __shfl_xor(most, o));
  if ((tid & 63) == 0) atomicMax(named, most);
  for (int m = tid; m < nmuscle; m += nt) cosp[m] = cosf(params[m * ldpar + 3]);
  constexpr int kPoints = AHEAD ? 14 : 1, kEntries = AHEAD ? 9 : 1;
  float points[kPoints], entries[kEntries], speed = 0.0f, excitation = 0.0f;
  int nq = 0;
  FvMuscle mine = {};
  auto hold = [&](int64_t w) __attribute__((always_inline)) {
    int t = tid;
    asm volatile("" : "+v"(t));  // (no address is kept from world to world)
    const float *pw = wp + w * ldw, *mw = moment + w * ldm;
#pragma unroll
    for (int k = 0; k < kPoints; ++k)
      if (t + k * nt < 3 * nwp) points[k] = pw[(unsigned)(t + k * nt)];
#pragma unroll
    for (int k = 0; k < kEntries; ++k)
      if (t + k * nt < ne) entries[k] = mw[(unsigned)(t + k * nt)];
    if (t < nq) speed = qvel[w * ldq + t];
    if (t < nmuscle) excitation = activation[w * lda + t];
  };
  auto muscle = [&](int m) __attribute__((always_inline)) {
    const float *par = params + (size_t)m * ldpar;
    return FvMuscle{waypoint_start[m], waypoint_start[m + 1] - 1, dof_offsets[m], dof_offsets[m + 1], par[0], par[2],
                    fmaxf(par[1], 1.0e-6f), fmaxf(rest[m], 1.0e-6f), fmaxf(length_scale[m] * fv.vmax, 1.0e-6f)};
  };
  if (AHEAD) {
    if (tid < nmuscle) mine = muscle(tid);
    __syncthreads();
    nq = min(__builtin_amdgcn_readfirstlane(*named), n.nqvel);
    hold(blockIdx.x);
  }
  for (int64_t w = blockIdx.x; w < nworld; w += gridDim.x) {
    __syncthreads();  // the tables are there, the world before is done with
    float active0 = excitation;
    if constexpr (AHEAD) {
      int t = tid;
      asm volatile("" : "+v"(t));
#pragma unroll
      for (int k = 0; k < kPoints; ++k)
        if (t + k * nt < 3 * nwp) row[t + k * nt] = points[k];
#pragma unroll
      for (int k = 0; k < kEntries; ++k)
        if (t + k * nt < ne) mom[t + k * nt] = entries[k];
      if (t < nq) qv[t] = speed;
      if (w + gridDim.x < nworld) hold(w + gridDim.x);
    } else {
      stage_row<nt>(row, wp + w * ldw, 3 * nwp, tid);
      stage_row<nt>(mom, moment + w * ldm, ne, tid);
      stage_row<nt>(qv, qvel + w * ldq, min(__builtin_amdgcn_readfirstlane(*named), n.nqvel), tid);
    }
    __syncthreads();
    for (int i = tid; i < nwp - 1; i += nt) dist[i] = length(sub(ld3(row + 3 * (i + 1)), ld3(row + 3 * i)));
    __syncthreads();
    for (int m = tid; m < nmuscle; m += nt) {
      FvMuscle k = mine;
      float active = active0;
      if (!AHEAD || m >= nt) {
        k = muscle(m);
        active = activation[w * lda + m];
      }
      float len = 0.0f, velocity = 0.0f;
      // both sums in order, the next terms asked for before these are added (a term past the last is the last again)
      if (k.i0 < k.i1) {
        float d[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) d[u] = dist[min(k.i0 + u, k.i1 - 1)];
        for (int i = k.i0; i < k.i1; i += 4) {
          float dn[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) dn[u] = dist[min(i + 4 + u, k.i1 - 1)];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            if (i + u < k.i1) len = len + d[u];
            d[u] = dn[u];
          }
        }
      }
      if (k.e0 < k.e1) {
        float a[4], v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int at = min(k.e0 + u, k.e1 - 1);
          a[u] = mom[at], v[u] = qv[dof[at]];
        }
        for (int e = k.e0; e < k.e1; e += 4) {
          float an[4], vn[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int at = min(e + 4 + u, k.e1 - 1);
            an[u] = mom[at], vn[u] = qv[dof[at]];
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            if (e + u < k.e1) velocity = __builtin_fmaf(-a[u], v[u], velocity);
            a[u] = an[u], v[u] = vn[u];
          }
        }
      }
      const float f0 = k.f0, lt0 = k.lt0, velocity_scale = k.velocity_scale;
      float mult, dmult;
      force_velocity_curve(velocity / velocity_scale, fv.fvmax, &mult, &dmult);
      if (fv.clamp_activation != 0.0f) active = fminf(fmaxf(active, 0.0f), 1.0f);
      const float lm = len / k.rest - lt0;
      const float ln = fminf(fmaxf(lm / k.lm0, model.length_norm_min), model.length_norm_max);
      const float unit = f0 * active_fl(ln, model.active) * cosp[m] * model.force_scale;
      out_length[w * ldo + m] = len;
      out_activation[w * ldo + m] = active * mult;
      out_velocity[w * ldo + m] = velocity;
      out_multiplier[w * ldo + m] = mult;
      out_slope[w * ldo + m] = fv.include_active * active * unit * dmult / velocity_scale;
    }
  }
}

__global__ __launch_bounds__(256) void force_kernel(
    const float *__restrict__ wp, int64_t ldw, const int32_t *__restrict__ seg_start,
    const int32_t *__restrict__ seg_offsets, const float *__restrict__ params, int ldpar,
    const float *__restrict__ rest, im_muscle_force_model model, int nmuscle,
    float *__restrict__ unit, int64_t ldu, float *__restrict__ passive, int64_t ldpa) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t w = blockIdx.y;
  if (m >= nmuscle) return;
  muscle_force_magnitudes(wp + w * ldw, seg_start, seg_offsets, params, ldpar, rest, model, m,
                          unit + w * ldu + m, passive ? passive + w * ldpa + m : nullptr);
}

// Waypoints and force magnitudes of one world in one workgroup: the waypoints go to memory and
// stay in LDS, from where the muscle lengths are taken.  Same operations as the two kernels
// above, so the results are theirs bit for bit.
__global__ __launch_bounds__(512) void waypoints_forces_kernel(
    const float *__restrict__ xpos, int64_t ldp, const float *__restrict__ xquat, int64_t ldq,
    const int32_t *__restrict__ wp_body, const float *__restrict__ wp_local, int nwp,
    float *__restrict__ out, int64_t ldo, const int32_t *__restrict__ seg_start,
    const int32_t *__restrict__ seg_offsets, const float *__restrict__ params, int ldpar,
    const float *__restrict__ rest, im_muscle_force_model model, int nmuscle,
    float *__restrict__ unit, int64_t ldu, float *__restrict__ passive, int64_t ldpa) {
  extern __shared__ float wpl[];  // [3 * nwp]
  const int64_t w = blockIdx.x;
  const int tid = threadIdx.x, nt = blockDim.x;
  for (int i = tid; i < nwp; i += nt) {
    const V3 p = world_waypoint(xpos + w * ldp, xquat + w * ldq, wp_body, wp_local, i);
    wpl[3 * i] = p.x;
    wpl[3 * i + 1] = p.y;
    wpl[3 * i + 2] = p.z;
  }
  __syncthreads();
  float *o = out + w * ldo;
  for (int k = tid; k < 3 * nwp; k += nt) o[k] = wpl[k];
  for (int m = tid; m < nmuscle; m += nt)
    muscle_force_magnitudes(wpl, seg_start, seg_offsets, params, ldpar, rest, model, m,
                            unit + w * ldu + m, passive ? passive + w * ldpa + m : nullptr);
}

__global__ __launch_bounds__(256) void torque_forward_kernel(
    Geo g, Seg s, const int32_t *__restrict__ offsets, const int32_t *__restrict__ e_seg,
    const int32_t *__restrict__ e_muscle, const float *__restrict__ e_a,
    const float *__restrict__ e_b, const float *__restrict__ unit, int64_t ldu,
    const float *__restrict__ passive, int64_t ldpa, const float *__restrict__ act, int64_t lda,
    int root, int ntorque, float *__restrict__ out, int64_t ldo) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t w = blockIdx.y;
  if (j >= ntorque) return;
  const float *cd = g.cdof + w * g.ldd + 6 * (int64_t)(j + root);
  const V3 ang = ld3(cd), lin = ld3(cd + 3);
  float total = 0.0f;
  for (int e = offsets[j]; e < offsets[j + 1]; ++e) {
    const int m = e_muscle[e];
    float f = unit[w * ldu + m] * act[w * lda + m];
    if (passive) f = f + passive[w * ldpa + m];
    if (f == 0.0f) continue;
    total = total + seg_term(g, s, w, e_seg[e], lin, ang, e_a[e], e_b[e], f);
  }
  out[w * ldo + j] = total;
}

__global__ __launch_bounds__(256) void activation_grad_kernel(
    Geo g, Seg s, const int32_t *__restrict__ offsets, const int32_t *__restrict__ e_seg,
    const int32_t *__restrict__ e_torque, const float *__restrict__ e_a,
    const float *__restrict__ e_b, const float *__restrict__ unit, int64_t ldu,
    const float *__restrict__ gout, int64_t ldg, int root, int nmuscle, float *__restrict__ gact,
    int64_t lda) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t w = blockIdx.y;
  if (m >= nmuscle) return;
  const float f = unit[w * ldu + m];
  float grad = 0.0f;
  // The reference returns before the store when f == 0 and relies on a zero-filled
  // output (muscle_dynamics_kernels.py:1817-1819); the store of 0 here is the same value.
  if (f != 0.0f) {
    for (int e = offsets[m]; e < offsets[m + 1]; ++e) {
      const int j = e_torque[e];
      const float *cd = g.cdof + w * g.ldd + 6 * (int64_t)(j + root);
      grad = grad + gout[w * ldg + j] *
                        seg_term(g, s, w, e_seg[e], ld3(cd + 3), ld3(cd), e_a[e], e_b[e], f);
    }
  }
  gact[w * lda + m] = grad;
}

__global__ __launch_bounds__(256) void sparse_moment_kernel(
    Geo g, Seg s, const int32_t *__restrict__ entry_torque, const int32_t *__restrict__ offsets,
    const int32_t *__restrict__ e_seg, const float *__restrict__ e_a,
    const float *__restrict__ e_b, int root, int nentry, float *__restrict__ moment, int64_t ldm) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t w = blockIdx.y;
  if (e >= nentry) return;
  const float *cd = g.cdof + w * g.ldd + 6 * (int64_t)(entry_torque[e] + root);
  const V3 ang = ld3(cd), lin = ld3(cd + 3);
  float total = 0.0f;
  for (int k = offsets[e]; k < offsets[e + 1]; ++k)
    total = total + seg_term(g, s, w, e_seg[k], lin, ang, e_a[k], e_b[k], 1.0f);
  moment[w * ldm + e] = total;
}

// Feasible torque box over activations in [0, 1]: per torque dof the entries are grouped by
// muscle (consecutive entries of one muscle); a muscle's total goes to the lower bound when
// negative, else to the upper (muscle_dynamics_kernels.py:1453-1528).
__global__ __launch_bounds__(256) void torque_bounds_kernel(
    Geo g, Seg s, const int32_t *__restrict__ offsets, const int32_t *__restrict__ e_seg,
    const int32_t *__restrict__ e_muscle, const float *__restrict__ e_a,
    const float *__restrict__ e_b, const float *__restrict__ unit, int64_t ldu, int root,
    int ntorque, float *__restrict__ lower, float *__restrict__ upper, int64_t ldo) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t w = blockIdx.y;
  if (j >= ntorque) return;
  const float *cd = g.cdof + w * g.ldd + 6 * (int64_t)(j + root);
  const V3 ang = ld3(cd), lin = ld3(cd + 3);
  int current = -1;
  float total = 0.0f, lo = 0.0f, hi = 0.0f;
  for (int e = offsets[j]; e < offsets[j + 1]; ++e) {
    const int m = e_muscle[e];
    if (current >= 0 && m != current) {
      if (total < 0.0f) lo = lo + total;
      else hi = hi + total;
      total = 0.0f;
    }
    current = m;
    total = total + seg_term(g, s, w, e_seg[e], lin, ang, e_a[e], e_b[e], unit[w * ldu + m]);
  }
  if (current >= 0) {
    if (total < 0.0f) lo = lo + total;
    else hi = hi + total;
  }
  lower[w * ldo + j] = lo;
  upper[w * ldo + j] = hi;
}

// ---- a workgroup per world, resident over worlds -------------------------------------------
// The four contractions above visit every applied segment once per (segment, dof) entry and
// redo its square root and three divisions each time, and they fetch a muscle's force and a
// dof's motion axis from memory once per entry.  Here a workgroup first leaves in LDS each
// segment's unit direction and its two lever vectors, every muscle's force and every torque
// dof's axis; then every thread evaluates entries (same operations, same order as
// contribution()), and a last pass adds each output's entries in list order, reading them
// several at a time so that only the additions wait on one another.  Results equal the
// one-thread-per-output kernels bit for bit.
//
// What bounds it is the vector issue rate: 41 instructions of an entry's arithmetic cannot be
// left out without changing bits, and a launch per world spent as many again on the entry lists
// (four table reads with their addresses, the entry's row, the products by the LDS records'
// sizes; 63 - 79 % of the cycles issued a vector instruction).  The lists are the same for every
// world, so the grid is what the chip holds at once, a workgroup walks over worlds, and a thread of
// a small rig keeps its TRIPS entries as LDS addresses and coefficients in registers.  An output's
// ordered sum runs beside the next world's staging: two barriers per world.
// Threads by the entries (launch_world).  The kernels alone, torque / gradient / moment, a launch per
// world with 512 threads -> this:
//    40 muscles ( 655 entries) x 8192 worlds  41.9 / 36.8 / 29.1 -> 24.8 / 22.0 / 20.3 us
//   120         (1882)                        70.5 / 53.9 / 51.2 -> 57.0 / 40.1 / 40.5
//   200         (3145)                        90.7 / 71.9 / 72.0 -> 83.6 / 66.5 / 65.6
//   284         (4445)                         133 / 98.1 /  108 ->  116 / 86.1 / 87.0
// 768 threads that keep six entries each, the best for the moment at 284 muscles alone (84.8 us), took
// 48.7 / 39.0 / 35.6 at 40 muscles and 116 / 78.6 / 75.8 at 200.
enum { MW_FORWARD, MW_GRAD, MW_BOUNDS, MW_MOMENT };

struct MwArgs {
  Geo g;
  Seg s;
  const int32_t *offsets, *e_seg, *e_other, *row_torque;  // row_torque: MW_MOMENT only
  const float *e_a, *e_b;
  const float *unit, *passive, *act, *gout;
  int64_t ldu, ldpa, lda, ldg;
  float *out0, *out1;
  int64_t ldo;
  int root, nrow, nentry, nseg;
  int ntorque, nmuscle;  // sizes of the staged axes and forces (nmuscle 0 for MW_MOMENT)
  int nworld;
};

constexpr int kContribPad = 4;  // floats read past the last entry by ordered_sum()
constexpr int kAxis = 7;        // floats of a dof's record: its cdof and, for MW_GRAD, grad_output
struct MwLds {
  float *segd;     // [nseg][9]: dir (0 for a degenerate segment), p0 - c0, p1 - c1
  float *contrib;  // [nentry]
  float *axis;     // [ntorque][kAxis]
  float *force;    // [nmuscle]: force of a muscle as the contraction sees it
  unsigned short *rowid;  // [nentry]: an entry's row; in contrib's place where registers keep the entries
};
__host__ __device__ inline size_t mw_lds_floats(const MwArgs &a) {
  return (size_t)9 * a.nseg + (size_t)a.nentry + kContribPad + (size_t)kAxis * a.ntorque + (size_t)a.nmuscle;
}

// One entry: word indices of its records in LDS, and its coefficients.
struct MwEntry {
  unsigned where;  // segment's record | dof's record << 16
  unsigned force;  // muscle's force
  float a, b;
};
template <int MODE>
__device__ __forceinline__ MwEntry load_entry(const MwArgs &a, const MwLds &l, const float *lds, int e) {
  const int row = l.rowid[e], other = MODE == MW_MOMENT ? 0 : a.e_other[e];
  const int torque = MODE == MW_GRAD ? other : MODE == MW_MOMENT ? a.row_torque[row] : row;
  const int muscle = MODE == MW_GRAD ? row : other;
  MwEntry t;
  t.where = (unsigned)(9 * a.e_seg[e]) | (unsigned)(l.axis - lds + kAxis * torque) << 16;
  t.force = (unsigned)(l.force - lds + muscle);
  t.a = a.e_a[e];
  t.b = a.e_b[e];
  return t;
}

template <int MODE>
__device__ __forceinline__ float entry_contribution(const float *lds, const MwEntry &t) {
  const float f = MODE == MW_MOMENT ? 1.0f : lds[t.force];
  const float *cd = lds + (t.where >> 16);
  const V3 ang = ld3(cd), lin = ld3(cd + 3);
  const float *sd = lds + (t.where & 0xFFFFu);
  const V3 dir = {sd[0], sd[1], sd[2]}, r0 = {sd[3], sd[4], sd[5]}, r1 = {sd[6], sd[7], sd[8]};
  const V3 fv = scale(f, dir);
  const V3 st = add(lin, cross(ang, r0));
  const V3 en = add(lin, cross(ang, r1));
  float c = dot(sub(scale(t.a, st), scale(t.b, en)), fv);
  // evaluated for every entry, without a branch around it: a thread's entries then proceed
  // side by side instead of one after the other
  asm volatile("" : "+v"(c));
  // an entry whose force is zero is skipped by the reference: it enters the sum as 0
  c = f == 0.0f ? 0.0f : c;
  if (MODE == MW_GRAD) c = cd[6] * c;
  return c;
}

// Sum of contrib[e0..e1) in list order from +0.  Whole groups of 16 (LONG) and of 4 entries are
// read with one address and added without a test; the last group reads up to three floats past
// e1 (contrib is padded for that) and enters them as +0, which leaves every bit of a sum that
// started at +0 (such a sum is never -0).
template <bool LONG>
__device__ __forceinline__ float ordered_sum(const float *contrib, int e0, int e1) {
  float total = 0.0f;
  int e = e0;
  if (LONG) {
    for (; e + 16 <= e1; e += 16) {
      float c[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) c[k] = contrib[e + k];
#pragma unroll
      for (int k = 0; k < 16; ++k) total = total + c[k];
    }
  }
  for (; e + 4 <= e1; e += 4) {
    float c[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) c[k] = contrib[e + k];
#pragma unroll
    for (int k = 0; k < 4; ++k) total = total + c[k];
  }
  if (e < e1) {
    float c[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) c[k] = contrib[e + k];
#pragma unroll
    for (int k = 0; k < 3; ++k) total = total + (e + k < e1 ? c[k] : 0.0f);
  }
  return total;
}

// The same with the next sixteen entries on their way while sixteen are added, for a kernel with the registers for them (torque of 284 muscles x 4096 worlds
// 68.2 -> 65.1 us in groups, gradient 61.2 -> 57.3; muscle_world_kernel with kept entries spilled: 90 muscles x 4096 41.3 -> 43.7 us).
// Words up to kSumAhead past the last entry are read and left out.
constexpr int kSumAhead = 16;
__device__ __forceinline__ float ordered_sum_ahead(const float *contrib, int e0, int e1) {
  float total = 0.0f, c[16];
  int e = e0;
#pragma unroll
  for (int k = 0; k < 16; ++k) c[k] = contrib[e + k];
  for (; e + 16 <= e1; e += 16) {
    float ahead[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) ahead[k] = contrib[e + 16 + k];
#pragma unroll
    for (int k = 0; k < 16; ++k) total = total + c[k];
#pragma unroll
    for (int k = 0; k < 16; ++k) c[k] = ahead[k];
  }
#pragma unroll
  for (int k = 0; k < 15; ++k) total = total + (e + k < e1 ? c[k] : 0.0f);
  return total;
}

// TRIPS: entries that a thread keeps in registers, nentry <= TRIPS * NT; 0: they are read from the
// lists for every world.
template <int MODE, int NT, int TRIPS>
__global__ __launch_bounds__(NT, 6) void muscle_world_kernel(MwArgs a) {
  extern __shared__ float lds[];
  MwLds l;
  l.segd = lds;
  l.contrib = l.segd + 9 * a.nseg;
  l.axis = l.contrib + a.nentry + kContribPad;
  l.force = l.axis + kAxis * a.ntorque;
  l.rowid = (unsigned short *)(TRIPS ? l.contrib : lds + mw_lds_floats(a));
  constexpr int nt = NT;
  const int tid = threadIdx.x;
  // staging starts at the last wavefront: the first one's sums of the world before take longest
  const int rid = nt - 1 - tid;
  if (a.nentry < 32 * a.nrow) {  // short rows: a thread writes its row's
    for (int r = tid; r < a.nrow; r += nt)
      for (int e = a.offsets[r]; e < a.offsets[r + 1]; ++e) l.rowid[e] = (unsigned short)r;
  } else {  // long rows: a wave writes a row's
    for (int r = tid >> 6; r < a.nrow; r += nt >> 6)
      for (int e = a.offsets[r] + (tid & 63); e < a.offsets[r + 1]; e += 64) l.rowid[e] = (unsigned short)r;
  }
  MwEntry kept[TRIPS ? TRIPS : 1];
  if (TRIPS) {
    __syncthreads();
#pragma unroll
    for (int k = 0; k < TRIPS; ++k) {
      kept[k] = load_entry<MODE>(a, l, lds, min(k * nt + tid, a.nentry - 1));
      if (k % 2) __builtin_amdgcn_sched_barrier(0);
    }
    // contrib takes the rows' place only behind the first world's barrier
  }
  for (int64_t w = blockIdx.x; w < a.nworld; w += gridDim.x) {
    const float *wp = a.g.wp + w * a.g.ldw, *com = a.g.com + w * a.g.ldc, *cdof = a.g.cdof + w * a.g.ldd;
    for (int sg = rid; sg < a.nseg; sg += nt) {
      const V3 p0 = ld3(wp + 3 * a.s.p0[sg]), p1 = ld3(wp + 3 * a.s.p1[sg]);
      const V3 c0 = ld3(com + 3 * a.s.b0[sg]), c1 = ld3(com + 3 * a.s.b1[sg]);
      const V3 seg = sub(p1, p0);
      const float len = length(seg);
      const bool ok = !(len < 1.0e-8f);
      const V3 r0 = sub(p0, c0), r1 = sub(p1, c1);
      // a degenerate segment contributes nothing: with a zero direction its entries come out as
      // +-0, and adding +-0 to a sum that started at +0 leaves every bit of it
      float *o = l.segd + 9 * sg;
      o[0] = ok ? seg.x / len : 0.0f;
      o[1] = ok ? seg.y / len : 0.0f;
      o[2] = ok ? seg.z / len : 0.0f;
      o[3] = r0.x; o[4] = r0.y; o[5] = r0.z;
      o[6] = r1.x; o[7] = r1.y; o[8] = r1.z;
    }
    for (int i = rid; i < 6 * a.ntorque; i += nt) l.axis[i + i / 6] = cdof[6 * a.root + i];
    // MW_GRAD reads force[r] in its sums of the world before: by the thread that overwrites it here
    for (int m = MODE == MW_GRAD ? tid : rid; m < a.nmuscle; m += nt) {
      float f = a.unit[w * a.ldu + m];
      if (MODE == MW_FORWARD) {
        f = f * a.act[w * a.lda + m];
        if (a.passive) f = f + a.passive[w * a.ldpa + m];
      }
      l.force[m] = f;
    }
    if (MODE == MW_GRAD)
      for (int j = tid; j < a.ntorque; j += nt) l.axis[kAxis * j + 6] = a.gout[w * a.ldg + j];
    __syncthreads();
    if (TRIPS) {
#pragma unroll
      for (int k = 0; k < TRIPS; ++k) {
        const float c = entry_contribution<MODE>(lds, kept[k]);
        if (k * nt + tid < a.nentry) l.contrib[k * nt + tid] = c;
      }
    } else {
      // four entries per thread and trip while whole trips remain (all their loads are issued
      // before the first is needed), then one entry per thread
      int base = 0;
      for (; base + 4 * nt <= a.nentry; base += 4 * nt) {
        MwEntry t[4];
        float c[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) t[k] = load_entry<MODE>(a, l, lds, base + k * nt + tid);
#pragma unroll
        for (int k = 0; k < 4; ++k) c[k] = entry_contribution<MODE>(lds, t[k]);
#pragma unroll
        for (int k = 0; k < 4; ++k) l.contrib[base + k * nt + tid] = c[k];
      }
      for (int e = base + tid; e < a.nentry; e += nt)
        l.contrib[e] = entry_contribution<MODE>(lds, load_entry<MODE>(a, l, lds, e));
    }
    __syncthreads();
    const float *contrib = l.contrib;
    for (int r = tid; r < a.nrow; r += nt) {
      const int e0 = a.offsets[r], e1 = a.offsets[r + 1];
      if (MODE == MW_FORWARD) {
        a.out0[w * a.ldo + r] = ordered_sum<true>(contrib, e0, e1);
      } else if (MODE == MW_MOMENT) {  // a (muscle, dof) pair has a few segments
        a.out0[w * a.ldo + r] = ordered_sum<false>(contrib, e0, e1);
      } else if (MODE == MW_GRAD) {
        // The one-thread-per-muscle kernel leaves 0 for a muscle without force; its entries are
        // 0 here as well (gout * 0), but an infinite gout would turn them into NaN
        a.out0[w * a.ldo + r] = l.force[r] != 0.0f ? ordered_sum<true>(contrib, e0, e1) : 0.0f;
      } else {
        int current = -1;
        float total = 0.0f, lo = 0.0f, hi = 0.0f;
        auto add = [&](int m, float c) __attribute__((always_inline)) {
          if (current >= 0 && m != current) {
            if (total < 0.0f) lo = lo + total;
            else hi = hi + total;
            total = 0.0f;
          }
          current = m;
          total = total + c;
        };
        int e = e0;
        for (; e + 8 <= e1; e += 8) {  // eight entries' muscles on their way at once
          int m[8];
          float c[8];
#pragma unroll
          for (int k = 0; k < 8; ++k) m[k] = a.e_other[e + k], c[k] = contrib[e + k];
#pragma unroll
          for (int k = 0; k < 8; ++k) add(m[k], c[k]);
        }
        for (; e < e1; ++e) add(a.e_other[e], contrib[e]);
        if (current >= 0) {
          if (total < 0.0f) lo = lo + total;
          else hi = hi + total;
        }
        a.out0[w * a.ldo + r] = lo;
        a.out1[w * a.ldo + r] = hi;
      }
    }
  }
}

// Launches the workgroup-per-world kernel when a world's segments and entries fit in LDS (which
// also keeps the records' word indices below 16 bits) and the entry list states the range of its
// `other` column; returns false for the caller to use the one-thread-per-output kernel instead.
template <int MODE, int NT, int TRIPS>
bool launch_world_on(MwArgs a, bool walk, int nworld, hipStream_t stream) {
  const size_t lds_bytes = 4 * mw_lds_floats(a) + (TRIPS ? 0 : 2 * (((size_t)a.nentry + 1) & ~(size_t)1));
  if (lds_bytes > 64 * 1024) return false;
  unsigned grid = (unsigned)nworld;
  if (walk && resident_grid((const void *)muscle_world_kernel<MODE, NT, TRIPS>, NT, lds_bytes, nworld, &grid) != IM_OK) return false;
  a.nworld = nworld;
  hipLaunchKernelGGL((muscle_world_kernel<MODE, NT, TRIPS>), dim3(grid), dim3(NT), lds_bytes, stream, a);
  return true;
}
template <int MODE>
bool launch_world(const MwArgs &a, int nworld, hipStream_t stream) {
  static const bool forced_off = [] {
    const char *e = std::getenv("IMHIP_MUSCLE_KERNEL");
    return e && std::strcmp(e, "simple") == 0;
  }();
  if (forced_off || a.nentry == 0 || a.nseg == 0 || a.nrow > 65535 || a.ntorque <= 0 || (MODE != MW_MOMENT && a.nmuscle <= 0)) return false;
  const bool small = a.nentry <= 6 * 256;
  // The bounds' rows are long chains of comparisons on a few lanes: a workgroup per world hides them behind other
  // worlds, one that stays does not (40 / 120 / 200 / 284 muscles x 8192 worlds: 33.6 / 102 / 161 / 274 us; on
  // workgroups that stay 57 / 124 / 197 / 268; 768 threads with an entry's muscle read at a time 112 / 272 / 426 / 594).
  if (MODE == MW_BOUNDS)
    return small ? launch_world_on<MODE, 256, 0>(a, false, nworld, stream) : launch_world_on<MODE, 512, 0>(a, false, nworld, stream);
  int ncu = 0;
  if (compute_units(&ncu) != IM_OK) return false;
  // Entries kept in registers pay from two worlds per workgroup on (six of 256 threads, three of 512 per CU), and up
  // to about 2000 entries; beyond, and with 512 threads throughout, reading them from the lists takes as long.
  if (small && nworld >= 2 * 6 * ncu)
    return a.nentry <= 2 * 256   ? launch_world_on<MODE, 256, 2>(a, true, nworld, stream)
           : a.nentry <= 4 * 256 ? launch_world_on<MODE, 256, 4>(a, true, nworld, stream)
                                 : launch_world_on<MODE, 256, 6>(a, true, nworld, stream);
  if (!small && a.nentry <= 4 * 512 && nworld >= 2 * 3 * ncu) return launch_world_on<MODE, 512, 4>(a, true, nworld, stream);
  return launch_world_on<MODE, 512, 0>(a, true, nworld, stream);
}

// ---- a world from its context in one launch --------------------------------------------------
// Torque, activation gradient and sparse moment straight from body poses: a workgroup takes a world's
// waypoints, segment records and muscle forces into LDS and contracts them there, so neither waypoints nor
// forces go to memory (15 KB a world at 284 muscles, written and read back by two launches before).
//
// What bounds it is the vector issue rate.  What is left out of a world's instructions, bits unchanged: a
// body's quaternion is normalised once and not once per waypoint; a muscle's cosine is taken once per
// workgroup; an entry whose one coefficient is 0 takes the lever of its other end only (0 * finite subtracted from or added to a number
// leaves it, and a zero's sign does not survive an ordered sum that starts at +0).  The lists come packed, the entries of a
// kind together, so that a wavefront's entries are of one kind and a thread keeps its entries in two
// registers each.  A world with a lever or an axis so large that their products may not be finite takes
// the full expression throughout (0 * inf is NaN there).
// Four barriers per world: poses and axes, waypoints, segments and forces, contributions; the ordered sums run beside
// the next world's poses.  4096 worlds of 284 muscles, three workgroups of 512 per CU: torque 80 us where the two
// launches took 35 + 64, gradient 74 (35 + 49), moment 65 (20 + 58); by counters the vector ALUs issue in 0.75, 0.79 and 0.71
// of the cycles, the LDS is busy in 0.63, 0.70 and 0.65 (three eighths of that bank conflicts).
// a value every lane holds alike, as a scalar
__device__ __forceinline__ float uniform(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}

struct CtxArgs {
  im_muscle_context c;
  const float *in;  // activation (MW_FORWARD) or grad_output (MW_GRAD)
  int64_t ldin;
  float *out;
  int64_t ldo;
  int root, nworld;
  int single_end, single;  // entries before these: end only; end or start only (multiples of 64)
};

constexpr float kCtxLarge = 1.0e18f;  // two factors below it have a finite product
constexpr int kCtxTrips = 10;     // packed entries of a thread
constexpr int kCtxMost = kCtxTrips * 512, kCtxMuscles = 512;
constexpr int kGroupTrips = 4, kRowTrips = 6;  // groups of a thread
constexpr int kPose = 8;  // floats of a body's record: u, s s - u.u, 2 s, position
struct CtxLds {
  int contrib, segd, axis, force, com, flags, dist, words;
};
// GROUPS: muscle_groups_kernel's, which keeps the segments' lengths too.
template <bool GROUPS>
__host__ __device__ inline CtxLds ctx_lds(const im_muscle_context &c, bool forces) {
  const int sums = c.nentry + kContribPad, points = 3 * c.nwaypoint, records = 9 * c.nsegment, poses = kPose * c.nbody;
  CtxLds l;
  l.contrib = 0;  // the waypoints lie here until the contributions take their place
  l.segd = sums > points ? sums : points;  // and the bodies' records until the segments' do
  if (GROUPS) l.segd = (l.segd + 3) & ~3;
  l.axis = l.segd + (records > poses ? records : poses);
  l.force = l.axis + kAxis * c.ntorque;
  l.com = l.force + (forces ? c.nmuscle : 0);
  l.flags = l.com + 3 * c.nbody;
  l.dist = l.flags + 2;
  l.words = l.dist + (GROUPS && forces ? c.nlength + 3 : 0);
  if (GROUPS && l.words < c.nentry + kSumAhead) l.words = c.nentry + kSumAhead;
  return l;
}

// An entry with both coefficients 1: contribution() less the products with 1.
__device__ __forceinline__ float both_ends(const float *cd, const float *sd, float f) {
  const V3 ang = ld3(cd), lin = ld3(cd + 3), fv = scale(f, ld3(sd));
  return dot(sub(add(lin, cross(ang, ld3(sd + 3))), add(lin, cross(ang, ld3(sd + 6)))), fv);
}
// An entry with one: its end's lever, and the sign bit that the end's term enters with.
__device__ __forceinline__ float one_end(const float *cd, const float *sd, const float *lever, unsigned sign, float f) {
  const V3 ang = ld3(cd), lin = ld3(cd + 3), fv = scale(f, ld3(sd));
  const float v = dot(add(lin, cross(ang, ld3(lever))), fv);
  return __builtin_bit_cast(float, __builtin_bit_cast(unsigned, v) ^ sign);
}

// A packed entry into its place by the whole expression, both levers whatever the coefficients.
template <int MODE>
__device__ __forceinline__ void full_contribution(float *lds, const CtxLds &l, uint2 e, bool end_only, bool start_only) {
  const float *sd = lds + l.segd + 9 * (e.x & 0xFFFFu), *cd = lds + l.axis + kAxis * (e.x >> 16);
  const float f = MODE == MW_MOMENT ? 1.0f : lds[l.force + (e.y >> 16)];
  const V3 ang = ld3(cd), lin = ld3(cd + 3), fv = scale(f, ld3(sd));
  const V3 st = add(lin, cross(ang, ld3(sd + 3))), en = add(lin, cross(ang, ld3(sd + 6)));
  float v = dot(sub(scale(end_only ? 0.0f : 1.0f, st), scale(start_only ? 0.0f : 1.0f, en)), fv);
  v = f == 0.0f ? 0.0f : v;
  if (MODE == MW_GRAD) v = cd[6] * v;
  lds[e.y & 0xFFFFu] = v;
}

// The kernel's argument block in its argument segment, through a pointer laundered once per phase: held in
// scalar registers over a world's phases its thirty pointers are spilled.
__device__ __forceinline__ const CtxArgs &ctx_args() {
  typedef const CtxArgs __attribute__((address_space(4))) Segment;
  Segment *p = (Segment *)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const CtxArgs *)p;
}

template <int MODE, int NT, int TRIPS>
__global__ __launch_bounds__(NT, TRIPS > kCtxTrips ? 5 : 6) void muscle_context_kernel(CtxArgs) {
  extern __shared__ float lds[];
  constexpr int nt = NT;
  constexpr bool FORCES = MODE != MW_MOMENT;
  int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) * 64;
  // a thread's entries: LDS byte offsets of the segment's and the dof's record, the entry's place and the force
  auto offsets_of = [](const CtxLds &l, uint2 e) __attribute__((always_inline)) {
    const unsigned seg = 4u * l.segd + 36u * (e.x & 0xFFFFu), axis = 4u * (l.axis + kAxis * (e.x >> 16));
    return make_uint2(seg | axis << 16, 4u * (e.y & 0xFFFFu) | 4u * (l.force + (e.y >> 16)) << 16);
  };
  uint2 kept[TRIPS];
  float cosine = 1.0f;  // of the pennation of the thread's muscle
  int turn = 0;
  {
    const CtxArgs &a = ctx_args();
    const im_muscle_context &c = a.c;
    const CtxLds l = ctx_lds<false>(c, FORCES);
#pragma unroll
    for (int k = 0; k < TRIPS; ++k) {
      const int e = k * nt + tid;
      kept[k] = offsets_of(l, ((const uint2 *)c.packed)[e < c.npacked ? e : 0]);
    }
    if (FORCES) cosine = cosf(c.params[min(tid, c.nmuscle - 1) * c.ld_params + 3]);
    if (tid < 2) ((int *)(lds + l.flags))[tid] = 0;
    __syncthreads();
  }
  // A phase's table entries are asked for a phase ahead of their use, behind its barrier (up to WT waypoints, ST
  // segments and a muscle of LT segments a thread; what is beyond is read where it is used).
  constexpr int WT = 3, ST = 3, LT = 4;
  for (int64_t w = blockIdx.x; w < ctx_args().nworld; w += gridDim.x, turn ^= 1) {
    asm volatile("" : "+v"(tid));  // (no address formed from it is kept from world to world)
    const int rid = nt - 1 - tid;
    int wp_body[WT];
    V3 wp_local[WT];
    {  // poses, centres, axes; activations where the forces will be
      const CtxArgs &a = ctx_args();
      const im_muscle_context &c = a.c;
      const CtxLds l = ctx_lds<false>(c, FORCES);
#pragma unroll
      for (int k = 0; k < WT; ++k) {
        const int i = min(tid + k * nt, c.nwaypoint - 1);
        wp_body[k] = c.waypoint_body[i];
        wp_local[k] = ld3(c.waypoint_local + 3 * i);
      }
      const float *com = c.subtree_com + w * c.ld_subtree_com, *cdof = c.cdof + w * c.ld_cdof + 6 * a.root;
      for (int i = rid; i < 6 * c.ntorque; i += nt) {
        const float v = cdof[i];
        lds[l.axis + i + i / 6] = v;
        if (!(fabsf(v) < kCtxLarge)) ((int *)(lds + l.flags))[turn] = 1;
      }
      for (int b = rid; b < c.nbody; b += nt) {
        const float *x = c.xpos + w * c.ld_xpos + 3 * b;
        const BodyTurn t = body_turn(c.xquat + w * c.ld_xquat + 4 * b);
        float *o = lds + l.segd + kPose * b;
        o[0] = t.u.x, o[1] = t.u.y, o[2] = t.u.z, o[3] = t.k, o[4] = t.s2;
        o[5] = x[0], o[6] = x[1], o[7] = x[2];
      }
      for (int i = rid; i < 3 * c.nbody; i += nt) lds[l.com + i] = com[i];
      if (MODE == MW_FORWARD)
        for (int m = rid; m < c.nmuscle; m += nt) lds[l.force + m] = a.in[w * a.ldin + m];
      if (MODE == MW_GRAD)
        for (int j = rid; j < c.ntorque; j += nt) lds[l.axis + kAxis * j + 6] = a.in[w * a.ldin + j];
    }
    __syncthreads();
    // the segments' wavefronts are the last ones, the muscles' the first: a muscle takes as long as three segments
    int nseg_threads = nt;
    int seg_tab[ST][4], length_tab[LT], first_segment = 0, last_segment = 0;
    float par[3], rest = 0.0f;
    {
      const im_muscle_context &c = ctx_args().c;
      const CtxLds l = ctx_lds<false>(c, FORCES);
      if (FORCES) nseg_threads = max(nt - ((c.nmuscle + 63) & ~63), nt / 4);
#pragma unroll
      for (int k = 0; k < ST; ++k) {
        const int sg = min(rid + k * nseg_threads, c.nsegment - 1);
        seg_tab[k][0] = c.start_waypoint[sg], seg_tab[k][1] = c.end_waypoint[sg];
        seg_tab[k][2] = c.start_root_body[sg], seg_tab[k][3] = c.end_root_body[sg];
      }
      if (FORCES) {
        const int m = min(tid, c.nmuscle - 1);
        first_segment = c.all_segment_offsets[m], last_segment = c.all_segment_offsets[m + 1];
#pragma unroll
        for (int k = 0; k < 3; ++k) par[k] = c.params[m * c.ld_params + k];
        rest = c.rest[m];
      }
      float *wpl = lds + l.contrib;
      auto waypoint = [&](int i, int body, V3 local) __attribute__((always_inline)) {
        const float *o = lds + l.segd + kPose * body;
        const V3 p = add({o[5], o[6], o[7]}, turned({{o[0], o[1], o[2]}, o[3], o[4]}, local));
        wpl[3 * i] = p.x, wpl[3 * i + 1] = p.y, wpl[3 * i + 2] = p.z;
      };
#pragma unroll
      for (int k = 0; k < WT; ++k)
        if (tid + k * nt < c.nwaypoint) waypoint(tid + k * nt, wp_body[k], wp_local[k]);
      for (int i = tid + WT * nt; i < c.nwaypoint; i += nt) waypoint(i, c.waypoint_body[i], ld3(c.waypoint_local + 3 * i));
      if (tid == 0) ((int *)(lds + l.flags))[turn ^ 1] = 0;
      if (FORCES)
#pragma unroll
        for (int k = 0; k < LT; ++k) length_tab[k] = first_segment + k < last_segment ? c.all_segment_start[first_segment + k] : 0;
    }
    __syncthreads();
    {
      const CtxArgs &a = ctx_args();
      const im_muscle_context &c = a.c;
      const CtxLds l = ctx_lds<false>(c, FORCES);
      const float *wpl = lds + l.contrib;
      if (FORCES) {
        const bool passives = MODE == MW_FORWARD && c.model.include_passive;
        auto distance = [&](int i) __attribute__((always_inline)) { return length(sub(ld3(wpl + 3 * (i + 1)), ld3(wpl + 3 * i))); };
        if (tid < c.nmuscle) {
          float d[LT], len = 0.0f;
#pragma unroll
          for (int k = 0; k < LT; ++k) d[k] = distance(length_tab[k]);
#pragma unroll
          for (int k = 0; k < LT; ++k) len = first_segment + k < last_segment ? len + d[k] : len;
          for (int s = first_segment + LT; s < last_segment; ++s) len = len + distance(c.all_segment_start[s]);
          float unit, passive;
          force_of_length(len, par, rest, cosine, passives ? expf(c.model.passive[1]) - 1.0f : 1.0f, c.model, &unit,
                          MODE == MW_FORWARD ? &passive : nullptr);
          if (MODE == MW_FORWARD) {
            unit = unit * lds[l.force + tid];
            if (passives) unit = unit + passive;
          }
          lds[l.force + tid] = unit;
        }
      }
      auto segment = [&](int sg, int w0, int w1, int b0, int b1) __attribute__((always_inline)) {
        const V3 p0 = ld3(wpl + 3 * w0), p1 = ld3(wpl + 3 * w1);
        const V3 r0 = sub(p0, ld3(lds + l.com + 3 * b0)), r1 = sub(p1, ld3(lds + l.com + 3 * b1));
        const V3 seg = sub(p1, p0);
        const float len = length(seg);
        const bool ok = !(len < 1.0e-8f);  // (as in muscle_world_kernel)
        float *o = lds + l.segd + 9 * sg;
        o[0] = ok ? seg.x / len : 0.0f;
        o[1] = ok ? seg.y / len : 0.0f;
        o[2] = ok ? seg.z / len : 0.0f;
        o[3] = r0.x, o[4] = r0.y, o[5] = r0.z;
        o[6] = r1.x, o[7] = r1.y, o[8] = r1.z;
        const float all = fabsf(r0.x) + fabsf(r0.y) + fabsf(r0.z) + fabsf(r1.x) + fabsf(r1.y) + fabsf(r1.z);
        if (!(all < kCtxLarge)) ((int *)(lds + l.flags))[turn] = 1;
      };
#pragma unroll
      for (int k = 0; k < ST; ++k)
        if (rid < nseg_threads && rid + k * nseg_threads < c.nsegment)
          segment(rid + k * nseg_threads, seg_tab[k][0], seg_tab[k][1], seg_tab[k][2], seg_tab[k][3]);
      for (int sg = rid + ST * nseg_threads; rid < nseg_threads && sg < c.nsegment; sg += nseg_threads)
        segment(sg, c.start_waypoint[sg], c.end_waypoint[sg], c.start_root_body[sg], c.end_root_body[sg]);
    }
    __syncthreads();
    float line = 0.0f;
    {  // the next world's rows are brought into the L2 beside what follows: a line each 16 floats of a row
      const CtxArgs &a = ctx_args();
      const im_muscle_context &c = a.c;
      const int64_t next = w + gridDim.x < a.nworld ? w + gridDim.x : w;
      int i = 16 * rid;
      auto touch = [&](const float *row, int n) __attribute__((always_inline)) {
        if (i >= 0 && i < n) line = row[i];
        i -= (n + 15) & ~15;
      };
      touch(c.xpos + next * c.ld_xpos, 3 * c.nbody);
      touch(c.xquat + next * c.ld_xquat, 4 * c.nbody);
      touch(c.subtree_com + next * c.ld_subtree_com, 3 * c.nbody);
      touch(c.cdof + next * c.ld_cdof + 6 * a.root, 6 * c.ntorque);
      if (MODE != MW_MOMENT) touch(a.in + next * a.ldin, MODE == MW_FORWARD ? c.nmuscle : c.ntorque);
    }
    {
      const CtxArgs &a = ctx_args();
      const int npacked = a.c.npacked, single_end = a.single_end, single = a.single;
      const char *base = (const char *)lds;
      if (__builtin_expect(__builtin_amdgcn_readfirstlane(((const int *)(lds + ctx_lds<false>(a.c, FORCES).flags))[turn]) == 0, 1)) {
#pragma unroll
        for (int k = 0; k < TRIPS; ++k) {
          const int first = k * nt + wave;  // the wavefront's entries of this trip are of one kind
          if (first < npacked) {
            unsigned records = kept[k].x, place = kept[k].y;
            asm volatile("" : "+v"(records), "+v"(place));  // (their parts are not kept from world to world)
            const float *sd = (const float *)(base + (records & 0xFFFFu)), *cd = (const float *)(base + (records >> 16));
            const float f = MODE == MW_MOMENT ? 1.0f : *(const float *)(base + (place >> 16));
            float v;
            if (first >= single)
              v = both_ends(cd, sd, f);
            else
              v = one_end(cd, sd, sd + (first < single_end ? 6 : 3), first < single_end ? 0x80000000u : 0u, f);
            if (MODE != MW_MOMENT) v = f == 0.0f ? 0.0f : v;
            if (MODE == MW_GRAD) v = cd[6] * v;
            if (k * nt + tid < npacked) *(float *)((char *)lds + (place & 0xFFFFu)) = v;
          }
          if (k % 2) __builtin_amdgcn_sched_barrier(0);
        }
      } else {
        const CtxLds l = ctx_lds<false>(a.c, FORCES);
        for (int e = tid; e < npacked; e += nt)
          full_contribution<MODE>(lds, l, ((const uint2 *)a.c.packed)[e], e < single_end, e >= single_end && e < single);
      }
    }
    asm volatile("" : : "v"(line));
    __syncthreads();
    {
      const CtxArgs &a = ctx_args();
      for (int r = tid; r < a.c.nrow; r += nt) {
        const float sum = ordered_sum<MODE != MW_MOMENT>(lds, a.c.offsets[r], a.c.offsets[r + 1]);
        a.out[w * a.ldo + r] = MODE == MW_GRAD && lds[ctx_lds<false>(a.c, FORCES).force + r] == 0.0f ? 0.0f : sum;
      }
    }
  }
}

// ---- the same with the list in groups ---------------------------------------------------------
// What bounds the kernel above is the vector issue rate and the LDS together, and of its 7800 instructions a world (284
// muscles, torque) the entries' own arithmetic is 2000: the others fetch and unpack each entry's two records, form
// table addresses for every world, take a muscle's lengths on a lane that waits for the longest.  Here up to three
// entries share what they have in common.  Torque and gradient: entries of one segment and kind (the dofs of a
// joint; 2.6 a group), so that the segment's record is read and the force put on its direction once a group.  Moment:
// a row's whole list on one thread, its dof's record read once and the ordered sum formed in a register.  The 64
// groups of a wavefront are of one kind and number.  A waypoint's, a segment's and a muscle's table entries are one
// aligned load each, from tables that are filled up to whole wavefronts; a body's record is two 16-byte reads; every
// segment's length is taken by a lane of its own, at the price of a barrier.
// 4096 worlds of 284 muscles, entry by entry -> in groups: torque 78.1 -> 63.1 us, gradient 68.5 -> 56.0, moment 57.9 -> 48.0; 120
// muscles x 8192 68.1 / 63.2 / 52.2 -> 56.5 / 52.7 / 44.3; 40 x 8192 31.6 / 30.4 / 24.9 -> 29.6 / 28.2 / 24.8.  Of the
// torque's time the entries are 21 us, waypoints, records and lengths 20, ordered sums 10, forces 6.  Not kept: the dofs'
// and the segments' records in 8 and 12 words for 16-byte reads (more bank conflicts: 65 / 63 / 53); groups by dof ahead of
// segment (70 / 64 / 60); eight wavefronts per SIMD for torque and gradient (64 registers, spills).
template <int MODE, int NT, int TRIPS, int WAVES>
__global__ __launch_bounds__(NT, WAVES) void muscle_groups_kernel(CtxArgs) {
  extern __shared__ float lds[];
  constexpr int nt = NT;
  constexpr bool FORCES = MODE != MW_MOMENT;
  int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint4 kept[TRIPS];  // LDS byte offsets, 16 bits each
  uint64_t kinds = 0;  // six bits a trip; 63: the wavefront has no groups in it
  float cosine = 1.0f, passive_scale = 1.0f;
  int turn = 0;
  {
    const CtxArgs &a = ctx_args();
    const im_muscle_context &c = a.c;
    const CtxLds l = ctx_lds<true>(c, FORCES);
    const unsigned segd = 4u * l.segd, axis = 4u * l.axis, force = 4u * l.force;
    auto both = [](unsigned lo, unsigned hi) __attribute__((always_inline)) { return lo | hi << 16; };
#pragma unroll
    for (int k = 0; k < TRIPS; ++k) {
      const int block = k * (nt / 64) + wave;
      const bool on = 64 * block < c.ngroup;
      kinds |= (uint64_t)(unsigned)__builtin_amdgcn_readfirstlane(on ? c.group_kinds[on ? block : 0] & 63 : 63) << (6 * k);
      const uint4 g = ((const uint4 *)c.groups)[(on ? 64 * block : 0) + (tid & 63)];
      const unsigned x0 = g.x & 0xFFFFu, x1 = g.x >> 16, y0 = g.y & 0xFFFFu, y1 = g.y >> 16, z0 = g.z & 0xFFFFu, z1 = g.z >> 16;
      if (FORCES)
        kept[k] = {both(segd + 36 * x0, axis + 4 * kAxis * x1), both(axis + 4 * kAxis * y0, axis + 4 * kAxis * y1), both(force + 4 * z0, 4 * z1),
                   both(4 * (g.w & 0xFFFFu), 4 * (g.w >> 16))};
      else
        kept[k] = {both(axis + 4 * kAxis * x0, 4 * x1), both(segd + 36 * y0, segd + 36 * y1), segd + 36 * z0, 0};
    }
    if (FORCES) cosine = cosf(c.params[min(tid, c.nmuscle - 1) * c.ld_params + 3]);
    if (MODE == MW_FORWARD) passive_scale = uniform(expf(c.model.passive[1]) - 1.0f);
    if (tid < 2) ((int *)(lds + l.flags))[tid] = 0;
    __syncthreads();
  }
  // Table entries of a phase are asked for a phase ahead, behind its barrier (this many a thread; what is beyond is read
  // where it is used).
  constexpr int WT = 3, ST = 2;
  for (int64_t w = blockIdx.x; w < ctx_args().nworld; w += gridDim.x, turn ^= 1) {
    asm volatile("" : "+v"(tid));  // (no address formed from it is kept from world to world)
    const int rid = nt - 1 - tid, rwave = nt - 64 - 64 * wave;
    float4 wp_tab[WT];
    {  // poses, centres, axes; activations where the forces will be
      const CtxArgs &a = ctx_args();
      const im_muscle_context &c = a.c;
      const CtxLds l = ctx_lds<true>(c, FORCES);
#pragma unroll
      for (int k = 0; k < WT; ++k)
        if (k * nt + 64 * wave < c.nwaypoint) wp_tab[k] = ((const float4 *)c.waypoint_table + k * nt)[(unsigned)tid];
      const float *com = c.subtree_com + w * c.ld_subtree_com, *cdof = c.cdof + w * c.ld_cdof + 6 * a.root;
      for (int i = rid; i < 6 * c.ntorque; i += nt) {
        const float v = cdof[(unsigned)i];
        lds[l.axis + i + i / 6] = v;
        if (!(fabsf(v) < kCtxLarge)) ((int *)(lds + l.flags))[turn] = 1;
      }
      for (int b = rid; b < c.nbody; b += nt) {
        const float *x = c.xpos + w * c.ld_xpos + 3 * b;
        const BodyTurn t = body_turn(c.xquat + w * c.ld_xquat + 4 * b);
        float *o = lds + l.segd + kPose * b;
        *(float4 *)o = {t.u.x, t.u.y, t.u.z, t.k};
        *(float4 *)(o + 4) = {t.s2, x[0], x[1], x[2]};
      }
      for (int i = rid; i < 3 * c.nbody; i += nt) lds[l.com + i] = com[(unsigned)i];
      const float *in = a.in + w * a.ldin;
      if (MODE == MW_FORWARD)
        for (int m = rid; m < c.nmuscle; m += nt) lds[l.force + m] = in[(unsigned)m];
      if (MODE == MW_GRAD)
        for (int j = rid; j < c.ntorque; j += nt) lds[l.axis + kAxis * j + 6] = in[(unsigned)j];
    }
    __syncthreads();
    uint2 seg_tab[ST];
    unsigned len_tab[ST];
    {
      const im_muscle_context &c = ctx_args().c;
      const CtxLds l = ctx_lds<true>(c, FORCES);
#pragma unroll
      for (int k = 0; k < ST; ++k) {
        if (k * nt + rwave < c.nsegment) seg_tab[k] = ((const uint2 *)c.segment_table + k * nt)[(unsigned)rid];
        if (FORCES && k * nt + 64 * wave < c.nlength) len_tab[k] = (c.length_table + k * nt)[(unsigned)tid];
      }
      float *wpl = lds + l.contrib;
      auto waypoint = [&](int i, float4 t) __attribute__((always_inline)) {
        const float *o = (const float *)((const char *)(lds + l.segd) + __builtin_bit_cast(unsigned, t.w));
        const float4 lo = *(const float4 *)o, hi = *(const float4 *)(o + 4);
        const V3 p = add({hi.y, hi.z, hi.w}, turned({{lo.x, lo.y, lo.z}, lo.w, hi.x}, {t.x, t.y, t.z}));
        wpl[3 * i] = p.x, wpl[3 * i + 1] = p.y, wpl[3 * i + 2] = p.z;
      };
#pragma unroll
      for (int k = 0; k < WT; ++k)
        if (tid + k * nt < c.nwaypoint) waypoint(tid + k * nt, wp_tab[k]);
      for (int i = tid + WT * nt; i < c.nwaypoint; i += nt) waypoint(i, ((const float4 *)c.waypoint_table)[(unsigned)i]);
      if (tid == 0) ((int *)(lds + l.flags))[turn ^ 1] = 0;
    }
    __syncthreads();
    uint4 run{};
    float4 par{};
    {  // segments' records, and every segment's length
      const im_muscle_context &c = ctx_args().c;
      const CtxLds l = ctx_lds<true>(c, FORCES);
      if (FORCES && 64 * wave < c.nmuscle) {
        run = ((const uint4 *)c.muscle_table)[2u * tid];
        par = ((const float4 *)c.muscle_table)[2u * tid + 1];
      }
      const char *points = (const char *)(lds + l.contrib), *centres = (const char *)(lds + l.com);
      auto point = [&](unsigned at) __attribute__((always_inline)) { return ld3((const float *)(points + at)); };
      auto segment = [&](int sg, uint2 t) __attribute__((always_inline)) {
        const V3 p0 = point(t.x & 0xFFFFu), p1 = point(t.x >> 16);
        const V3 r0 = sub(p0, ld3((const float *)(centres + (t.y & 0xFFFFu)))), r1 = sub(p1, ld3((const float *)(centres + (t.y >> 16))));
        const V3 seg = sub(p1, p0);
        const float len = length(seg);
        const bool ok = !(len < 1.0e-8f);  // (as in muscle_world_kernel)
        float *o = lds + l.segd + 9 * sg;
        o[0] = ok ? seg.x / len : 0.0f;
        o[1] = ok ? seg.y / len : 0.0f;
        o[2] = ok ? seg.z / len : 0.0f;
        o[3] = r0.x, o[4] = r0.y, o[5] = r0.z;
        o[6] = r1.x, o[7] = r1.y, o[8] = r1.z;
        const float all = fabsf(r0.x) + fabsf(r0.y) + fabsf(r0.z) + fabsf(r1.x) + fabsf(r1.y) + fabsf(r1.z);
        if (!(all < kCtxLarge)) ((int *)(lds + l.flags))[turn] = 1;
      };
      auto distance = [&](unsigned at) __attribute__((always_inline)) { return length(sub(point(at + 12), point(at))); };
#pragma unroll
      for (int k = 0; k < ST; ++k)
        if (rid + k * nt < c.nsegment) segment(rid + k * nt, seg_tab[k]);
      for (int sg = rid + ST * nt; sg < c.nsegment; sg += nt) segment(sg, ((const uint2 *)c.segment_table)[(unsigned)sg]);
      if (FORCES) {
#pragma unroll
        for (int k = 0; k < ST; ++k)
          if (tid + k * nt < c.nlength) lds[l.dist + tid + k * nt] = distance(len_tab[k]);
        for (int i = tid + ST * nt; i < c.nlength; i += nt) lds[l.dist + i] = distance(c.length_table[(unsigned)i]);
      }
    }
    __syncthreads();
    float line = 0.0f;
    int e0 = 0, e1 = 0;  // the list of the thread's first row
    {  // the next world's rows are brought into the L2 beside what follows: a line each 16 floats of a row
      const CtxArgs &a = ctx_args();
      const im_muscle_context &c = a.c;
      const int64_t next = w + gridDim.x < a.nworld ? w + gridDim.x : w;
      const int nin = MODE == MW_MOMENT ? 0 : MODE == MW_FORWARD ? c.nmuscle : c.ntorque;
      if (16 * rwave < 10 * c.nbody + 6 * c.ntorque + nin + 5 * 16) {  // (no lane of the other wavefronts has a line)
        int i = 16 * rid;
        auto touch = [&](const float *row, int n) __attribute__((always_inline)) {
          if (i >= 0 && i < n) line = row[i];
          i -= (n + 15) & ~15;
        };
        touch(c.xpos + next * c.ld_xpos, 3 * c.nbody);
        touch(c.xquat + next * c.ld_xquat, 4 * c.nbody);
        touch(c.subtree_com + next * c.ld_subtree_com, 3 * c.nbody);
        touch(c.cdof + next * c.ld_cdof + 6 * a.root, 6 * c.ntorque);
        if (MODE != MW_MOMENT) touch(a.in + next * a.ldin, nin);
      }
      if (64 * wave < c.nrow && tid < c.nrow) e0 = c.offsets[(unsigned)tid], e1 = c.offsets[(unsigned)tid + 1];
    }
    if constexpr (FORCES) {
      const im_muscle_context &c = ctx_args().c;
      const CtxLds l = ctx_lds<true>(c, FORCES);
      const bool passives = MODE == MW_FORWARD && c.model.include_passive;
      if (tid < c.nmuscle) {
        const float *dist = lds + l.dist + run.x;
        const int count = (int)run.y;
        float len = 0.0f;
        for (int s = 0; s < count; s += 4) {  // (up to three past the muscle's last one are read and left out)
          float d[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) d[k] = dist[s + k];
#pragma unroll
          for (int k = 0; k < 4; ++k) len = s + k < count ? len + d[k] : len;
        }
        const float lengths[3] = {__builtin_bit_cast(float, run.z), __builtin_bit_cast(float, run.w), par.x};
        float unit, passive;
        force_of_length(len, lengths, par.y, cosine, passive_scale, c.model, &unit, MODE == MW_FORWARD ? &passive : nullptr);
        if (MODE == MW_FORWARD) {
          unit = unit * lds[l.force + tid];
          if (passives) unit = unit + passive;
        }
        lds[l.force + tid] = unit;
      }
      __syncthreads();
    }
    const bool large = __builtin_amdgcn_readfirstlane(((const int *)(lds + ctx_lds<true>(ctx_args().c, FORCES).flags))[turn]) != 0;
    {
      char *base = (char *)lds;
      auto at = [&](unsigned byte) __attribute__((always_inline)) { return (const float *)(base + byte); };
      auto vec = [&](unsigned byte) __attribute__((always_inline)) { return ld3(at(byte)); };
      struct Dof {
        V3 ang, lin;
        float gout;
      };
      auto dof = [&](unsigned byte) __attribute__((always_inline)) {
        return Dof{vec(byte), vec(byte + 12), MODE == MW_GRAD ? at(byte)[6] : 0.0f};
      };
      if (__builtin_expect(!large, 1)) {
        asm volatile("" : "+s"(kinds));  // (nor is what follows from these)
#pragma unroll
        for (int k = 0; k < TRIPS; ++k) {
          const int kind = (int)(kinds >> (6 * k)) & 63;
          if (kind == 63) break;
          uint4 g = kept[k];
          asm volatile("" : "+v"(g.x), "+v"(g.y), "+v"(g.z), "+v"(g.w));  // (their parts are not kept from world to world)
          if constexpr (FORCES) {
            const unsigned sd = g.x & 0xFFFFu;
            const float f = *at(g.z & 0xFFFFu);
            const V3 fv = scale(f, vec(sd));
            auto put = [&](unsigned place, float v, float gout) __attribute__((always_inline)) {
              v = f == 0.0f ? 0.0f : v;
              if (MODE == MW_GRAD) v = gout * v;
              *(float *)(base + place) = v;
            };
            auto all = [&](auto one) __attribute__((always_inline)) {
              if (kind >> 2 == 3) {
                const Dof d0 = dof(g.x >> 16), d1 = dof(g.y & 0xFFFFu), d2 = dof(g.y >> 16);
                put(g.z >> 16, one(d0), d0.gout), put(g.w & 0xFFFFu, one(d1), d1.gout), put(g.w >> 16, one(d2), d2.gout);
              } else {
                const Dof d0 = dof(g.x >> 16);
                put(g.z >> 16, one(d0), d0.gout);
                if (kind >> 2 == 2) {
                  const Dof d1 = dof(g.y & 0xFFFFu);
                  put(g.w & 0xFFFFu, one(d1), d1.gout);
                }
              }
            };
            if ((kind & 3) == 2) {
              const V3 r0 = vec(sd + 12), r1 = vec(sd + 24);
              all([&](const Dof &d) __attribute__((always_inline)) { return dot(sub(add(d.lin, cross(d.ang, r0)), add(d.lin, cross(d.ang, r1))), fv); });
            } else {
              const V3 r = vec(sd + ((kind & 3) == 0 ? 24 : 12));
              const unsigned sign = (kind & 3) == 0 ? 0x80000000u : 0u;
              all([&](const Dof &d) __attribute__((always_inline)) {
                return __builtin_bit_cast(float, __builtin_bit_cast(unsigned, dot(add(d.lin, cross(d.ang, r)), fv)) ^ sign);
              });
            }
          } else {
            const Dof d = dof(g.x & 0xFFFFu);
            float total = 0.0f;
#pragma unroll
            for (int s = 0; s < 3; ++s) {
              const int one = (kind >> (2 * s)) & 3;
              if (one == 3) break;
              const unsigned sd = s == 0 ? g.y & 0xFFFFu : s == 1 ? g.y >> 16 : g.z;
              const V3 dir = vec(sd);
              float v;
              if (one == 2) {
                v = dot(sub(add(d.lin, cross(d.ang, vec(sd + 12))), add(d.lin, cross(d.ang, vec(sd + 24)))), dir);
              } else {
                v = dot(add(d.lin, cross(d.ang, vec(sd + (one == 0 ? 24 : 12)))), dir);
                v = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, v) ^ (one == 0 ? 0x80000000u : 0u));
              }
              total = total + v;
            }
            *(float *)(base + (g.x >> 16)) = total;
          }
        }
      } else {
        const CtxArgs &a = ctx_args();
        const CtxLds l = ctx_lds<true>(a.c, FORCES);
        for (int e = tid; e < a.c.npacked; e += nt) full_contribution<MODE>(lds, l, ((const uint2 *)a.c.packed)[e], e < a.single_end, e >= a.single_end && e < a.single);
      }
    }
    asm volatile("" : : "v"(line));
    __syncthreads();
    {
      const CtxArgs &a = ctx_args();
      float *out = a.out + w * a.ldo;
      for (int r = tid; r < a.c.nrow; r += nt) {
        if (r != tid) e0 = a.c.offsets[r], e1 = a.c.offsets[r + 1];
        if (MODE == MW_MOMENT)
          out[(unsigned)r] = large ? ordered_sum<false>(lds, e0, e1) : lds[r];
        else
          out[(unsigned)r] = MODE == MW_GRAD && lds[ctx_lds<true>(a.c, FORCES).force + r] == 0.0f ? 0.0f : ordered_sum_ahead(lds, e0, e1);
      }
    }
  }
}

template <int NT>
int launch_resident(void (*kernel)(CtxArgs), int words, const CtxArgs &a, hipStream_t stream, int waves = 24) {
  const size_t bytes = 4 * (size_t)words;
  unsigned grid = 0;
  if (const int st = resident_grid((const void *)kernel, NT, bytes, a.nworld, &grid, waves)) return st;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(NT), bytes, stream, a);
  IM_HIP_CHECK(hipGetLastError());
  return IM_OK;
}
// The fewest threads that hold a world at ten entries each, a muscle a thread at most: a world's barriers cost
// less with fewer wavefronts to wait for, and the CU holds more worlds side by side.  Torque / gradient / moment x 8192
// worlds by threads, us: 40 muscles (655 entries) 128: 28.2 / 27.5 / 23.2, 256: 39.6 / 38.0 / 30.7, 512: 61.1 / 58.6 /
// 45.2; 120 (1882) 256: 61.9 / 59.8 / 51.2, 512: 82.9 / 76.9 / 65.6.  Between 2560 and 3584 entries 256 threads with
// fourteen each where the batch does not fit the chip at once: 200 muscles (3145) x 8192 103 / 99.7 / 76.5 against
// 112 / 103 / 84.8 with 512, but x 500 15.5 / 14.0 / 11.3 against 14.1 / 12.5 / 10.4.
template <int MODE>
int launch_context(const CtxArgs &a, hipStream_t stream) {
  const int packed = a.c.npacked, muscles = MODE == MW_MOMENT ? 0 : a.c.nmuscle;
  int ncu = 0;
  if (const int st = compute_units(&ncu)) return st;
  constexpr int trips = MODE == MW_MOMENT ? kRowTrips : kGroupTrips;
  const int groups = a.c.ngroup, with_lengths = ctx_lds<true>(a.c, MODE != MW_MOMENT).words, words = ctx_lds<false>(a.c, MODE != MW_MOMENT).words;
  // Groups: the same, with four groups a thread (six rows for the moment); for batches beyond six workgroups a CU also
  // 128 threads with five each (75 muscles x 8192 42.5 / 41.2 us with 256 of four, 38.3 / 38.2; with six each 90 muscles x 8192 gained, x 4096
  // lost) and 256 with six: 200 muscles x 8192 97.1 / 84.4 -> 88.7 / 82.4, x 2048 28.1 / 24.8 -> 26.7 / 25.2.
  // Where 128 threads take the entries one by one, groups are not always less: their fills make up whole wavefronts of each kind, and
  // a moment's rows cost more before the first world.  Entry by entry / in groups, us: torque of 60 muscles (977 entries, 576 groups) x
  // 4096 19.1 / 19.7, of 65 (1082, 576) 21.1 / 20.9, of 57 (931, 512) 19.9 / 17.7; moment of 10 muscles (198, 384) x 8192 16.5 / 18.2,
  // of 40 (657, 576) x 8192 22.5 / 23.1, of 57 (931, 640) x 1100 8.6 / 9.0, x 2000 10.6 / 10.2, of 75 (1276, 896) x 8192 31.9 / 34.9.
  const bool many = a.nworld > 6 * ncu, few_entries = packed <= kCtxTrips * 128 && muscles <= 128;
  bool grouped = groups > 0 && 4 * (size_t)with_lengths <= 64 * 1024;
  if (MODE == MW_MOMENT && few_entries) grouped = grouped && a.nworld > 7 * ncu && groups <= trips * 128 && 5 * groups <= 4 * packed;
  if (MODE != MW_MOMENT && few_entries && many && groups > trips * 128 && packed <= 8 * 128) grouped = false;
  if (grouped) {
    if (groups <= trips * 128 && muscles <= 128) return launch_resident<128>(muscle_groups_kernel<MODE, 128, trips, 6>, with_lengths, a, stream, 32);
    if constexpr (MODE != MW_MOMENT)
      if (groups <= 5 * 128 && muscles <= 128 && many) return launch_resident<128>(muscle_groups_kernel<MODE, 128, 5, 5>, with_lengths, a, stream, 32);
    if (groups <= trips * 256 && muscles <= 256) return launch_resident<256>(muscle_groups_kernel<MODE, 256, trips, 6>, with_lengths, a, stream, 32);
    if constexpr (MODE != MW_MOMENT)
      if (groups <= 6 * 256 && muscles <= 256 && many) return launch_resident<256>(muscle_groups_kernel<MODE, 256, 6, 5>, with_lengths, a, stream, 32);
    if (groups <= trips * 512) return launch_resident<512>(muscle_groups_kernel<MODE, 512, trips, 6>, with_lengths, a, stream, 32);
  }
  if (packed <= kCtxTrips * 128 && muscles <= 128) return launch_resident<128>(muscle_context_kernel<MODE, 128, kCtxTrips>, words, a, stream);
  if (packed <= kCtxTrips * 256 && muscles <= 256) return launch_resident<256>(muscle_context_kernel<MODE, 256, kCtxTrips>, words, a, stream);
  if (packed <= 14 * 256 && muscles <= 256 && many) return launch_resident<256>(muscle_context_kernel<MODE, 256, 14>, words, a, stream);
  return launch_resident<512>(muscle_context_kernel<MODE, 512, kCtxTrips>, words, a, stream);
}

bool geo_ok(const im_muscle_geometry *g) {
  return g && g->waypoints && g->subtree_com && g->cdof && g->ld_waypoints >= 0 &&
         g->ld_subtree_com >= 0 && g->ld_cdof >= 0;
}
bool seg_ok(const im_muscle_segments *s) {
  return s && s->start_waypoint && s->end_waypoint && s->start_root_body && s->end_root_body;
}
Geo geo(const im_muscle_geometry *g) {
  return {g->waypoints, g->subtree_com, g->cdof, g->ld_waypoints, g->ld_subtree_com, g->ld_cdof};
}
Seg seg(const im_muscle_segments *s) {
  return {s->start_waypoint, s->end_waypoint, s->start_root_body, s->end_root_body};
}
dim3 grid2(int n, int nworld) { return dim3((unsigned)((n + 255) / 256), (unsigned)nworld); }
constexpr int kMaxGridY = 65535;
int slab_count(int nworld, int w0) { return nworld - w0 < kMaxGridY ? nworld - w0 : kMaxGridY; }

}  // namespace
}  // namespace im

using namespace im;

// The y dimension of a grid carries the world; launches are split so that it stays within
// the limit of 65535.
#define IM_FOR_WORLD_SLABS(nworld, w0, nw)                                     \
  for (int w0 = 0, nw = slab_count(nworld, 0); w0 < (nworld); \
       w0 += kMaxGridY, nw = slab_count(nworld, w0))

extern "C" int im_muscle_waypoints(const float *xpos, int64_t ld_xpos, const float *xquat,
                                   int64_t ld_xquat, const int32_t *waypoint_body,
                                   const float *waypoint_local, int nwaypoint, float *waypoints,
                                   int64_t ld_waypoints, int nworld, void *stream) {
  if (nworld < 0 || nwaypoint < 0) return IM_ERR_ARG;
  if (nworld == 0 || nwaypoint == 0) return IM_OK;
  if (!xpos || !xquat || !waypoint_body || !waypoint_local || !waypoints) return IM_ERR_ARG;
  if (ld_waypoints < 3 * (int64_t)nwaypoint) return IM_ERR_STRIDE;
  IM_FOR_WORLD_SLABS(nworld, w0, nw) {
    hipLaunchKernelGGL(waypoints_kernel, grid2(nwaypoint, nw), dim3(256), 0, (hipStream_t)stream,
                       xpos + w0 * ld_xpos, ld_xpos, xquat + w0 * ld_xquat, ld_xquat,
                       waypoint_body, waypoint_local, nwaypoint, waypoints + w0 * ld_waypoints,
                       ld_waypoints, nw);
  }
  IM_HIP_CHECK(hipGetLastError());
  return IM_OK;
}

extern "C" int im_muscle_force_magnitudes(const float *waypoints, int64_t ld_waypoints,
                                          const int32_t *all_segment_start_idx,
                                          const int32_t *all_muscle_segment_offsets,
                                          const float *muscle_params, int ld_params,
                                          const float *muscle_rest_length,
                                          const im_muscle_force_model *model, int nmuscle,
                                          float *unit_force, int64_t ld_unit,
                                          float *passive_force, int64_t ld_passive, int nworld,
                                          void *stream) {
  if (nworld < 0 || nmuscle < 0 || !model) return IM_ERR_ARG;
  if (nworld == 0 || nmuscle == 0) return IM_OK;
  if (!waypoints || !all_segment_start_idx || !all_muscle_segment_offsets || !muscle_params ||
      !muscle_rest_length || !unit_force || ld_params < 4)
    return IM_ERR_ARG;
  if (ld_unit < nmuscle || (passive_force && ld_passive < nmuscle)) return IM_ERR_STRIDE;
  IM_FOR_WORLD_SLABS(nworld, w0, nw) {
    hipLaunchKernelGGL(force_kernel, grid2(nmuscle, nw), dim3(256), 0, (hipStream_t)stream,
                       waypoints + w0 * ld_waypoints, ld_waypoints, all_segment_start_idx,
                       all_muscle_segment_offsets, muscle_params, ld_params, muscle_rest_length,
                       *model, nmuscle, unit_force + w0 * ld_unit, ld_unit,
                       passive_force ? passive_force + w0 * ld_passive : nullptr, ld_passive);
  }
  IM_HIP_CHECK(hipGetLastError());
  return IM_OK;
}

extern "C" int im_muscle_force_velocity_state(
    const float *waypoints, int64_t ld_waypoints, const int32_t *muscle_waypoint_start,
    const float *muscle_params, int ld_params, const float *muscle_rest_length,
    const float *force_velocity_length_scale, const float *activation, int64_t ld_activation,
    const float *qvel, int64_t ld_qvel, const float *moment, int64_t ld_moment,
    const int32_t *muscle_dof_offsets, const int32_t *muscle_dof_torque_idx, int root_dof_count,
    const im_muscle_force_model *model, const im_muscle_force_velocity_model *fv, int nmuscle,
    float *muscle_length, float *effective_activation, float *length_velocity,
    float *force_velocity_multiplier, float *force_velocity_slope, int64_t ld_out, int nworld, void *stream) {
  if (nworld < 0 || nmuscle < 0 || root_dof_count < 0) return IM_ERR_ARG;
  if (nworld == 0 || nmuscle == 0) return IM_OK;
  if (!waypoints || !muscle_waypoint_start || !muscle_params || !muscle_rest_length ||
      !force_velocity_length_scale || !activation || !qvel || !moment || !muscle_dof_offsets ||
      !muscle_dof_torque_idx || !model || !fv || !muscle_length || !effective_activation || !length_velocity ||
      !force_velocity_multiplier || !force_velocity_slope || ld_params < 4)
    return IM_ERR_ARG;
  if (ld_out < nmuscle || ld_activation < nmuscle) return IM_ERR_STRIDE;
  // a world's rows of waypoints, moments and velocities staged in LDS when they fit (the rows'
  // strides bound what the tables can address); IMHIP_MUSCLE_KERNEL=simple keeps the lane-per-muscle kernel
  static const bool forced_off = [] {
    const char *e = std::getenv("IMHIP_MUSCLE_KERNEL");
    return e && std::strcmp(e, "simple") == 0;
  }();
  // Beside the distances, the entries' dofs and a cosine per muscle.  Up to 80 KB, where a CU holds two
  // workgroups: 4096 worlds of 284 muscles with velocities in rows of 56 / 8000 / 12000 floats (37 / 69 / 85 KB)
  // take 38.0 / 53.6 / 92.4 us here and 81 - 83 us on the lane-per-muscle kernel.
  const FvLds n{(int)std::min<int64_t>(ld_waypoints, 1 << 20), (int)std::min<int64_t>(ld_moment, 1 << 20),
                (int)std::min<int64_t>(ld_qvel, 1 << 20), nmuscle};
  if (!forced_off && ld_waypoints > 0 && ld_moment > 0 && ld_qvel > 0 && nmuscle <= 16 * 1024 && n.bytes() <= 80 * 1024) {
    // (a batch of up to four workgroups per CU, all resident at once, has the threads to spare: 1000 worlds of
    // 100 muscles 7.7 us with 320 threads, 8.4 with 128)
    int ncu = 0;
    if (const int st = compute_units(&ncu)) return st;
    const int threads = nworld <= 4 * ncu ? 320 : std::min(std::max((nmuscle + 63) / 64 * 64, 128), 320);
    const bool ahead = n.words_wp <= 14 * threads && n.nentry <= 9 * threads && n.nqvel <= threads;
#define IM_FV(NT) (ahead ? force_velocity_state_world_kernel<NT, true> : force_velocity_state_world_kernel<NT, false>)
    auto kernel = threads == 128 ? IM_FV(128) : threads == 192 ? IM_FV(192) : threads == 256 ? IM_FV(256) : IM_FV(320);
#undef IM_FV
    if (n.bytes() > 64 * 1024)
      IM_HIP_CHECK(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, n.bytes()));
    unsigned grid = 0;
    if (const int st = resident_grid((const void *)kernel, threads, (size_t)n.bytes(), nworld, &grid)) return st;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads),
                       (size_t)n.bytes(), (hipStream_t)stream, waypoints, ld_waypoints, muscle_waypoint_start,
                       muscle_params, ld_params, muscle_rest_length, force_velocity_length_scale, activation,
                       ld_activation, qvel, ld_qvel, moment, ld_moment, muscle_dof_offsets, muscle_dof_torque_idx,
                       root_dof_count, *model, *fv, n, muscle_length, effective_activation, length_velocity,
                       force_velocity_multiplier, force_velocity_slope, ld_out, nworld);
    IM_HIP_CHECK(hipGetLastError());
    return IM_OK;
  }
  IM_FOR_WORLD_SLABS(nworld, w0, nw) {
    hipLaunchKernelGGL(force_velocity_state_kernel, grid2(nmuscle, nw), dim3(256), 0, (hipStream_t)stream,
                       waypoints + w0 * ld_waypoints, ld_waypoints, muscle_waypoint_start, muscle_params, ld_params,
                       muscle_rest_length, force_velocity_length_scale, activation + w0 * ld_activation,
                       ld_activation, qvel + w0 * ld_qvel, ld_qvel, moment + w0 * ld_moment, ld_moment,
                       muscle_dof_offsets, muscle_dof_torque_idx, root_dof_count, *model, *fv, nmuscle,
                       muscle_length + w0 * ld_out, effective_activation + w0 * ld_out, length_velocity + w0 * ld_out,
                       force_velocity_multiplier + w0 * ld_out, force_velocity_slope + w0 * ld_out, ld_out);
  }
  IM_HIP_CHECK(hipGetLastError());
  return IM_OK;
}

extern "C" int im_muscle_waypoints_forces(
    const float *xpos, int64_t ld_xpos, const float *xquat, int64_t ld_xquat,
    const int32_t *waypoint_body, const float *waypoint_local, int nwaypoint, float *waypoints,
    int64_t ld_waypoints, const int32_t *all_segment_start_idx,
    const int32_t *all_muscle_segment_offsets, const float *muscle_params, int ld_params,
    const float *muscle_rest_length, const im_muscle_force_model *model, int nmuscle,
    float *unit_force, int64_t ld_unit, float *passive_force, int64_t ld_passive, int nworld,
    void *stream) {
  const size_t lds_bytes = (size_t)12 * (nwaypoint > 0 ? nwaypoint : 0);
  if (nworld <= 0 || nwaypoint <= 0 || nmuscle <= 0 || lds_bytes > 64 * 1024) {
    // nothing to share between the two, or a world's waypoints do not fit in LDS
    const int rc = im_muscle_waypoints(xpos, ld_xpos, xquat, ld_xquat, waypoint_body,
                                       waypoint_local, nwaypoint, waypoints, ld_waypoints, nworld,
                                       stream);
    if (rc != IM_OK) return rc;
    return im_muscle_force_magnitudes(waypoints, ld_waypoints, all_segment_start_idx,
                                      all_muscle_segment_offsets, muscle_params, ld_params,
                                      muscle_rest_length, model, nmuscle, unit_force, ld_unit,
                                      passive_force, ld_passive, nworld, stream);
  }
  if (!model || !xpos || !xquat || !waypoint_body || !waypoint_local || !waypoints ||
      !all_segment_start_idx || !all_muscle_segment_offsets || !muscle_params ||
      !muscle_rest_length || !unit_force || ld_params < 4)
    return IM_ERR_ARG;
  if (ld_waypoints < 3 * (int64_t)nwaypoint || ld_unit < nmuscle ||
      (passive_force && ld_passive < nmuscle))
    return IM_ERR_STRIDE;
  hipLaunchKernelGGL(waypoints_forces_kernel, dim3((unsigned)nworld), dim3(512), lds_bytes,
                     (hipStream_t)stream, xpos, ld_xpos, xquat, ld_xquat, waypoint_body,
                     waypoint_local, nwaypoint, waypoints, ld_waypoints, all_segment_start_idx,
                     all_muscle_segment_offsets, muscle_params, ld_params, muscle_rest_length,
                     *model, nmuscle, unit_force, ld_unit, passive_force, ld_passive);
  IM_HIP_CHECK(hipGetLastError());
  return IM_OK;
}

static Geo slab(const im_muscle_geometry *g, int64_t w0) {
  Geo r = geo(g);
  r.wp += w0 * r.ldw;
  r.com += w0 * r.ldc;
  r.cdof += w0 * r.ldd;
  return r;
}

extern "C" int im_muscle_torque_forward(const im_muscle_geometry *geometry,
                                        const im_muscle_segments *segments,
                                        const im_muscle_entries *torque_entries,
                                        const float *unit_force, int64_t ld_unit,
                                        const float *passive_force, int64_t ld_passive,
                                        const float *activation, int64_t ld_activation,
                                        int root_dof_count, float *torque, int64_t ld_torque,
                                        int nworld, void *stream) {
  if (nworld < 0 || !torque_entries || torque_entries->nrow < 0 || root_dof_count < 0)
    return IM_ERR_ARG;
  const int nt = torque_entries->nrow;
  if (nworld == 0 || nt == 0) return IM_OK;
  if (!geo_ok(geometry) || !seg_ok(segments) || !torque_entries->offsets || !unit_force ||
      !activation || !torque)
    return IM_ERR_ARG;
  if (torque_entries->nentry > 0 && (!torque_entries->segment || !torque_entries->other ||
                                     !torque_entries->start_coeff || !torque_entries->end_coeff))
    return IM_ERR_ARG;
  if (ld_torque < nt) return IM_ERR_STRIDE;
  {
    MwArgs a{geo(geometry), seg(segments), torque_entries->offsets, torque_entries->segment,
             torque_entries->other, nullptr, torque_entries->start_coeff, torque_entries->end_coeff,
             unit_force, passive_force, activation, nullptr, ld_unit, ld_passive, ld_activation, 0,
             torque, nullptr, ld_torque, root_dof_count, nt, torque_entries->nentry,
             segments->nsegment, nt, torque_entries->nother};
    if (launch_world<MW_FORWARD>(a, nworld, (hipStream_t)stream)) {
      IM_HIP_CHECK(hipGetLastError());
      return IM_OK;
    }
  }
  IM_FOR_WORLD_SLABS(nworld, w0, nw) {
    hipLaunchKernelGGL(torque_forward_kernel, grid2(nt, nw), dim3(256), 0, (hipStream_t)stream,
                       slab(geometry, w0), seg(segments), torque_entries->offsets,
                       torque_entries->segment, torque_entries->other,
                       torque_entries->start_coeff, torque_entries->end_coeff,
                       unit_force + w0 * ld_unit, ld_unit,
                       passive_force ? passive_force + w0 * ld_passive : nullptr, ld_passive,
                       activation + w0 * ld_activation, ld_activation, root_dof_count, nt,
                       torque + w0 * ld_torque, ld_torque);
  }
  IM_HIP_CHECK(hipGetLastError());
  return IM_OK;
}

extern "C" int im_muscle_activation_grad(const im_muscle_geometry *geometry,
                                         const im_muscle_segments *segments,
                                         const im_muscle_entries *muscle_entries,
                                         const float *unit_force, int64_t ld_unit,
                                         const float *grad_output, int64_t ld_grad_output,
                                         int root_dof_count, float *grad_activation,
                                         int64_t ld_grad_activation, int nworld, void *stream) {
  if (nworld < 0 || !muscle_entries || muscle_entries->nrow < 0 || root_dof_count < 0)
    return IM_ERR_ARG;
  const int nm = muscle_entries->nrow;
  if (nworld == 0 || nm == 0) return IM_OK;
  if (!geo_ok(geometry) || !seg_ok(segments) || !muscle_entries->offsets || !unit_force ||
      !grad_output || !grad_activation)
    return IM_ERR_ARG;
  if (muscle_entries->nentry > 0 && (!muscle_entries->segment || !muscle_entries->other ||
                                     !muscle_entries->start_coeff || !muscle_entries->end_coeff))
    return IM_ERR_ARG;
  if (ld_grad_activation < nm || ld_unit < nm) return IM_ERR_STRIDE;
  {
    MwArgs a{geo(geometry), seg(segments), muscle_entries->offsets, muscle_entries->segment,
             muscle_entries->other, nullptr, muscle_entries->start_coeff, muscle_entries->end_coeff,
             unit_force, nullptr, nullptr, grad_output, ld_unit, 0, 0, ld_grad_output,
             grad_activation, nullptr, ld_grad_activation, root_dof_count, nm, muscle_entries->nentry,
             segments->nsegment, muscle_entries->nother, nm};
    if (launch_world<MW_GRAD>(a, nworld, (hipStream_t)stream)) {
      IM_HIP_CHECK(hipGetLastError());
      return IM_OK;
    }
  }
  IM_FOR_WORLD_SLABS(nworld, w0, nw) {
    hipLaunchKernelGGL(activation_grad_kernel, grid2(nm, nw), dim3(256), 0, (hipStream_t)stream,
                       slab(geometry, w0), seg(segments), muscle_entries->offsets,
                       muscle_entries->segment, muscle_entries->other,
                       muscle_entries->start_coeff, muscle_entries->end_coeff,
                       unit_force + w0 * ld_unit, ld_unit, grad_output + w0 * ld_grad_output,
                       ld_grad_output, root_dof_count, nm,
                       grad_activation + w0 * ld_grad_activation, ld_grad_activation);
  }
  IM_HIP_CHECK(hipGetLastError());
  return IM_OK;
}

extern "C" int im_muscle_sparse_moment(const im_muscle_geometry *geometry,
                                       const im_muscle_segments *segments,
                                       const int32_t *muscle_dof_torque_idx,
                                       const im_muscle_entries *entry_segments,
                                       int root_dof_count, float *moment, int64_t ld_moment,
                                       int nworld, void *stream) {
  if (nworld < 0 || !entry_segments || entry_segments->nrow < 0 || root_dof_count < 0)
    return IM_ERR_ARG;
  const int ne = entry_segments->nrow;
  if (nworld == 0 || ne == 0) return IM_OK;
  if (!geo_ok(geometry) || !seg_ok(segments) || !muscle_dof_torque_idx ||
      !entry_segments->offsets || !moment)
    return IM_ERR_ARG;
  if (entry_segments->nentry > 0 && (!entry_segments->segment || !entry_segments->start_coeff ||
                                     !entry_segments->end_coeff))
    return IM_ERR_ARG;
  if (ld_moment < ne) return IM_ERR_STRIDE;
  {
    MwArgs a{geo(geometry), seg(segments), entry_segments->offsets, entry_segments->segment, nullptr,
             muscle_dof_torque_idx, entry_segments->start_coeff, entry_segments->end_coeff, nullptr,
             nullptr, nullptr, nullptr, 0, 0, 0, 0, moment, nullptr, ld_moment, root_dof_count, ne,
             entry_segments->nentry, segments->nsegment, entry_segments->nother, 0};
    if (launch_world<MW_MOMENT>(a, nworld, (hipStream_t)stream)) {
      IM_HIP_CHECK(hipGetLastError());
      return IM_OK;
    }
  }
  IM_FOR_WORLD_SLABS(nworld, w0, nw) {
    hipLaunchKernelGGL(sparse_moment_kernel, grid2(ne, nw), dim3(256), 0, (hipStream_t)stream,
                       slab(geometry, w0), seg(segments), muscle_dof_torque_idx,
                       entry_segments->offsets, entry_segments->segment,
                       entry_segments->start_coeff, entry_segments->end_coeff, root_dof_count, ne,
                       moment + w0 * ld_moment, ld_moment);
  }
  IM_HIP_CHECK(hipGetLastError());
  return IM_OK;
}

extern "C" int im_muscle_torque_bounds(const im_muscle_geometry *geometry,
                                       const im_muscle_segments *segments,
                                       const im_muscle_entries *torque_entries,
                                       const float *unit_force, int64_t ld_unit, int root_dof_count,
                                       float *lower, float *upper, int64_t ld_bounds, int nworld,
                                       void *stream) {
  if (nworld < 0 || !torque_entries || torque_entries->nrow < 0 || root_dof_count < 0)
    return IM_ERR_ARG;
  const int nt = torque_entries->nrow;
  if (nworld == 0 || nt == 0) return IM_OK;
  if (!geo_ok(geometry) || !seg_ok(segments) || !torque_entries->offsets || !unit_force || !lower ||
      !upper)
    return IM_ERR_ARG;
  if (torque_entries->nentry > 0 && (!torque_entries->segment || !torque_entries->other ||
                                     !torque_entries->start_coeff || !torque_entries->end_coeff))
    return IM_ERR_ARG;
  if (ld_bounds < nt) return IM_ERR_STRIDE;
  {
    MwArgs a{geo(geometry), seg(segments), torque_entries->offsets, torque_entries->segment,
             torque_entries->other, nullptr, torque_entries->start_coeff, torque_entries->end_coeff,
             unit_force, nullptr, nullptr, nullptr, ld_unit, 0, 0, 0, lower, upper, ld_bounds,
             root_dof_count, nt, torque_entries->nentry, segments->nsegment, nt,
             torque_entries->nother};
    if (launch_world<MW_BOUNDS>(a, nworld, (hipStream_t)stream)) {
      IM_HIP_CHECK(hipGetLastError());
      return IM_OK;
    }
  }
  IM_FOR_WORLD_SLABS(nworld, w0, nw) {
    hipLaunchKernelGGL(torque_bounds_kernel, grid2(nt, nw), dim3(256), 0, (hipStream_t)stream,
                       slab(geometry, w0), seg(segments), torque_entries->offsets,
                       torque_entries->segment, torque_entries->other,
                       torque_entries->start_coeff, torque_entries->end_coeff,
                       unit_force + w0 * ld_unit, ld_unit, root_dof_count, nt,
                       lower + w0 * ld_bounds, upper + w0 * ld_bounds, ld_bounds);
  }
  IM_HIP_CHECK(hipGetLastError());
  return IM_OK;
}

extern "C" int im_muscle_from_context(const im_muscle_context *context, int what, const float *in, int64_t ld_in,
                                      int root_dof_count, float *out, int64_t ld_out, int nworld, void *stream) {
  if (!context || nworld < 0 || root_dof_count < 0 || what < 0 || what > 2) return IM_ERR_ARG;
  const im_muscle_context &c = *context;
  const int packed = c.kind_count[0] + c.kind_count[1] + c.kind_count[2];
  if (c.nbody <= 0 || c.nwaypoint <= 0 || c.nsegment <= 0 || c.ntorque <= 0 || c.nmuscle <= 0 || c.nrow <= 0 || c.nentry <= 0 || c.npacked != packed ||
      c.kind_count[0] < 0 || c.kind_count[1] < 0 || c.kind_count[2] < 0 || c.kind_count[0] % 64 || c.kind_count[1] % 64 || c.ld_params < 4)
    return IM_ERR_ARG;
  if (c.npacked > kCtxMost || (what != IM_MUSCLE_MOMENT && c.nmuscle > kCtxMuscles) || 4 * (size_t)c.nentry + 16 * (size_t)c.nwaypoint + 36 * (size_t)c.nsegment + 28 * (size_t)c.ntorque + 8 * (size_t)c.nmuscle > 256 * 1024 ||
      c.nbody > 65535 || 4 * (size_t)ctx_lds<false>(c, true).words > 64 * 1024)
    return IM_ERR_UNSUPPORTED;
  static const bool forced_off = [] {
    const char *e = std::getenv("IMHIP_MUSCLE_KERNEL");
    return e && std::strcmp(e, "simple") == 0;
  }();
  if (forced_off) return IM_ERR_UNSUPPORTED;
  if (nworld == 0) return IM_OK;
  if (!c.xpos || !c.xquat || !c.subtree_com || !c.cdof || !c.waypoint_body || !c.waypoint_local || !c.start_waypoint || !c.end_waypoint ||
      !c.start_root_body || !c.end_root_body || !c.offsets || !c.packed || ((uintptr_t)c.packed & 7) || !out)
    return IM_ERR_ARG;
  if (c.ngroup < 0 || c.ngroup % 64 || (c.ngroup > 0 && (c.nlength < 0 || c.nlength > 256 * 1024))) return IM_ERR_ARG;
  if (c.ngroup > 0 && (!c.waypoint_table || !c.segment_table || !c.muscle_table || !c.length_table || !c.groups || !c.group_kinds ||
                       (((uintptr_t)c.waypoint_table | (uintptr_t)c.segment_table | (uintptr_t)c.muscle_table | (uintptr_t)c.groups) & 15)))
    return IM_ERR_ARG;
  if (what != IM_MUSCLE_MOMENT && (!c.all_segment_start || !c.all_segment_offsets || !c.params || !c.rest || !in)) return IM_ERR_ARG;
  if (c.ld_xpos < 0 || c.ld_xquat < 0 || c.ld_subtree_com < 0 || c.ld_cdof < 0 || ld_in < 0 || ld_out < c.nrow ||
      (what == IM_MUSCLE_GRAD && c.nrow > c.nmuscle))
    return IM_ERR_STRIDE;
  const CtxArgs a{c, in, ld_in, out, ld_out, root_dof_count, nworld, c.kind_count[0], c.kind_count[0] + c.kind_count[1]};
  return what == IM_MUSCLE_TORQUE ? launch_context<MW_FORWARD>(a, (hipStream_t)stream)
         : what == IM_MUSCLE_GRAD ? launch_context<MW_GRAD>(a, (hipStream_t)stream)
                                  : launch_context<MW_MOMENT>(a, (hipStream_t)stream);
}
