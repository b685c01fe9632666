// What the launches of one whole constraint solve (im_newton_solve) share: the start, the first factor
// stage and the resident loop, three launches on the caller's stream.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cstdint>

#include "../../include/imhip.h"
#include "common.h"

namespace im {

// What the launch of the start also does for a whole solve.
struct WholeSolve {
  const float *start = nullptr;  // (nworld, ld_start): where a world with rows starts (null: qacc as it lies there)
  int64_t ld_start = 0;
  int *counter = nullptr;  // the resident loop's counter of worlds handed out, set to counter_value
  int counter_value = 0;
  int active = 0;  // nsolving = nworld; a world without rows gets a zero constraint force
};
int newton_init_launch(const im_newton_args *p, const float *qacc_smooth, int64_t ld_qacc_smooth, const float *efc_aref,
                       int64_t ld_aref, int nv, int nM, const WholeSolve &whole, hipStream_t stream);

// The resident loops' launchers.  With `before`, it is called once the launch's shape is known (it issues
// the start, which also sets `counter`, and the first factor stage); without, the counter is set by a
// launch of its own.  A world then writes its final constraint force itself.
struct Before {
  virtual int operator()(int *counter, int value) = 0;
};
int newton_solve_tree(const im_tree_plan *plan, const im_newton_args *p, hipStream_t stream, Before *before);
int newton_solve_sparse(const im_sparse_plan *plan, const im_newton_args *p, float *hfactor, int32_t *dof_union,
                        hipStream_t stream, Before *before);
int newton_solve_dense_tile(const im_newton_args *p, float *H, int32_t *dof_union, int nv, int nv_pad, int nM,
                            int32_t *next_world, hipStream_t stream, Before *before);
int newton_solve_dense_column(const im_newton_args *p, float *H, float *U, int32_t *dof_union, int nv, int nv_pad, int nM,
                              int32_t *next_world, hipStream_t stream, Before *before);
// im_dense_init_factor, and with 80 columns as well, which that entry point leaves to three launches
int dense_init_factor(const uint8_t *done, const int32_t *nefc, const float *J, int njmax, const float *D, const
                      int32_t *state, int quad, const float *M, int64_t ldM, const int32_t *elemid, const float *grad,
                      int64_t ldg, float *H, float *U, int nv, int nv_pad, int32_t *dof_union, float *search, int64_t
                      ld_search, float *search_dot, float *decrement, int nworld, void *stream);
// the tree stage of a solve's start, without the two sums (the resident loop forms them)
int newton_tree_first(const im_tree_plan *plan, const im_newton_args *p, hipStream_t stream);

// Workgroups of a kernel that a CU keeps resident, kept after the first question: the runtime's answer costs as
// much host time as a launch.  In `plans` for a kernel of a plan's loaded module, null for one of the library's.
int resident_per_cu(const void *fn, Occupancy *plans, int threads, size_t lds, int *per_cu);
// Compute units of the current device.
int compute_units(int *ncu);
int current_device(int *device);
// Whether a resident kernel keeps to registers on the current device (one that parks more than a few values of its
// prologue in memory is left out) and may use a CU's whole LDS, which is asked for.
bool usable_resident(const void *fn);
// usable[i] of variants[i].fn on the current device, asked once per device.
template <class Variant, size_t N>
int usable_variants(Kept<int, std::array<bool, N>> &kept, const Variant (&variants)[N], std::array<bool, N> *usable) {
  int device = 0;
  if (const int st = current_device(&device)) return st;
  return kept.get(device, [&](std::array<bool, N> &u) {
    for (size_t i = 0; i < N; ++i) u[i] = usable_resident(variants[i].fn);
    return (int)IM_OK;
  }, usable);
}
// Workgroups of a resident loop over nworld worlds, up to `waves` of them to a workgroup and `per_cu` workgroups to a CU,
// and the worlds that each starts with: a batch smaller than the chip is spread over its compute units and SIMDs.
// Neighbours in a workgroup are worlds next to one another (70 dofs x 2048 worlds with a workgroup's worlds 512 apart,
// so that their matrices share memory channels: 906 us per solve against 819), and every CU gets as many (683
// workgroups of three on 256 CUs: 890 us).  `together` (the tree kernels): a workgroup's wavefronts work on its worlds'
// factors in step, so a second workgroup on a CU does that work twice (35 dofs x 700 worlds, a world each: 217 us
// against 210): only behind full ones.  Full workgroups always, and now: sparse 35 dofs x 500 worlds 452 -> 420 us,
// dense 27 x 1000 304 -> 273, tree 27 x 64 174 -> 164.
inline int resident_worlds_grid(int nworld, int waves, int ncu, int per_cu, bool together, int *group_worlds) {
  const int each = (int)(((int64_t)nworld + ncu - 1) / ncu);  // worlds of a CU
  int k = waves;
  if (together) {
    k = std::min(waves, each);
  } else if (each < waves * per_cu) {  // the fewest places for them, in the largest workgroups
    for (int m = 1, places = waves * per_cu; m <= per_cu; ++m) {
      const int of_m = (each + m - 1) / m;
      if (of_m <= waves && of_m * m < places) k = of_m, places = of_m * m;
    }
  }
  k = std::max(1, k);
  *group_worlds = k;
  return (int)std::min<int64_t>((int64_t)ncu * per_cu, ((int64_t)nworld + k - 1) / k);
}
// *counter = value, as a launch
void set_counter(int *counter, int value, hipStream_t stream);

}  // namespace im
