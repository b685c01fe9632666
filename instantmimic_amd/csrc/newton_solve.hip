// One call for a whole constraint solve with a resident loop: the start (everything of init_context
// before the first Hessian), the first factor stage, the loop with the final constraint force -- three
// launches on the caller's stream, in the order of the reference's step
// (src/instantmimic/utils/mjw_step_optimized.py:2588-2683).  The pieces stay callable by themselves;
// issued one by one from a host language a solve is eight launches (start point, fills, sums and force
// among them), whose issue took longer than a small batch's work: 117 us per solve of 64 worlds.
#include <hip/hip_runtime.h>

#include <tuple>

#include "common.h"
#include "newton_solve.h"
#include "sparse_plan.h"

namespace im {
namespace {
__global__ void set_counter_kernel(int *counter, int value) { *counter = value; }
}  // namespace

void set_counter(int *counter, int value, hipStream_t stream) {
  hipLaunchKernelGGL(set_counter_kernel, dim3(1), dim3(1), 0, stream, counter, value);
}

int current_device(int *device) {
  IM_HIP_CHECK(hipGetDevice(device));
  return IM_OK;
}

int resident_per_cu(const void *fn, Occupancy *plans, int threads, size_t lds, int *per_cu) {
  static Occupancy library;
  int device = 0;
  if (const int st = current_device(&device)) return st;
  return (plans ? *plans : library).get(std::make_tuple(device, fn, threads, lds), [&](int &n) {
    if (plans)
      IM_HIP_CHECK(hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&n, (hipFunction_t)fn, threads, lds));
    else
      IM_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, fn, threads, lds));
    return (int)IM_OK;
  }, per_cu);
}

int compute_units(int *ncu) {
  static Kept<int, int> known;
  int device = 0;
  if (const int st = current_device(&device)) return st;
  return known.get(device, [&](int &n) {
    IM_HIP_CHECK(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device));
    n = n > 0 ? n : 1;
    return (int)IM_OK;
  }, ncu);
}

// Bytes of private memory a lane of a resident kernel may have: four values parked from the prologue to the next world.
// The kernels of this library have 12 at most; one beyond the limit spills within a round and is left out.
constexpr size_t kResidentPrivate = 16;
bool usable_resident(const void *fn) {
  hipFuncAttributes fa{};
  const bool ok = hipFuncGetAttributes(&fa, fn) == hipSuccess && fa.localSizeBytes <= kResidentPrivate &&
                  hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - (int)fa.sharedSizeBytes) == hipSuccess;
  (void)hipGetLastError();
  return ok;
}

namespace {
// the start and the first factor stage of a solve
struct FirstStage : Before {
  const im_newton_args *p;
  const im_newton_start *s;
  const im_newton_model *m;
  hipStream_t stream;
  int operator()(int *counter, int value) override {
    WholeSolve whole;
    whole.start = s->qacc_start, whole.ld_start = s->ld_start;
    whole.counter = counter, whole.counter_value = value;
    whole.active = 1;
    const int st = newton_init_launch(p, s->qacc_smooth, s->ld_smooth, s->efc_aref, s->ld_aref, m->nv, m->nM, whole, stream);
    if (st != IM_OK) return st;
    if (m->tree) return newton_tree_first(m->tree, p, stream);
    if (m->sparse)
      return im_sparse_init_factor(m->sparse, p->done, p->nefc, p->efc_J, p->njmax, p->efc_D, p->efc_state, p->quad, p->M,
                                   (int)p->ldM, p->grad, (int)p->ld_grad, m->U, p->search, p->search_dot, p->newton_decrement,
                                   p->nworld, stream);
    return dense_init_factor(p->done, p->nefc, p->efc_J, p->njmax, p->efc_D, p->efc_state, p->quad, p->M, p->ldM, m->elemid,
                                p->grad, p->ld_grad, m->H, m->U, m->nv, m->nv_pad, m->dof_union, p->search, m->nv, p->search_dot,
                                p->newton_decrement, p->nworld, stream);
  }
};
}  // namespace
}  // namespace im

extern "C" int im_newton_solve(const im_newton_args *args, const im_newton_start *start, const im_newton_model *model,
                               void *stream) {
  if (!args || !start || !model || !start->qacc_smooth || !start->efc_aref || model->nv <= 0 || model->nM <= 0) return IM_ERR_ARG;
  if (args->iterations <= 0 || (model->tree && model->sparse)) return IM_ERR_ARG;
  // A plan's kernels take their row lengths from the plan, the start and the arrays from the model: a plan
  // of other sizes would walk rows of the wrong length.
  if (model->tree && (model->tree->nv != model->nv || model->tree->nM > model->nM)) return IM_ERR_ARG;
  if (model->sparse && (model->sparse->nv != model->nv || model->sparse->nv_pad != model->nv_pad || model->sparse->nM > model->nM))
    return IM_ERR_ARG;
  if (args->nworld == 0) return IM_OK;
  const hipStream_t st = (hipStream_t)stream;
  im::FirstStage first;
  first.p = args, first.s = start, first.m = model, first.stream = st;
  if (model->tree) return im::newton_solve_tree(model->tree, args, st, &first);
  if (model->sparse) return im::newton_solve_sparse(model->sparse, args, model->U, model->dof_union, st, &first);
  if (!model->H || !model->U || !model->elemid || !model->dof_union || !model->next_world) return IM_ERR_ARG;
  if (model->nv <= 32)
    return im::newton_solve_dense_tile(args, model->H, model->dof_union, model->nv, model->nv_pad, model->nM, model->next_world, st, &first);
  return im::newton_solve_dense_column(args, model->H, model->U, model->dof_union, model->nv, model->nv_pad, model->nM,
                                       model->next_world, st, &first);
}
