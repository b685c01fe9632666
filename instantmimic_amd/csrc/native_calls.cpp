// The hot entry points' host path in native code: a CPython module (instantmimic_amd/_native.so) whose
// functions take the caller's tensors, check them and issue the library's launch on the current stream.
// In Python the checks and the marshalling of a call's arguments took 9 - 14 us per launch and
// 120 us per constraint solve, longer than the kernels they launch on small batches (a tree solve of
// 1000 worlds runs 4 us); here a call is 2 - 5 us, most of it the runtime's launch.
//
// Every function returns None when it has launched, a positive library status, or -1 when the
// arguments are not what it takes at once (another dtype, a stride, a missing array, another current
// device): the Python caller then goes through its own checks, which name the error or handle the case.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdlib>
#include <cstring>

#include "../../include/imhip.h"

namespace {

using at::Tensor;

const Tensor *tensor_of(PyObject *o) { return o && THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

// Runs the launch without the interpreter's lock: it may wait for room in the stream's queue.
template <class F>
int unlocked(F &&launch) {
  int status = -1;  // (what torch throws, for a tensor without storage, declines the call)
  PyThreadState *const state = PyEval_SaveThread();
  try {
    status = launch();
  } catch (...) {
  }
  PyEval_RestoreThread(state);
  return status;
}
// Whatever Python exception a declined argument left behind goes: the caller's own checks raise theirs.
PyObject *declined() {
  PyErr_Clear();
  return PyLong_FromLong(-1);
}
PyObject *answer(int status) {
  if (status == IM_OK) Py_RETURN_NONE;
  return status < 0 ? declined() : PyLong_FromLong(status);
}

// The checks of one call: every tensor on the first one's device, which is the current one.
struct Call {
  bool ok = true;
  int device = -2;

  bool on(const Tensor *t, at::ScalarType type) {
    if (!t || !t->is_cuda() || t->scalar_type() != type) return ok = false;
    const int d = t->get_device();
    if (device == -2) {
      device = d;
      if (c10::hip::current_device() != d) ok = false;
    } else if (d != device) {
      ok = false;
    }
    return ok;
  }
  // a 2-D float tensor with contiguous rows of at least `width` floats for `nworld` worlds (-1: any)
  bool rows(const Tensor *t, int64_t nworld, int64_t width) {
    if (!on(t, at::kFloat) || t->dim() != 2 || t->stride(1) != 1 || t->size(1) < width) return ok = false;
    return ok = ok && (nworld < 0 || t->size(0) == nworld);
  }
  bool whole(const Tensor *t, at::ScalarType type, int64_t count) {
    if (!on(t, type) || !t->is_contiguous() || t->numel() != count) return ok = false;
    return ok;
  }
  // a contiguous (nworld, pad, pad) float tensor
  bool squares(const Tensor *t, int64_t nworld, int64_t pad) {
    if (!on(t, at::kFloat) || t->dim() != 3 || t->size(0) != nworld || t->size(1) != pad || t->size(2) != pad) return ok = false;
    return ok = ok && t->is_contiguous();
  }
  // rows of at least `width` floats for `nworld` worlds, given as (nworld, width) with contiguous rows or as any contiguous shape
  bool vectors(const Tensor *t, int64_t nworld, int64_t width, int64_t *ld) {
    if (!on(t, at::kFloat) || t->dim() < 1 || nworld <= 0) return ok = false;
    if (t->dim() == 2 && t->stride(1) == 1) {
      *ld = t->stride(0);
      return ok = ok && t->size(0) == nworld && t->size(1) >= width;
    }
    if (!t->is_contiguous() || t->size(0) != nworld) return ok = false;
    *ld = t->numel() / nworld;
    return ok = ok && *ld >= width;
  }
  void *stream() const { return (void *)c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }
};

template <class T = float>
T *ptr(const Tensor *t) { return (T *)t->data_ptr(); }
template <class T = float>
T *ptr_or_null(const Tensor *t) { return t ? (T *)t->data_ptr() : nullptr; }

// An integer, or an object that stands for one (__index__).  False for anything else: a float, say,
// which the Python callers convert.
bool as_int(PyObject *o, int64_t *v) {
  *v = PyLong_AsLongLong(o);
  if (*v != -1 || !PyErr_Occurred()) return true;
  PyErr_Clear();
  return false;
}
void *as_address(PyObject *o) {
  void *p = PyLong_AsVoidPtr(o);
  if (!p && PyErr_Occurred()) PyErr_Clear();
  return p;
}

// ---- tree_ldl -----------------------------------------------------------------------------------

// (plan, nv, nM, M, x, y)
PyObject *tree_factor_solve(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (n != 6) return declined();
  const auto *plan = (const im_tree_plan *)as_address(a[0]);
  int64_t nv, nM;
  if (!as_int(a[1], &nv) || !as_int(a[2], &nM)) return declined();
  const Tensor *M = tensor_of(a[3]), *x = tensor_of(a[4]), *y = tensor_of(a[5]);
  Call c;
  if (!plan || !c.rows(M, -1, nM) || !c.rows(x, M->size(0), nv) || !c.rows(y, M->size(0), nv)) return declined();
  void *const stream = c.stream();
  return answer(unlocked([&] {
    return im_tree_factor_solve(plan, ptr(M), M->stride(0), ptr(y), y->stride(0), ptr(x), x->stride(0), (int)M->size(0), stream);
  }));
}

// (plan, nv, nM, M, J, D, state, nefc, grad, x, negate, quad)
PyObject *assemble_tree_factor_solve(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (n != 12) return declined();
  const auto *plan = (const im_tree_plan *)as_address(a[0]);
  int64_t nv, nM, quad;
  const int negate = PyObject_IsTrue(a[10]);
  if (!as_int(a[1], &nv) || !as_int(a[2], &nM) || negate < 0 || !as_int(a[11], &quad)) return declined();
  const Tensor *M = tensor_of(a[3]), *J = tensor_of(a[4]), *D = tensor_of(a[5]), *state = tensor_of(a[6]), *nefc = tensor_of(a[7]),
               *grad = tensor_of(a[8]), *x = tensor_of(a[9]);
  Call c;
  if (!plan || !c.rows(M, -1, nM) || (!nefc && a[7] != Py_None)) return declined();
  const int64_t nworld = M->size(0);
  if (!c.on(J, at::kFloat) || J->dim() != 3 || J->size(0) != nworld || J->size(2) != nv || J->size(1) < 1 || !J->is_contiguous()) return declined();
  const int64_t njmax = J->size(1);
  auto per_row = [&](const Tensor *t, at::ScalarType type) {
    return c.whole(t, type, nworld * njmax) && t->dim() == 2 && t->size(0) == nworld;
  };
  if (!per_row(D, at::kFloat) || !per_row(state, at::kInt) || (nefc && !c.whole(nefc, at::kInt, nworld)) || !c.rows(grad, nworld, nv) ||
      !c.rows(x, nworld, nv))
    return declined();
  void *const stream = c.stream();
  const unsigned flags = negate ? IM_FLAG_NEGATE : 0;
  return answer(unlocked([&] {
    return im_assemble_tree_ldl_solve(plan, ptr(M), M->stride(0), ptr(J), (int)njmax, ptr(D), ptr<int32_t>(state),
                                           ptr_or_null<int32_t>(nefc), (int)quad, ptr(grad), grad->stride(0), ptr(x),
                                           x->stride(0), nullptr, (int)nworld, flags, stream);
  }));
}

// ---- blocked_dense ------------------------------------------------------------------------------

// (nworld, nv, pad, block, nM, indices, U, M, x, y)
PyObject *blocked_factor_solve(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (n != 10) return declined();
  int64_t nworld, nv, pad, block, nM;
  if (!as_int(a[0], &nworld) || !as_int(a[1], &nv) || !as_int(a[2], &pad) || !as_int(a[3], &block) || !as_int(a[4], &nM)) return declined();
  const Tensor *indices = tensor_of(a[5]), *U = tensor_of(a[6]), *M = tensor_of(a[7]), *x = tensor_of(a[8]), *y = tensor_of(a[9]);
  Call c;
  int64_t ldx = 0, ldy = 0;
  if (nworld <= 0 || !c.rows(M, nworld, nM) || !c.squares(U, nworld, pad) || !c.whole(indices, at::kInt, pad * pad) ||
      !c.vectors(x, nworld, nv, &ldx) || !c.vectors(y, nworld, nv, &ldy))
    return declined();
  void *const stream = c.stream();
  return answer(unlocked([&] {
    return im_blocked_factor_solve(ptr(M), M->stride(0), (int)nM, ptr<int32_t>(indices), (int)block, (int)nv, (int)pad, ptr(y), ldy,
                                        ptr(U), ptr(x), ldx, (int)nworld, stream);
  }));
}

// (M_dense, J, D, state, nefc, H, y, x, factor, quad)
PyObject *dense_hessian_factor_solve(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (n != 10) return declined();
  const Tensor *M = tensor_of(a[0]), *J = tensor_of(a[1]), *D = tensor_of(a[2]), *state = tensor_of(a[3]), *nefc = tensor_of(a[4]),
               *H = tensor_of(a[5]), *y = tensor_of(a[6]), *x = tensor_of(a[7]), *U = tensor_of(a[8]);
  Call c;
  int64_t quad;
  if (!as_int(a[9], &quad) || !c.on(J, at::kFloat) || J->dim() != 3 || !J->is_contiguous() || J->size(1) < 1 || (!nefc && a[4] != Py_None) || (!H && a[5] != Py_None) ||
      (!U && a[8] != Py_None))
    return declined();
  const int64_t nworld = J->size(0), njmax = J->size(1), nv = J->size(2), pad = (nv + 15) / 16 * 16;
  int64_t ldx = 0, ldy = 0;
  auto per_row = [&](const Tensor *t, at::ScalarType type) {
    return c.whole(t, type, nworld * njmax) && t->dim() == 2 && t->size(0) == nworld;
  };
  if (!c.whole(M, at::kFloat, nworld * nv * nv) || !per_row(D, at::kFloat) || !per_row(state, at::kInt) ||
      (nefc && !c.whole(nefc, at::kInt, nworld)) || !c.vectors(y, nworld, nv, &ldy) || !c.vectors(x, nworld, nv, &ldx) ||
      (U && !c.squares(U, nworld, pad)) || (H && (H->dim() != 3 || H->size(1) < nv || !c.squares(H, nworld, H->size(1)))))
    return declined();
  void *const stream = c.stream();
  return answer(unlocked([&] {
    return im_jtdj_factor_solve(ptr(M), ptr(J), (int)njmax, ptr(D), ptr<int32_t>(state), ptr_or_null<int32_t>(nefc), (int)quad,
                                     ptr_or_null(H), (int)nv, H ? (int)H->size(1) : 0, ptr(y), ldy, ptr_or_null(U), (int)pad, ptr(x), ldx,
                                     (int)nworld, stream);
  }));
}

// ---- newton_fusion ------------------------------------------------------------------------------

#define IM_NAMES(X)                                                                                                              \
  X(opt) X(stat) X(meaninertia) X(tolerance) X(ls_tolerance) X(ls_iterations) X(iterations) X(disableflags) X(nv) X(nv_pad)     \
  X(block_dim) X(linesearch_iterative) X(M_mulm_rowadr) X(M_mulm_col) X(M_mulm_madr) X(nworld) X(M) X(ne) X(nf) X(nefc)         \
  X(qfrc_smooth) X(qacc_smooth) X(qacc_warmstart) X(qacc) X(qfrc_constraint) X(solver_niter) X(overflow) X(efc) X(J) X(D)       \
  X(frictionloss) X(aref) X(Ma) X(force) X(state) X(search) X(search_dot) X(mv) X(jv) X(Jaref) X(done) X(alpha)                 \
  X(improvement) X(ls_exhausted) X(quad_changed_ids) X(quad_changed_count) X(state_changed_count) X(search_unchanged) X(grad)   \
  X(grad_dot) X(grad_scale) X(newton_decrement) X(h) X(hfactor) X(newton_tree_scratch) X(sparse_hessian_plan)                   \
  X(newton_elemid) X(newton_dof_union) X(newton_next_world) X(kernel) X(address) X(path) X(block) X(nM)
struct Names {
#define IM_FIELD(x) PyObject *x = nullptr;
  IM_NAMES(IM_FIELD)
#undef IM_FIELD
  bool make() {
#define IM_MAKE(x) \
  if (!(x = PyUnicode_InternFromString(#x))) return false;
    IM_NAMES(IM_MAKE)
#undef IM_MAKE
    return true;
  }
} names;

// Attributes of the model, the data and the context: every reference is held until the launches are issued.
struct Holder {
  PyObject *held[96];
  int count = 0;
  bool missing = false;
  ~Holder() {
    while (count) Py_DECREF(held[--count]);
  }
  // the attribute, or null (and `missing` unless it may be absent) where there is none
  PyObject *get(PyObject *from, PyObject *name, bool optional = false) {
    PyObject *v = from && count < 96 ? PyObject_GetAttr(from, name) : nullptr;
    if (!v) {
      PyErr_Clear();
      if (!optional) missing = true;
      return nullptr;
    }
    held[count++] = v;
    return v;
  }
  PyObject *maybe(PyObject *from, PyObject *name) {  // null for None or absent
    PyObject *v = get(from, name, true);
    return v == Py_None ? nullptr : v;
  }
  const Tensor *tensor(PyObject *from, PyObject *name) {
    const Tensor *t = tensor_of(get(from, name));
    if (!t) missing = true;
    return t;
  }
  // null for None, and for an attribute that is not there where that is allowed (`absent`)
  const Tensor *maybe_tensor(PyObject *from, PyObject *name, bool absent) {
    PyObject *v = get(from, name, absent);
    if (v == Py_None) return nullptr;
    const Tensor *t = tensor_of(v);
    if (v && !t) missing = true;
    return t;
  }
  int64_t integer(PyObject *from, PyObject *name, bool optional = false, int64_t otherwise = 0) {
    PyObject *v = get(from, name, optional);
    if (!v) return otherwise;
    int64_t i;
    if (!as_int(v, &i)) missing = true;
    return i;
  }
};

// (m, d, ctx, nsolving, disable_warmstart, ls_overflow_bit, iterations_overflow_bit): the whole solve
PyObject *newton_solve(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (n != 7) return declined();
  const char *form = std::getenv("IMHIP_NEWTON");
  if (form && std::strcmp(form, "stages") == 0) return declined();
  PyObject *m = a[0], *d = a[1], *ctx = a[2];
  int64_t no_warmstart, ls_bit, iterations_bit;
  if (!as_int(a[4], &no_warmstart) || !as_int(a[5], &ls_bit) || !as_int(a[6], &iterations_bit)) return declined();
  Holder h;
  Call c;
  im_newton_args p{};
  im_newton_start s{};
  im_newton_model k{};
  PyObject *opt = h.get(m, names.opt), *efc = h.get(d, names.efc), *stat = h.get(m, names.stat);
  if (h.missing) return declined();
  const int64_t nv = h.integer(m, names.nv), pad = h.integer(m, names.nv_pad), nworld = h.integer(d, names.nworld);
  const Tensor *J = h.tensor(efc, names.J), *M = h.tensor(d, names.M);
  if (h.missing || nworld <= 0 || nv <= 0 || !c.on(J, at::kFloat) || J->dim() != 3 || !J->is_contiguous() || J->size(0) != nworld ||
      J->size(2) != nv || !c.rows(M, nworld, 1))
    return declined();
  const int64_t njmax = J->size(1);
  p.efc_J = ptr(J), p.njmax = (int32_t)njmax, p.M = ptr(M), p.ldM = M->stride(0), p.nworld = (int32_t)nworld;
  // options
  auto option = [&](PyObject *from, PyObject *name, const float **out, int32_t *count) {
    const Tensor *t = h.tensor(from, name);
    if (h.missing || !c.on(t, at::kFloat) || !t->is_contiguous() || t->numel() < 1) return false;
    *out = ptr(t), *count = (int32_t)t->numel();
    return true;
  };
  if (!option(opt, names.tolerance, &p.opt_tolerance, &p.ntolerance) || !option(opt, names.ls_tolerance, &p.opt_ls_tolerance, &p.nls_tolerance) ||
      !option(stat, names.meaninertia, &p.stat_meaninertia, &p.nmeaninertia))
    return declined();
  p.ls_iterations = (int32_t)h.integer(opt, names.ls_iterations), p.iterations = (int32_t)h.integer(opt, names.iterations);
  const int64_t flags = h.integer(opt, names.disableflags, true);
  p.block = 64;
  if (pad < 64) p.block = (int32_t)h.integer(h.get(m, names.block_dim), names.linesearch_iterative);
  p.quad = 1, p.ls_overflow_bit = (int32_t)ls_bit, p.iterations_overflow_bit = (int32_t)iterations_bit;
  const Tensor *radr = h.tensor(m, names.M_mulm_rowadr), *col = h.tensor(m, names.M_mulm_col), *madr = h.tensor(m, names.M_mulm_madr);
  if (h.missing || p.iterations <= 0 || !c.whole(radr, at::kInt, nv + 1) || !c.whole(col, at::kInt, col->numel()) ||
      !c.whole(madr, at::kInt, col->numel()))
    return declined();
  p.M_mulm_rowadr = ptr<int32_t>(radr), p.M_mulm_col = ptr<int32_t>(col), p.M_mulm_madr = ptr<int32_t>(madr), p.nterm = (int32_t)col->numel();
  // arrays: (nworld, width) contiguous, or one element per world
  enum Presence { REQUIRED, MAY_BE_NONE, MAY_BE_ABSENT };
  auto rows = [&](PyObject *from, PyObject *name, int64_t width, auto **out, Presence presence = REQUIRED) {
    const Tensor *t = presence == REQUIRED ? h.tensor(from, name) : h.maybe_tensor(from, name, presence == MAY_BE_ABSENT);
    *out = nullptr;
    if (h.missing) return false;
    if (!t) return true;
    using T = std::remove_const_t<std::remove_pointer_t<std::remove_pointer_t<decltype(out)>>>;
    const at::ScalarType type = std::is_same_v<T, float> ? at::kFloat : at::kInt;
    if (!c.whole(t, type, nworld * width) || (width != 1 && (t->dim() != 2 || t->size(0) != nworld))) return false;
    *out = (T *)t->data_ptr();
    return true;
  };
  auto bytes = [&](PyObject *name, uint8_t **out) {
    const Tensor *t = h.tensor(ctx, name);
    if (h.missing || (t->scalar_type() != at::kByte && t->scalar_type() != at::kBool) || !c.whole(t, t->scalar_type(), nworld)) return false;
    *out = (uint8_t *)t->data_ptr();
    return true;
  };
  if (!rows(d, names.ne, 1, &p.ne, MAY_BE_NONE) || !rows(d, names.nf, 1, &p.nf, MAY_BE_NONE) || !rows(d, names.nefc, 1, &p.nefc) ||
      !rows(efc, names.D, njmax, &p.efc_D) || !rows(efc, names.frictionloss, njmax, &p.efc_frictionloss, MAY_BE_NONE) ||
      !rows(d, names.qfrc_smooth, nv, &p.qfrc_smooth) || !rows(d, names.qacc, nv, &p.qacc) || !rows(efc, names.Ma, nv, &p.efc_Ma) ||
      !rows(efc, names.force, njmax, &p.efc_force) || !rows(efc, names.state, njmax, &p.efc_state) ||
      !rows(ctx, names.Jaref, njmax, &p.Jaref) || !rows(ctx, names.jv, njmax, &p.jv) || !rows(ctx, names.search, nv, &p.search) ||
      !rows(ctx, names.mv, nv, &p.mv) || !rows(d, names.qfrc_constraint, nv, &p.qfrc_constraint) ||
      !rows(ctx, names.search_dot, 1, &p.search_dot) || !rows(ctx, names.alpha, 1, &p.alpha) ||
      !rows(ctx, names.improvement, 1, &p.improvement) || !rows(ctx, names.grad_dot, 1, &p.grad_dot) ||
      !rows(ctx, names.grad_scale, 1, &p.grad_scale) || !rows(ctx, names.newton_decrement, 1, &p.newton_decrement) ||
      !rows(ctx, names.quad_changed_count, 1, &p.quad_changed_count) || !rows(ctx, names.state_changed_count, 1, &p.state_changed_count) ||
      !rows(d, names.solver_niter, 1, &p.solver_niter) || !rows(d, names.overflow, 1, &p.overflow, MAY_BE_ABSENT) || !bytes(names.done, &p.done) ||
      !bytes(names.ls_exhausted, &p.ls_exhausted) || !bytes(names.search_unchanged, &p.search_unchanged))
    return declined();
  const Tensor *grad = h.tensor(ctx, names.grad), *ids = h.tensor(ctx, names.quad_changed_ids), *left = tensor_of(a[3]);
  if (h.missing || grad->dim() != 2 || grad->size(0) != nworld || grad->size(1) < nv || !c.whole(grad, at::kFloat, grad->numel()) ||
      ids->dim() != 2 || ids->size(0) != nworld || !c.whole(ids, at::kInt, ids->numel()) || !c.whole(left, at::kInt, 1))
    return declined();
  p.grad = ptr(grad), p.ld_grad = grad->size(1), p.quad_changed_ids = ptr<int32_t>(ids), p.ld_ids = (int32_t)ids->size(1);
  p.nsolving = ptr<int32_t>(left);
  // the start
  const Tensor *smooth = h.tensor(d, names.qacc_smooth), *aref = h.tensor(efc, names.aref);
  const Tensor *warm = (flags & no_warmstart) ? nullptr : h.maybe_tensor(d, names.qacc_warmstart, true);
  if (h.missing || !c.rows(smooth, nworld, nv) || !c.rows(aref, nworld, njmax) || (warm && !c.rows(warm, nworld, nv)) ||
      smooth->size(1) != nv || (warm && warm->size(1) != nv))
    return declined();
  s.qacc_smooth = ptr(smooth), s.ld_smooth = smooth->stride(0), s.efc_aref = ptr(aref), s.ld_aref = aref->stride(0);
  s.qacc_start = warm ? ptr(warm) : s.qacc_smooth, s.ld_start = warm ? warm->stride(0) : s.ld_smooth;
  // the factor stage
  k.nv = (int32_t)nv, k.nv_pad = (int32_t)pad, k.nM = (int32_t)M->size(1);
  auto square = [&](PyObject *name, float **out) {
    const Tensor *t = h.tensor(ctx, name);
    if (h.missing || !c.squares(t, nworld, pad)) return false;
    *out = ptr(t);
    return true;
  };
  PyObject *tree = h.maybe(ctx, names.newton_tree_scratch), *plan = h.maybe(ctx, names.sparse_hessian_plan);
  if (plan) {
    PyObject *path = h.get(plan, names.path);
    if (h.missing || !PyUnicode_Check(path)) return declined();
    if (PyUnicode_CompareWithASCIIString(path, "fused") != 0) plan = nullptr;
  }
  if (tree && plan) return declined();
  if (tree) {
    PyObject *kernel = h.get(tree, names.kernel);
    k.tree = (const im_tree_plan *)as_address(h.get(kernel, names.address));
    // a plan of another model, or an M shorter than its rows: the Python checks name the error
    if (h.missing || !k.tree || h.integer(kernel, names.nv) != nv || h.integer(kernel, names.nM) > M->size(1)) return declined();
  } else {
    if (!square(names.hfactor, &k.U) || !rows(ctx, names.newton_dof_union, nv + 1, &k.dof_union)) return declined();
    if (plan) {
      k.sparse = (const im_sparse_plan *)as_address(h.get(plan, names.address));
      if (h.missing || !k.sparse || h.integer(plan, names.nv) != nv || h.integer(plan, names.nv_pad) != pad || !M->is_contiguous())
        return declined();
    } else {
      const Tensor *elemid = h.tensor(ctx, names.newton_elemid), *next = h.tensor(ctx, names.newton_next_world);
      if (h.missing || !square(names.h, &k.H) || ((uintptr_t)k.H & 15) || (pad & 3) || !c.whole(elemid, at::kInt, nv * nv) || !c.whole(next, at::kInt, 1)) return declined();
      k.elemid = ptr<int32_t>(elemid), k.next_world = ptr<int32_t>(next);
    }
  }
  if (h.missing || !c.ok) return declined();
  void *const stream = c.stream();
  const int status = unlocked([&] { return im_newton_solve(&p, &s, &k, stream); });
  return status == IM_ERR_UNSUPPORTED ? declined() : answer(status);
}

using Body = PyObject *(*)(PyObject *, PyObject *const *, Py_ssize_t);
// an exception out of torch (a tensor without storage, as under tracing) sends the caller to its own path
template <Body F>
PyObject *guarded(PyObject *self, PyObject *const *a, Py_ssize_t n) {
  try {
    return F(self, a, n);
  } catch (...) {
    return declined();
  }
}

PyMethodDef methods[] = {
    {"tree_factor_solve", (PyCFunction)(void *)guarded<tree_factor_solve>, METH_FASTCALL, nullptr},
    {"assemble_tree_factor_solve", (PyCFunction)(void *)guarded<assemble_tree_factor_solve>, METH_FASTCALL, nullptr},
    {"blocked_factor_solve", (PyCFunction)(void *)guarded<blocked_factor_solve>, METH_FASTCALL, nullptr},
    {"dense_hessian_factor_solve", (PyCFunction)(void *)guarded<dense_hessian_factor_solve>, METH_FASTCALL, nullptr},
    {"newton_solve", (PyCFunction)(void *)guarded<newton_solve>, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", "Host path of the hot entry points.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
  if (!names.make()) return nullptr;
  PyObject *m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch_version", IM_TORCH_VERSION) < 0) Py_CLEAR(m);
  return m;
}
