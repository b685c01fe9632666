"""The native host path (csrc/native_calls.cpp) hands over to the Python checks what it does not
take at once: views with a row stride run, and wrong dtypes, shapes and layouts raise as before."""

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from instantmimic_amd import synth
from instantmimic_amd.mjw_kernels import blocked_dense as BD
from instantmimic_amd.mjw_kernels import newton_fusion as NF
from instantmimic_amd.mjw_kernels import tree_ldl as T
from oracle import planner as P
from oracle import ref as R

import newton_chain as NC

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nworld", [1, 5, 257])
@pytest.mark.parametrize("layout", ["contiguous", "row stride", "no nefc"])
def test_gpu_assemble_and_solve_take_any_row_stride(device, nworld, layout):
    b = synth.make_batch("humanoid", nworld)
    nv, nM = b.shape.nv, b.colind.size
    sc = T.create_tree_factor_solve_scratch(type("m", (), dict(nv=nv, M_rowadr=b.rowadr, M_rownnz=b.rownnz, M_colind=b.colind)), device)
    wide = 7 if layout == "row stride" else 0

    def rows(a):
        t = torch.zeros((a.shape[0], a.shape[1] + wide), device=device)
        t[:, : a.shape[1]] = torch.from_numpy(a).to(device)
        return t[:, : a.shape[1]]

    up = lambda a: torch.from_numpy(a).to(device)  # noqa: E731
    M, g, x = rows(b.M), rows(b.grad), rows(np.zeros((nworld, nv), np.float32))
    T.assemble_tree_factor_solve(sc, M, up(b.J), up(b.D), up(b.state[0]), None if layout == "no nefc" else up(b.nefc), g, x, negate=True)
    st = P.tree_ldl_structure(b.rowadr, b.rownnz, b.colind)
    want = R.assemble_tree_ldl_solve(*st, P.best_tree_ldl_plan(*st), b.M, b.J, b.D, b.state[0], b.nefc, b.grad)
    np.testing.assert_array_equal(x.cpu().numpy(), -want)
    y = torch.zeros((nworld, nv), device=device)
    T.tree_factor_solve(sc, M, y, g)
    assert M.shape[1] == nM and torch.isfinite(y).all() and (wide == 0 or not M.is_contiguous() or nworld == 1)


def test_gpu_the_python_checks_still_name_the_error(device):
    b = synth.make_batch("humanoid", 8)
    nv = b.shape.nv
    sc = T.create_tree_factor_solve_scratch(type("m", (), dict(nv=nv, M_rowadr=b.rowadr, M_rownnz=b.rownnz, M_colind=b.colind)), device)
    M, y = torch.from_numpy(b.M).to(device), torch.from_numpy(b.grad).to(device)
    x = torch.zeros_like(y)
    with pytest.raises(TypeError):
        T.tree_factor_solve(sc, M.double(), x, y)
    with pytest.raises(ValueError):
        T.tree_factor_solve(sc, M, x[:4], y)
    with pytest.raises(ValueError):
        T.tree_factor_solve(sc, M, x.t().contiguous().t(), y)
    with pytest.raises(TypeError):
        T.tree_factor_solve(sc, M.cpu(), x, y)
    J, D, st = torch.zeros((8, 4, nv), device=device), torch.ones((8, 4), device=device), torch.zeros((8, 4), dtype=torch.int32, device=device)
    with pytest.raises(TypeError):
        T.assemble_tree_factor_solve(sc, M, J, D, st.long(), None, y, x)
    with pytest.raises(ValueError):
        T.assemble_tree_factor_solve(sc, M, J[:, :, :5].contiguous(), D, st, None, y, x)


def _snapshot(d, ctx):
    return {k: v.clone() for o in (d, d.efc, ctx) for k, v in vars(o).items() if isinstance(v, torch.Tensor)}


def _same(before, d, ctx):
    return all(torch.equal(torch.nan_to_num(before[k]) if before[k].is_floating_point() else before[k],
                           torch.nan_to_num(v) if v.is_floating_point() else v)
               for o in (d, d.efc, ctx) for k, v in vars(o).items() if isinstance(v, torch.Tensor))  # fmt: skip


@pytest.mark.parametrize("call", ["solve", "run", "init_context"])
def test_gpu_newton_with_a_tree_scratch_of_another_model(device, call):
    """A scratch of a smaller or a larger tree, and an M shorter than the plan's rows, are refused
    before anything is launched or written."""
    go = {"solve": NF.solve, "run": NF.run, "init_context": lambda m, d, ctx, left: NF.init_context(m, d, ctx)}[call]
    scratch_of = lambda name: T.create_tree_factor_solve_scratch(synth.model_from_parents(synth.SHAPES[name].parents), device)  # noqa: E731
    p = NC.problem("humanoid", 9, "tree")
    m, d, ctx, left = NC.device_objects(p, device)
    own = ctx.newton_tree_scratch
    before = _snapshot(d, ctx)
    for name in ("ant", "g1"):
        ctx.newton_tree_scratch = scratch_of(name)
        with pytest.raises(ValueError, match="another model"):
            go(m, d, ctx, left)
    ctx.newton_tree_scratch, M = own, d.M
    before["M"] = d.M = M[:, :-1]
    with pytest.raises(ValueError, match="elements"):
        go(m, d, ctx, left)
    assert _same(before, d, ctx) and int(left.item()) == 0


def _linear_step(device, nworld=5):
    b = synth.make_batch("humanoid", nworld)
    m = type("m", (), dict(nv=b.shape.nv, M_rowadr=b.rowadr, M_rownnz=b.rownnz, M_colind=b.colind))
    up = lambda a: torch.from_numpy(a).to(device)  # noqa: E731
    return T.create_tree_factor_solve_scratch(m, device), [up(a) for a in (b.M, b.J, b.D, b.state[0], b.nefc, b.grad)]


def _dense_step(device, nv=35, rows=40, nworld=5, seed=3):
    g = torch.Generator(device="cpu").manual_seed(seed)
    a = torch.randn((nworld, nv, nv), generator=g) * 0.2
    M = (a @ a.transpose(1, 2).contiguous() + torch.eye(nv)).to(device)
    J, D = torch.randn((nworld, rows, nv), generator=g).to(device), (torch.rand((nworld, rows), generator=g) + 0.5).to(device)
    state = torch.randint(0, 2, (nworld, rows), generator=g, dtype=torch.int32).to(device)
    nefc = torch.full((nworld,), rows - 3, dtype=torch.int32, device=device)
    return [M, J, D, state, nefc, torch.randn((nworld, nv), generator=g).to(device)]


@pytest.mark.parametrize("one", [1.0, np.float32(1.0), np.int64(1), True, torch.tensor(1), torch.tensor(1.0)], ids=repr)
def test_gpu_quad_is_converted_as_int_does(device, one):
    """``quad`` goes through ``int()``: any number that equals the state selects its rows."""
    sc, (M, J, D, state, nefc, grad) = _linear_step(device)
    x, want = torch.zeros_like(grad), torch.zeros_like(grad)
    T.assemble_tree_factor_solve(sc, M, J, D, state, nefc, grad, want, quad=1)
    T.assemble_tree_factor_solve(sc, M, J, D, state, nefc, grad, x, quad=one)
    assert torch.equal(x, want)
    M, J, D, state, nefc, y = _dense_step(device)
    x, want = torch.zeros_like(y), torch.zeros_like(y)
    BD.dense_hessian_factor_solve(M, J, D, state, nefc, None, y, want, quad=1)
    BD.dense_hessian_factor_solve(M, J, D, state, nefc, None, y, x, quad=one)
    assert torch.equal(x, want)


def test_gpu_arguments_that_are_no_numbers_raise_their_own_error(device):
    sc, (M, J, D, state, nefc, grad) = _linear_step(device)
    x = torch.full_like(grad, 7.0)
    for wrong in ("one", None):
        with pytest.raises((TypeError, ValueError)):
            T.assemble_tree_factor_solve(sc, M, J, D, state, nefc, grad, x, quad=wrong)

    class Undecided:
        def __bool__(self):
            raise LookupError("neither")

    with pytest.raises(LookupError, match="neither"):
        T.assemble_tree_factor_solve(sc, M, J, D, state, nefc, grad, x, negate=Undecided())
    assert bool((x == 7.0).all())


@pytest.mark.parametrize("missing", ["ne", "nf", "frictionloss"])
def test_gpu_solve_asks_for_every_array_of_the_step(device, missing):
    """None stands for no equality rows, no friction rows; an attribute that is not there is an error."""
    p = NC.problem("humanoid", 5, "tree")
    m, d, ctx, left = NC.device_objects(p, device)
    delattr(d.efc if missing == "frictionloss" else d, missing)
    with pytest.raises(AttributeError, match=missing):
        NF.solve(m, d, ctx, left)
    m, d, ctx, left = NC.device_objects(p, device)
    d.ne = d.nf = d.efc.frictionloss = None
    NF.solve(m, d, ctx, left)
    assert bool(ctx.done.all()) and bool(torch.isfinite(d.qacc).all())


def _blocked(device, nworld=5, nv=35, block=8):
    g = torch.Generator(device="cpu").manual_seed(4)
    a = torch.randn((nworld, nv, nv), generator=g) * 0.2
    M = (a @ a.transpose(1, 2).contiguous() + torch.eye(nv)).reshape(nworld, -1).to(device)
    tile = SimpleNamespace(size=nv, elemid=torch.arange(nv * nv, dtype=torch.int32))
    d = SimpleNamespace(nworld=nworld, M=M)
    sc = BD.create_blocked_dense_factor_solve_scratch(SimpleNamespace(nv=nv, M_tiles=[tile]), d, device, block_size=block)
    return d, M, sc, torch.randn((nworld, nv), generator=g).to(device)


@pytest.mark.parametrize("shape", ["rows", "flat", "planes"])
def test_gpu_a_factor_workspace_has_the_shape_of_the_factor(device, shape):
    """As many floats in another shape are refused, for the factor of each of the two solves."""
    d, M, sc, y = _blocked(device)
    x, n, pad = torch.zeros_like(y), d.nworld, sc.pad
    shapes = lambda n, pad: dict(rows=(n * pad, pad), flat=(n * pad * pad,), planes=(n, pad // 2, 2 * pad))[shape]  # noqa: E731
    with pytest.raises(ValueError):
        BD._blocked_dense_factor_solve(d, M, x, y, sc, factor_workspace=torch.zeros(shapes(n, pad), device=device))
    M, J, D, state, nefc, y = _dense_step(device)
    with pytest.raises(ValueError):
        BD.dense_hessian_factor_solve(M, J, D, state, nefc, None, y, x, factor=torch.zeros(shapes(n, 48), device=device))
    assert not bool(x.any())


@pytest.mark.parametrize("stage,name", [("sparse", "hfactor"), ("dense", "hfactor"), ("dense", "h")])
def test_gpu_the_solves_squares_have_the_shape_of_the_factor(device, stage, name):
    p = NC.problem("g1", 6, stage)
    m, d, ctx, left = NC.device_objects(p, device)
    setattr(ctx, name, getattr(ctx, name).reshape(3, p.pad, 2 * p.pad))
    with pytest.raises((TypeError, ValueError)):
        NF.solve(m, d, ctx, left)


_WRONG = {
    "double": lambda t: t.double() if t.is_floating_point() else t.long(),
    "half": lambda t: t.half() if t.is_floating_point() else t.short(),
    "one world less": lambda t: t[:-1],
    "on the host": lambda t: t.cpu(),
    "every other column": lambda t: torch.zeros((*t.shape[:-1], 2 * t.shape[-1]), dtype=t.dtype, device=t.device)[..., ::2],
}


@pytest.mark.parametrize("wrong", sorted(_WRONG))
@pytest.mark.parametrize("call", ["solve", "matrix"])
def test_gpu_dense_hessian_refuses_what_its_kernels_cannot_read(device, call, wrong):
    """Each array of the dense J'DJ in turn in another type, length, place or layout: an error, and
    nothing written."""
    M, J, D, state, nefc, y = _dense_step(device)
    x, H, U = torch.full_like(y, 7.0), torch.full((5, 48, 48), 7.0, device=device), torch.full((5, 48, 48), 7.0, device=device)
    args = dict(M=M, J=J, D=D, state=state, nefc=nefc, H=H, y=y, x=x, U=U)
    for name in args if call == "solve" else ("M", "J", "D", "state", "nefc", "H"):
        a = {**args, name: _WRONG[wrong](args[name])}
        with pytest.raises((TypeError, ValueError)):
            if call == "solve":
                BD.dense_hessian_factor_solve(a["M"], a["J"], a["D"], a["state"], a["nefc"], a["H"], a["y"], a["x"], factor=a["U"])
            else:
                BD.dense_hessian(a["M"], a["J"], a["D"], a["state"], a["nefc"], a["H"])
    assert all(bool((t == 7.0).all()) for t in (x, H, U))


@pytest.mark.parametrize("where", ["elemid", "dof_union", "nefc", "done"])
def test_gpu_first_dense_factor_leaves_arrays_on_the_host(device, where):
    """The one launch takes no address of host memory: False, with nothing written."""
    p = NC.problem("g1", 4, "dense")
    m, d, ctx, _ = NC.device_objects(p, device)
    a = dict(elemid=ctx.newton_elemid, dof_union=ctx.newton_dof_union, nefc=d.nefc, done=ctx.done)
    a[where] = a[where].cpu()
    before = ctx.h.clone()
    assert not BD.dense_init_factor(d.M, a["elemid"], d.efc.J, d.efc.D, d.efc.state, a["nefc"], a["done"], ctx.grad, ctx.h, ctx.hfactor,
                                    ctx.search, ctx.search_dot, ctx.newton_decrement, a["dof_union"])  # fmt: skip
    assert torch.equal(torch.nan_to_num(before), torch.nan_to_num(ctx.h))


_SOLVE_ARRAYS = {
    "m": "M_mulm_rowadr M_mulm_col M_mulm_madr", "opt": "tolerance ls_tolerance", "stat": "meaninertia",
    "d": "M ne nf nefc qfrc_smooth qacc_smooth qacc qfrc_constraint solver_niter overflow",
    "efc": "J D frictionloss aref Ma force state",
    "ctx": "search search_dot mv jv Jaref done alpha improvement ls_exhausted quad_changed_ids quad_changed_count "
           "state_changed_count search_unchanged grad grad_dot grad_scale newton_decrement",
}  # fmt: skip
_STAGE_ARRAYS = {"tree": "", "sparse": " hfactor newton_dof_union", "dense": " hfactor newton_dof_union h newton_elemid newton_next_world"}


@pytest.mark.parametrize("wrong", sorted(_WRONG))
@pytest.mark.parametrize("stage,name", [("tree", "humanoid"), ("sparse", "g1"), ("dense", "humanoid"), ("dense", "g1")])
def test_gpu_solve_refuses_what_its_kernels_cannot_read(device, stage, name, wrong):
    """Each array of a whole solve in turn in another type, length, place or layout: an error from the
    Python checks, whichever of them it reaches first."""
    p = NC.problem(name, 6, stage)
    m, d, ctx, left = NC.device_objects(p, device)
    for where, names in _SOLVE_ARRAYS.items():
        owner = dict(m=m, opt=m.opt, stat=m.stat, d=d, efc=d.efc, ctx=ctx)[where]
        for attr in (names + (_STAGE_ARRAYS[stage] if where == "ctx" else "")).split():
            kept = getattr(owner, attr)
            if wrong == "every other column" and kept.numel() == 1:
                continue  # (contiguous whatever its stride)
            setattr(owner, attr, _WRONG[wrong](kept))
            with pytest.raises((TypeError, ValueError, RuntimeError)):
                NF.solve(m, d, ctx, left)
                pytest.fail(f"{where}.{attr} {wrong} was taken")
            setattr(owner, attr, kept)
    for bad in (left.long(), left.cpu(), torch.zeros(2, dtype=torch.int32, device=device)):
        with pytest.raises((TypeError, ValueError, RuntimeError)):
            NF.solve(m, d, ctx, bad)
    NF.solve(m, d, ctx, left)
    NC.compare(p, NC.oracle_solve(p), d, ctx)


@pytest.mark.parametrize("wrong", sorted(_WRONG))
@pytest.mark.parametrize("block", [8, 16])
def test_gpu_blocked_solve_refuses_what_its_kernels_cannot_read(device, block, wrong):
    d, M, sc, y = _blocked(device, block=block)
    args = dict(M=M, x=torch.full_like(y, 7.0), y=y, U=torch.full((d.nworld, sc.pad, sc.pad), 7.0, device=device))
    for name in args:
        a = {**args, name: _WRONG[wrong](args[name])}
        with pytest.raises((TypeError, ValueError)):
            BD._blocked_dense_factor_solve(d, a["M"], a["x"], a["y"], sc, factor_workspace=a["U"])
    for short in (dict(M=M[:, :-1]), dict(y=y[:, :-1])):
        a = {**args, **short}
        with pytest.raises(ValueError):
            BD._blocked_dense_factor_solve(d, a["M"], a["x"], a["y"], sc, factor_workspace=a["U"])
    assert bool((args["x"] == 7.0).all()) and bool((args["U"] == 7.0).all())


def test_gpu_views_run_through_the_dense_entry_points(device):
    """Rows with a stride, and right-hand sides with a third axis, give what plain rows give."""
    d, M, sc, y = _blocked(device)
    want, wide = torch.zeros_like(y), torch.zeros((d.nworld, 3 * y.shape[1]), device=device)
    BD._blocked_dense_factor_solve(d, M, want, y, sc)
    Mw = torch.zeros((d.nworld, M.shape[1] + 5), device=device)
    Mw[:, : M.shape[1]] = M
    view = wide[:, y.shape[1] : 2 * y.shape[1]]
    BD._blocked_dense_factor_solve(d, Mw[:, : M.shape[1]], view, y, sc)
    cube = torch.zeros((*y.shape, 1), device=device)
    BD._blocked_dense_factor_solve(d, M, cube, y[:, :, None].contiguous(), sc)
    assert torch.equal(view, want) and torch.equal(cube[:, :, 0], want) and bool((wide[:, : y.shape[1]] == 0).all())
    M, J, D, state, nefc, y = _dense_step(device)
    BD.dense_hessian_factor_solve(M, J, D, state, nefc, None, y, want)
    wide.zero_()
    BD.dense_hessian_factor_solve(M, J, D, state, nefc, None, y, view)
    cube.zero_()
    BD.dense_hessian_factor_solve(M, J, D, state, nefc, None, y[:, :, None].contiguous(), cube)
    assert torch.equal(view, want) and torch.equal(cube[:, :, 0], want) and bool((wide[:, : y.shape[1]] == 0).all())
