"""Sparse plans on a wavefront per world: the steps of a level, where launches keep them, and the kernels with them in
LDS and in memory, against the oracle bit for bit."""

from types import SimpleNamespace

import numpy as np
import pytest

import newton_chain as NC
from instantmimic_amd import synth
from instantmimic_amd.mjw_kernels import newton_stages as NS
from instantmimic_amd.mjw_kernels import sparse_hessian as S
from oracle import ref as R
from sparse_layout import Layout
from test_newton_solve import _solve_on_gpu
from test_newton_stages import _changes
from test_sparse_hessian import _batch, _random_model


def _forest(nv: int, seed: int):
    """Parents of a random forest of joints of one to three dofs, a tenth of them roots."""
    return [int(p) for p in _random_model(np.random.default_rng(seed), nv).dof_parentid]


# (parents, words of steps): chains from the smallest that the solver takes a sparse plan for to the largest on a wavefront, and
# forests whose entries have several runs
TREES = {
    "g1": list(synth.SHAPES["g1"].parents), "snu": list(synth.SHAPES["snu"].parents),
    **{f"chain{n}": [-1] + list(range(n - 1)) for n in (33, 40, 42, 43, 44, 46, 48, 56, 64)},
    "forest57": _forest(57, 1022), "forest40": _forest(40, 1053), "forest63": _forest(63, 1040),
}  # fmt: skip


def _plan(name, device=None):
    m = synth.model_from_parents(TREES[name])
    return m, S.build_plan(m, [], S.block_width(m.nv_pad), **({} if device is None else {"device": device}))


def _layout(m, plan):
    return Layout(plan, m.nv, 2 * len(m.M_colind) - m.nv)


@pytest.mark.parametrize("name", list(TREES))
def test_steps_factor_and_solve(name):
    """The steps read as the kernels read them, in 64 bits: H and the gradient on the slots, the factor's steps, the
    backward solve's, against a dense solve."""
    m, plan = _plan(name)
    t, nv, lay = plan.tables, m.nv, _layout(m, plan)
    rng = np.random.default_rng(1)
    H, g = np.zeros((nv, nv)), rng.normal(size=nv)
    sa, sb = t["SH_SA"], t["SH_SB"]
    H[sa, sb] = H[sb, sa] = rng.normal(size=len(sa))
    H += np.diag(np.abs(H).sum(1) + 1.0)
    rhs = plan.nfac
    N = np.concatenate([H[sa, sb], g[t["SH_ORIG"]], np.zeros(256)])
    iD = np.zeros(nv + 256)
    steps = lay.words[: 128 * (lay.nfactor + 1)].reshape(-1, 64, 2)
    assert not steps[-1].any()
    v = np.zeros(64)
    for x, y in (s.T for s in steps[:-1]):
        assert len(set(y >> 25)) == 1
        most = int((y >> 6 & 127).max())
        assert (y[0] >> 25 & 1, y[0] >> 31) == (most < 2, most == 2)
        width = 1 << int(y[0] >> 26 & 7)
        if y[0] >> 29 & 1:
            v[:] = 0.0
        for lane in range(64):
            at = np.arange(int(y[lane] >> 6 & 127)) * width
            v[lane] += (N[int(x[lane] & 0xFFF) + at] * N[int(x[lane] >> 12 & 0xFFF) + at] * iD[int(y[lane] & 63) + at]).sum()
        if y[0] >> 30 & 1:
            for lane in np.flatnonzero(y >> 13 & 0xFFF):
                assert lane % width == 0
                slot, col = int(y[lane] >> 13 & 0xFFF) - 1, int(x[lane] >> 24) - 1
                N[slot] -= v[lane : lane + width].sum()
                if col >= 0:
                    iD[col] = 1.0 / N[slot]
    back = lay.words[128 * (lay.nfactor + 1) :].reshape(-1, 64)
    assert len(back) == lay.nbackward + 1 and not back[-1].any()
    for r in back[:-1]:
        r = r[r >> 31 == 1]
        i, j = rhs + (r >> 12 & 63), rhs + (r >> 18 & 63)
        np.subtract.at(N, j, N[r & 0xFFF] * N[i] * iD[r >> 12 & 63])
    x = np.zeros(nv)
    x[t["SH_ORIG"]] = N[rhs : rhs + nv] * iD[:nv]
    np.testing.assert_allclose(x, np.linalg.solve(H, g), rtol=1e-9, atol=1e-12)


def test_no_plan_loses_its_wavefront_kernel_or_worlds_to_its_steps():
    """The kernels of a single pass read the steps from memory, so that no plan's size of them takes it to the kernel of a
    workgroup per world; a resident loop keeps them in LDS up to where they cost a large batch worlds."""
    for name in TREES:
        m, plan = _plan(name)
        lay = _layout(m, plan)
        words = lay.sizes[2]
        # the first factor: the factor and the rows' list of four worlds, no more than the slack beside them
        for rows in (16, 64, 256):
            factor = plan.nslots + m.nv + 2 * rows
            assert 16 * factor <= lay.init_bytes(rows) <= 16 * (factor + 8) + 4 * max(0, 192 - 2 * rows)
        assert lay.init_bytes(256) <= 64 * 1024
        # the update stage
        for worlds in (1, 100, 10**6):
            waves, rows, lds = lay.update(worlds)
            assert waves in (4, 8, 16) and rows in (16, 32) and lds <= 160 * 1024
        # the resident loop
        for rows in (32, 64, 96, 160):
            one, many = lay.resident(rows, 1), lay.resident(rows, 10**6)
            assert one[0] and one[2] == words and many[2] in (0, words) and max(one[3], many[3]) <= 158 * 1024
            assert many[2] == words or many[0] * many[4] > one[0] * one[4]
            held = 256 * one[0] * one[4]
            assert lay.resident(rows, held) == one and lay.resident(rows, held + 1) == many
    side = lambda name, rows, worlds: _layout(*_plan(name)).resident(rows, worlds)[:3]  # noqa: E731
    assert side("g1", 96, 8192)[::2] == (16, 3200)
    assert side("forest57", 66, 100)[::2] == (12, 8448) and side("forest57", 66, 3200)[::2] == (16, 0)
    assert side("chain48", 40, 100)[::2] == (8, 9344) and side("chain48", 40, 2100)[::2] == (12, 0)


# ---------------------------------------------------------------------------------- GPU


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["chain33", "chain40", "chain42", "chain43", "chain44", "chain46", "chain48", "chain64", "forest57", "forest40", "forest63"])
@pytest.mark.parametrize("nworld", [45, 1101])
def test_gpu_update_stage_bitwise(device, name, nworld):
    """Changed rows, none (a solve with the factor that lies there) and untouched worlds."""
    import torch

    m, plan = _plan(name, device)
    b = _batch(m, [], nworld, 24, 5)
    b.state = np.stack([b.state[0], np.where(np.random.default_rng(3).random(b.state[0].shape) < 0.2, synth.QUADRATIC - b.state[0], b.state[0])]).astype(np.int32)
    new, ids, changes, sc, done, grad = _changes(b, np.random.default_rng(5))
    assert changes.max() > 2 and not changes.min()
    oplan = R.sparse_plan(m, [], plan.block)
    hf0, *_ = R.sparse_init_factor(oplan, b.nefc, b.J, b.D, b.state[0], b.M, b.grad)
    want = R.sparse_update_factor(oplan, sc, changes, ids, b.J, b.D, new, grad, hf0, done=done)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    hf, uni = t(hf0), torch.zeros((nworld, m.nv + 1), dtype=torch.int32, device=device)
    search, sdot, decr = torch.zeros((nworld, m.nv), device=device), torch.zeros(nworld, device=device), torch.zeros(nworld, device=device)
    NS.factor_factory(m.nv, m.nv_pad, plan)(t(b.J), t(b.D), t(new), t(ids), t(changes), t(sc), t(done), t(grad), None, hf, search, sdot, decr, uni)
    torch.cuda.synchronize()
    n_used = 2 * plan.nfac + m.nv
    np.testing.assert_array_equal(hf.cpu().numpy().reshape(nworld, -1)[:, :n_used], want[0].reshape(nworld, -1)[:, :n_used])
    for g, r in zip((search, sdot, decr), want[2:]):
        np.testing.assert_array_equal(g.cpu().numpy(), r)


@pytest.mark.gpu
@pytest.mark.parametrize("name,rows,nworld,near", [
    ("chain42", 40, 60, True), ("chain48", 40, 60, True), ("chain48", 40, 2100, False), ("chain64", 24, 30, True),
    ("forest57", 66, 60, True), ("forest57", 66, 3200, False), ("forest40", 40, 4200, True),
])  # fmt: skip
def test_gpu_solve_with_steps_in_lds_and_in_memory(device, monkeypatch, name, rows, nworld, near):
    import torch

    m, plan = _plan(name)
    ncu = torch.cuda.get_device_properties(device).multi_processor_count
    assert (_layout(m, plan).resident(rows, nworld, ncu)[2] > 0) == near
    monkeypatch.setitem(synth.SHAPES, name, synth.Shape(name, tuple(TREES[name]), rows, nworld, (0.5, 8.0), 0.02, (-4.0, 4.0), 0.6, 1, 77))
    monkeypatch.setattr(S, "plan_for_model", lambda m, ctx, groups, block, device: (S.build_plan(m, groups, block, device=device), "enabled"))
    p = NC.problem(name, nworld, "sparse", empty_every=11)
    s = NC.oracle_solve(p)
    m, d, ctx, nsolving = _solve_on_gpu(p, device, graph=False)
    NC.compare(p, s, d, ctx)
