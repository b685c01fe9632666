"""The dense Newton stage on one wavefront's matrix-core tiles (33 to 79 dofs) at the edges of its
block rows, with row counts on both sides of its steps of four rows and chunks of 64, against the
CPU restatement bit for bit; and the solve with the stored factor behind it."""

import numpy as np
import pytest
from test_newton_stages import Q, _toggled  # noqa: F401

from instantmimic_amd import synth
from instantmimic_amd.mjw_kernels import blocked_dense as BD
from instantmimic_amd.mjw_kernels import newton_stages as NS
from oracle import ref as R

_COUNTS = (0, 1, 3, 4, 5, 63, 64, 65, 130)


@pytest.mark.gpu
@pytest.mark.parametrize("nv", [33, 47, 48, 63, 64, 79])
def test_gpu_dense_wave_stage_at_block_edges(device, nv):
    import torch

    parents = tuple([-1] + list(range(nv - 1)))
    nworld, pad = 2 * len(_COUNTS) + 1, (nv // 16 + 1) * 16
    b = synth.make_batch(synth.Shape(f"chain{nv}", parents, 130, nworld, (0.5, 8.0), 0.02, (-3.0, 3.0), 0.6, 1, 1200 + nv))
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    Md = synth.dense_from_csr(b.M, b.rowadr, b.rownnz, b.colind).astype(np.float32).reshape(nworld, -1)
    H0 = R.jtdj_dense(Md, b.J, b.D, b.state[0], b.nefc, pad)
    new, ids, changes, sc, done, grad = _toggled(b, np.random.default_rng(3), _COUNTS)
    first = np.full(nworld, -1, np.int32)
    H1, U1, *_ = R.dense_update_factor(sc, first, ids, b.J, b.D, b.state[0], b.grad, H0, np.zeros_like(H0), done=done)
    want = R.dense_update_factor(sc, changes, ids, b.J, b.D, new, grad, H1, U1, done=done)
    H, U = t(H0), torch.zeros((nworld, pad, pad), device=device)
    uni = torch.zeros((nworld, nv + 1), dtype=torch.int32, device=device)
    search, sdot, decr = torch.zeros((nworld, nv), device=device), torch.zeros(nworld, device=device), torch.zeros(nworld, device=device)
    stage = NS.factor_factory(nv, pad)
    J, D, ids_d, sc_d, done_d = t(b.J), t(b.D), t(ids), t(sc), t(done)
    stage(J, D, t(b.state[0]), ids_d, t(first), sc_d, done_d, t(b.grad), H, U, search, sdot, decr, uni)  # the factor of H as it lies there
    stage(J, D, t(new), ids_d, t(changes), sc_d, done_d, t(grad), H, U, search, sdot, decr, uni)  # zero changes: the stored factor
    torch.cuda.synchronize()
    np.testing.assert_array_equal(H.cpu().numpy(), want[0])
    np.testing.assert_array_equal(U.cpu().numpy(), want[1])
    np.testing.assert_array_equal(uni.cpu().numpy()[changes > 0], want[2][changes > 0])
    np.testing.assert_array_equal(search.cpu().numpy(), want[3])
    np.testing.assert_array_equal(sdot.cpu().numpy(), want[4])
    np.testing.assert_array_equal(decr.cpu().numpy(), want[5])


@pytest.mark.gpu
@pytest.mark.parametrize("nv,pad", [(33, 48), (48, 64), (63, 64)])
def test_gpu_first_hessian_lists_the_contributing_rows(device, nv, pad):
    """The first Hessian and its factor with more rows than one listing holds: rows in none, the first,
    the last and all of three listings, counts on both sides of a step and of a group of steps."""
    import torch

    parents = tuple([-1] + list(range(nv - 1)))
    nefc = np.array([0, 1, 256, 257, 520, 520, 520, 520, 520, 515, 300, 255, 64], np.int32)
    nworld, njmax = len(nefc), 520
    b = synth.make_batch(synth.Shape(f"chain{nv}", parents, njmax, nworld, (0.5, 8.0), 0.02, (-3.0, 3.0), 0.3, 1, 2400 + nv))
    state = np.where(b.state[0] == Q, Q, 0).astype(np.int32)
    state[1:4], state[4], state[5, :256], state[6, 256:] = Q, 0, 0, 0  # all; none; but the first listing's; only those
    state[7], state[8] = 0, Q
    state[7, [0, 100, 255, 256, 511]] = Q  # counts of 3, 1 + 1 and 0
    Md = synth.dense_from_csr(b.M, b.rowadr, b.rownnz, b.colind).astype(np.float32).reshape(nworld, -1)
    every, grad, done = np.ones(nworld, np.int32), b.grad, (nefc == 0).astype(np.uint8)
    H0 = R.jtdj_dense(Md, b.J, b.D, state, nefc, pad)
    ids = np.zeros((nworld, njmax), np.int32)
    H1, U1, _, search1, sdot1, decr1 = R.dense_update_factor(every, -every, ids, b.J, b.D, state, grad, H0, np.zeros_like(H0), done=done)
    elemid = np.full((nv, nv), -1, np.int32)
    for i in range(nv):
        for k in range(b.rowadr[i], b.rowadr[i] + b.rownnz[i]):
            elemid[i, b.colind[k]] = elemid[b.colind[k], i] = k
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    H, U = torch.zeros((nworld, pad, pad), device=device), torch.zeros((nworld, pad, pad), device=device)
    uni = torch.zeros((nworld, nv + 1), dtype=torch.int32, device=device)
    search, sdot, decr = torch.zeros((nworld, nv), device=device), torch.zeros(nworld, device=device), torch.zeros(nworld, device=device)
    M = t(b.M.reshape(nworld, -1))
    assert BD.dense_init_factor(M, t(elemid), t(b.J), t(b.D), t(state), t(nefc), t(done), t(grad), H, U, search, sdot, decr, uni)
    torch.cuda.synchronize()
    # the upper triangle is the oracle's chain; the lower is its mirror image (the oracle's own lower triangle weights the other factor)
    Hu = H.cpu().numpy()[:, :nv, :nv]
    np.testing.assert_array_equal(np.triu(Hu), np.triu(H1[:, :nv, :nv]))
    np.testing.assert_array_equal(Hu, Hu.transpose(0, 2, 1))
    live = nefc > 0
    np.testing.assert_array_equal(U.cpu().numpy()[live], U1[live])
    np.testing.assert_array_equal(search.cpu().numpy()[live], search1[live])
    np.testing.assert_array_equal(sdot.cpu().numpy()[live], sdot1[live])
    np.testing.assert_array_equal(decr.cpu().numpy()[live], decr1[live])
