"""The dense Newton stage on one wavefront's matrix-core tiles (33 to 79 dofs) at the edges of its
block rows, with row counts on both sides of its steps of four rows and chunks of 64, against the
CPU restatement bit for bit; and the solve with the stored factor behind it."""

import numpy as np
import pytest
from test_newton_stages import Q, _toggled  # noqa: F401

from instantmimic_amd import synth
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
