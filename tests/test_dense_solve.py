"""The factor and solve of dense matrices on one wavefront's matrix-core tiles at the edges of its block
rows, with and without a spare column for the right-hand side, with pivots outside the range of the short
square root, and with contributing rows on both sides of its steps of four, against the CPU restatement."""

import numpy as np
import pytest

from instantmimic_amd import _lib
from instantmimic_amd.mjw_kernels import blocked_dense as BD
from oracle import ref as R


def _spd(rng, nworld, nv):
    a = rng.standard_normal((nworld, nv, nv))
    M = (a @ a.transpose(0, 2, 1) / nv + np.eye(nv)).astype(np.float32)
    M[-1] *= np.float32(2.0**-110)  # every pivot below 2^-96
    return M


@pytest.mark.gpu
@pytest.mark.parametrize("B", [8, 16])
@pytest.mark.parametrize("nv", [1, 8, 9, 16, 17, 31, 32, 33, 40, 41, 64, 65, 80, 81, 96, 112, 113, 127, 128])
def test_gpu_blocked_solve_at_block_edges(device, nv, B):
    import torch

    rng, nworld = np.random.default_rng(nv), 6
    M, y = _spd(rng, nworld, nv).reshape(nworld, -1), rng.standard_normal((nworld, nv)).astype(np.float32)
    pad, layout, _ = BD.block_index_layout(np.arange(nv * nv), nv, nv * nv, B)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    Md, yd, idx, x, U = t(M), t(y), t(layout), torch.full((nworld, nv), np.nan, device=device), torch.zeros((nworld, pad, pad), device=device)
    st = _lib.lib().im_blocked_factor_solve(Md.data_ptr(), nv * nv, nv * nv, idx.data_ptr(), B, nv, pad, yd.data_ptr(), nv, U.data_ptr(), x.data_ptr(), nv, nworld, None)
    assert st == 0
    torch.cuda.synchronize()
    x_ref, U_ref = R.blocked_factor_solve(M, layout, nv, pad, B, y)
    np.testing.assert_array_equal(U.cpu().numpy(), U_ref)
    np.testing.assert_array_equal(x.cpu().numpy(), x_ref)


@pytest.mark.gpu
@pytest.mark.parametrize("B", [8, 16])
@pytest.mark.parametrize("nv", [7, 24, 35, 56, 101, 128])
def test_gpu_blocked_solve_of_a_sparse_matrix(device, nv, B):
    """Elements whose id is past the matrix's (by one, by many, by more than a byte count of 32 bits holds) are zero; the values lie
    in another order, in rows of a wider array whose other words are poison."""
    import torch

    rng, nworld, wide = np.random.default_rng(nv), 5, 3
    A = rng.standard_normal((nworld, nv, nv)).astype(np.float32) / np.float32(nv)
    A = A + A.transpose(0, 2, 1) + 4 * np.eye(nv, dtype=np.float32)
    drop = np.triu(rng.random((nv, nv)) < 0.3, 1)
    drop |= drop.T
    A[:, drop] = 0.0
    keep = np.argwhere(~drop)
    keep = keep[rng.permutation(len(keep))]
    nM = len(keep)
    elemid = rng.choice(np.array([nM, nM + 9, 1 << 30, 2**31 - 1], np.int32), (nv, nv))
    elemid[keep[:, 0], keep[:, 1]] = np.arange(nM)
    M = np.full((nworld, nM + wide), np.nan, np.float32)
    M[:, :nM] = A[:, keep[:, 0], keep[:, 1]]
    y = rng.standard_normal((nworld, nv)).astype(np.float32)
    pad, layout, _ = BD.block_index_layout(elemid, nv, nM, B)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    Md, yd, idx, x, U = t(M), t(y), t(layout), torch.full((nworld, nv), np.nan, device=device), torch.zeros((nworld, pad, pad), device=device)
    st = _lib.lib().im_blocked_factor_solve(Md.data_ptr(), nM + wide, nM, idx.data_ptr(), B, nv, pad, yd.data_ptr(), nv, U.data_ptr(), x.data_ptr(), nv, nworld, None)
    assert st == 0
    torch.cuda.synchronize()
    x_ref, U_ref = R.blocked_factor_solve(M[:, :nM], layout, nv, pad, B, y)
    np.testing.assert_array_equal(U.cpu().numpy(), U_ref)
    np.testing.assert_array_equal(x.cpu().numpy(), x_ref)


@pytest.mark.gpu
@pytest.mark.parametrize("nv", [1, 15, 16, 17, 33, 48, 64, 79, 80, 96, 112, 127, 128])
def test_gpu_dense_hessian_solve_at_block_edges(device, nv):
    import torch

    counts = np.array([0, 1, 3, 4, 5, 8, 63, 64, 65, 130], np.int32)
    rng, nworld, rows = np.random.default_rng(nv), len(counts), 130
    pad, hpad = -(-nv // 16) * 16, (nv // 16 + 1) * 16
    M, y = _spd(rng, nworld, nv), rng.standard_normal((nworld, nv)).astype(np.float32)
    M[-1] *= np.float32(2.0**110)
    J = rng.standard_normal((nworld, rows, nv)).astype(np.float32)
    D = rng.uniform(0.1, 10.0, (nworld, rows)).astype(np.float32)
    state = (rng.uniform(size=(nworld, rows)) < 0.7).astype(np.int32)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    H, x, U = torch.zeros((nworld, hpad, hpad), device=device), torch.zeros((nworld, nv), device=device), torch.zeros((nworld, pad, pad), device=device)
    BD.dense_hessian_factor_solve(t(M), t(J), t(D), t(state), t(counts), H, t(y), x, factor=U)
    torch.cuda.synchronize()
    H_ref = H.cpu().numpy()  # the factor's input: its sums' order is the matrix cores' own
    assert R.rel_l2(H_ref, R.jtdj_dense(M.reshape(nworld, -1), J, D, state, counts, hpad)) <= 1e-6
    np.testing.assert_array_equal(H_ref, H_ref.transpose(0, 2, 1))
    _, layout, _ = BD.block_index_layout(np.arange(nv * nv), nv, nv * nv, 16)
    x_ref, U_ref = R.blocked_factor_solve(np.ascontiguousarray(H_ref[:, :nv, :nv]).reshape(nworld, -1), layout, nv, pad, 16, y)
    np.testing.assert_array_equal(U.cpu().numpy(), U_ref)
    np.testing.assert_array_equal(x.cpu().numpy(), x_ref)


def _hessian_case(nv, rows, counts, seed):
    rng, nworld = np.random.default_rng(seed), len(counts)
    M, y = _spd(rng, nworld, nv), rng.standard_normal((nworld, nv)).astype(np.float32)
    M[-1] *= np.float32(2.0**110)
    J = rng.standard_normal((nworld, rows, nv)).astype(np.float32)
    D = rng.uniform(0.1, 10.0, (nworld, rows)).astype(np.float32)
    state = (rng.uniform(size=(nworld, rows)) < 0.7).astype(np.int32)
    return M, J, D, state, np.asarray(counts, np.int32), y


@pytest.mark.gpu
@pytest.mark.parametrize("nv,hpad,offset", [(9, 9, 0), (15, 15, 0), (17, 18, 0), (33, 35, 0), (48, 48, 1), (64, 67, 0), (79, 80, 3), (127, 127, 0), (128, 128, 2)])
def test_gpu_dense_hessian_in_rows_that_take_no_wide_store(device, nv, hpad, offset):
    """H with a row length that is no multiple of four, or off 16 bytes: the bits of an aligned H, nothing
    written beyond the dofs."""
    import torch

    c = [torch.from_numpy(np.ascontiguousarray(a)).to(device) for a in _hessian_case(nv, 70, [0, 5, 64, 70, 33], nv)]
    nworld, apad = 5, -(-nv // 16) * 16
    x, xa = torch.zeros((nworld, nv), device=device), torch.zeros((nworld, nv), device=device)
    flat = torch.full((nworld * hpad * hpad + 4,), 7.0, device=device)
    H = flat[offset : offset + nworld * hpad * hpad].view(nworld, hpad, hpad)
    aligned = torch.full((nworld, apad, apad), 7.0, device=device)
    assert (hpad % 4 or H.data_ptr() % 16) and aligned.data_ptr() % 16 == 0
    BD.dense_hessian_factor_solve(*c[:5], H, c[5], x)
    BD.dense_hessian_factor_solve(*c[:5], aligned, c[5], xa)
    assert torch.equal(H[:, :nv, :nv], aligned[:, :nv, :nv]) and torch.equal(x, xa)
    H[:, :nv, :nv] = 7.0
    assert bool((flat == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("nv", [16, 33, 79])
def test_gpu_dense_hessian_of_long_row_lists(device, nv):
    """More rows than four worlds' lists fit a workgroup's LDS (a wavefront per workgroup then), and more
    than one world's list fits a CU's: refused."""
    import torch

    rows, nworld = 5301, 3
    M, J, D, state, counts, y = _hessian_case(nv, rows, [rows, 1, 4099], nv)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    pad = -(-nv // 16) * 16
    H, x, U = torch.zeros((nworld, pad, pad), device=device), torch.zeros((nworld, nv), device=device), torch.zeros((nworld, pad, pad), device=device)
    BD.dense_hessian_factor_solve(t(M), t(J), t(D), t(state), t(counts), H, t(y), x, factor=U)
    H_ref = H.cpu().numpy()
    # 3700 terms an element in another order: about sqrt(3700) half-ulps of 6e-8, 3.6e-6
    assert R.rel_l2(H_ref, R.jtdj_dense(M.reshape(nworld, -1), J, D, state, counts, pad)) <= 1e-5
    np.testing.assert_array_equal(H_ref, H_ref.transpose(0, 2, 1))
    _, layout, _ = BD.block_index_layout(np.arange(nv * nv), nv, nv * nv, 16)
    x_ref, U_ref = R.blocked_factor_solve(np.ascontiguousarray(H_ref[:, :nv, :nv]).reshape(nworld, -1), layout, nv, pad, 16, y)
    np.testing.assert_array_equal(U.cpu().numpy(), U_ref)
    np.testing.assert_array_equal(x.cpu().numpy(), x_ref)
    many = 20500
    with pytest.raises(_lib.ImhipError):
        BD.dense_hessian_factor_solve(t(M[:1]), torch.zeros((1, many, nv), device=device), torch.zeros((1, many), device=device),
                                      torch.zeros((1, many), dtype=torch.int32, device=device), None, None, t(y[:1]), x[:1])  # fmt: skip


@pytest.mark.gpu
@pytest.mark.parametrize("nv", [111, 112, 113, 121, 128])
def test_gpu_small_batches_of_large_matrices_equal_the_same_worlds_in_a_large_one(device, nv):
    """Up to a world per CU (two with 192 rows) a workgroup has a world, beyond that a wavefront: on both
    sides of the line the same worlds give the same bits, H, factor and solution, with H off 16 bytes and
    without one."""
    import torch

    ncu = torch.cuda.get_device_properties(device).multi_processor_count
    few, pad = 9, -(-nv // 16) * 16
    for rows, line in ((70, ncu), (191, ncu), (192, 2 * ncu), (215, 2 * ncu)):
        c = [torch.from_numpy(np.ascontiguousarray(a)).to(device) for a in _hessian_case(nv, rows, [0, 1, 5, 32, 33, 64, 65, 70, rows], nv)]

        def solve(n, offset, with_h):
            w = [t.repeat(-(-n // few), *[1] * (t.dim() - 1))[:n].contiguous() for t in c]
            flat = torch.zeros(n * pad * pad + 4, device=device)
            H = flat[offset : offset + n * pad * pad].view(n, pad, pad) if with_h else None
            x, U = torch.full((n, nv), 7.0, device=device), torch.full((n, pad, pad), 7.0, device=device)
            BD.dense_hessian_factor_solve(*w[:5], H, w[5], x, factor=U)
            return [t[:few] for t in (x, U, *([H[:, :nv, :nv]] if with_h else []))], x, U

        want, x, U = solve(line + 1, 0, True)
        for n, offset, with_h in ((few, 0, True), (line, 1, True), (line, 0, False)):
            got, x, U = solve(n, offset, with_h)
            for a, b in zip(got, want):
                np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy())
            reps = n // few
            for t in (x, U):
                assert torch.equal(t[: reps * few].view(reps, few, -1).nan_to_num(), t[:few].reshape(1, few, -1).expand(reps, -1, -1).nan_to_num())
    rng = np.random.default_rng(nv)
    _, layout, _ = BD.block_index_layout(np.arange(nv * nv), nv, nv * nv, 16)
    idx = torch.from_numpy(layout).to(device)
    M, y = _spd(rng, few, nv).reshape(few, -1), rng.standard_normal((few, nv)).astype(np.float32)
    for n in (ncu, ncu + 1):
        Md, yd = (torch.from_numpy(a).to(device).repeat(-(-n // few), 1)[:n].contiguous() for a in (M, y))
        x, U = torch.full((n, nv), np.nan, device=device), torch.zeros((n, pad, pad), device=device)
        st = _lib.lib().im_blocked_factor_solve(Md.data_ptr(), nv * nv, nv * nv, idx.data_ptr(), 16, nv, pad, yd.data_ptr(), nv, U.data_ptr(), x.data_ptr(), nv, n, None)
        assert st == 0
        x_ref, U_ref = R.blocked_factor_solve(M, layout, nv, pad, 16, y)
        np.testing.assert_array_equal(U[:few].cpu().numpy(), U_ref)
        np.testing.assert_array_equal(x[:few].cpu().numpy(), x_ref)
        np.testing.assert_array_equal(x[-few:].cpu().numpy(), np.tile(x_ref, (-(-n // few), 1))[:n][-few:])
