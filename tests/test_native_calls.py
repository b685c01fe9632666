"""The native host path (csrc/native_calls.cpp) hands over to the Python checks what it does not
take at once: views with a row stride run, and wrong dtypes, shapes and layouts raise as before."""

import numpy as np
import pytest

from instantmimic_amd import synth
from instantmimic_amd.mjw_kernels import tree_ldl as T
from oracle import planner as P
from oracle import ref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nworld", [1, 5, 257])
@pytest.mark.parametrize("layout", ["contiguous", "row stride", "no nefc"])
def test_gpu_assemble_and_solve_take_any_row_stride(device, nworld, layout):
    import torch

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
    import torch

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
