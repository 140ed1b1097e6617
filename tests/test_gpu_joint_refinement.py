"""Refinement residuals of several right-hand sides: the buffers of the joint
form, and the joint form against the residuals formed one by one.

Tolerance: both solutions have ||r|| <= stol ||b||, so they differ by at most
2 cond(K) stol, plus rounding; cond(K) from the dense matrix.
"""

import pytest
import torch

from test_gpu_persist import model_of
from torchfem.sparse import PCGSolver

pytestmark = pytest.mark.gpu
DT = torch.float64


def test_a_handle_holds_five_krylov_vectors():
    """x, r, u, p and s of n x 16, and vectors of n (fewer than 16 of them
    together): the joint form's two of n x 16 come with the first solve that
    uses them."""
    n = 1_000_000
    PCGSolver(n, 16).close()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    s = PCGSolver(n, 16)
    used = free - torch.cuda.mem_get_info()[0]
    s.close()
    assert 5 * 16 * n * 8 <= used < 6 * 16 * n * 8


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("cases", [2, 3, 8, 11, 16])
def test_joint_against_one_by_one(cases, precision, monkeypatch):
    m = model_of("hexa1", (5, 4, 6))
    g = torch.Generator().manual_seed(cases)
    F = torch.randn(cases, m.n_nod, 3, generator=g, dtype=DT).cuda()
    F[0] = 1.0  # a smooth load reaches its targets at other iterations
    F[:, m.constraints] = 0.0
    us = []
    for mode in ("0", "1"):
        monkeypatch.setenv("TFM_PCG_JOINT", mode)
        us.append(m.solve_load_cases(F, precision=precision, stol=1e-9)[0])
    cond = float(torch.linalg.cond(m.K.to_dense()))
    d = (us[0] - us[1]).reshape(cases, -1).norm(dim=1)
    assert bool((d <= 2.0 * cond * 1e-9 * 1.01 * us[1].reshape(cases, -1).norm(dim=1)).all())
