"""Several right-hand sides through every team width of the products and the
joint refinement, against dense solves: right-hand sides of different scales,
one of them zero, nodes of no element.

Tolerance: ||x - x*|| / ||x*|| <= cond(K) ||r|| / ||b|| with ||r|| <= stol ||b||
by the stopping rule; the dense reference is good to cond(K) 1e-16.
"""

import pytest
import torch

from test_gpu_persist import dense, model_of

pytestmark = pytest.mark.gpu
DT = torch.float64

CASES = [("quad1", (13, 9), 2), ("tetra1_heat", (5, 5, 5), 1), ("tetra1", (3, 3, 3), 0),
         ("hexa1", (5, 4, 6), 3), ("hexa2", (3, 2, 3), 0)]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nrhs", [2, 4, 7, 9, 16])
@pytest.mark.parametrize("kind,n,orphans", CASES)
def test_against_dense(kind, n, orphans, nrhs, precision):
    m = model_of(kind, n, orphans)
    m.solve(stol=1e-8)
    K, _, cond = dense(m)
    g = torch.Generator().manual_seed(nrhs)
    F = torch.randn(nrhs, *m._neumann.shape, generator=g, dtype=DT).cuda()
    F = F * (10.0 ** torch.linspace(-3, 3, nrhs, dtype=DT).cuda()).reshape(-1, 1, 1)
    F[1] = 0.0
    stol = 1e-9  # joint refinement: one FP64 product for all
    u, _ = m.solve_load_cases(F, precision=precision, preconditioner="block_jacobi", stol=stol)
    b = torch.where(m.constraints.reshape(1, -1), 0.0, F.reshape(nrhs, -1))
    x = torch.linalg.solve(K, b.T).T
    u = u.reshape(nrhs, -1)
    assert float(u[1].abs().max()) == 0.0
    for r in range(nrhs):
        if r != 1:
            assert float((u[r] - x[r]).norm() / x[r].norm()) <= cond * (stol + 1e-14)
