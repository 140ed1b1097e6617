"""A wait of the persistent small-system solver (csrc/persist.hip) that is given
up: TFM_PCG_PERSIST_QUIT makes the last block leave at one point of the solve, as
it would after 50 ms without the others: 2 k - 1 where it waits for the k-th
residual, 2 k before it folds its k-th correction into x. Every block then leaves
and the general path finishes the solve from whatever x the blocks have left.

Tolerance of a solution: as in test_gpu_persist.py, cond(K) (stol + 1e-14).
"""

import threading
import time

import pytest
import torch

from test_gpu_persist import dense, grid_matrix, model_of
from torchfem.sparse import PCGSolver, _csr_arrays

pytestmark = pytest.mark.gpu
DT = torch.float64


@pytest.fixture(autouse=True)
def no_rest(monkeypatch):
    """The solves after one that gave up take the persistent kernel again."""
    monkeypatch.setenv("TFM_PCG_PERSIST_REST_MS", "0")


@pytest.mark.parametrize("quit_at", [1, 2])
def test_zero_load_from_a_warm_start(quit_at, monkeypatch):
    """b = 0 gives x = 0 whatever the guess, also where the last block leaves
    before it has cleared its part (the first residual tells that b = 0)."""
    A, b = grid_matrix(3000)
    rowptr, col, val = _csr_arrays(A, b.device)
    monkeypatch.setenv("TFM_PCG_PERSIST_QUIT", str(quit_at))
    solver = PCGSolver(3000, 1, b.device)
    x = torch.ones_like(b)
    solver.solve_csr(rowptr, col, val, torch.zeros_like(b), x, 1e-10)
    solver.close()
    assert float(x.abs().max()) == 0.0


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kind,n", [("hexa1", (6, 6, 6)), ("quad1", (37, 23))])
def test_solution_after_a_wait_given_up(kind, n, precision, monkeypatch):
    """Before and within the folds, where x holds the correction of some blocks
    only; from zero and from a warm start."""
    m = model_of(kind, n)
    f = m._neumann
    m.solve()
    _, x, cond = dense(m)
    for quit_at in range(1, 9):
        m = model_of(kind, n)  # its own solver handle
        monkeypatch.setenv("TFM_PCG_PERSIST_QUIT", str(quit_at))
        for stol, scale in ((1e-9, 1.0), (1e-12, 1.5)):
            m._neumann = scale * f
            u = m.solve(precision=precision, preconditioner="block_jacobi", stol=stol,
                        use_cached_solve=True)[0].reshape(-1) / scale
            assert float((u - x).norm() / x.norm()) <= cond * (stol + 1e-14), quit_at


def test_rest_after_a_wait_given_up(monkeypatch):
    """The next solves of the thread do not wait again, whatever their handle;
    other threads' do as before, and so does the thread's after the rest."""
    A, b = grid_matrix(3000)
    rowptr, col, val = _csr_arrays(A, b.device)

    def path(out):
        solver = PCGSolver(3000, 1, b.device)  # as sparse_solve: a handle per solve
        out.append(solver.solve_csr(rowptr, col, val, b, torch.zeros_like(b), 1e-10)["path"])
        solver.close()
        return out[-1]

    assert path([]) == "persistent"
    monkeypatch.setenv("TFM_PCG_PERSIST_REST_MS", "2000")
    monkeypatch.setenv("TFM_PCG_PERSIST_QUIT", "2")
    t0 = time.monotonic()
    assert path([]) == "gave_up"
    monkeypatch.setenv("TFM_PCG_PERSIST_QUIT", "0")
    seen = path([])
    other = []
    thread = threading.Thread(target=path, args=(other,))
    thread.start()
    thread.join()
    assert time.monotonic() - t0 < 1.9  # all of this within the rest
    assert seen == "general" and other == ["persistent"]
    time.sleep(2.1)
    assert path([]) == "persistent"
