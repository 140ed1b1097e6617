"""Which solves run in the persistent small-system solver (csrc/persist.hip): the
path that a solve reports, for the cases that test_gpu_persist.py compares with
the general path."""

import pytest
import torch

from test_gpu_persist import CASES, DT, grid_matrix, model_of
from torchfem import Solid
from torchfem.elements import linear_to_quadratic
from torchfem.materials import IsotropicElasticity3D
from torchfem.mesh import cube_hexa
from torchfem.sparse import PCGSolver, _csr_arrays

pytestmark = pytest.mark.gpu


def fem_path(m, **kw):
    m.solve(**kw)
    return m.last_solve_info["forward"]["pcg"][-1]["path"]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kind,n,orphans", CASES)
def test_fem_solves(kind, n, orphans, precision, monkeypatch):
    m = model_of(kind, n, orphans)
    for pc in ("block_jacobi", "jacobi"):
        for stol in (1e-8, 1e-12):
            assert fem_path(m, precision=precision, preconditioner=pc, stol=stol) == "persistent"
    monkeypatch.setenv("TFM_PCG_PERSIST", "0")
    assert fem_path(m, precision=precision, preconditioner="block_jacobi") == "general"


@pytest.mark.parametrize("n", [(16, 16, 15), (16, 16, 16), (31, 31, 30), (33, 32, 34)])
def test_block_counts_around_the_cu_count(n):
    assert fem_path(model_of("hexa1", n), preconditioner="block_jacobi", stol=1e-9) == "persistent"


def test_beyond_the_size_rule():
    """More values per CU than the rule of persist_solve takes (420 KB in FP32)."""
    m = model_of("hexa1", (60, 60, 60))
    assert m._pattern.nnz * 4 > 256 * 420 * 1024
    assert fem_path(m, preconditioner="block_jacobi", stol=1e-3) == "general"


@pytest.mark.parametrize("n,path", [(1, "persistent"), (2, "persistent"), (129, "persistent"),
                                    (4097, "persistent"), (70001, "persistent"),
                                    (250007, "no_fit")])
def test_csr_rows(n, path):
    A, b = grid_matrix(n) if n > 1 else (torch.eye(1, dtype=DT).cuda().to_sparse() * 3.0,
                                         torch.ones(1, dtype=DT).cuda())
    rowptr, col, val = _csr_arrays(A, b.device)
    solver = PCGSolver(n, 1, b.device)
    assert solver.solve_csr(rowptr, col, val, b, torch.zeros_like(b), 1e-10)["path"] == path
    solver.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_a_mesh_that_does_not_fit_is_tried_once(precision):
    """Hexa2 with its nodes numbered at random: too many distinct neighbours for
    a block's LDS. The model's next solves do not try again."""
    nodes, el = linear_to_quadratic(*cube_hexa(19, 19, 19))
    p = torch.randperm(len(nodes), generator=torch.Generator().manual_seed(0))
    inv = torch.empty_like(p)
    inv[p] = torch.arange(len(p))
    m = Solid(nodes.to(DT)[p].cuda(), inv[el].cuda(),
              IsotropicElasticity3D(torch.tensor(1000.0, dtype=DT, device="cuda"),
                                    torch.tensor(0.3, dtype=DT, device="cuda")))
    m.constraints[m.nodes[:, 0] == 0.0] = True
    m.forces[m.nodes[:, 0] == 1.0, 1] = 1.0
    paths = []
    for _ in range(2):  # one or more linear solves each
        m.solve(precision=precision, preconditioner="block_jacobi", stol=1e-6)
        paths += [p["path"] for p in m.last_solve_info["forward"]["pcg"]]
    assert paths == ["no_fit"] + ["general"] * (len(paths) - 1)


def test_a_wait_given_up_is_reported(monkeypatch):
    monkeypatch.setenv("TFM_PCG_PERSIST_QUIT", "2")
    monkeypatch.setenv("TFM_PCG_PERSIST_REST_MS", "0")
    assert fem_path(model_of("hexa1", (6, 6, 6)), stol=1e-9) == "gave_up"
