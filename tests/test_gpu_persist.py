"""The persistent small-system solver (csrc/persist.hip) against the general
path and dense solves: block edges, remainders, orphans, every element type,
both precisions, general CSR rows and the cases it hands back.

Tolerance of a solution: ||x - x*|| / ||x*|| <= cond(K) ||r|| / ||b||, with
||r|| <= stol ||b|| by the stopping rule; the dense reference is itself good
to cond(K) 1e-16, so cond(K) (stol + 1e-14) bounds the sum.
"""

import threading

import pytest
import torch

from torchfem import Planar, Solid, SolidHeat
from torchfem.elements import linear_to_quadratic
from torchfem.materials import (IsotropicConductivity3D, IsotropicElasticity3D,
                                IsotropicElasticityPlaneStress)
from torchfem.mesh import cube_hexa, cube_tetra6, rect_quad
from torchfem.sparse import PCGSolver, _csr_arrays, sparse_solve

pytestmark = pytest.mark.gpu
DT = torch.float64


def model_of(kind, n, orphans=0):
    g = torch.Generator().manual_seed(sum(n))
    if kind == "quad1":
        nodes, el = rect_quad(n[0] + 1, n[1] + 1)
    elif kind.startswith("tetra1"):
        nodes, el = cube_tetra6(n[0], jitter=0.1)
    else:
        nodes, el = cube_hexa(*(v + 1 for v in n))
        if kind == "hexa2":
            nodes, el = linear_to_quadratic(nodes, el)
    if orphans:  # nodes of no element, before, between and after the others
        keep = torch.ones(len(nodes) + orphans, dtype=torch.bool)
        keep[torch.linspace(0, len(keep) - 1, orphans).long()] = False
        new = torch.nonzero(keep).reshape(-1)
        full = torch.zeros(len(keep), nodes.shape[1], dtype=DT)
        full[keep] = nodes.to(DT)
        nodes, el = full, new[el]
    rho = 0.2 + torch.rand(len(el), generator=g, dtype=DT)
    nodes, el, rho = nodes.to(DT).cuda(), el.cuda(), rho.cuda()
    nu = torch.tensor(0.3, dtype=DT, device="cuda")
    if kind == "tetra1_heat":
        m = SolidHeat(nodes, el, IsotropicConductivity3D(rho))
    elif kind == "quad1":
        m = Planar(nodes, el, IsotropicElasticityPlaneStress(1000.0 * rho, nu))
    else:
        m = Solid(nodes, el, IsotropicElasticity3D(1000.0 * rho, nu))
    used = torch.zeros(m.n_nod, dtype=torch.bool, device="cuda")
    used[el.reshape(-1)] = True
    m.constraints[(m.nodes[:, 0] == 0.0) & used] = True
    m.constraints[~used] = True
    f = torch.zeros_like(m._neumann)
    f[:, 0] = torch.randn(m.n_nod, generator=g, dtype=DT).cuda() * used
    m._neumann = f
    return m


def dense(m):
    K = m.K.to_dense()
    b = torch.where(m.constraints.reshape(-1), 0.0, m._neumann.reshape(-1))
    return K, torch.linalg.solve(K, b), float(torch.linalg.cond(K))


CASES = [("hexa1", (1, 1, 1), 0), ("hexa1", (3, 2, 4), 0), ("hexa1", (5, 5, 5), 3),
         ("hexa1", (9, 7, 8), 0), ("hexa2", (1, 1, 1), 0), ("hexa2", (4, 3, 3), 0),
         ("tetra1", (4, 4, 4), 2), ("tetra1_heat", (2, 2, 2), 0), ("tetra1_heat", (11, 11, 11), 1),
         ("quad1", (1, 1), 0), ("quad1", (37, 23), 2)]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("pc", ["block_jacobi", "jacobi"])
@pytest.mark.parametrize("kind,n,orphans", CASES)
def test_persistent_against_dense_and_general(kind, n, orphans, pc, precision, monkeypatch):
    m = model_of(kind, n, orphans)
    m.solve(stol=1e-8)
    K, x, cond = dense(m)
    for stol in (1e-8, 1e-12):  # 1e-12: double-double refinement residuals
        its = {}
        for mode in ("0", "1"):
            monkeypatch.setenv("TFM_PCG_PERSIST", mode)
            u = m.solve(precision=precision, preconditioner=pc, stol=stol)[0].reshape(-1)
            its[mode] = m.last_solve_info["forward"]["pcg"][0]["iterations"][0]
            assert float((u - x).norm() / x.norm()) <= cond * (stol + 1e-14)
        # the same recurrence in another summation order
        assert abs(its["0"] - its["1"]) <= 2 + 0.1 * its["0"]


@pytest.mark.parametrize("n", [(16, 16, 15), (16, 16, 16), (31, 31, 30), (33, 32, 34)])
def test_block_counts_around_the_cu_count(n, monkeypatch):
    """Grids from fewer blocks than CUs to rows that stream from L2 instead of
    LDS: the true residual meets the tolerance and repeats bit for bit."""
    m = model_of("hexa1", n)
    out = {}
    for mode in ("0", "1", "1 again"):
        monkeypatch.setenv("TFM_PCG_PERSIST", mode[0])
        out[mode] = m.solve(preconditioner="block_jacobi", stol=1e-9)[0].reshape(-1)
        b = torch.where(m.constraints.reshape(-1), 0.0, m._neumann.reshape(-1))
        r = b - torch.mv(m.K, out[mode])
        assert float(r.norm() / b.norm()) <= 1e-9 * 1.01
    assert torch.equal(out["1"], out["1 again"])


def test_zero_load_and_warm_start():
    m = model_of("hexa1", (6, 6, 6))
    f = m._neumann
    m._neumann = torch.zeros_like(f)
    assert float(m.solve()[0].abs().max()) == 0.0
    m._neumann = f
    u = m.solve(stol=1e-11, use_cached_solve=True)[0]
    first = m.last_solve_info["forward"]["pcg"][0]["iterations"][0]
    v = m.solve(stol=1e-11, use_cached_solve=True)[0]
    again = m.last_solve_info["forward"]["pcg"][0]["iterations"][0]
    assert again <= first // 4
    # two solves, each off by at most cond * stol
    assert float((u - v).norm() / u.norm()) <= 2.0 * dense(m)[2] * 1.1e-11


def grid_matrix(n, seed=0):
    """SPD matrix of an n-node path plus random long-range couplings, columns
    unsorted within a row."""
    g = torch.Generator().manual_seed(seed)
    i = torch.arange(n - 1)
    far = torch.randint(0, n, (n,), generator=g)
    rows = torch.cat([i, i + 1, torch.arange(n), far])
    cols = torch.cat([i + 1, i, far, torch.arange(n)])
    vals = torch.cat([-torch.ones(2 * (n - 1), dtype=DT), -0.3 * torch.ones(2 * n, dtype=DT)])
    keep = rows != cols
    A = torch.sparse_coo_tensor(torch.stack([rows[keep], cols[keep]]), vals[keep], (n, n)).coalesce()
    d = -torch.sparse.sum(A, 1).to_dense() + 0.05
    A = (A + torch.sparse_coo_tensor(torch.arange(n).repeat(2, 1), d, (n, n))).coalesce()
    return A.cuda(), torch.randn(n, generator=g, dtype=DT).cuda()


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 127, 128, 129, 1024, 4097, 70001, 250007])
def test_csr_rows(n, monkeypatch):
    """General CSR rows from one unknown to row sets whose distinct columns do
    not fit in LDS (those go back to the general path)."""
    A, b = grid_matrix(n) if n > 1 else (torch.eye(1, dtype=DT).cuda().to_sparse() * 3.0,
                                         torch.ones(1, dtype=DT).cuda())
    xs = []
    for mode in ("0", "1"):
        monkeypatch.setenv("TFM_PCG_PERSIST", mode)
        x, _ = sparse_solve(A, b, method="cg", stol=1e-10)
        assert float((b - torch.mv(A, x)).norm() / b.norm()) <= 1e-10 * 1.01
        xs.append(x)
    if n <= 4097:
        xd = torch.linalg.solve(A.to_dense(), b)
        cond = float(torch.linalg.cond(A.to_dense()))
        assert float((xs[1] - xd).norm() / xd.norm()) <= cond * (1e-10 + 1e-14)


def test_indefinite_matrix_fails_fast():
    A, b = grid_matrix(500)
    A = (A - torch.sparse_coo_tensor(torch.arange(500).repeat(2, 1).cuda(),
                                     torch.full((500,), 2.0, dtype=DT, device="cuda"),
                                     (500, 500))).coalesce()
    with pytest.raises(RuntimeError, match="not positive definite"):
        sparse_solve(A, b, method="cg")


def test_iteration_limit():
    A, b = grid_matrix(3000)
    rowptr, col, val = _csr_arrays(A, b.device)
    solver = PCGSolver(3000, 1, b.device, max_iter=5)
    with pytest.raises(RuntimeError, match="after 5 iterations"):
        solver.solve_csr(rowptr, col, val, b, torch.zeros_like(b), 1e-12)
    solver.close()


def test_threads_and_streams():
    """Two threads on streams of their own: one holds the persistent path, the
    other takes the general one or waits its turn; both are right."""
    models = [model_of("hexa1", (8, 8, 8)), model_of("hexa1", (7, 9, 8))]
    want = [m.solve(stol=1e-10)[0] for m in models]
    conds = [dense(m)[2] for m in models]
    torch.cuda.synchronize()
    errors = []

    def work(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(5):
                    u = models[k].solve(stol=1e-10)[0]
                    torch.cuda.current_stream().synchronize()
                    if float((u - want[k]).norm() / want[k].norm()) > 2.0 * conds[k] * 1.1e-10:
                        errors.append(k)
        except Exception as e:  # noqa: BLE001 - reported by the assertion
            errors.append(repr(e))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
