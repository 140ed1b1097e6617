"""The fused kernels of the two-level iteration (update with restriction,
coarse rows with prolongation) at the edges of their shapes: one, two and four
chunks per aggregate, aggregate counts that leave a block's last rows empty,
and every padded right-hand side count.

The preconditioner only steers the iteration, so what is checked is what a
solve promises (the true relative residual meets stol) and that the coarse
correction works (its iterations stay below those of block-Jacobi alone; a
restriction and prolongation that disagree lose this at once).
"""

import pytest
import torch

from torchfem import Planar, Solid, SolidHeat
from torchfem._coarse import CoarseSpace
from torchfem.materials import (IsotropicConductivity3D, IsotropicElasticity3D,
                                IsotropicElasticityPlaneStress)
from torchfem.mesh import cube_hexa, cube_tetra6, rect_quad

pytestmark = pytest.mark.gpu
DT = torch.float64


def build(kind):
    g = torch.Generator().manual_seed(1)
    nu = torch.tensor(0.3, dtype=DT, device="cuda")
    if kind == "heat":
        nodes, el = cube_tetra6(13, jitter=0.1)
        m = SolidHeat(nodes.cuda(), el.cuda(),
                      IsotropicConductivity3D(0.5 + torch.rand(len(el), generator=g, dtype=DT).cuda()))
    elif kind == "plane":
        nodes, el = rect_quad(61, 46)
        m = Planar(nodes.cuda(), el.cuda(), IsotropicElasticityPlaneStress(
            500.0 + 500.0 * torch.rand(len(el), generator=g, dtype=DT).cuda(), nu))
    else:
        nodes, el = cube_hexa(13, 14, 12)
        m = Solid(nodes.cuda(), el.cuda(), IsotropicElasticity3D(
            500.0 + 500.0 * torch.rand(len(el), generator=g, dtype=DT).cuda(), nu))
    m.constraints[m.nodes[:, 0] == 0.0] = True
    return m, g


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nrhs", [1, 2, 3, 7, 16])
@pytest.mark.parametrize("kind,size", [
    ("solid", 6 * 30), ("solid", 6 * 8), ("solid", 6),      # ~70, ~270 and 2,184 nodes each
    ("plane", 3 * 37), ("plane", 3 * 9), ("plane", 3 * 2),
    ("heat", 201), ("heat", 26), ("heat", 1)])              # four aggregates per block
def test_fused_two_level_iteration(kind, size, nrhs, precision):
    m, g = build(kind)
    space = CoarseSpace(m._pattern, size=size)
    m._coarse_spaces = {id(m._pattern): space}
    F = torch.randn(nrhs, m.n_nod, m.n_dof_per_node, generator=g, dtype=DT).cuda()
    con = m.constraints.reshape(-1)
    stol = 1e-9
    its = {}
    for pc in ("block_jacobi", "two_level"):
        u, _ = m.solve_load_cases(F, precision=precision, preconditioner=pc, stol=stol)
        info = m.last_solve_info["forward"]["pcg"][0]
        assert "two_level_fallback" not in info and info["fp64_fallback"] == 0
        its[pc] = max(info["iterations"])
        for f, x in zip(F, u):
            b = torch.where(con, 0.0, f.reshape(-1))
            r = b - torch.mv(m.K, x.reshape(-1))
            assert float(r.norm() / b.norm()) <= stol * 1.01
    assert m._coarse_for(m._last_system) is space.h
    assert its["two_level"] < its["block_jacobi"]
