"""Sensitivities of general layouts on one-point elements (8 or 16 elements to a
block): element counts around a block, and around the line between the two.

Reference: d/dC[i,j,k,l] = w detJ s dlam_i/dx_j sym(grad u)_kl, d/dKAPPA[i,j] = w
detJ s dlam/dx_i dT/dx_j, and the energies lam_e K_e u_e of the scale, in torch from
eval_shape_functions and k0. Every value is a product of sums of 4 nodes x 3
components (12 x 12 terms of energies): 144 eps = 3.2e-14, times 6 for J^{-1}.
"""

import pytest
import torch

from torchfem import Solid, SolidHeat
from torchfem.base import _MatHolder, _SensView
from torchfem.materials import IsotropicConductivity3D, IsotropicElasticity3D
from torchfem.mesh import cube_tetra6

pytestmark = pytest.mark.gpu
DT = torch.float64
TOL = 2e-13


@pytest.mark.parametrize("nrhs", [1, 3])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 17, 16383, 16384, 16385, 16401])
@pytest.mark.parametrize("heat", [False, True])
def test_one_point_elements(heat, n, nrhs):
    g = torch.Generator().manual_seed(n)
    nodes, el = cube_tetra6(3 if n < 100 else 15, jitter=0.1)
    el = el[:n]
    used, el = torch.unique(el, return_inverse=True)
    nodes, el = nodes[used].to(DT).cuda(), el.cuda()
    E = 800.0 + 400.0 * torch.rand(n, generator=g, dtype=DT)
    if heat:
        mat = IsotropicConductivity3D(E).vectorize(n)
        mat.KAPPA = mat.KAPPA + 100.0 * torch.rand(n, 3, 3, generator=g, dtype=DT)
        m, nd = SolidHeat(nodes, el, mat), 1
    else:
        mat = IsotropicElasticity3D(E, torch.tensor(0.3, dtype=DT)).vectorize(n)
        mat.C = mat.C.clone()
        mat.C[:, 0, 0, 0, 0] *= 1.5
        m, nd = Solid(nodes, el, mat), 3
    h = _MatHolder(*m._material_params())
    u = torch.randn(nrhs, m.n_dofs, generator=g, dtype=DT).cuda()
    lam = torch.randn(nrhs, m.n_dofs, generator=g, dtype=DT).cuda()
    out = _SensView(m, h).sensitivity(u, lam, -1.0)
    xi = torch.full((1, 3), 0.25, dtype=DT, device="cuda")
    _, B, detJ = m.eval_shape_functions(xi)
    B, w = B.reshape(n, 3, 4), detJ.reshape(n) / 6.0
    k0 = m.k0().reshape(n, 4 * nd, 4 * nd)
    for r in range(nrhs):
        ue, le = (v[r].reshape(-1, nd)[el] for v in (u, lam))  # [n, 4, nd]
        Hu, Hl = (torch.matmul(v.transpose(1, 2).contiguous(), B.transpose(1, 2).contiguous())
                  for v in (ue, le))  # [n, nd, 3]
        if not heat:
            Hu = 0.5 * (Hu + Hu.transpose(1, 2))
        ref = -w[:, None, None] * Hl.reshape(n, -1, 1) * Hu.reshape(n, 1, -1)
        assert float((out[r, :, :-1] - ref.reshape(n, -1)).abs().max()) <= TOL * float(ref.abs().max())
        en = -(le.reshape(n, -1) * (k0 * ue.reshape(n, 1, -1)).sum(2)).sum(1)
        assert float((out[r, :, -1] - en).abs().max()) <= TOL * float(en.abs().max())
