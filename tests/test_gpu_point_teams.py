"""Kernels that give an element one lane per Gauss point (csrc/assembly.hip):
element counts around the 64 / n_gp elements of a wave, several right-hand
sides, a previous flux.

Tolerances: every result is a sum of at most 8 points x 20 nodes x 9 products
of FP64 numbers, so n eps = 1440 * 1.1e-16 = 1.6e-13 of the largest
magnitude, times 6 for the conditioning of J^{-1} on these elements.
"""

import pytest
import torch

import oracle as O
from torchfem import Planar, Solid, SolidHeat
from torchfem.base import _MatHolder, _SensView
from torchfem.materials import (IsotropicConductivity3D, IsotropicElasticity3D,
                                IsotropicElasticityPlaneStress)

pytestmark = pytest.mark.gpu
DT = torch.float64
TOL = 1e-12


def model(name, n, general):
    """The first n elements of a distorted mesh, with per-element materials."""
    g = torch.Generator().manual_seed(n)
    if name == "Quad1":
        nodes, el = O.rect_quad(n + 1, 2, 1.0 * n, 1.0)
    elif name.startswith("Tetra1"):
        nodes, el = O.cube_tetra6(4, jitter=0.1, seed=1)
        el = el[:n]
    else:
        nodes, el = O.cube_hexa(n + 1, 2, 2)
        if name == "Hexa2":
            nodes, el = O.linear_to_quadratic(nodes, el)
    used, el = torch.unique(el, return_inverse=True)
    nodes = nodes[used].to(DT)
    nodes = nodes + 0.02 / n * torch.sin(3.0 * nodes.roll(1, dims=1))
    E = 800.0 + 400.0 * torch.rand(n, generator=g, dtype=DT)
    if name == "Tetra1-heat":
        m = SolidHeat(nodes.cuda(), el.cuda(), IsotropicConductivity3D(E))
        return m, O.OracleModel(nodes, el, O.Tetra1, "heat", O.iso_KAPPA(E))
    nu = torch.tensor(0.3, dtype=DT)
    C = O.plane_stress_C(E, nu) if name == "Quad1" else O.iso3d_C(E, nu)
    iso = IsotropicElasticityPlaneStress if name == "Quad1" else IsotropicElasticity3D
    mat = iso(E, nu).vectorize(n)
    if general:
        C = C * (1.0 + 0.3 * torch.rand(n, 1, 1, 1, 1, generator=g, dtype=DT))
        C[:, 0, 0, 0, 0] *= 1.5
        mat.C = C.clone()
    cls = Planar if name == "Quad1" else Solid
    m = cls(nodes.cuda(), el.cuda(), mat)
    if name == "Quad1":
        return m, O.OracleModel(nodes, el, O.Quad1, "planar", C, thickness=torch.ones(n, dtype=DT))
    return m, O.OracleModel(nodes, el, O.ELEMENTS[name], "solid", C)


SIZES = [("Quad1", 15, False), ("Quad1", 17, True), ("Tetra1", 63, False), ("Tetra1", 65, True),
         ("Tetra1-heat", 64, False), ("Hexa1", 1, False), ("Hexa1", 7, True), ("Hexa1", 8, False),
         ("Hexa1", 9, True), ("Hexa1", 65, False), ("Hexa2", 1, True), ("Hexa2", 9, False)]


def close(a, b):
    return float((a.cpu() - b).abs().max()) <= TOL * float(b.abs().max())


@pytest.mark.parametrize("name,n,general", SIZES)
def test_forces_fluxes_and_sensitivities(name, n, general):
    m, o = model(name, n, general)
    kind, p0, p1, sc = m._material_params()
    h = _MatHolder(kind, p0, p1, sc)
    g = torch.Generator().manual_seed(7)
    u = torch.randn(3, o.n_dofs, generator=g, dtype=DT)
    lam = torch.randn(3, o.n_dofs, generator=g, dtype=DT)
    k0, f, grad, flux = o.integrate(u[0], need_k=True)
    nq = m.n_dof_per_node * m.n_dim
    prev = torch.randn(m.n_int, n, nq, generator=g, dtype=DT) * float(flux.abs().max())
    F, fe, gm, qm, gg, qg = m._forces(h.mat, u[0].cuda(), means=True, per_gp=True)
    H = grad.reshape(gg.shape)
    if m.n_dof_per_node > 1:
        H = H - torch.eye(m.n_dim, dtype=DT).reshape(-1)
    assert close(gg, H) and close(gm, H.mean(0))
    assert close(qg, flux.reshape(qg.shape)) and close(qm, flux.reshape(qg.shape).mean(0))
    assert close(fe.reshape(f.shape), f)
    assert close(F, o.assemble_rhs(f))
    # a previous flux adds to the flux and, through the same weights, to the forces
    _, fe2, _, _, _, qg2 = m._forces(h.mat, u[0].cuda(), per_gp=True, flux_prev=prev.cuda())
    assert close(qg2, flux.reshape(prev.shape) + prev)
    _, fe1, _, _, _, _ = m._forces(h.mat, 0.0 * u[0].cuda(), flux_prev=prev.cuda())
    assert close(fe2, (fe + fe1).cpu())
    # K is linear in its parameters: their sensitivities times the parameters,
    # and the one of the scale, are lam_e K_e u_e
    out = _SensView(m, h).sensitivity(u.cuda(), lam.cuda(), -1.0).cpu()
    pars = torch.stack([p0, p1], 1) if p1 is not None else p0
    pars = pars.reshape(n, -1).cpu()
    idx = o.idx.reshape(n, -1)
    for r in range(3):
        ref = -torch.einsum("ei,eij,ej->e", lam[r][idx], k0.reshape(n, idx.shape[1], -1), u[r][idx])
        assert close(out[r, :, -1], ref)
        assert close((out[r, :, :-1] * pars).sum(1), ref)


@pytest.mark.parametrize("name,n,general", SIZES)
def test_element_matrices(name, n, general):
    """Element counts around the elements of a block (16, 4, 1)."""
    m, o = model(name, n, general)
    k0 = o.integrate(torch.zeros(o.n_dofs, dtype=DT), need_k=True)[0]
    assert close(m.k0().reshape(k0.shape), k0)


@pytest.mark.parametrize("orphans", [False, True])
@pytest.mark.parametrize("name,n,general", SIZES)
def test_assembly_of_element_matrices(name, n, general, orphans):
    """Any (unsymmetric) element matrices; nodes of no element first and last.
    At most 24 terms per entry: 24 eps = 2.7e-15 of the largest sum."""
    m, o = model(name, n, general)
    if orphans:
        X, el = m.nodes, m.elements
        X = torch.cat([X[:1], X[:1], X, X[:2]])
        m = type(m)(X, el + 2, None)
    g = torch.Generator().manual_seed(3)
    W = m._pattern.npe * m.n_dof_per_node
    k = torch.randn(n, W, W, generator=g, dtype=DT)
    con = torch.nonzero(torch.rand(m.n_dofs, generator=g) < 0.2).reshape(-1)
    K = m.assemble_matrix(k.cuda(), con.cuda()).to_dense().cpu()
    idx = m.idx.cpu().long()
    ref = torch.zeros(m.n_dofs, m.n_dofs, dtype=DT)
    ref.index_put_((idx[:, :, None].expand_as(k), idx[:, None, :].expand_as(k)), k, accumulate=True)
    ref[con], ref[:, con] = 0.0, 0.0
    ref[con, con] = 1.0
    assert float((K - ref).abs().max()) <= 3e-15 * float(ref.abs().max()) * 24
