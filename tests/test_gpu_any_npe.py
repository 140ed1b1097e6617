"""tfm_pattern_expand and tfm_assemble_elements on elements of any number of
nodes (the library's own have 4, 8 and 20), and on a stated max_deg beyond what
the tiled kernel holds in LDS, against dense sums.

Tolerance: every entry is a sum of at most max_inc terms in another order:
max_inc eps sum |terms|, bounded with |k| <= 1 by max_inc^2 eps.
"""

import ctypes as C

import pytest
import torch

from torchfem import _lib as L
from torchfem._pattern import build_host_pattern

pytestmark = pytest.mark.gpu
DT = torch.float64


@pytest.mark.parametrize("ndof", [1, 2, 3])
@pytest.mark.parametrize("npe,stated", [(1, 0), (2, 0), (3, 0), (4, 0), (5, 0), (8, 0), (10, 0),
                                        (20, 0), (27, 0), (4, 4000), (8, 2500), (20, 2500)])
def test_element_matrices_of_any_width(npe, stated, ndof):
    g = torch.Generator().manual_seed(npe * 10 + ndof)
    n_nod, n_elem = 60 + npe, 41
    el = torch.stack([torch.randperm(n_nod - 3, generator=g)[:npe] for _ in range(n_elem)])
    pat = build_host_pattern(el, n_nod, ndof)  # the last three nodes are orphans
    W, n = npe * ndof, n_nod * ndof
    k = 2.0 * torch.rand(n_elem, W, W, generator=g, dtype=DT) - 1.0
    con = torch.rand(n, generator=g) < 0.2

    dev = {q: torch.as_tensor(pat[q]).cuda() for q in
           ("adj_ptr", "adj", "val_ptr", "ne_ptr", "ne_elem", "ne_loc")}
    epos = torch.as_tensor(pat["epos"].astype("int16")).cuda()  # the same 16 bits
    el32, nodes = el.to(torch.int32).cuda(), torch.zeros(n_nod, 3, dtype=DT, device="cuda")
    inc = int(torch.bincount(el.reshape(-1)).max())
    deg = int((pat["adj_ptr"][1:] - pat["adj_ptr"][:-1]).max())
    nnz = int(pat["val_ptr"][-1])
    mesh = L.Mesh(nodes=L.ptr(nodes), elements=L.ptr(el32), n_nod=n_nod, n_elem=n_elem, dim=3,
                  npe=npe, ndof=ndof, etype=0, max_deg=max(deg, stated), max_inc=inc, nnz=nnz,
                  epos=L.ptr(epos), **{q: L.ptr(v) for q, v in dev.items()})
    assert inc * mesh.max_deg <= 48 * 1024  # what the entry point takes
    s = torch.cuda.current_stream().cuda_stream

    rows, cols = (torch.empty(nnz, dtype=torch.int64, device="cuda") for _ in range(2))
    k_map = torch.empty(n_elem, W, W, dtype=torch.int32, device="cuda")
    L.check(L.lib().tfm_pattern_expand(s, C.byref(mesh), L.ptr(rows), L.ptr(cols), None,
                                       L.ptr(k_map), None))
    dofs = (el[:, :, None] * ndof + torch.arange(ndof)).reshape(n_elem, W)
    slot = k_map.long().cpu()
    assert torch.equal(rows.cpu()[slot], dofs[:, :, None].expand(-1, W, W))
    assert torch.equal(cols.cpu()[slot], dofs[:, None, :].expand(-1, W, W))

    K = torch.zeros(n * n, dtype=DT).index_add_(
        0, (dofs[:, :, None] * n + dofs[:, None, :]).reshape(-1), k.reshape(-1)).reshape(n, n)
    K[con, :] = 0.0
    K[:, con] = 0.0
    K[con, con] = 1.0
    kd, con8 = k.cuda(), con.to(torch.uint8).cuda()
    tol = inc * inc * torch.finfo(DT).eps
    for form in (L.FP32_PLAIN, L.FP32_DIFF):
        v64 = torch.empty(nnz, dtype=DT, device="cuda")
        v32 = torch.empty(nnz, dtype=torch.float32, device="cuda")
        blk = torch.empty(n_nod, ndof, ndof, dtype=DT, device="cuda")
        L.check(L.lib().tfm_assemble_elements(s, C.byref(mesh), L.ptr(kd), L.ptr(con8), L.ptr(v64),
                                              L.ptr(v32), L.ptr(blk), form))
        got = torch.zeros(n, n, dtype=DT)
        got[rows.cpu(), cols.cpu()] = v64.cpu()
        assert float((got - K).abs().max()) <= tol
        want = torch.stack([K[i * ndof:(i + 1) * ndof, i * ndof:(i + 1) * ndof] for i in range(n_nod)])
        assert float((blk.cpu() - want).abs().max()) <= tol
        r, c = rows.cpu(), cols.cpu()
        ref = v64.cpu()
        if form == L.FP32_DIFF:  # diagonal blocks hold the row sums (nodes of elements)
            used = torch.zeros(n_nod, dtype=torch.bool)
            used[el.reshape(-1)] = True
            b = torch.arange(n) % ndof
            sums = torch.stack([got[:, b == q].sum(1) for q in range(ndof)], 1)
            here = (r // ndof == c // ndof) & used[r // ndof]
            ref = torch.where(here, sums[r, c % ndof], ref)
        eps32 = torch.finfo(torch.float32).eps
        bound = eps32 * ref.abs() + deg * inc * inc * torch.finfo(DT).eps
        assert bool(((v32.cpu().double() - ref).abs() <= bound).all())
