"""The device pattern builder at the edges of its sorts (csrc/pattern.hip): 64,
128 and 256 candidates per node, merged pieces beyond, and the most adjacent
nodes. Integers: equal to the host builder's."""

import numpy as np
import pytest
import torch

from torchfem import _lib as L
from torchfem._pattern import build_device_pattern, build_host_pattern

pytestmark = pytest.mark.gpu


def fan(n_elem, npe, pool, repeats=False):
    """Elements that all hold node 3, and others of nodes 4 .. pool + 3."""
    g = torch.Generator().manual_seed(n_elem * npe + pool)
    if repeats:
        el = torch.randint(3, pool + 4, (n_elem, npe), generator=g)
    else:
        el = torch.stack([torch.randperm(pool, generator=g)[:npe] + 4 for _ in range(n_elem)])
    el[:, 1] = 3
    return el, pool + 6  # nodes of no element first and last


@pytest.mark.parametrize("n_elem,npe,pool,repeats", [
    (1, 4, 10, False), (16, 4, 60, False), (17, 4, 60, False), (32, 4, 120, False),
    (33, 4, 120, False), (64, 4, 188, False), (65, 4, 188, False), (400, 4, 191, False),
    (8, 8, 50, False), (9, 8, 50, False), (13, 20, 191, False), (60, 20, 191, False),
    (40, 8, 30, True)])
def test_equals_the_host_builder(n_elem, npe, pool, repeats):
    el, n = fan(n_elem, npe, pool, repeats)
    host = build_host_pattern(el, n, 3)
    dev = build_device_pattern(el.int().cuda().contiguous(), n, 3, torch.device("cuda", 0))
    n_adj = int(host["adj_ptr"][-1])
    for key in ("ne_ptr", "ne_elem", "ne_loc", "adj_ptr", "val_ptr"):
        assert np.array_equal(dev[key].cpu().numpy(), host[key]), key
    assert np.array_equal(dev["adj"].cpu().numpy()[:n_adj], host["adj"])
    assert np.array_equal(dev["epos"].cpu().numpy().view(np.uint16), host["epos"])
    for key in ("nnz", "max_deg", "max_inc"):
        assert dev[key] == host[key], key


def test_more_than_192_neighbours_are_refused():
    el, n = fan(400, 4, 300)
    with pytest.raises(L.HIPError, match="192"):
        build_device_pattern(el.int().cuda().contiguous(), n, 3, torch.device("cuda", 0))
