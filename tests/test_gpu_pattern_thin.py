"""The device pattern of meshes whose nodes have few candidates, a thread per
node from 8,192 nodes and up to 32 candidates per node on average, and a wave
per node on the other side of both lines. Integers: equal to the host builder's."""

import numpy as np
import pytest
import torch

from test_gpu_pattern_sort import fan
from torchfem import _lib as L
from torchfem._pattern import build_device_pattern, build_host_pattern

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def mesh(n_nod, npe, n_elem, hub):
    """Random elements (one names a node twice) over n_nod nodes, some of them in
    none; `hub`: elements around the nodes of `fan`, one of them in all."""
    g = torch.Generator().manual_seed(n_elem)
    el = torch.randint(0, n_nod - 2, (n_elem, npe), generator=g)
    el = el[torch.tensor([len(set(e)) == npe for e in el.tolist()])]
    el[7, 2] = el[7, 0]
    if hub:
        el = torch.cat([el, fan(400, npe, hub)[0] + n_nod - 2])
        n_nod += hub + 6
    return el, n_nod


@pytest.mark.parametrize("n_nod,npe,per_node,hub", [
    (8192, 4, 1.0, 0), (8191, 4, 1.0, 0), (8192, 4, 1.99, 0), (8192, 4, 2.02, 0),
    (20000, 8, 0.499, 0), (20000, 8, 0.502, 0), (20000, 20, 0.075, 0), (20000, 4, 1.0, 190),
    (20000, 8, 0.3, 190)])
def test_equals_the_host_builder(n_nod, npe, per_node, hub):
    el, n = mesh(n_nod, npe, int(per_node * n_nod), hub)
    host = build_host_pattern(el, n, 2)
    dev = build_device_pattern(el.int().cuda().contiguous(), n, 2, DEV)
    n_adj = int(host["adj_ptr"][-1])
    for key in ("ne_ptr", "ne_elem", "ne_loc", "adj_ptr", "val_ptr"):
        assert np.array_equal(dev[key].cpu().numpy(), host[key]), key
    assert np.array_equal(dev["adj"].cpu().numpy()[:n_adj], host["adj"])
    assert np.array_equal(dev["epos"].cpu().numpy().view(np.uint16), host["epos"])
    for key in ("nnz", "max_deg", "max_inc"):
        assert dev[key] == host[key], key


def test_more_than_192_neighbours_are_refused():
    el, n = mesh(20000, 4, 20000, 300)
    with pytest.raises(L.HIPError, match="192"):
        build_device_pattern(el.int().cuda().contiguous(), n, 2, DEV)
