"""The point gather where its short cuts end: cells on the faces, edges and corners of
leaves, beside the leaf table's box, far outside, and with coordinates that are not finite,
with the one-level table (one lookup a cell, none off the box) against the two-level one
(a leaf cache, corner by corner): equal bit for bit, as are rows that are not 16-byte
aligned."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _points(rng):
    """Index coordinates around a 3 x 3 x 3 block of leaves with its origin at 16."""
    edge = np.array([7.5, 8.0, 14.9, 15.0, 15.25, 16.0, 22.75, 23.0, 23.5, 24.0, 31.5, 38.9, 39.0, 39.5,
                     40.0, 47.25, 48.0])
    g = np.stack(np.meshgrid(edge, edge, edge, indexing="ij"), -1).reshape(-1, 3)
    p = [g, rng.uniform(10, 45, (3000, 3)), rng.uniform(-300, 300, (500, 3))]
    odd = rng.uniform(16, 40, (60, 3))
    odd[np.arange(60), np.arange(60) % 3] = np.tile([np.nan, np.inf, -np.inf, 1e9, -1e9], 12)
    p = np.concatenate([*p, odd]).astype(np.float32)
    return p[rng.permutation(len(p))]


@pytest.mark.parametrize("channels,order", [(1, 0), (1, 1), (3, 1), (12, 1)])
def test_layouts_agree(channels, order):
    from plenvdb_amd import lib
    from plenvdb_amd.topology import Topology

    rng = np.random.default_rng(channels)
    on = rng.random((3, 3, 3)) < 0.6
    on[1, 1, 1], on[1, 1, 2], on[0, 0, 0] = True, False, True
    mask = np.zeros((64, 64, 64), bool)
    mask[16:40, 16:40, 16:40] = np.kron(on, np.ones((8, 8, 8), bool))
    one = Topology.from_mask(mask)
    two = Topology.from_leaves(*one.leaves(), [64] * 3, layout=2)
    assert two.two_level and not one.two_level
    pts = torch.from_numpy(_points(rng).T.copy()).cuda()
    n = pts.shape[1]
    store = torch.randn(one.nslots * channels + 1, device="cuda")
    got = []
    for topo, shift in ((one, 0), (two, 0), (one, 1)):
        vals = torch.empty(one.nslots * channels + 1, device="cuda")
        vals[shift:shift + one.nslots * channels] = store[:-1]
        out = torch.empty(n, channels, device="cuda")
        lib.call("pvdb_trilinear_fwd", topo.handle, vals.data_ptr() + 4 * shift, channels, order,
                 *[pts[a].data_ptr() for a in range(3)], n, out.data_ptr(), lib.stream())
        got.append(out)
    torch.testing.assert_close(got[0], got[1], rtol=0, atol=0, equal_nan=True)
    torch.testing.assert_close(got[2], got[1], rtol=0, atol=0, equal_nan=True)
    assert bool(got[0].isnan().any()) and int((got[0] != 0).any(1).sum()) > 1000
