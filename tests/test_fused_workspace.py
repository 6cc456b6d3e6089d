"""The fused step's workspace: room for some rays, records and leaves is room for
fewer of any of them, also where the smaller step would scatter by cell and the
larger one's workspace holds no room for that."""
import ctypes as C

import numpy as np
import pytest
import torch


def _bytes(n_rays, capacity, nleaf):
    from plenvdb_amd.fused import _workspace_bytes

    return _workspace_bytes(n_rays, capacity, nleaf)


@pytest.mark.parametrize("capacity,nleaf", [(64, 1), (1 << 20, 600), (25 << 20, 600)])
def test_bytes_grow_with_the_rays(capacity, nleaf):
    b = [_bytes(n, capacity, nleaf) for n in (1, 4095, 4096, 4097, 4110, 8192, 65536)]
    assert b == sorted(b)


def test_bytes_grow_with_the_records():
    b = [_bytes(1000, c, 600) for c in (1, 32, 33, 1 << 20, (12 << 20) - 1, 12 << 20, 15 << 20, 64 << 20)]
    assert b == sorted(b)


@pytest.mark.gpu
def test_a_larger_leaf_sets_workspace_serves_a_smaller_one():
    """The step by chunks in place of the one by cell: the same terms in other orders
    (tolerance as in test_gpu_scatter_cells.py)."""
    from test_gpu_scatter_cells import _scene

    from plenvdb_amd import lib
    from plenvdb_amd.fused import FusedTrainer
    from plenvdb_amd.topology import Topology

    sc = _scene(500, True)
    topo = Topology.from_mask(sc["mask"])
    cap = 13 << 20
    large = _bytes(500, cap, 20000)  # of leaves that would not be scattered to by cell
    tr, ch = (FusedTrainer(sc, topo=topo, capacity=cap) for _ in range(2))
    assert tr.ws_bytes > large
    ch.workspace = torch.full((large,), 255, dtype=torch.uint8, device="cuda")
    ch.desc.workspace, ch.desc.workspace_bytes = ch.workspace.data_ptr(), large
    lib.call("pvdb_fused_init", topo.handle, C.byref(ch.desc), lib.stream())
    for t in (tr, ch):
        t.step()
    torch.cuda.synchronize()
    assert ch.records()["total"] == tr.records()["total"] > 0
    assert torch.equal(tr.loss, ch.loss) and torch.equal(tr.mlp, ch.mlp)
    for k in ("m_density", "m_color"):
        a, b = (getattr(t, k).cpu().numpy() for t in (tr, ch))
        assert np.linalg.norm(a - b) <= 1e-4 * np.linalg.norm(b), k
        np.testing.assert_array_equal(a != 0, b != 0)


def test_models_without_the_mlp_reserve_no_cells():
    from plenvdb_amd.fused import _workspace_bytes

    sizes = (8192, 25 << 20, 600)
    assert _workspace_bytes(*sizes, 3) == _workspace_bytes(*sizes, 12) < _workspace_bytes(*sizes, 0) - (12 * 25 << 20)
