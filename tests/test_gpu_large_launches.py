"""Calls of more items than one launch holds (2^32 work items; more run modulo 2^32 and
report nothing): the items past it are computed too.  The results are exact."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _topo():
    from plenvdb_amd.topology import Topology

    mask = np.zeros((16, 16, 16), bool)
    mask[:8, :8, :8] = True
    return Topology.from_mask(mask)


def test_point_scatter():
    """64 points to a workgroup of 256: 2^30 points.  All but the last lie outside."""
    from plenvdb_amd import lib

    topo = _topo()
    n = (1 << 30) + 640
    x = torch.full((n,), -100.0, device="cuda")  # coordinates and gradients
    x[-3:] = 2.0
    grad = torch.zeros(topo.nslots, device="cuda")
    lib.call("pvdb_trilinear_bwd", topo.handle, lib.ptr(grad), 1, 0, *[lib.ptr(x)] * 4, n, lib.stream())
    want = torch.zeros_like(grad)
    want[2 * 64 + 2 * 8 + 2] = 6.0
    assert topo.nleaf == 1 and torch.equal(grad, want)


def test_alphas_to_weights():
    """2^26 rays, for which a wavefront to a ray would be too many work items.  The last has
    two samples, the first one."""
    from plenvdb_amd import render_utils as ru

    n = (1 << 26) + 5
    alpha = torch.tensor([0.25, 0.5, 0.5], device="cuda")
    rid = torch.tensor([0, n - 1, n - 1], device="cuda")
    w, t, last, i0, i1 = ru.alpha2weight(alpha, rid, n)
    assert w.tolist() == [0.25, 0.5, 0.25] and t.tolist() == [1.0, 1.0, 0.5]
    assert float(last[0]) == 0.75 and float(last[-1]) == 0.25 and bool((last[1:-1] == 1).all())
    gw = torch.tensor([1.0, 2.0, 4.0], device="cuda")
    g = ru.alpha2weight_backward(alpha, w, t, last, i0, i1, n, gw, torch.zeros_like(last))
    # dL/dalpha_i = gw_i T_i - sum of the later gw_j w_j over 1 - alpha_i (+ 1e-10, in doubles)
    assert g.tolist() == [1.0, float(np.float32(2.0 - 4.0 * 0.25 / (0.5 + 1e-10))), 2.0]


def test_zero_active():
    """A thread to a value: 512 slots of 2^23 + 1 channels."""
    from plenvdb_amd import lib

    topo, ch = _topo(), (1 << 23) + 1
    g = torch.full((topo.nslots * ch,), 1.0, device="cuda")
    lib.call("pvdb_zero_active", topo.handle, lib.ptr(g), ch, lib.stream())
    assert not bool(g.any())


def test_workspace_init():
    """A thread to a byte: a workspace of 6 GB."""
    import ctypes as C

    from plenvdb_amd import lib, scenes
    from plenvdb_amd.fused import FusedTrainer, _workspace_bytes

    tr = FusedTrainer(scenes.make_scene("c2", n_rays=16))
    tr.desc.capacity = 26_000_000
    n = _workspace_bytes(16, tr.desc.capacity, tr.topo.nleaf, 12)  # without room for cells
    ws = torch.full((n,), 7, dtype=torch.uint8, device="cuda")
    tr.desc.workspace, tr.desc.workspace_bytes = ws.data_ptr(), n
    lib.call("pvdb_fused_init", tr.topo.handle, C.byref(tr.desc), lib.stream())
    assert n > 1 << 32 and not bool(ws.any())
