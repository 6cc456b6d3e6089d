"""The scatter by cell beyond the few leaves of test_gpu_scatter_cells.py, each time
against the scatter by chunks on the same records: more leaves than one pass of the
leaves' scan takes, whole steps with the MLP's Adam in the counting launch (launched, and
replayed from a captured step), the two-level leaf table, and records whose nearest
voxel's leaf does not exist.

Tolerances: the two scatters add the same fp32 terms in other orders, 1e-4 as in
test_gpu_scatter_cells.py.  From the second step on the parameters differ in their last
bits, so a weight on a bf16 rounding boundary can turn a few records' terms over: 1e-3.
"""
import numpy as np
import pytest
import torch

from test_gpu_fused import rel_l2

pytestmark = pytest.mark.gpu


def _pair(sc, topo, capacity):
    """A trainer that scatters by cell, and one by chunks that holds its records."""
    from plenvdb_amd.fused import FusedTrainer

    tr = FusedTrainer(sc, topo=topo, capacity=capacity)
    assert tr.scatters_by_cell()
    tr.forward_backward()
    total = tr.records()["total"]
    tr.zero_grad()
    ch = FusedTrainer(sc, topo=topo, capacity=total)
    assert not ch.scatters_by_cell()
    return tr, ch, total


def _same_grads(tr, ch):
    for t in (tr, ch):
        t.zero_grad()
        t.forward_backward()
    torch.cuda.synchronize()
    for k in ("grad_density", "grad_color"):
        a, b = (getattr(t, k).cpu().numpy() for t in (tr, ch))
        assert np.abs(b).sum() > 0 and rel_l2(a, b) <= 1e-4, k
        np.testing.assert_array_equal(a != 0, b != 0)
    assert torch.equal(tr.mlp_grad, ch.mlp_grad) and torch.equal(tr.loss, ch.loss)


def test_more_leaves_than_one_scan_pass():
    from plenvdb_amd import scenes
    from plenvdb_amd.topology import Topology

    nleaf = 2100  # three passes of 1024
    sc = scenes.make_scene("c2", n_rays=2000)
    on = np.zeros(20 ** 3, bool)
    on[np.random.default_rng(5).permutation(20 ** 3)[:nleaf]] = True
    sc["mask"] = np.kron(on.reshape(20, 20, 20), np.ones((8, 8, 8), bool)).astype(sc["mask"].dtype)
    topo = Topology.from_mask(sc["mask"])
    assert topo.nleaf == nleaf
    tr, ch, total = _pair(sc, topo, nleaf * (24 << 10))
    print("[case]", total, "records", flush=True)
    _same_grads(tr, ch)
    hit = (tr.grad_density.reshape(nleaf, 512) != 0).any(1)
    assert all(bool(hit[a:a + 1024].any()) for a in (0, 1024, 2048))
    for t in (tr, ch):
        t.adam_only()  # the touched leaves
    for k in ("m_density", "m_color"):
        a, b = (getattr(t, k).cpu().numpy() for t in (tr, ch))
        np.testing.assert_array_equal(a != 0, b != 0)


@pytest.mark.parametrize("layout", [1, 2])
def test_whole_steps(layout):
    from test_gpu_scatter_cells import _scene

    from plenvdb_amd.topology import Topology

    sc = _scene(600, True)
    origins, masks = Topology.from_mask(sc["mask"]).leaves()
    topo = Topology.from_leaves(origins, masks, sc["reso"], layout=layout)
    assert topo.two_level == (layout == 2)
    tr, ch, total = _pair(sc, topo, 13 << 20)
    print("[case] layout", layout, total, "records", flush=True)
    _same_grads(tr, ch)
    for t in (tr, ch):
        t.zero_grad()
    for step in range(4):
        if step == 2:
            tr.capture_graph()
        tr.step()
        ch.step()
        torch.cuda.synchronize()
        if step == 0:
            assert torch.equal(tr.mlp, ch.mlp) and torch.equal(tr.mlp_m, ch.mlp_m)
        for k in ("m_density", "v_density", "m_color", "v_color", "mlp_m", "mlp_v", "mlp"):
            a, b = (getattr(t, k).cpu().numpy() for t in (tr, ch))
            assert rel_l2(a, b) <= (1e-4 if step == 0 else 1e-3), (step, k)
        assert not tr.grad_rows.any()
        assert bool(torch.isfinite(torch.randn(1 << 16, device="cuda").sum()))  # eager work between


def _between(j, reso, mn, mx):
    """A coordinate whose occupancy voxel is j and whose nearest voxel is j + 1: the two
    formulas round differently next to j + 1/2."""
    f = np.float32
    ln, rm1 = f(mx) - f(mn), f(reso - 1)
    ms = rm1 / ln
    mb = -f(mn) * ms
    y = f(mn + (j + 0.5) / (reso - 1) * (mx - mn))
    c = [y]
    for d in (np.inf, -np.inf):
        v = y
        for _ in range(64):
            v = np.nextafter(v, f(d), dtype=f)
            c.append(v)
    p = np.array(c, f)
    occ = np.floor((p * ms + mb).astype(f) + f(0.5))
    near = np.floor(((p - f(mn)) / ln * rm1).astype(f) + f(0.5))
    return p[(occ == j) & (near == j + 1)]


def test_records_of_missing_leaves():
    from plenvdb_amd import scenes
    from plenvdb_amd.topology import Topology

    n = 96
    sc = scenes.make_scene("c2", n_rays=n)
    reso = sc["reso"][1]
    mn, mx = float(sc["xyz_min"][1]), float(sc["xyz_max"][1])
    tops = [j for j in range(39, reso - 9, 8) if len(_between(j, reso, mn, mx))]
    assert tops
    j = tops[len(tops) // 2]  # the last voxel of its leaf
    mask = np.zeros_like(sc["mask"])
    mask[64:96, j - 7:j + 1, 64:96] = True
    sc["mask"] = mask
    rng = np.random.default_rng(1)
    y = np.where(np.arange(n) % 3 == 0, rng.choice(_between(j, reso, mn, mx), n),
                 np.float32(mn + (j - 3.3) / (reso - 1) * (mx - mn))).astype(np.float32)
    z = rng.uniform(66, 94, n) / (reso - 1) * (mx - mn) + mn
    sc["rays_o"] = np.stack([np.full(n, -4.0), y, z], 1).astype(np.float32)
    sc["rays_d"] = sc["viewdirs"] = np.tile(np.array([1, 0, 0], np.float32), (n, 1))
    tr, ch, total = _pair(sc, Topology.from_mask(mask), 13 << 20)
    xyz = tr.records()["xyze"]
    lost = np.floor(xyz[:, 1] + np.float32(0.5)) == j + 1
    print("[case]", total, "records,", int(lost.sum()), "of a missing leaf", flush=True)
    assert lost.sum() >= 100 and (~lost).sum() >= 100
    _same_grads(tr, ch)
