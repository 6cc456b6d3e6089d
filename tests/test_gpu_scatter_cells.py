"""The scatter by cell, which a step takes when its record capacity is large, also
for its leaves: few leaves (a block of 2 x 2 x 2 with a diagonal neighbour, so that cells
reach over faces, edges and corners into present and missing leaves), against the
FP64 oracle, and against the scatter by chunks on the same records, which the
same step takes with a capacity that just holds them.

Tolerances: the oracle's as in the fused tests (1e-3).  The two scatters add the
same fp32 terms in other orders, up to a few thousand to a voxel: n 2^-24 of their
magnitudes' sum at worst, 1e-4 of the result with n = 1700 and no cancellation.
"""
import numpy as np
import pytest
import torch

from test_gpu_fused import oracle_for, rel_l2

pytestmark = pytest.mark.gpu


def _scene(n_rays, holes):
    from plenvdb_amd import scenes

    sc = scenes.make_scene("c2", n_rays=n_rays)
    mask = np.zeros_like(sc["mask"])
    mask[72:88, 72:88, 72:88] = True
    mask[88:96, 88:96, 88:96] = True
    if holes:
        mask &= np.random.default_rng(n_rays).random(mask.shape) < 0.8
    sc["mask"] = mask
    return sc


@pytest.mark.parametrize("n_rays,bf16,holes", [(500, False, False), (1700, True, True),
                                               (9000, False, True)])
def test_cells_vs_oracle_and_chunks(oracle_mod, n_rays, bf16, holes):
    from plenvdb_amd.fused import FusedTrainer
    from plenvdb_amd.topology import Topology

    sc = _scene(n_rays, holes)
    topo = Topology.from_mask(sc["mask"])
    tr = FusedTrainer(sc, topo=topo, color_bf16=bf16, capacity=13 << 20)
    assert topo.nleaf == 9
    for _ in range(2):  # the second pass meets the first one's counts and buffers
        tr.zero_grad()
        tr.forward_backward()
    total = tr.records()["total"]
    print("[case]", n_rays, "rays,", total, "records", flush=True)
    ch = FusedTrainer(sc, topo=topo, color_bf16=bf16, capacity=total)
    assert ch.ws_bytes < tr.ws_bytes // 8
    ch.forward_backward()
    torch.cuda.synchronize()
    assert ch.records()["total"] == total
    for k in ("grad_density", "grad_color"):
        a, b = (getattr(t, k).cpu().numpy() for t in (tr, ch))
        assert np.abs(b).sum() > 0 and rel_l2(a, b) <= 1e-4, k
        np.testing.assert_array_equal(a != 0, b != 0)
    assert torch.equal(tr.mlp_grad, ch.mlp_grad) and torch.equal(tr.loss, ch.loss)
    if n_rays <= 1700:
        ref = oracle_for(oracle_mod, tr, sc)
        assert rel_l2(tr.grad_density.cpu().numpy(), ref["grad_density"]) <= 1e-3
        assert rel_l2(tr.grad_color.cpu().numpy(), ref["grad_color"]) <= 1e-3
    # the touched leaves: both optimizers move the same voxels
    tr.adam_only()
    ch.adam_only()
    for k in ("m_density", "m_color"):
        a, b = (getattr(t, k).cpu().numpy() for t in (tr, ch))
        assert rel_l2(a, b) <= 1e-4, k
        np.testing.assert_array_equal(a != 0, b != 0)
    assert not tr.grad_rows.any()
