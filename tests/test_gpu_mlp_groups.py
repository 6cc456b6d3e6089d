"""The MLP kernels where their groups of 32 records end: a few rays give record
counts on both sides of a group's edge, down to a part of one group, and more
groups than wavefronts (the full sizes are in test_gpu_fused_full.py).  Biases
of size 1 and both leaf-table layouts, against the FP64 oracle.

Tolerances: the forward carries at least 16 bits per product, so rgb and loss
stay within the fused tests' 1e-3, as do density and colour gradients (pairs,
16 bits).  The MLP's own gradients take both factors of each product in bf16
(half an ulp of 2^-8 each): 2^-8 relative for a single record, to which few
records add no averaging, and as much again for the recomputed activations.
"""
import numpy as np
import pytest
import torch

from test_gpu_fused import oracle_for, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rays,bf16,layout", [(1, False, 1), (2, True, 1), (3, False, 2),
                                                (5, False, 1), (6, True, 2), (41, False, 1)])
def test_few_records_vs_fp64_oracle(oracle_mod, n_rays, bf16, layout):
    from plenvdb_amd import scenes
    from plenvdb_amd.fused import FusedTrainer, unpack_mlp
    from plenvdb_amd.topology import Topology

    sc = scenes.make_scene("c2", n_rays=n_rays)
    rng = np.random.default_rng(n_rays)
    sc["mlp"] = dict(sc["mlp"], b0=rng.normal(size=128).astype(np.float32),
                     b1=rng.normal(size=128).astype(np.float32),
                     b2=rng.normal(size=3).astype(np.float32))
    origins, vmask = Topology.from_mask(sc["mask"]).leaves()
    tr = FusedTrainer(sc, topo=Topology.from_leaves(origins, vmask, sc["reso"], layout=layout),
                      color_bf16=bf16)
    assert tr.topo.two_level == (layout == 2)
    for _ in range(2):  # the second pass meets the first one's records in the workspace
        tr.zero_grad()
        tr.forward_backward()
    torch.cuda.synchronize()
    ref = oracle_for(oracle_mod, tr, sc)
    print("[case]", n_rays, "rays,", tr.records()["total"], "records", flush=True)
    assert tr.records()["total"] == ref["n_mask"]
    assert float(np.abs(tr.ray_out[:, :3].cpu().numpy() - ref["rgb_marched"]).max()) <= 1e-3
    assert abs(float(tr.loss.item()) - ref["loss"]) <= 1e-3 * abs(ref["loss"])
    assert rel_l2(tr.grad_density.cpu().numpy(), ref["grad_density"]) <= 1e-3
    assert rel_l2(tr.grad_color.cpu().numpy(), ref["grad_color"]) <= 1e-3
    gm = unpack_mlp(tr.mlp_grad.cpu().numpy())
    for k in gm:
        assert rel_l2(gm[k], ref["grad_mlp"][k]) <= 2 ** -7, k
