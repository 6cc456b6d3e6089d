"""The step's VDB Adam on gradients that leave voxels out: untouched voxels keep
their values and moments, every gradient (inactive voxels' too) ends at zero."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _trainer(reso, modes, mlp):
    from plenvdb_amd import scenes
    from plenvdb_amd.fused import FusedTrainer
    from plenvdb_amd.topology import Topology

    cfg = scenes.SceneConfig("t", reso, 0, 0.0, 0.0, 64, mlp, 1e-4 if mlp else 0.0,
                             channels=12 if mlp else 3)
    rng = np.random.default_rng(3)
    n = (reso + 7) // 8
    g = np.argwhere(rng.random((n, n, n)) < 0.8)
    inside = [8 * g[:, a, None] + np.arange(8) < reso for a in range(3)]
    word = np.packbits((inside[1][:, :, None] & inside[2][:, None, :]).reshape(-1, 64), axis=1,
                       bitorder="little").view(np.uint64)
    masks = np.ascontiguousarray(np.where(inside[0], word, np.uint64(0)))
    topo = Topology.from_leaves((8 * g).astype(np.int32), masks, [reso] * 3)
    d = rng.normal(size=(64, 3)).astype(np.float32)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    sc = {"cfg": cfg, "mask": None, "reso": [reso] * 3, "xyz_min": np.full(3, -1.5, np.float32),
          "xyz_max": np.full(3, 1.5, np.float32), "rays_o": -4 * d, "rays_d": d, "viewdirs": d,
          "far_per_ray": None, "near": 2.0, "stepsize": 0.5, "voxel_size": 3.0 / reso,
          "target": rng.random((64, 3)).astype(np.float32), "voxel_size_ratio": 1.0,
          "act_shift": -4.6, "fast_color_thres": cfg.fast_color_thres, "bg": 1.0}
    if mlp:
        sc["mlp"] = {k: rng.normal(size=s).astype(np.float32) * 0.1 for k, s in
                     (("w0", (39, 128)), ("b0", 128), ("w1", (128, 128)), ("b1", 128),
                      ("w2", (128, 3)), ("b2", 3))}
    tr = FusedTrainer(sc, topo=topo, stepmode_density=modes[0], stepmode_color=modes[1])
    active = torch.from_numpy(np.unpackbits(masks.view(np.uint8), bitorder="little")).bool().cuda()
    return tr, active


@pytest.mark.parametrize("reso,modes,mlp", [(21, (1, 1), True), (24, (1, 1), False),
                                            (21, (0, 1), True), (19, (1, 0), False)])
def test_sparse_gradients(reso, modes, mlp):
    tr, active = _trainer(reso, modes, mlp)
    tr.forward_backward()  # marks the leaves that the step will visit
    ns, nc = tr.color.shape
    leaf = (tr.grad_rows.reshape(ns // 512, -1) != 0).any(1).repeat_interleave(512)
    gen = torch.Generator(device="cuda").manual_seed(5)
    rnd = lambda *s: torch.rand(*s, generator=gen, device="cuda")  # noqa: E731
    gd = torch.where(leaf & (rnd(ns) < 0.3), rnd(ns) - 0.5, 0.0)
    # whole Vec3 groups left out, single components of others zero
    keep = (rnd(ns, nc // 3) < 0.3).repeat_interleave(3, 1) & (rnd(ns, nc) < 0.7)
    gc = torch.where(leaf[:, None] & keep, rnd(ns, nc) - 0.5, 0.0)
    tr.grad_density.copy_(gd)
    tr.grad_color.copy_(gc)
    for t in (tr.m_density, tr.m_color):
        t.copy_(rnd(*t.shape) - 0.5)
    for t in (tr.v_density, tr.v_color):
        t.copy_(rnd(*t.shape))
    visited = leaf if modes == (1, 1) else torch.ones_like(leaf)
    sz = tr._stepsz(tr.lr_grid, 1)
    want = []
    for p, m, v, g, mode in ((tr.density[:, None], tr.m_density[:, None], tr.v_density[:, None],
                              gd[:, None], modes[0]), (tr.color, tr.m_color, tr.v_color, gc, modes[1])):
        grp = 3 if g.shape[1] > 1 else 1
        on = (g.reshape(ns, -1, grp) != 0).any(-1).repeat_interleave(grp, 1) if mode == 1 else g == g
        on = on & (active & visited)[:, None]
        p, m, v, g = (t.double() for t in (p, m, v, g))
        nm, nv = 0.9 * m + 0.1 * g, 0.99 * v + 0.01 * g * g
        want += [torch.where(on, a, b) for a, b in ((p - sz * nm / (1e-8 + nv.sqrt()), p), (nm, m),
                                                    (nv, v))]
    tr.adam_only()
    torch.cuda.synchronize()
    got = (tr.density[:, None], tr.m_density[:, None], tr.v_density[:, None], tr.color, tr.m_color,
           tr.v_color)
    for a, b in zip(got, want):
        # a few roundings of values up to 1 (and step sizes up to 0.1 times |m| / sqrt(v))
        assert torch.allclose(a.double(), b, rtol=2e-6, atol=1e-6)
    assert not bool(tr.grad_rows[:, : nc + 1][visited].any())
