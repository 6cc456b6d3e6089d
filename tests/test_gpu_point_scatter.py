"""The aggregated per-point scatter and the optimizer's row passes at the edges
of their blocks: fewer points than one workgroup's 64, one more, many points in
one cell (one long list), points outside every leaf."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _topo(R, seed):
    from plenvdb_amd.topology import Topology

    rng = np.random.default_rng(seed)
    mask = np.zeros((R, R, R), bool)
    for a, b, c in rng.integers(0, (R + 7) // 8, size=(12, 3)):
        mask[8 * a: 8 * a + 8, 8 * b: 8 * b + 8, 8 * c: 8 * c + 8] = True
    mask &= rng.random((R, R, R)) < 0.9  # inactive voxels of existing leaves
    return Topology.from_mask(mask)


@pytest.mark.parametrize("C", [1, 3, 12])
@pytest.mark.parametrize("n", [1, 63, 65, 1000])
def test_scatter_sums(oracle_mod, C, n):
    from plenvdb_amd.plenvdb import ColorVDB, DensityVDB

    R = 37
    topo = _topo(R, n)
    o, m = topo.leaves()
    bits = np.unpackbits(m.view(np.uint8).reshape(-1, 64), axis=1, bitorder="little").astype(bool)
    dom = oracle_mod.SlotDomain(o, bits)
    rng = np.random.default_rng(10 * C + n)
    p = rng.uniform(-2, R + 1, size=(n, 3)).astype(np.float32)
    p[: n // 2] = p[0].astype(np.int32) + rng.random((n // 2, 3), dtype=np.float32)  # one cell
    xs, ys, zs = (torch.from_numpy(np.ascontiguousarray(p[:, i])).cuda() for i in range(3))
    g = rng.normal(size=(n, C)).astype(np.float32)
    vdb = DensityVDB([R] * 3, 1, topology=topo) if C == 1 else ColorVDB([R] * 3, C, topology=topo)
    vdb.backward(xs, ys, zs, torch.from_numpy(g).cuda())
    order = 0 if C == 1 else 1
    args = (dom, C, p[:, 0], p[:, 1], p[:, 2])
    want = oracle_mod.trilinear_bwd(*args, g.astype(np.float64), order, "f64").reshape(-1, C)
    size = oracle_mod.trilinear_bwd(*args, np.abs(g).astype(np.float64), order, "f64").reshape(-1, C)
    # each of at most n terms of a slot has four roundings of its own and takes
    # part in at most n additions; the fractions carry one of the position's
    # size, R 2^-24 absolute, on weights' factors of at most one
    bound = 2.0 ** -24 * (n + 6) * size + 3 * R * 2.0 ** -24 * np.abs(g).sum(0)
    assert np.all(np.abs(vdb.grad.cpu().numpy() - want) <= bound)
    vdb.grad.fill_(1.0)
    from plenvdb_amd.plenvdb import ColorOpt, DensityOpt

    (DensityOpt if C == 1 else ColorOpt)(vdb, 0.1, 1e-8, 0.9, 0.99).zero_grad()
    np.testing.assert_array_equal(vdb.grad.cpu().numpy(),
                                  np.repeat(~bits.reshape(-1, 1), C, 1).astype(np.float32))


def test_scatter_keeps_nan_and_infinity():
    from plenvdb_amd.plenvdb import ColorVDB

    topo = _topo(24, 5)
    o, _ = topo.leaves()
    p = (o[0] + 3.5).astype(np.float32)
    x = [torch.full((3,), float(v), device="cuda") for v in p]
    g = torch.zeros(3, 12, device="cuda")
    g[0, 0], g[1, 1], g[2, 11] = float("nan"), float("inf"), -1.0
    v = ColorVDB([24] * 3, 12, topology=topo)
    v.backward(*x, g)
    row = v.grad[int((3 << 6) | (3 << 3) | 3)].cpu()
    assert torch.isnan(row[0]) and torch.isinf(row[1]) and row[11] == -0.125
    assert (row[2:11] == 0).all()


@pytest.mark.parametrize("n", [0, 1, 255, 257])
def test_index_points_equal_tensor_operations(n):
    from plenvdb_amd.grid import VDBGrid

    g = VDBGrid(1, [37, 20, 9], [-1.5, -0.25, 0.1], [1.5, 0.75, 2.0], topology=_topo(37, 1)).to("cuda")
    xyz = torch.randn(n, 3, device="cuda") * 2
    xyz[: n // 4] = float("inf")
    want = g.wld2idx(xyz).t().contiguous()
    torch.testing.assert_close(g._index_points(xyz), want, rtol=0, atol=0, equal_nan=True)
    strided = torch.empty(3, n, device="cuda").copy_(xyz.t()).t()
    torch.testing.assert_close(g._index_points(strided), want, rtol=0, atol=0, equal_nan=True)
    assert not xyz.requires_grad
    lead = g._index_points(xyz.requires_grad_())  # keeps its place in the caller's graph
    assert lead.requires_grad


def test_step_refuses_a_foreign_capture(monkeypatch):
    from plenvdb_amd import scenes
    from plenvdb_amd.fused import FusedTrainer

    tr = FusedTrainer(scenes.make_scene("c2", n_rays=8))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    with pytest.raises(RuntimeError, match="capture_graph"):
        tr.step()
