"""The autotuner on a step that scatters by cell: the scatter's workgroup count and
chunk length are choices of the scatter by chunks alone, so they are neither timed nor
reported there."""
import pytest
import torch

from test_gpu_scatter_cells import _scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("capacity,cells", [(13 << 20, True), (1 << 16, False)])
def test_choices_follow_the_scatter(capacity, cells):
    from plenvdb_amd import autotune
    from plenvdb_amd.fused import FusedTrainer
    from plenvdb_amd.topology import Topology

    sc = _scene(300, False)
    tr = FusedTrainer(sc, topo=Topology.from_mask(sc["mask"]), capacity=capacity)
    assert tr.scatters_by_cell() == cells
    for source in ("tuned", "cache"):
        out = tr.autotune(reps=1, force=source == "tuned")
        assert out["source"] == source
        want = {"mlp_fwd_workgroups", "ray_waves"}
        if not cells:
            want |= {"scatter_workgroups", "scatter_chunk_records"}
        assert set(out["launch"]) == want
        if source == "tuned":
            assert set(out["stage_ms"]) == want
    tr.forward_backward()
    torch.cuda.synchronize()
