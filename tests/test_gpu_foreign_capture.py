"""A step called while the caller captures its stream is refused before it changes
anything: the counter (and with it every later bias correction), the learning rates
and the descriptor's step sizes stay, launched or replayed."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _state(tr):
    d = tr.desc
    return (tr.step_count, tr.lr_grid, tr.lr_mlp, d.stepsz_density, d.stepsz_color, d.step_size_mlp,
            d.adam_scalars, tr.adam_scalars.tolist(), tr.density.clone(), tr.mlp.clone())


def _same(a, b):
    return all(torch.equal(x, y) if isinstance(x, torch.Tensor) else x == y for x, y in zip(a, b))


@pytest.mark.parametrize("replayed", [False, True])
def test_refusal_leaves_the_trainer_as_it_was(monkeypatch, replayed):
    from plenvdb_amd import scenes
    from plenvdb_amd.fused import FusedTrainer

    tr = FusedTrainer(scenes.make_scene("c2", n_rays=64))
    tr.step()
    if replayed:
        tr.capture_graph()
        tr.step()
    before = _state(tr)
    with monkeypatch.context() as m:
        m.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
        for call in (tr.step, tr.adam_only):
            with pytest.raises(RuntimeError, match="capture_graph"):
                call()
    torch.cuda.synchronize()
    assert _same(_state(tr), before)
    tr.step()
    assert tr.step_count == before[0] + 1
