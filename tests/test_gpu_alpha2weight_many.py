"""Alphas2Weights on both sides of the ray counts at which it goes over from a wavefront
to a thread per ray (8192 forward, 16,384 backward): the same rays, with one more empty
ray to take the other path, equal bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rays", [8192, 16384])
def test_both_paths_agree(n_rays):
    from plenvdb_amd import render_utils as ru

    g = torch.Generator().manual_seed(n_rays)
    lengths = torch.randint(0, 12, (n_rays,), generator=g)
    lengths[::97] = torch.randint(60, 200, (len(lengths[::97]),), generator=g)  # past a wavefront's 64
    lengths[5::31] = 0
    lengths[-1] = 3
    rid = torch.repeat_interleave(torch.arange(n_rays), lengths).cuda()
    n = rid.numel()
    alpha = torch.rand(n, generator=g) ** 3
    alpha[::501] = 1.0  # early stops
    alpha = alpha.cuda()
    gw = torch.randn(n, generator=g).cuda()
    got = []
    for extra in (0, 1):
        out = ru.alpha2weight(alpha, rid, n_rays + extra)
        gl = torch.linspace(-1, 1, n_rays).cuda()
        gl = torch.cat([gl, gl.new_zeros(extra)])
        grad = ru.alpha2weight_backward(alpha, *out, n_rays + extra, gw, gl)
        got.append([*out[:2], *(t[:n_rays] for t in out[2:]), grad])
    for a, b in zip(*got):
        assert torch.equal(a, b)
    assert bool((got[0][0] > 0).any()) and bool((got[0][2] < 1).any())
