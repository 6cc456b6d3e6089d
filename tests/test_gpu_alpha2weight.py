"""Alphas2Weights over rays of every length around a wavefront's 64 samples, with
early stops inside, at and past its edge, against the same sequential products
and sums in numpy: equal bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("big", [0.02, 0.3])
def test_sequential_products_and_sums(big):
    from plenvdb_amd import render_utils

    lengths = [0, 1, 2, 63, 64, 65, 127, 128, 129, 300, 0, 5]
    rng = np.random.default_rng(int(100 * big))
    ray_id = np.repeat(np.arange(len(lengths)), lengths)
    n = len(ray_id)
    f = np.float32
    alpha = rng.uniform(0, big, n).astype(f)
    start = np.cumsum([0] + lengths)
    alpha[start[4] + 63] = alpha[start[5] + 63] = alpha[start[6] + 64] = 1.0  # stops at the edges
    w, T, last = np.zeros(n, f), np.ones(n, f), np.ones(len(lengths), f)
    stop = np.zeros(len(lengths), np.int64)
    for r, m in enumerate(lengths):
        t, i = f(1), start[r]
        while i < start[r] + m:
            T[i], w[i] = t, t * alpha[i]
            t = f(np.float64(t) * (1.0 - np.float64(alpha[i])))
            i += 1
            if np.float64(t) < 1e-3:
                break
        last[r], stop[r] = t, i
    gw, gl = rng.normal(size=n).astype(f), rng.normal(size=len(lengths)).astype(f)
    ga = np.zeros(n, f)
    for r in range(len(lengths)):
        back = gl[r] * last[r]
        for i in range(stop[r] - 1, start[r] - 1, -1):
            den = np.float64(f(1) - alpha[i]) + 1e-10
            ga[i] = f(np.float64(gw[i] * T[i]) - np.float64(back) / den)
            back = f(back + f(gw[i] * w[i]))
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    out = render_utils.alpha2weight(dev(alpha), dev(ray_id), len(lengths))
    for got, want in zip(out[:3], (w, T, last)):
        np.testing.assert_array_equal(got.cpu().numpy(), want)
    some = np.array(lengths) > 0
    np.testing.assert_array_equal(out[4].cpu().numpy()[some], stop[some])
    got = render_utils.alpha2weight_backward(dev(alpha), *out, len(lengths), dev(gw), dev(gl))
    np.testing.assert_array_equal(got.cpu().numpy(), ga)
