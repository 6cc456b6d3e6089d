"""The MLP's ReLU pattern: the order in which the forward sums a pre-activation, and
the backward's use of the same pattern for its own recomputed activations.

The order is the bias, then for every 32 inputs the products with their hi, their mid
and their lo bf16 parts, eight inputs at a time.  Weights and inputs are powers of two
2^10 apart, so a term 2^30 below the sum so far (or below another of its eight) is
lost and one 2^20 below it kept exactly, whatever the rounding: the order alone
decides which small terms survive where large ones cancel, and with them the sign.
A bias gradient is zero exactly where a mask is off for every sample (all samples
have the same encoding inputs, and the colour's weights are zero).

With recomputed activations r from hi parts and the forward's mask on everywhere,
dW = sum of r g over samples for the bias gradient's sum of g: r is exact, and the
products take g in bf16, half an ulp of 2^-8 off.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

V = np.float32(1 + 2.0 ** -10 + 2.0 ** -20)  # parts 1, 2^-10 and 2^-20
PARTS = {0.0: (0, 0, 0), 1.0: (1, 0, 0), float(V): (1, 2.0 ** -10, 2.0 ** -20)}
BIG = 2.0 ** 40
# a view direction (V, 0, 0): column 12, and the cosines of the zeros
ENC = [31, 32, 33, 34, 35, 36, 37, 38]


def _inputs():
    x = np.zeros(40)
    x[12] = V
    x[ENC] = 1.0
    return x


def _preact(x, w, b):
    """[N] pre-activations of x [K] (values of PARTS) under w [K, N], b [N], in order."""
    parts = np.array([PARTS[float(v)] for v in x])
    acc = b.astype(np.float64)
    for k0 in range(0, len(x), 32):
        for p in range(3):
            for k in range(k0, min(k0 + 32, len(x)), 8):
                t = np.concatenate([acc[None], w[k:k + 8] * parts[k:k + 8, p, None]])
                t[np.abs(t) < np.abs(t).max(0) * 2.0 ** -25] = 0.0
                acc = t.sum(0).astype(np.float32).astype(np.float64)
    return acc


def _patterns(rng, inputs, n):
    """w [len(inputs), n], b [n]: large terms that cancel, and small ones."""
    w, b = np.zeros((len(inputs), n)), np.zeros(n)
    for o in range(n):
        at = rng.permutation(len(inputs))[:4]
        big = BIG * (1 if rng.random() < 0.5 else -1)
        w[at[0], o] = big
        if rng.random() < 0.5:
            w[at[1], o] = -big
        else:
            b[o] = -big
        w[at[2], o] = 1.0
        w[at[3], o] = rng.choice([0.0, 1.0, 2.0 ** 20])
    return w, b


def _trainer(mlp):
    from plenvdb_amd import scenes
    from plenvdb_amd.fused import FusedTrainer, unpack_mlp

    sc = scenes.make_scene("c2", n_rays=48)
    sc["viewdirs"] = np.tile(np.array([V, 0, 0], np.float32), (48, 1))
    sc["mlp"] = {k: np.asarray(v, np.float32) for k, v in mlp.items()}
    tr = FusedTrainer(sc)
    tr.forward_backward()
    torch.cuda.synchronize()
    assert tr.records()["total"] > 64
    return unpack_mlp(tr.mlp_grad.cpu().numpy())


def _signs(rng, *shape):
    return rng.choice([-1.0, 1.0], size=shape) * rng.uniform(0.5, 1, size=shape)


@pytest.mark.parametrize("seed", [0, 1])
def test_layer0_order(seed):
    rng = np.random.default_rng(seed)
    w0 = np.zeros((39, 128))
    cols = [12] + ENC
    w0[cols], b0 = _patterns(rng, cols, 128)
    pre = _preact(_inputs(), np.concatenate([w0, np.zeros((1, 128))]), b0)
    exact = b0 + w0.T @ _inputs()[:39]
    assert ((pre > 0) != (exact > 0)).sum() >= 16  # the order matters here
    g = _trainer({"w0": w0, "b0": b0, "w1": _signs(rng, 128, 128) * 2.0 ** -50, "b1": _signs(rng, 128),
                  "w2": _signs(rng, 128, 3) * 0.1, "b2": np.zeros(3)})
    print("[case] layer 0, units on:", int((pre > 0).sum()), flush=True)
    np.testing.assert_array_equal(g["b0"] != 0, pre > 0)


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_layer1_order(seed):
    rng = np.random.default_rng(seed)
    b0 = rng.choice([1.0, V], size=128)
    w1, b1 = _patterns(rng, np.arange(128), 128)
    near = rng.random(128) < 0.5  # half of them within one block of 32 inputs
    blk = rng.integers(0, 4, 128)
    for o in np.flatnonzero(near):
        k = np.flatnonzero(w1[:, o])
        v = w1[k, o]
        w1[:, o] = 0.0
        w1[32 * blk[o] + rng.permutation(32)[:len(k)], o] = v
    pre = _preact(b0, w1, b1)
    exact = b1 + w1.T @ b0
    assert ((pre > 0) != (exact > 0)).sum() >= 8
    g = _trainer({"w0": np.zeros((39, 128)), "b0": b0, "w1": w1, "b1": b1,
                  "w2": _signs(rng, 128, 3) * 2.0 ** -50, "b2": np.zeros(3)})
    print("[case] layer 1, units on:", int((pre > 0).sum()), flush=True)
    np.testing.assert_array_equal(g["b1"] != 0, pre > 0)


def test_dw_operands_take_the_forward_pattern():
    """Units whose pre-activation is 1/2 + 2^-10 .., but -1/2 from the hi parts alone: the
    forward has them on, and the dW products take the recomputed -1/2.  And units that are
    off, but 1/2 from the hi parts: no gradient."""
    rng = np.random.default_rng(3)
    on = np.arange(128) % 2 == 0
    w0 = np.zeros((39, 128))
    w0[12] = np.where(on, 1024.0, -1024.0)           # times V: +-(1024 + 1 + 2^-10)
    w0[31] = -w0[12]
    w0[38] = np.where(on, -0.5, 0.5)
    g = _trainer({"w0": w0, "b0": np.zeros(128), "w1": _signs(rng, 128, 128) * 0.1,
                  "b1": np.ones(128), "w2": _signs(rng, 128, 3) * 0.1, "b2": np.zeros(3)})
    np.testing.assert_array_equal(g["b0"] != 0, on)
    assert np.all(g["w1"][~on] == 0)
    want = -0.5 * np.broadcast_to(g["b1"], (64, 128))
    print("[case] dW1", float(np.abs(g["w1"][on] / want - 1).max()), flush=True)
    assert np.abs(g["b1"]).min() > 0 and np.abs(g["w1"][on] - want).max() <= 2 ** -8 * np.abs(want).max()

    b0 = np.where(np.arange(128) % 4 == 0, V, 1.0)   # H0, exactly
    w1 = np.zeros((128, 128))
    w1[0] = np.where(on, 1024.0, -1024.0)            # H0[0] = V, the other two 1
    w1[1] = -w1[0]
    w1[2] = np.where(on, -0.5, 0.5)
    g = _trainer({"w0": np.zeros((39, 128)), "b0": b0, "w1": w1, "b1": np.zeros(128),
                  "w2": _signs(rng, 128, 3) * 0.1, "b2": np.zeros(3)})
    np.testing.assert_array_equal(g["b1"] != 0, on)
    assert np.all(g["w2"][~on] == 0)
    want = -0.5 * np.broadcast_to(g["b2"], (64, 3))
    print("[case] dW2", float(np.abs(g["w2"][on] / want - 1).max()), flush=True)
    assert np.abs(g["b2"]).min() > 0 and np.abs(g["w2"][on] - want).max() <= 2 ** -8 * np.abs(want).max()
