"""The all-layers forward and backward kernels at the edges of their row tiles
(32, 64 and 128 rows), against the CPU oracle.

Prediction: the oracle's bfloat16 form rounds the same activations, so a value
differs by single flipped roundings (2^-9 of an activation) that travel on;
1e-2 of the largest output, as in the parity tests.  The gradient of every row
count: relative L2 error 2e-2 (the same reasoning, per whole gradient)."""
import numpy as np
import pytest

from fvs2d_amd.mlp import WarmStartNet
from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


def _data(n, seed):
    rng = np.random.default_rng(seed)
    raw = np.stack([rng.uniform(-20, 20, n), rng.uniform(-20, 20, n), rng.uniform(0, 20, n),
                    rng.uniform(0.5, 0.85, n), rng.uniform(-2, 4, n), rng.uniform(0.1, 0.15, n)], 1)
    return raw.astype(np.float32), rng.normal(0, 0.3, (n, 4)).astype(np.float32)


def _rows(raw):
    return mo.features(raw.astype(np.float64)).astype(np.float32).astype(np.float64)


# tiles of 32, 64 (from 16,384 rows) and 128 (from 65,536), whole and ragged
@pytest.mark.parametrize("depth,n", [(1, 1), (3, 31), (8, 97), (2, 16384), (2, 16449), (1, 65536), (2, 65601)])
def test_predict_at_tile_edges(depth, n):
    net = WarmStartNet(depth=depth, batch=66048, seed=depth)
    raw, _ = _data(n, n)
    y = net.predict(raw)
    rows = np.unique(np.concatenate([np.arange(min(n, 200)), np.arange(max(0, n - 200), n)]))
    ref, _ = mo.forward(net.get_params().astype(np.float64), _rows(raw[rows]), depth, bf16_mode=True)
    assert np.max(np.abs(y[rows] - ref)) <= 1e-2 * np.max(np.abs(ref))


# weight gradient: 1, 4, 26, 43 and 64 row slices of 2, 1, 5, 12 and 8 slabs, in
# one group (slab counts not a multiple of 4) and in four
@pytest.mark.parametrize("depth,n", [(1, 1), (2, 65), (3, 4097), (2, 16449), (3, 16384)])
def test_gradient_at_tile_edges(depth, n):
    net = WarmStartNet(depth=depth, batch=16512, seed=depth)
    raw, tgt = _data(n, n)
    loss, g = net.grad(raw, tgt)
    ref_loss, ref = mo.loss_and_grad(net.get_params().astype(np.float64), _rows(raw), tgt.astype(np.float64), depth,
                                     bf16_mode=True)
    assert abs(loss - ref_loss) <= 1e-3 * ref_loss
    assert np.linalg.norm(g - ref) <= 2e-2 * np.linalg.norm(ref)


@pytest.mark.parametrize("n", [3, 100, 192, 1088, 4160])
def test_output_bias_gradient_adds_rounded_terms(n):
    """With a row count that is no power of two, 1/(4n) is inexact, and the output
    layer's bias gradient shows whether each row's term was rounded before it was
    added.  Terms recomputed in numpy's float32 from the device's own predictions,
    added in the kernel's order: rows rs, rs + 8, ... of 128, pairs of the eight
    sums, the four pairs; then the blocks' sums by 16 groups and a tree."""
    net = WarmStartNet(depth=2, batch=4160, seed=4)
    raw, tgt = _data(n, n)
    _, g = net.grad(raw, tgt)
    rows = (n + 63) // 64 * 64
    f = np.float32
    d = np.zeros(((rows + 127) // 128 * 128, 4), f)
    d[:n] = net.predict(raw) - tgt
    dy = (f(2) * d) * f(1.0 / (4.0 * n))
    part = []
    for b in range(0, len(d), 128):
        s = np.zeros((8, 4), f)
        for k in range(0, 128, 8):
            s = s + dy[b + k:b + k + 8]
        s = s[0::2] + s[1::2]
        part.append(((s[0] + s[1]) + s[2]) + s[3])
    red = np.zeros((16, 4), f)
    for b, p in enumerate(part):
        red[b % 16] = red[b % 16] + p
    h = 8
    while h:
        red[:h] = red[:h] + red[h:2 * h]
        h //= 2
    assert np.array_equal(g[-4:], red[0])
