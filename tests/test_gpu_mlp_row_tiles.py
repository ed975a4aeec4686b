"""The all-layers kernels in each of their row tiles, against the CPU oracle: 32
rows below 32,768, 64 rows from there to 65,535, 128 rows from 65,536 on, with
whole and with ragged last tiles, in prediction and in training.  Tolerances as
at the other edges: a prediction differs by single flipped bfloat16 roundings
that travel on (1e-2 of the largest output), a whole gradient by 2e-2 in
relative L2 norm."""
import numpy as np
import pytest

from fvs2d_amd.mlp import WarmStartNet
from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


def _data(n):
    rng = np.random.default_rng(n)
    raw = np.stack([rng.uniform(-20, 20, n), rng.uniform(-20, 20, n), rng.uniform(0, 20, n),
                    rng.uniform(0.5, 0.85, n), rng.uniform(-2, 4, n), rng.uniform(0.1, 0.15, n)], 1)
    return raw.astype(np.float32), rng.normal(0, 0.3, (n, 4)).astype(np.float32)


def _rows(raw):
    return mo.features(raw.astype(np.float64)).astype(np.float32).astype(np.float64)


@pytest.mark.parametrize("depth,n", [(2, 32704), (2, 32768), (3, 32769), (1, 65472), (2, 65473)])
def test_predict(depth, n):
    net = WarmStartNet(depth=depth, batch=65664, seed=depth)
    raw, _ = _data(n)
    y = net.predict(raw)
    rows = np.unique(np.concatenate([np.arange(200), np.arange(n // 2, n // 2 + 100), np.arange(n - 200, n)]))
    ref, _ = mo.forward(net.get_params().astype(np.float64), _rows(raw[rows]), depth, bf16_mode=True)
    assert np.max(np.abs(y[rows] - ref)) <= 1e-2 * np.max(np.abs(ref))


@pytest.mark.parametrize("depth,n", [(2, 32704), (2, 32768), (1, 32769), (2, 65472), (2, 65536), (2, 65601)])
def test_gradient(depth, n):
    net = WarmStartNet(depth=depth, batch=65664, seed=depth)
    raw, tgt = _data(n)
    loss, g = net.grad(raw, tgt)
    ref_loss, ref = mo.loss_and_grad(net.get_params().astype(np.float64), _rows(raw), tgt.astype(np.float64), depth,
                                     bf16_mode=True)
    assert abs(loss - ref_loss) <= 1e-3 * ref_loss
    assert np.linalg.norm(g - ref) <= 2e-2 * np.linalg.norm(ref)
