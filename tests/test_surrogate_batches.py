"""The batched network kernel at the edges of its sample tiles (32) and of its workgroup
count (256 tiles), against the float64 network oracle."""
import numpy as np
import pytest

import mlp_np as R
import pmfmhd as M
from pmfmhd.surrogate import Surrogate

pytestmark = pytest.mark.gpu


def setup(rows, seed=3):
    rng = np.random.default_rng(seed)
    X = rng.normal(0, 1, (rows, 16)).astype(np.float32)
    Y = rng.normal(0, 0.5, (rows, 9)).astype(np.float32)
    s = M.allocate_state((16, 16, 16), 1 / 16, dtype=np.float32)
    net = Surrogate(s, seed=7)
    net.reserve(rows)
    net.upload(X, Y)
    return net, X, Y


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("rows", [1, 31, 32, 33, 257, 32 * 256 + 33])
def test_gradient_and_outputs_at_tile_edges(rows, bf16):
    """float32: 2e-5 of the largest entry, as the repository's gradient test; bfloat16 against the
    oracle with rounded operands: a last-bit difference flips the rounding of some operands
    (2^-8 of each), so 2e-3 (2e-2 against the unrounded network)."""
    net, X, Y = setup(rows)
    w = net.weights()
    want, _ = R.forward(w, X, round_bf16=bf16)
    loss, g = R.loss_and_grad(w, X, Y, round_bf16=bf16)
    tol = 2e-3 if bf16 else 2e-5
    got = net.predict(bf16=bf16)
    assert np.abs(got - want).max() <= tol * np.abs(want).max()
    l, gg = net.grad(bf16=bf16)
    assert abs(l - loss) <= tol * loss
    assert np.abs(gg - g).max() <= tol * np.abs(g).max()
    # a range that starts inside the dataset
    if rows > 40:
        l, gg = net.grad(first=7, count=33, bf16=bf16)
        loss, g = R.loss_and_grad(w, X[7:40], Y[7:40], round_bf16=bf16)
        assert abs(l - loss) <= tol * loss and np.abs(gg - g).max() <= tol * np.abs(g).max()


@pytest.mark.parametrize("batch", [5, 32, 100])
def test_first_training_step_uses_the_hashed_minibatch(batch):
    """Adam's first step moves every weight by lr against its gradient's sign: checked on the
    entries whose gradient is clear of rounding (a thousandth of the largest); lr 0 moves none."""
    net, X, Y = setup(200)
    w = net.weights()
    seed = 11
    mask = (1 << 64) - 1
    key = (seed * 0xD1B54A32D192ED03 + 0x9E3779B97F4A7C15) & mask
    idx = []
    for r in range(batch):
        z = (key + r * 0x9E3779B97F4A7C15) & mask
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & mask
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
        idx.append((z ^ (z >> 31)) % 200)
    loss, g = R.loss_and_grad(w, X[idx], Y[idx])
    losses = net.train(1, batch=batch, lr=1e-3, seed=seed, bf16=False)
    assert abs(losses[0] - loss) <= 2e-5 * loss
    moved = net.weights().astype(np.float64) - w
    clear = np.abs(g) > 1e-3 * np.abs(g).max()
    assert clear.sum() > 1000
    # the float32 weight rounds its move by 2^-24 of itself, eps = 1e-8 shortens it by eps / |g|
    slack = 2.0 ** -23 * np.abs(w) + 1e-3 * 1e-8 / np.maximum(np.abs(g), 1e-30) + 1e-3 * 1e-5
    assert np.all(np.abs(moved + 1e-3 * np.sign(g))[clear] <= slack[clear])
    still = net.weights()
    net.train(1, batch=batch, lr=0.0, seed=seed, bf16=False)
    assert np.array_equal(net.weights(), still)
