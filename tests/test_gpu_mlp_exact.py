"""GPU: the network's products where no rounding can differ from the oracle's
(oracle/mlp_ref.py): inputs, weights and errors are small integers (times 32 in
front of tanh, which then is -1, 0 or 1), so that every product and sum is exact
in FP32 in any order, and what is rounded to BF16 is the same number on both
sides.  Outputs and gradients have to be equal.  Layers of one input or one
hidden value (whose two strides are both 1), ragged remainders of every tile,
of the 256-row parts of the weight gradients and of the row of ones behind the
biases."""
import numpy as np
import pytest

import edus

mlp_ref = pytest.importorskip("mlp_ref")

pytestmark = pytest.mark.gpu

SHAPES = [(1, 16, 4, 65), (5, 1, 3, 67), (5, 1, 3, 66), (1, 1, 1, 1), (1, 64, 64, 300), (64, 1, 8, 515),
          (4, 16, 1, 1), (63, 65, 67, 256), (66, 80, 9, 65), (52, 33, 36, 1025), (148, 256, 64, 515)]


def _ints(rng, shape, nonzero):
    """-1, 0 and 1, about `nonzero` values of each column not zero."""
    p = min(1.0, nonzero / shape[0])
    return rng.choice([-1.0, 0.0, 1.0], size=shape, p=[p / 2, 1 - p, p / 2])


def _case(din, dh, dout, rows):
    rng = np.random.default_rng(din + 7 * dh + rows)
    # a layer of one input needs a bias to reach 0, where tanh has a derivative,
    # from an input that is not 0
    parts = [32 * _ints(rng, (din, dh), 2), 32 * _ints(rng, (dh,), dh / 2 if din > 1 else dh),
             32 * _ints(rng, (dh, dh), 2), 32 * _ints(rng, (dh,), dh / 2 if dh > 1 else rows % 2),
             _ints(rng, (dh, dout), 3), _ints(rng, (dout,), dout / 2)]
    params = np.concatenate([a.ravel() for a in parts]).astype(np.float32)
    X = rng.choice([-1.0, 0.0, 1.0], size=(rows, din)).astype(np.float32)
    y, _ = mlp_ref.forward(params, X, din, dh, dout)
    # 2 (Y - T) / n is a small integer
    T = (y - 0.5 * y.size * rng.choice([-2, -1, 1, 2], size=y.shape)).astype(np.float32)
    loss, grads = mlp_ref.grads(params, X, T, din, dh, dout)
    assert np.abs(y).max() < 2 ** 24 and np.abs(T).max() < 2 ** 23 and np.abs(grads).max() < 2 ** 24
    return params, X, T, y, loss, grads


@pytest.mark.parametrize("din,dh,dout,rows", SHAPES)
def test_equal(din, dh, dout, rows):
    print("case", din, dh, dout, rows, flush=True)
    params, X, T, y, loss_ref, g_ref = _case(din, dh, dout, rows)
    net = edus.Mlp(din, dh, dout, 3)
    net.set_params(params)
    assert np.array_equal(net.forward(X), y)
    loss, g = net.gradients(X, T)
    assert abs(loss - loss_ref) <= 1e-5 * loss_ref
    assert np.array_equal(g, g_ref)


@pytest.mark.parametrize("din,dh", [(1, 8), (6, 1)])
def test_width_one_trains(din, dh):
    rng = np.random.default_rng(3)
    X = rng.uniform(-1, 1, size=(2048, din)).astype(np.float32)
    T = np.tanh(X.sum(1, keepdims=True) / din).astype(np.float32)
    hist = edus.Mlp(din, dh, 1, seed=1).train(X, T, epochs=20, batch=256, lr=1e-2, seed=2)
    assert hist[-1] < hist[0]
