"""GPU: the network's products at the edges of their tiles against the numpy
oracle of the same roundings (oracle/mlp_ref.py): rows below, at and above the
64-row tile and the 256-row parts of the weight gradient, sizes that are no
multiple of 4 (element loads) or 16, one output.

Tolerances: both sides round the same values to BF16 and sum in FP32, in another
order: 1e-5 of the largest output, and for gradients, whose BF16 operands may
fall on the other side of a rounding, 2^-8 of the largest gradient (as
tests/test_gpu_mlp.py's bars or tighter)."""
import numpy as np
import pytest

import edus

mlp_ref = pytest.importorskip("mlp_ref")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("din,dh,dout,rows", [(4, 16, 1, 1), (5, 7, 3, 63), (12, 64, 16, 64), (66, 80, 9, 65),
                                              (148, 256, 64, 515), (52, 33, 36, 1025), (63, 65, 67, 256)])
def test_shapes(din, dh, dout, rows):
    print("case", din, dh, dout, rows, flush=True)
    rng = np.random.default_rng(din + rows)
    net = edus.Mlp(din, dh, dout, 3)
    params = net.get_params()
    X = rng.standard_normal((rows, din)).astype(np.float32)
    T = rng.standard_normal((rows, dout)).astype(np.float32)
    ref, _ = mlp_ref.forward(params, X, din, dh, dout)
    got = net.forward(X)
    hidden = 2.0 ** -8 * np.abs(params).max() * dh ** 0.5  # a hidden value rounded the other way
    assert np.abs(got - ref).max() <= 1e-5 * max(1.0, np.abs(ref).max()) + hidden
    loss_ref, g_ref = mlp_ref.grads(params, X, T, din, dh, dout)
    loss, g = net.gradients(X, T)
    assert abs(loss - loss_ref) <= 1e-3 * loss_ref
    assert np.abs(g - g_ref).max() <= 2.0 ** -8 * np.abs(g_ref).max() * 4
    small = net.forward(X[: max(1, rows // 2)])  # a smaller call after a larger one
    assert np.array_equal(small, got[: max(1, rows // 2)])
