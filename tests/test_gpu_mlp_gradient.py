"""The gradient on the matrix instructions at sample counts around a tile (32), a
block (128) and a grid, against the FP64 gradient."""
import numpy as np
import pytest

import hbtx
import mlp_oracle as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 127, 128, 129, 1000, 32767, 32768, 32769, 100_003])
def test_gradient_sizes(ctx, n):
    rng = np.random.default_rng(n)
    net = hbtx.MLP(ctx, 1)
    w = rng.normal(0, 0.3, M.NPAR).astype(np.float32)
    net.set_weights(w)
    X = rng.normal(0, 1, (n, M.NIN)).astype(np.float32)
    y = (rng.random(n) < 0.4).astype(np.uint8)
    g, loss = net.gradient(X, y)
    gref, lref = M.gradient(M.bf16_round(w).astype(np.float64), X.astype(np.float64), y)
    # three 64-term products in FP32 before the sum over the samples, and the hardware
    # exponential in the logistic: about 200 half-ulps of 2^-24, norm-wise
    assert np.linalg.norm(g - gref) <= 200 * 2.0 ** -24 * np.linalg.norm(gref) + 1e-12
    assert abs(loss - lref) <= 200 * 2.0 ** -24 * abs(lref) + 1e-6
    # the same samples again: the same bits
    g2, loss2 = net.gradient(X, y)
    assert np.array_equal(g, g2) and loss == loss2
