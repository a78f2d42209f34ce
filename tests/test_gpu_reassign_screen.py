"""The search's sorted list of k nearest (its keys held as doubles) at every unrolled size
and the numbers about it, with coincident tracers (distance zero, and ties by index), and
leaves that wrap, do not, and lie at half the box from a query."""
import numpy as np
import pytest

import pyoracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("box,spread", [(0.0, 0.2), (4.0, 0.2), (4.0, 2.2), (4.0, 1.0)])
@pytest.mark.parametrize("k", [1, 7, 8, 9, 10, 11, 16, 17, 31, 32])
def test_k_and_wraps(ctx, k, box, spread):
    rng = np.random.default_rng(k)
    n = 1500
    x = rng.normal(0, spread, (n, 3))
    x[:60] = x[60:120]  # coincident pairs
    if box:
        x = np.mod(x, box)
        x[-20:, 0] = np.mod(x[-40:-20, 0] + 0.5 * box, box)
    pos = x.astype(np.float32)
    if box:
        pos[pos >= box] = 0.0
    tracer = (rng.random(n) < 0.5).astype(np.int32)
    sub = rng.integers(0, 12, n).astype(np.int32)
    goff = np.array([0, 900, 900, n])
    prm = dict(periodic=1, box_size=box) if box else {}
    g, _ = ctx.reassign_targets(pos, tracer, sub, goff, k=k, params=prm)
    o = O.reassign_targets(pos, tracer, sub, goff, k=k, params=O.default_params(**prm))
    np.testing.assert_array_equal(g, o)
