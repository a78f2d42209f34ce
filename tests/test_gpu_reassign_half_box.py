"""Tracers beyond half the box from a particle by less than a float can tell: NEAREST goes
by the exact difference of the coordinates, so such a tracer is the nearer image's."""
import numpy as np
import pytest

import pyoracle as O

pytestmark = pytest.mark.gpu
BOX = 4.0
ULP = 2.0 ** -23


@pytest.mark.parametrize("order", [(0, 1, 2), (0, 2, 1)])
@pytest.mark.parametrize("above", [True, False])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_just_beyond_half(ctx, axis, above, order):
    # the difference is 2 + 2^-23, which rounds to 2 in float: distance^2 is 4 - 2^-21 of
    # the nearer image, and the other tracer's is 4
    q, t = np.ones(3), np.ones(3)
    q[axis], t[axis] = (1.0 + ULP, 3.0 + 2.0 * ULP) if above else (3.0 + 2.0 * ULP, 1.0 + ULP)
    u = q.copy()
    u[(axis + 1) % 3] += 2.0
    pos = np.array([q, t, u]).astype(np.float32)[list(order)]
    sub = np.array([0, 1, 2], np.int32)[list(order)]
    tracer = np.array([0, 1, 1], np.int32)
    prm = dict(periodic=1, box_size=BOX)
    got, _ = ctx.reassign_targets(pos, tracer, sub, [0, 3], k=1, params=prm)
    ref = O.reassign_targets(pos, tracer, sub, [0, 3], k=1, params=O.default_params(**prm))
    assert ref[0] == 1
    np.testing.assert_array_equal(got, ref)
