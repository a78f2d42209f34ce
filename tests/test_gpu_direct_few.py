"""The periodic exact sum over few sources, to either side of the 32 from which on a block
asks whether its pairs can wrap: where none can, the non-periodic bits either way."""
import numpy as np
import pytest

import hbtx
import pyoracle as O

pytestmark = pytest.mark.gpu
BOX = 4.0


@pytest.mark.parametrize("nt", [1, 130])
@pytest.mark.parametrize("n", [1, 3, 31, 32, 33])
def test_few_sources(ctx, n, nt):
    rng = np.random.default_rng(n)
    src = rng.uniform(1.5, 2.5, (n, 3)).astype(np.float32)
    tgt = rng.uniform(1.5, 2.5, (nt, 3)).astype(np.float32)
    mass = rng.uniform(0.5, 1.5, n).astype(np.float32)
    tm = np.zeros(nt, np.float32)
    prm = dict(softening=0.01)
    per = dict(prm, periodic=1, box_size=BOX)
    plain = ctx.direct_potential(src, mass, tgt, tm, params=hbtx.make_params(**prm))
    assert np.array_equal(ctx.direct_potential(src, mass, tgt, tm, params=hbtx.make_params(**per)), plain)
    # about the box corner: FP32 terms in compensated sums against FP64, 2e-6
    src, tgt = np.mod(src - 2.0, BOX).astype(np.float32), np.mod(tgt - 2.0, BOX).astype(np.float32)
    got = ctx.direct_potential(src, mass, tgt, tm, params=hbtx.make_params(**per))
    exact = O.direct_potential(src, mass, tgt, tm, params=per)
    assert (np.abs(got - exact) / np.abs(exact)).max() < 2e-6
