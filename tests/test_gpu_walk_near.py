"""The walk's records four at a time: cells around the softening length (a batch that
holds one below it takes its cells one by one), particles near and far within a group,
and record counts about the group size, against the oracle's FP64 walk of the same tree."""
import numpy as np
import pytest

import hbtx
import pyoracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("periodic", [0, 1])
@pytest.mark.parametrize("n,softening,theta", [(n, 0.01, 0.7) for n in (2, 3, 4, 5, 7, 8, 9, 63, 64, 65, 257)] +
                         [(3000, e, t) for e in (1e-4, 0.01, 0.05, 0.3) for t in (0.5, 2.0)])
def test_walk_near_softening(ctx, n, softening, theta, periodic):
    rng = np.random.default_rng(n)
    pos = np.concatenate([rng.normal(0.5, 0.02, (n // 2, 3)), rng.uniform(0, 1, (n - n // 2, 3))]).astype(np.float32)
    mass = rng.uniform(0.5, 1.5, n).astype(np.float32)
    prm = dict(theta=theta, softening=softening, periodic=periodic, box_size=4.0)
    ref, _ = O.tree_potential(pos, mass, pos, mass, params=prm)
    t = ctx.tree(pos, mass, hbtx.make_params(**prm))
    got = t.potential(pos, mass)
    t.close()
    # FP32 terms against FP64 ones: some 1e-7; an opening test decided differently in
    # FP32 moves a particle by one cell's monopole error
    rel = np.abs(got - ref) / np.maximum(np.abs(ref), 1e-3 * np.median(np.abs(ref)))
    assert np.quantile(rel, 0.99) < 1e-5 and rel.max() < 1e-3, np.quantile(rel, [0.5, 0.99, 1.0])
