"""The walk's work queue: every item is walked once whatever the number of chunks, items
and waves (fewer items than chunks, than waves, and more)."""
import numpy as np
import pytest

import hbtx
import pyoracle as O
import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt", [1, 64, 65, 448, 512, 513, 577, 8000, 70001])
def test_point_counts(ctx, nt):
    rng = np.random.default_rng(nt)
    pos = rng.uniform(0, 1, (300, 3)).astype(np.float32)
    mass = rng.uniform(0.5, 1.5, 300).astype(np.float32)
    tgt = rng.uniform(0, 1, (nt, 3)).astype(np.float32)
    zero = np.zeros(nt, np.float32)
    prm = dict(theta=0.0, softening=0.01)
    t = ctx.tree(pos, mass, hbtx.make_params(**prm))
    got = t.potential(tgt, zero)
    t.close()
    ref = O.direct_potential(pos, mass, tgt, zero, params=prm)
    # FP32 terms in compensated sums against FP64
    assert (np.abs(got - ref) / np.abs(ref)).max() < 2e-6


@pytest.mark.parametrize("chunks", [1, 3, 16])
@pytest.mark.parametrize("sizes", [[40], [300, 20, 20], [20] * 700, [30000, 5000] + [25] * 300])
def test_chunk_counts_give_the_same(ctx, sizes, chunks):
    rng = np.random.default_rng(len(sizes))
    off = np.concatenate([[0], np.cumsum(sizes)])
    n = off[-1]
    sub = np.repeat(np.arange(len(sizes)), sizes)
    centre = rng.uniform(0, 50, (len(sizes), 3))
    pop = synth.Population(pos=(centre[sub] + rng.normal(0, 0.05, (n, 3))).astype(np.float32),
                           vel=rng.normal(0, 30, (n, 3)).astype(np.float32),
                           mass=np.full(n, 0.01, np.float32), offsets=off, pid=np.arange(n))
    saved = ctx.tuning()
    try:
        res = []
        for ch in (8, chunks):
            ctx.set_tuning(saved["direct_cutoff"], ch)
            res.append(ctx.unbind(pop, hbtx.workload_params()))
    finally:
        ctx.set_tuning(saved["direct_cutoff"], saved["walk_chunks"])
    for k in ("order", "energy", "result"):
        assert np.array_equal(res[0][k], res[1][k]), k
