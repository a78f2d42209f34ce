"""Batches whose number of subhaloes lies at the edges of the tile lists' forms (one
launch, two launches, passes over many blocks): every subhalo's result is what it is
in a batch of a few subhaloes."""
import numpy as np
import pytest

import hbtx
import synth

pytestmark = pytest.mark.gpu


def tiled(pop, reps):
    n, ns = pop.n * reps, pop.nsub * reps
    off = np.concatenate([[0], np.cumsum(np.tile(pop.counts(), reps))])
    t = lambda a: np.tile(a, (reps,) + (1,) * (a.ndim - 1))  # noqa: E731
    out = synth.Population(t(pop.pos), t(pop.vel), t(pop.mass), off, np.arange(n), ref_pos=t(pop.ref_pos),
                           ref_vel=t(pop.ref_vel))
    assert out.nsub == ns
    return out


# one block's threads (1024), a step (8192), the longest list of one block (32768)
@pytest.mark.parametrize("nsub", [1, 2, 1023, 1024, 1025, 8191, 8193, 32767, 32768, 32769, 70001])
def test_many_subhaloes(ctx, nsub):
    base = synth.population(seed=61, nsub=1 if nsub < 3 else 7, nmin=21, nmax=60)
    # one larger subhalo, so that ranges of many tiles are in the list too
    big = synth.population(seed=62, nsub=1, nmin=30000, nmax=40000)
    reps = (nsub - 1) // base.nsub
    rest = nsub - 1 - reps * base.nsub
    parts = ([tiled(base, reps)] if reps else []) + ([base.subset(np.arange(rest))] if rest else []) + [big]
    off = np.concatenate([[0], np.cumsum(np.concatenate([p.counts() for p in parts]))])
    cat = lambda f: np.concatenate([getattr(p, f) for p in parts])  # noqa: E731
    pop = synth.Population(cat("pos"), cat("vel"), cat("mass"), off, np.arange(off[-1]), ref_pos=cat("ref_pos"),
                           ref_vel=cat("ref_vel"))
    assert pop.nsub == nsub
    prm = hbtx.workload_params(direct_cutoff=-1)
    got, few, one = (ctx.unbind(p, prm) for p in (pop, base, big))
    res = got["result"]
    for name in ("nbound", "mbound", "com_pos", "com_vel", "spec_pot", "spec_am", "iterations", "core_pos"):
        want = np.concatenate([np.tile(few["result"][name], (reps + 1,) + (1,) * (few["result"][name].ndim - 1))[:nsub - 1],
                               one["result"][name]])
        assert np.array_equal(res[name], want, equal_nan=True), name
    assert np.array_equal(got["energy"][-big.n:], one["energy"])
    assert np.array_equal(got["order"][-big.n:], one["order"])
    k = min(reps, 1) * base.n
    assert np.array_equal(got["order"][:k], few["order"][:k])
