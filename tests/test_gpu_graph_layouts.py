"""Round graphs when a context's next batch has as many particles and subhaloes as the
last one, in other shares: buffers stay from load to load, so whatever the captured
launches depend on has to be told apart by the graphs' own key."""
import numpy as np
import pytest

import hbtx
import synth

pytestmark = pytest.mark.gpu


def batch(counts, seed):
    """NFW subhaloes, a third of each one's particles too fast to be bound: the first
    round removes more than 16,384 of 60,000, and leaves more than 2,048 of 15,000."""
    rng = np.random.default_rng(seed)
    pos, vel = [], []
    for n in counts:
        fast = n // 3
        one = synth.single_nfw(seed=int(rng.integers(1 << 30)), n_halo=n - fast, n_inter=fast,
                               rs=0.02 * (n / 1e4) ** (1 / 3))
        v = one.vel.copy()
        v[n - fast:] *= 20.0
        pos.append(one.pos + rng.uniform(0, 40, 3))
        vel.append(v)
    n = int(np.sum(counts))
    off = np.concatenate([[0], np.cumsum(counts)])
    return synth.Population(np.concatenate(pos), np.concatenate(vel), np.full(n, synth.PARTICLE_MASS), off,
                            np.arange(n))


def same(a, b):
    assert np.array_equal(a["order"], b["order"])
    assert np.array_equal(a["energy"], b["energy"])
    assert np.array_equal(a["result"], b["result"])


# pairs of equal particle count, subhalo count and summed entry bound; the largest source
# set of their second rounds lies to either side of a sort form's limit
EVEN = [15000] * 10
SKEW = [60000] + [10000] * 9


@pytest.mark.parametrize("first,second", [(EVEN, SKEW), (SKEW, EVEN), ([16384] * 8, [49152] + [11700] * 6 + [11720])])
def test_same_size_other_shares(first, second):
    assert sum(first) == sum(second) and len(first) == len(second)
    c = hbtx.Context(0)
    try:
        prm = hbtx.workload_params(direct_cutoff=512)
        c.unbind(batch([90000] + [15000] * 10, 1), prm)  # (nothing grows afterwards)
        for k, counts in enumerate((first, second, first)):
            pop = batch(counts, 2 + k)
            got = c.unbind(pop, prm)
            st = c.stats()
            assert st["graph_rounds"] == st["rounds"] - 1 > 0
            same(got, c.unbind(pop, prm, hbtx.BATCHED | hbtx.NO_GRAPH))
            # (a third is unbound)
            assert (got["result"]["nbound"] < 0.7 * np.asarray(counts)).all()
            same(got, c.unbind(pop, prm))
    finally:
        c.close()
