"""Host arrays through the pinned staging: round trips at sizes around a chunk and
the threads' shares, and a batch whose upload spans several chunks against the same
subhaloes in smaller batches."""
import numpy as np
import pytest

import hbtx
import synth

pytestmark = pytest.mark.gpu
CHUNK = 4 << 20


# elements of 8 bytes (and 4 for the values): one chunk, its edges, more chunks than slots
@pytest.mark.parametrize("n", [1, 511, CHUNK // 8 - 1, CHUNK // 8, CHUNK // 8 + 1, CHUNK // 4 + 3, 11 * CHUNK // 8 + 5])
def test_round_trip(ctx, n):
    rng = np.random.default_rng(n)
    keys = rng.integers(0, 1 << 62, n, dtype=np.uint64)
    vals = rng.integers(0, 1 << 30, n).astype(np.int32)
    # one segment per element: nothing moves
    k, v = ctx.segmented_sort(keys, vals, np.arange(n + 1))
    assert np.array_equal(k, keys) and np.array_equal(v, vals)


def test_batch_over_several_chunks_equals_its_halves(ctx):
    pop = synth.population(seed=91, target_particles=400_000, nmax=3000, hydro=True)
    pop.pid[:] = np.random.default_rng(1).permutation(pop.n) + (1 << 40)
    assert pop.n * 44 > 4 * CHUNK
    prm = hbtx.workload_params(direct_cutoff=-1, dm_only=0, thermal=1)
    whole = ctx.unbind(pop, prm)
    cut = pop.nsub // 3
    for ids in (np.arange(cut), np.arange(cut, pop.nsub)):
        part = pop.subset(ids)
        got = ctx.unbind(part, prm)
        a, b = pop.offsets[ids[0]], pop.offsets[ids[-1] + 1]
        assert np.array_equal(got["order"], whole["order"][a:b])
        assert np.array_equal(got["energy"], whole["energy"][a:b])
        for name in hbtx.RESULT_DTYPE.names:
            assert np.array_equal(got["result"][name], whole["result"][name][ids]), name


def test_refused_batch_leaves_nothing_loaded(ctx):
    pop = synth.population(seed=92, nsub=20, nmax=300, hydro=True)
    prm = hbtx.workload_params(dm_only=0)
    for field, at, value in (("mass", 17, -0.01), ("mass", 3, np.nan), ("ptype", 40, 6), ("ptype", 5, -1)):
        bad = pop.subset(np.arange(pop.nsub))
        getattr(bad, field)[at] = value
        with pytest.raises(hbtx.HbtxError) as e:
            ctx.load(bad)
        assert e.value.code == hbtx.E_INVALID
        with pytest.raises(hbtx.HbtxError):
            ctx.run(prm)
    out = ctx.unbind(pop, prm)
    assert out["result"]["nbound"].sum() > 0


def test_ids_default_to_the_index_in_the_subhalo(ctx):
    import ctypes as C
    pop = synth.population(seed=93, nsub=50, nmax=2000)
    prm = hbtx.make_params(**hbtx.workload_params())
    p = hbtx._p
    order, energy = np.zeros(pop.n, np.int64), np.zeros(pop.n, np.float32)
    res = np.zeros(pop.nsub, hbtx.RESULT_DTYPE)
    for flags in (hbtx.BATCHED, hbtx.PLAIN):
        rc = hbtx.lib().hbtx_unbind_batch(ctx._h, C.byref(prm), pop.n, p(pop.pos), p(pop.vel), p(pop.mass), None, None,
                                          None, pop.nsub, p(pop.offsets), p(pop.ref_pos), p(pop.ref_vel), None, None,
                                          flags, p(order), p(energy), None, p(res))
        assert rc == hbtx.OK
        alive = res["nbound"] > 0
        assert alive.any()
        first = order[pop.offsets[:-1]]
        assert np.array_equal(res["mostbound_id"], np.where(alive, first, -1))
