"""Device memory that a context keeps from call to call is given back where it is no
longer used."""
import numpy as np
import pytest

import hbtx
import synth

pytestmark = pytest.mark.gpu


def test_entry_buffers_after_a_large_batch():
    prm = hbtx.workload_params()
    big = synth.single_nfw(seed=1, n_halo=250_000, n_inter=50_000)
    small = synth.population(seed=2, nsub=20, nmax=500)
    c = hbtx.Context(0)
    try:
        first = c.unbind(small, prm)
        want = c.unbind(big, prm)
        held = hbtx.device_bytes()
        # small batches between large ones leave the buffers as they are
        for _ in range(2):
            for _ in range(10):
                c.unbind(small, prm)
            got = c.unbind(big, prm)
            assert hbtx.device_bytes() == held
        for k in ("order", "energy", "result"):
            assert np.array_equal(got[k], want[k])
        for _ in range(16):
            got = c.unbind(small, prm)
        # octree entries: at most n / 2 at each of 22 depths and the particles, 49 bytes each
        assert held - hbtx.device_bytes() > 300_000 * 5 * 49
        for k in ("order", "energy", "result"):
            assert np.array_equal(got[k], first[k])
        got = c.unbind(big, prm)
        for k in ("order", "energy", "result"):
            assert np.array_equal(got[k], want[k])
    finally:
        c.close()
