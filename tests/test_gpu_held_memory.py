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


def test_workspaces_after_a_large_call():
    src = np.random.default_rng(3).normal(0, 0.1, (200, 3)).astype(np.float32)
    one = np.ones(200, np.float32)
    tgt = np.tile(src, (110_000, 1))  # 22 million targets: 52 bytes each
    c = hbtx.Context(0)
    try:
        tree = c.tree(src, one, hbtx.workload_params())
        before = hbtx.device_bytes()
        got = tree.potential(tgt)
        # (the sort's scratch stays: 12 bytes a target and its tiles' counts, less than half as much)
        assert hbtx.device_bytes() - before < (1 << 29)
        # (another order of the terms in plain FP32 sums of about 16: 2^-24 each, both sides)
        want = tree.potential(src)
        assert np.allclose(got.reshape(-1, 200), want, rtol=3e-6)
        # a small call keeps what it made
        held = hbtx.device_bytes()
        tree.potential(src)
        assert hbtx.device_bytes() == held
        tree.close()
    finally:
        c.close()
