"""Trees that take over a freed tree's buffers: the same potentials as from fresh ones, several
trees alive at once, frees from another thread and after the context."""
import gc
import threading

import numpy as np
import pytest

import hbtx

pytestmark = pytest.mark.gpu
PRM = dict(theta=0.7, softening=0.01)


def points(n):
    rng = np.random.default_rng(n)
    return rng.normal(0, 1, (n, 3)).astype(np.float32), rng.uniform(0.5, 1.5, n).astype(np.float32)


def test_grow_shrink_and_several_alive(ctx):
    prm = hbtx.make_params(**PRM)
    want = {}
    for n in (1, 70, 5000, 300):
        c = hbtx.Context()
        t = c.tree(*points(n), prm)
        want[n] = t.potential(*points(n))
        t.close()
        c.close()
    for n in (5000, 300, 1, 70, 5000):
        t = ctx.tree(*points(n), prm)
        assert np.array_equal(t.potential(*points(n)), want[n]), n
        t.close()
    alive = [ctx.tree(*points(n), prm) for n in (300, 5000, 70)]
    alive[1].close()
    again = ctx.tree(*points(5000), prm)
    for t, n in ((alive[0], 300), (alive[2], 70), (again, 5000)):
        assert np.array_equal(t.potential(*points(n)), want[n]), n
        t.close()


def test_free_elsewhere_and_later():
    prm = hbtx.make_params(**PRM)
    c = hbtx.Context()
    before = hbtx.device_bytes()
    t = c.tree(*points(2000), prm)
    th = threading.Thread(target=t.close)
    th.start()
    th.join()
    t = c.tree(*points(1000), prm)
    held = hbtx.device_bytes()
    assert held > before
    c.close()
    assert hbtx.device_bytes() < held
    t.close()  # after its context
    del t, c
    gc.collect()
    assert hbtx.device_bytes() <= before
