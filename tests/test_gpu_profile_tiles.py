"""Profiles of bound sets at the sizes where the tiles change: one wave's tiles (up to 512
slots), whole and part tiles of 4096, against the oracle."""
import numpy as np
import pytest

import hbtx
import pyoracle as O
import synth
from test_gpu_profiles import compare

pytestmark = pytest.mark.gpu


def test_tile_edges(ctx):
    sizes = np.array([0, 1, 2, 3, 15, 16, 17, 63, 64, 65, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 2000, 4095, 4096,
                      4097, 4608, 4609, 8192, 8193, 40000])
    off = np.concatenate([[0], np.cumsum(sizes)])
    n = off[-1]
    rng = np.random.default_rng(5)
    pos = (np.repeat(rng.uniform(5, 45, (len(sizes), 3)), sizes, axis=0) + rng.normal(0, 0.05, (n, 3))).astype(np.float32)
    mass = rng.uniform(0.005, 0.015, n).astype(np.float32)
    mbound = np.array([mass[a:b].sum() for a, b in zip(off[:-1], off[1:])], np.float32)
    prm = hbtx.workload_params(hz=70.0)
    g = ctx.profiles_of(pos, mass, off, sizes, mbound, prm)
    r = O.profiles(pos, mass, off[:-1], sizes, mbound,
                   O.default_params(**{k: v for k, v in prm.items() if k != "direct_cutoff"}))
    compare(g, r, sizes)
