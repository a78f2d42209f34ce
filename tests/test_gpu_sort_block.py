"""Segments at the edges of the block sort (2049 to 16,384 elements, where none is
longer) with the forms beside it: the permutation of a stable sort, whatever the key bits, with ties, equal
digits and many such segments at once."""
import numpy as np
import pytest

import hbtx  # noqa: F401

pytestmark = pytest.mark.gpu
EDGES = [2049, 2050, 3000, 4095, 4096, 4097, 8191, 12345, 15361, 16383, 16384]


def check(ctx, keys, off):
    n = len(keys)
    vals = np.random.default_rng(n).permutation(n).astype(np.int32)
    k, v = ctx.segmented_sort(keys, vals, off)
    for s in range(len(off) - 1):
        a, e = off[s], off[s + 1]
        o = np.argsort(keys[a:e], kind="stable")
        assert np.array_equal(k[a:e], keys[a:e][o]), (s, e - a)
        if e - a > 2048:
            assert np.array_equal(v[a:e], vals[a:e][o]), (s, e - a)
        else:  # (a network: equal keys in any order)
            key_of = dict(zip(vals[a:e], keys[a:e]))
            assert np.array_equal(np.sort(v[a:e]), np.sort(vals[a:e]))
            assert all(key_of[x] == y for x, y in zip(v[a:e], k[a:e])), (s, e - a)


@pytest.mark.parametrize("more", [[], [5, 700, 2048], [16385], [20000]])
@pytest.mark.parametrize("bits", [1, 7, 8, 9, 31, 33, 36, 63, 64])
def test_edges(ctx, bits, more):
    rng = np.random.default_rng(bits)
    off = np.concatenate([[0], np.cumsum(EDGES + more)])
    keys = rng.integers(0, 1 << 63, off[-1], dtype=np.uint64) * np.uint64(2) + rng.integers(0, 2, off[-1], dtype=np.uint64)
    check(ctx, keys >> np.uint64(64 - bits), off)


@pytest.mark.parametrize("what", ["equal", "few", "sorted", "reversed", "one digit apart"])
def test_distributions(ctx, what):
    rng = np.random.default_rng(3)
    off = np.concatenate([[0], np.cumsum([5000, 16384, 2500])])
    n = off[-1]
    keys = {"equal": np.full(n, 12345, np.uint64),
            "few": rng.integers(0, 3, n).astype(np.uint64) << np.uint64(40),
            "sorted": np.arange(n, dtype=np.uint64),
            "reversed": np.arange(n, dtype=np.uint64)[::-1].copy(),
            "one digit apart": (rng.integers(0, 256, n).astype(np.uint64) << np.uint64(24)) + np.uint64(7)}[what]
    check(ctx, keys, off)


@pytest.mark.parametrize("run", [2, 31, 32, 33, 1000])
def test_runs_of_equal_top_bits(ctx, run):
    # runs whose keys differ (or not) below the top 32 of 63 bits, about the length at
    # which the passes of the lower bits go first
    rng = np.random.default_rng(run)
    off = np.concatenate([[0], np.cumsum([6000, 16384, 2049])])
    n = off[-1]
    top = rng.permutation(np.arange(n, dtype=np.uint64) // np.uint64(run)) + np.uint64(1 << 31)
    low = rng.integers(0, 8, n).astype(np.uint64) * np.uint64(0x0FFFFFF1)
    check(ctx, (top << np.uint64(31)) | low, off)


def test_more_segments_than_blocks(ctx):
    rng = np.random.default_rng(4)
    sizes = rng.integers(2049, 3000, 700)
    off = np.concatenate([[0], np.cumsum(sizes)])
    check(ctx, rng.integers(0, 1 << 40, off[-1], dtype=np.uint64), off)
