"""The exact sum's two kernels: several waves per 64 targets (few targets) and one
wave per 64 targets (many).  Both add the same sums in the same order, so a target's
potential does not depend on how many targets came with it, and both agree with
the FP64 sum."""
import numpy as np
import pytest

import hbtx

pytestmark = pytest.mark.gpu


# source counts around a group (4 sources), the adder's batch (128) and a stage (256), targets around a wave
@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("ns,nt", [(1, 1), (3, 64), (4, 65), (5, 63), (127, 2), (128, 64), (129, 130), (131, 65),
                                   (255, 7), (256, 64), (257, 65), (4099, 129)])
def test_split_sum_equals_the_wave_sum(ctx, ns, nt, periodic):
    rng = np.random.default_rng(ns * 1000 + nt)
    src = (rng.normal(0, 0.05, (ns, 3)) + 2.0).astype(np.float32)
    mass = rng.uniform(0.005, 0.02, ns).astype(np.float32)
    tgt = (rng.normal(0, 0.08, (nt, 3)) + 2.0).astype(np.float32)
    prm = hbtx.workload_params(**(dict(periodic=1, box_size=4.0) if periodic else {}))
    few = ctx.direct_potential(src, mass, tgt, params=prm)
    # the same targets among more than 64 x 12 a CU of them
    reps = 64 * 12 * 256 // nt + 2
    many = ctx.direct_potential(src, mass, np.tile(tgt, (reps, 1)), params=prm).reshape(reps, nt)
    assert np.array_equal(many, np.broadcast_to(few, many.shape))
    d = tgt.astype(np.float64)[:, None, :] - src.astype(np.float64)[None, :, :]
    if periodic:
        d = np.where(d > 2.0, d - 4.0, np.where(d < -2.0, d + 4.0, d))
    r = np.sqrt((d * d).sum(2))
    h = 2.8 * float(np.float32(0.001))
    u = r / h
    near = np.where(u < 0.5, -2.8 + u * u * (16 / 3 + u * u * (6.4 * u - 9.6)),
                    -3.2 + 1 / (15 * np.maximum(u, 1e-9)) + u * u * (32 / 3 + u * (-16 + u * (9.6 - 32 / 15 * u)))) / h
    ref = (np.where(u < 1, near, -1 / np.maximum(r, 1e-12)) * mass.astype(np.float64)).sum(1) * 43.0071
    # per term: three rounded differences, r2, 1/r (one ulp) and the product, then three
    # rounded additions in the group: under 16 half-ulps of 2^-24 of same-signed terms
    assert np.max(np.abs(few - ref) / np.abs(ref)) < 16 * 2.0 ** -24
