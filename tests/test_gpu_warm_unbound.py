"""Warm rounds in a periodic box that leave nothing bound, or that had nothing proposed:
there is no first particle to wrap a frame about, and the subhalo iterates from all its
particles as a plain unbinding does."""
import numpy as np
import pytest

import hbtx
import synth

pytestmark = pytest.mark.gpu
BOX = 40.0


def batch():
    """Two haloes about the box corner; the first's last 80 particles stream through it
    at many times the escape speed, with a dispersion their own mass cannot hold."""
    rng = np.random.default_rng(3)
    pos, vel = [], []
    for n, fast in ((3000, 80), (1500, 0)):
        one = synth.single_nfw(seed=n, n_halo=n - fast, n_inter=fast)
        v = one.vel.copy()
        vmax = np.abs(v).max()
        v[n - fast:] = 50.0 * vmax * np.array([1.0, 0.0, 0.0]) + 5.0 * vmax * rng.normal(0, 1, (fast, 3))
        pos.append(np.mod(one.pos - 1.0, BOX))
        vel.append(v)
    pos = np.concatenate(pos).astype(np.float32)
    pos[pos >= BOX] = 0.0
    off = np.array([0, 3000, 4500])
    return synth.Population(pos, np.concatenate(vel), np.full(4500, synth.PARTICLE_MASS), off, np.arange(4500),
                            ref_pos=np.zeros((2, 3)), ref_vel=np.zeros((2, 3)))


@pytest.mark.parametrize("flags", [0, hbtx.NO_GRAPH])
@pytest.mark.parametrize("cutoff", [10, 512])  # octrees, exact sums
@pytest.mark.parametrize("proposed,min_part", [(80, 20), (0, 0)])
def test_rejected_proposal(proposed, min_part, cutoff, flags):
    pop = batch()
    prm = hbtx.workload_params(periodic=1, box_size=BOX, direct_cutoff=cutoff, min_num_part=min_part)
    c = hbtx.Context(0)
    try:
        plain = c.unbind(pop, prm, hbtx.BATCHED | flags)
        assert (plain["result"]["nbound"] > 1000).all()
        pro = np.zeros(pop.n, np.uint8)
        pro[3000 - proposed:3000] = 1
        pro[3000 + plain["order"][3000:3000 + plain["result"]["nbound"][1]]] = 1
        c.load(pop)
        c.set_proposal(pro)
        c.run(prm, hbtx.BATCHED | hbtx.WARMSTART | flags)
        warm = c.fetch()
    finally:
        c.close()
    # the first subhalo: the plain iteration's bits after one more round
    assert warm["result"]["iterations"][0] == plain["result"]["iterations"][0] + 1
    for k in hbtx.RESULT_DTYPE.names:
        if k != "iterations":
            assert np.array_equal(warm["result"][k][0], plain["result"][k][0]), k
    assert np.array_equal(warm["order"][:3000], plain["order"][:3000])
    assert np.array_equal(warm["energy"][:3000], plain["energy"][:3000])
    # the second: its own bound set as the proposal is accepted
    assert abs(int(warm["result"]["nbound"][1]) - int(plain["result"]["nbound"][1])) <= 2
