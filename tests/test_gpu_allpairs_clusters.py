"""All-pairs forces of particles with more pairs in range than k_ap_force lists
(96): the oracle's sums bit for bit at list lengths around 32, 64 and 96 and over
every block size, and a droplet under a long cutoff no slower than the
thread-per-particle kernel that dense boxes take."""
import time

import numpy as np
import pytest

import moldyn_amd as M
from oracle import oracle as O
from tests.common import AR_MASS, engine_for

pytestmark = pytest.mark.gpu


def check(s, table=None, engine=None, steps=0):
    e = engine or engine_for(s, "fp64_allpairs")
    e.update_force()
    O.update_force(s, table)
    if steps:
        e.step(0.0005, steps)
        for _ in range(steps):
            O.verlet_step(s, 0.0005, table)
    d = e.download()
    for got, want in ((d["force"], s.force), (d["pot"], s.pot), (d["virial"], s.temp), (d["x"], s.pos)):
        assert np.array_equal(got, want)
    e.close()


def with_clusters(sizes, n, seed):
    """n particles far apart but for clusters of `sizes` particles, each within
    0.5 nm of one another."""
    rng = np.random.default_rng(seed)
    side = int(np.ceil(n ** (1 / 3)))
    box = side * 2.0
    pos = (np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n] + 0.5) * 2.0
    at = 0
    for k, m in enumerate(sizes):
        pos[at:at + m] = pos[at] + rng.uniform(-0.14, 0.14, (m, 3))
        at += m
    order = rng.permutation(n)
    return O.State([n], [AR_MASS], [box] * 3, pos=pos[order], vel=np.zeros((n, 3)))


@pytest.mark.parametrize("block_size", [64, 128, 256, 512])
@pytest.mark.parametrize("n", [1007, 1040])
def test_list_lengths(n, block_size):
    s = with_clusters([32, 33, 34, 64, 65, 66, 96, 97, 98, 129], n, n)
    check(s, engine=engine_for(s, "fp64_allpairs", block_size=block_size))


def test_steps_and_tiles_per_block():
    s = with_clusters([2, 100, 31], 700, 5)
    s.pos += np.random.default_rng(6).uniform(-0.001, 0.001, s.pos.shape)
    check(s, engine=engine_for(s, "fp64_allpairs", block_size=64, tiles_per_block=3), steps=2)


def test_types():
    """Clusters of three types with their own cutoffs, crossing the box."""
    counts, masses = [350, 33, 417], [AR_MASS, 20.0, 40.0]
    s1 = with_clusters([140, 120, 3], 800, 7)
    box = s1.box
    s = O.State(counts, masses, list(box), pos=s1.pos + np.array([0.4, -1.0, 0.0]), vel=np.zeros((800, 3)))
    e = M.Engine(counts, masses, box, force_mode="fp64_allpairs")
    pairs = {(0, 1): (0.3, 1.0), (1, 2): (0.25, 2.0), (2, 2): (0.31, 0.5)}
    for (a, b), (sigma, eps) in pairs.items():
        e.set_pair_potential(a, b, sigma, eps)
    e.upload(s.pos, s.vel, box)
    check(s, O.potential_table(3, {k: O.new_lennard_jones(*v) for k, v in pairs.items()}), e)


def test_droplet_under_a_long_cutoff():
    """20,000 particles in a droplet and 7,000 around it, cutoff 5 sigma: few
    pairs in range on average in a large box, the same droplet in a small one
    goes to the thread-per-particle kernel."""
    rng = np.random.default_rng(1)
    sigma, side = 0.3418, 28
    drop = (O.lattice_u([side] * 3, 0.40) + rng.uniform(-0.03, 0.03, (side ** 3, 3)))[:20000]
    best = []
    for box in (90.0, 21.0):
        x = np.concatenate([drop + (box - 0.4 * side) / 2, rng.uniform(0.0, box, (7000, 3))])
        e = M.Engine([27000], [AR_MASS], [box] * 3, force_mode="fp64_allpairs")
        e.set_pair_potential(0, 0, sigma, 1.712, r_cut=5 * sigma, u_cut=0.0)
        e.upload(x, np.zeros_like(x), [box] * 3)
        t = []
        for _ in range(4):
            t0 = time.perf_counter()
            e.update_force()
            t.append(time.perf_counter() - t0)
        best.append(min(t))
        e.close()
    assert best[0] < 1.3 * best[1], best
