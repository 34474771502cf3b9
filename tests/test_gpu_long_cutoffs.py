"""Dense lists where a cell's stencil holds more particles than a wave sorts at
once (1,024): long cutoffs and crowds, slots in the order of space and shuffled,
several types, cells of more than 64 particles.  FP64 list forces against the
oracle, bit for bit, and the build's cost across that size."""
import time

import numpy as np
import pytest

import moldyn_amd as M
from oracle import oracle as O
from tests.common import AR_MASS

pytestmark = pytest.mark.gpu
SIGMA, EPS = 0.3418, 1.712


def liquid(n_side, a, seed, shuffled):
    rng = np.random.default_rng(seed)
    n = n_side ** 3
    pos = O.lattice_u([n_side] * 3, a) + rng.uniform(-0.03, 0.03, (n, 3))
    pos = np.mod(pos, n_side * a)
    return pos[rng.permutation(n)] if shuffled else pos, [n_side * a] * 3


def check(pos, box, counts, masses, pairs):
    """pairs: (i, j) -> (sigma, eps, r_cut)"""
    s = O.State(counts, masses, box, pos=pos, vel=np.zeros_like(pos))
    e = M.Engine(counts, masses, box, force_mode="fp64_list")
    table = {}
    for (i, j), (sigma, eps, rc) in pairs.items():
        u_cut = 4.0 * eps * ((sigma / rc) ** 12 - (sigma / rc) ** 6)
        e.set_pair_potential(i, j, sigma, eps, r_cut=rc, u_cut=u_cut)
        table[(i, j)] = (sigma, eps, rc, u_cut)
    e.upload(pos, s.vel, box)
    e.update_force()
    d = e.download(("force", "pot", "virial"))
    O.update_force(s, O.potential_table(len(counts), table))
    for name, want in (("force", s.force), ("pot", s.pot), ("virial", s.temp)):
        assert np.array_equal(d[name], want), name
    mean = e.stats()["mean_list_len"]
    e.close()
    return mean


@pytest.mark.parametrize("shuffled", [False, True])
@pytest.mark.parametrize("n_side,rc", [(12, 4.0), (13, 5.0), (17, 5.0), (15, 6.5)])
def test_one_type(n_side, rc, shuffled):
    pos, box = liquid(n_side, 0.40, n_side, shuffled)
    assert check(pos, box, [len(pos)], [AR_MASS], {(0, 0): (SIGMA, EPS, rc * SIGMA)}) > 100


@pytest.mark.parametrize("shuffled", [False, True])
def test_types(shuffled):
    pos, box = liquid(14, 0.40, 3, shuffled)
    counts = [1000, 44, 1700]
    pairs = {(i, j): (SIGMA, EPS, (5.0 if i == j else 3.0) * SIGMA) for i in range(3) for j in range(i, 3)}
    check(pos, box, counts, [AR_MASS, 20.0, 40.0], pairs)


def test_crowd_in_a_liquid():
    """700 particles inside one cell of a liquid, the rest around them."""
    pos, box = liquid(14, 0.45, 4, True)
    pos[900:1600] = 3.1 + np.random.default_rng(5).uniform(-0.2, 0.2, (700, 3))
    check(pos, box, [len(pos)], [AR_MASS], {(0, 0): (SIGMA, EPS, 2.5 * SIGMA)})


def test_cost_across_the_size():
    best = []
    for rc in (3.5, 4.0):
        pos, box = liquid(33, 0.40, 1, True)
        e = M.Engine([len(pos)], [AR_MASS], box, force_mode="fp32_list")
        e.set_pair_potential(0, 0, SIGMA, EPS, r_cut=rc * SIGMA, u_cut=0.0)
        e.upload(pos, np.zeros_like(pos), box)
        t = []
        for _ in range(5):
            t0 = time.perf_counter()
            e.update_force()
            t.append(time.perf_counter() - t0)
        best.append(min(t))
        e.close()
    assert best[1] < 12.0 * best[0], best
