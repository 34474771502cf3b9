"""The all-pairs path's two ways of summing (spread over the chip with
per-particle lists, or a thread per particle) against the oracle, bit for bit:
sizes at the edges of the particle tiles (16, 32, 64) and of the 512-candidate
tiles, several types, particles outside the box, and a cluster with more pairs
in range than a list holds."""
import numpy as np
import pytest

import moldyn_amd as M
from oracle import oracle as O
from tests.common import AR_MASS, engine_for, gas_state

pytestmark = pytest.mark.gpu


def liquid(n, seed):
    """n particles in random order on a jittered simple-cubic lattice (a = 0.5
    nm, about 20 neighbours each)."""
    side = int(np.ceil(n ** (1.0 / 3.0))) + (1 if n < 300 else 0)
    rng = np.random.default_rng(seed)
    pos = O.lattice_u([side] * 3, 0.5) + rng.uniform(0.0, 0.1, (side ** 3, 3))
    pos = pos[rng.permutation(side ** 3)[:n]]
    box = max(side * 0.5, 2.0)
    return O.State([n], [AR_MASS], [box] * 3, pos=pos, vel=O.mb_velocities(n, 120.0, AR_MASS, seed))


def check(s, steps=0, table=None, engine=None):
    e = engine or engine_for(s, "fp64_allpairs")
    e.update_force()
    O.update_force(s, table)
    if steps:
        e.step(0.002, steps)
        for _ in range(steps):
            O.verlet_step(s, 0.002, table)
    d = e.download()
    for got, want in ((d["force"], s.force), (d["pot"], s.pot), (d["virial"], s.temp), (d["x"], s.pos), (d["v"], s.vel)):
        assert np.array_equal(got, want)
    e.close()


@pytest.mark.parametrize("n", [2, 15, 17, 63, 65, 511, 512, 513, 1025, 3001])
def test_tile_edges(n):
    check(liquid(n, n), steps=3)


@pytest.mark.parametrize("n", [8500, 16700, 33000])
def test_every_particle_tile(n):
    """Sizes that take 16, 32 and 64 particles per block."""
    check(liquid(n, n))


def test_outside_the_box():
    s = liquid(700, 1)
    s.pos[::3] += np.array([1.3, -1.3, 0.2]) * s.box
    check(s)


def test_cluster_overflows_the_lists():
    """300 particles within a cutoff of one another in a dilute gas."""
    s = gas_state(2300, 14.0, 2)
    rng = np.random.default_rng(3)
    s.pos[1000:1300] = 7.0 + rng.uniform(-0.2, 0.2, (300, 3))
    check(s)


@pytest.mark.parametrize("box", [8.0, 3.2])
def test_types(box):
    """Three types with their own cutoffs; box 3.2 holds more than 48 pairs in
    range per particle (a thread per particle)."""
    counts, masses = [700, 65, 513], [AR_MASS, 20.0, 40.0]
    rng = np.random.default_rng(4)
    pos = rng.uniform(0.0, box, (sum(counts), 3))
    vel = rng.normal(0.0, 0.1, pos.shape)
    s = O.State(counts, masses, [box] * 3, pos=pos, vel=vel)
    e = M.Engine(counts, masses, s.box, force_mode="fp64_allpairs")
    pairs = {(0, 1): (0.3, 1.0), (1, 2): (0.25, 2.0), (2, 2): (0.4, 0.5)}
    for (a, b), (sigma, eps) in pairs.items():
        e.set_pair_potential(a, b, sigma, eps)
    table = O.potential_table(3, {k: O.new_lennard_jones(*v) for k, v in pairs.items()})
    e.upload(pos, vel, s.box)
    check(s, table=table, engine=e)
