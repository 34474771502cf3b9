"""The wave-per-cell list builder of dense systems: FP64 list forces against
the oracle, bit for bit, where its paths change: one, two, three and more cells
per axis, candidate counts on both sides of 256, 512 and 1024, cells of more
than 64 particles, several types, particles outside the box, and lists rebuilt
while stepping."""
import numpy as np
import pytest

import moldyn_amd as M
from oracle import oracle as O
from tests.common import AR_MASS, engine_for

pytestmark = pytest.mark.gpu


def random_state(box, density, seed, counts=None, masses=None):
    box = np.asarray(box, dtype=np.float64)
    n = int(density * box.prod())
    counts = counts or [n]
    rng = np.random.default_rng(seed)
    pos = rng.uniform(0.0, 1.0, (sum(counts), 3)) * box
    return O.State(counts, masses or [AR_MASS], list(box), pos=pos, vel=np.zeros_like(pos))


def check(s, engine=None, table=None):
    e = engine or engine_for(s, "fp64_list")
    e.update_force()
    d = e.download(("force", "pot", "virial"))
    O.update_force(s, table)
    assert np.array_equal(d["force"], s.force)
    assert np.array_equal(d["pot"], s.pot) and np.array_equal(d["virial"], s.temp)
    e.close()


@pytest.mark.parametrize("density", [4.0, 10.0, 21.0, 40.0, 90.0])
@pytest.mark.parametrize("box", [(1.8, 1.8, 1.8), (2.0, 2.9, 1.8), (2.9, 2.9, 2.9), (3.9, 2.0, 5.1)])
def test_grid_shapes_and_candidate_counts(box, density):
    check(random_state(box, density, int(density)))


def test_crowded_cell():
    """200 particles within 0.3 nm in a liquid: more than a wave holds per cell."""
    s = random_state((6.0, 6.0, 6.0), 8.0, 1)
    s.pos[300:500] = 3.3 + np.random.default_rng(2).uniform(-0.15, 0.15, (200, 3))
    check(s)


def test_outside_the_box():
    s = random_state((5.0, 5.0, 5.0), 9.0, 3)
    s.pos[::4] += np.array([5.0, -5.0, 0.0])
    check(s)


def test_types():
    counts, masses = [300, 70, 800], [AR_MASS, 20.0, 40.0]
    s = random_state((4.6, 4.6, 4.6), 12.0, 4, counts, masses)
    e = M.Engine(counts, masses, s.box, force_mode="fp64_list")
    pairs = {(0, 1): (0.3, 1.0), (1, 2): (0.25, 2.0), (2, 2): (0.3, 0.5)}
    for (a, b), (sigma, eps) in pairs.items():
        e.set_pair_potential(a, b, sigma, eps)
    e.upload(s.pos, s.vel, s.box)
    check(s, e, O.potential_table(3, {k: O.new_lennard_jones(*v) for k, v in pairs.items()}))


def test_sparse_gas_compressed_to_a_liquid():
    """A run whose barostat takes it from brick-built (sparse) to cell-built
    lists, against the all-pairs path."""
    side = 10
    rng = np.random.default_rng(5)
    pos = O.lattice_u([side] * 3, 0.95) + rng.uniform(0.0, 0.1, (side ** 3, 3))
    s = O.State([side ** 3], [AR_MASS], [side * 0.95] * 3, pos=pos, vel=O.mb_velocities(side ** 3, 120.0, AR_MASS, 6))
    out = []
    for mode in ("fp64_list", "fp64_allpairs"):
        e = engine_for(s, mode)
        e.update_force()
        th, ba = M.thermostat("berendsen", tau=0.5, target_t=120.0), M.barostat("berendsen", 1.0, 5.0, 200.0)
        for _ in range(4):
            e.step(0.002, 60, th, ba)
        out.append(e.download())
        e.close()
    a, b = out
    density = side ** 3 / float(np.prod(a["box"]))
    assert density * 4 / 3 * np.pi * 0.957 ** 3 > 6.0
    for k in ("x", "v", "force", "box"):
        assert np.allclose(a[k], b[k], rtol=1e-9, atol=1e-9 * np.abs(b[k]).max())
