"""Steps of dense systems (each lane walks its particle's own list, several
entries at a time) against the oracle, bit for bit: one, two, three and eight
types, lists of every length from none on, and particles that cross the box."""
import numpy as np
import pytest

import moldyn_amd as M
from oracle import oracle as O
from tests.common import AR_MASS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [[1000], [999, 1], [1, 64, 935], [125] * 8, [343], [301, 42]])
def test_steps(counts):
    n = sum(counts)
    side = round(n ** (1 / 3))
    a = 0.40
    box = [side * a] * 3
    rng = np.random.default_rng(n + len(counts))
    pos = O.lattice_u([side] * 3, a) + rng.uniform(-0.03, 0.03, (n, 3))
    pos = np.mod(pos[rng.permutation(n)], side * a)
    # spread the last particles of the first type out: short lists beside long ones
    box[2] *= 3.0
    lone = min(counts[0], 12)
    pos[counts[0] - lone:counts[0], 2] = side * a * (1.2 + 1.6 * np.arange(lone) / 12)
    masses = [AR_MASS * (1 + 0.3 * t) for t in range(len(counts))]
    vel = np.concatenate([O.mb_velocities(c, 150.0, m, 3 + t) for t, (c, m) in enumerate(zip(counts, masses))])
    s = O.State(counts, masses, box, pos=pos, vel=vel)
    table = {(i, j): (0.30 + 0.004 * (i + 2 * j), 0.5 + 0.1 * j)
             for i in range(len(counts)) for j in range(i, len(counts))}
    e = M.Engine(counts, masses, box, force_mode="fp64_list")
    for (i, j), (sigma, eps) in table.items():
        e.set_pair_potential(i, j, sigma, eps)
    tab = O.potential_table(len(counts), {k: O.new_lennard_jones(*v) for k, v in table.items()})
    e.upload(s.pos, s.vel, s.box)
    e.update_force()
    O.update_force(s, tab)
    for k in (1, 7, 32):
        e.step(0.002, k)
        for _ in range(k):
            O.verlet_step(s, 0.002, tab)
        d = e.download()
        for name, ref in (("x", s.pos), ("v", s.vel), ("force", s.force), ("pot", s.pot), ("virial", s.temp)):
            assert np.array_equal(d[name], ref), name
    e.close()
