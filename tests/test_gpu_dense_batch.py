"""Batches of many small dense replicas, whose list builds share the grid's waves
out over the building replicas' cells 64 and 256 replicas at a time: forces and
steps of every replica against the oracle, bit for bit, and the cost of a batch's
launches against that of the same number of particles in few replicas."""
import time

import numpy as np
import pytest

import moldyn_amd as M
from oracle import oracle as O
from tests.common import AR_MASS

pytestmark = pytest.mark.gpu


def replicas(counts, a, seed):
    rng = np.random.default_rng(seed)
    out = []
    for k, n in enumerate(counts):
        side = int(np.ceil(n ** (1 / 3) - 1e-9))
        edge = a * rng.uniform(0.9, 1.1)
        pos = (O.lattice_u([side] * 3, edge) + rng.uniform(-0.02, 0.02, (side ** 3, 3)))[:n]
        box = max(side * edge, 1.8)
        out.append(O.State([n], [AR_MASS], [box] * 3, pos=np.mod(pos, box), vel=O.mb_velocities(n, 120.0, AR_MASS, k)))
    return out


def batch(states):
    e = M.Engine([[s.counts[0]] for s in states], [AR_MASS], [list(s.box) for s in states], force_mode="fp64_list")
    e.upload(np.concatenate([s.pos for s in states]), np.concatenate([s.vel for s in states]),
             [list(s.box) for s in states])
    return e


@pytest.mark.parametrize("r", [2, 63, 65, 256, 257, 330])
def test_every_replica(r):
    rng = np.random.default_rng(r)
    counts = rng.integers(1, 90, r)
    counts[rng.integers(0, r)] = 900
    states = replicas(counts, 0.42, r)
    e = batch(states)
    e.update_force()
    e.step(0.002, 6)
    d = e.download()
    at = 0
    for s in states:
        O.update_force(s)
        for _ in range(6):
            O.verlet_step(s, 0.002)
        n = len(s.pos)
        for name, want in (("x", s.pos), ("v", s.vel), ("force", s.force), ("pot", s.pot)):
            assert np.array_equal(d[name][at:at + n], want), (at, name)
        at += n
    e.close()


def test_cost_of_many_replicas():
    best = []
    for r, n in ((1000, 64), (16, 4000)):
        e = batch(replicas([n] * r, 0.5, 1))
        e.update_force()
        e.step(0.002, 20)
        t = []
        for _ in range(3):
            t0 = time.perf_counter()
            e.step(0.002, 60)
            t.append(time.perf_counter() - t0)
        best.append(min(t))
        e.close()
    assert best[0] < 4.0 * best[1], best
