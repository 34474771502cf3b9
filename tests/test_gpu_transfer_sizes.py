"""Uploads and downloads where they change their way: pinned memory (up to 256
KB: 2,978 atoms of everything), its halves in turn (downloads up to 256 KB an
array: 14,894 atoms of everything, 10,922 of positions and velocities), device
staging, and pieces of that (128 MB).  The same bits come back, and a download
costs no jump at the first of these sizes."""
import time

import numpy as np
import pytest

import moldyn_amd as M
from tests.common import AR_MASS

pytestmark = pytest.mark.gpu


def engine(n, mode="fp64_list"):
    rng = np.random.default_rng(n)
    box = [10.0 * n ** (1 / 3)] * 3
    x, v = rng.uniform(0.0, box[0], (n, 3)), rng.normal(size=(n, 3))
    e = M.Engine([n], [AR_MASS], box, force_mode=mode)
    e.upload(x, v, box)
    return e, x, v, rng


@pytest.mark.parametrize("n", [2978, 2979, 4468, 7447, 10922, 10923, 14894, 14895, 30000])
def test_round_trip(n):
    e, x, v, rng = engine(n)
    f, pot, vir = rng.normal(size=(n, 3)), rng.normal(size=n), rng.normal(size=n)
    e.upload_forces(f, pot, vir)
    d = e.download()
    for name, want in (("x", x), ("v", v), ("force", f), ("pot", pot), ("virial", vir)):
        assert np.array_equal(d[name], want), name
    d = e.download(("x", "v"))
    assert np.array_equal(d["x"], x) and np.array_equal(d["v"], v)
    e.close()


@pytest.mark.parametrize("mode", ["fp64_list", "fp32_list"])
def test_round_trip_in_pieces(mode):
    """3.3 million atoms of three replicas and two types: more than 128 MB, which
    move in pieces that end inside waves, groups and replicas."""
    counts = np.array([[700001, 399990], [1, 1100003], [650000, 450007]])
    n, rng = int(counts.sum()), np.random.default_rng(2)
    box = [[400.0] * 3, [410.0] * 3, [420.0] * 3]
    x, v, f = rng.uniform(0.0, 400.0, (n, 3)), rng.normal(size=(n, 3)), rng.normal(size=(n, 3))
    if mode == "fp32_list":
        f = f.astype(np.float32).astype(np.float64)
    pot, vir = rng.normal(size=n), rng.normal(size=n)
    e = M.Engine(counts, [AR_MASS, 20.0], box, force_mode=mode)
    e.upload(x, v, box)
    e.upload_forces(f, pot, vir)
    d = e.download()
    for name, want in (("x", x), ("v", v), ("force", f), ("pot", pot), ("virial", vir), ("box", np.array(box))):
        assert np.array_equal(d[name], want), name
    e.upload_forces(None, pot, None)
    d = e.download(("force", "pot", "virial"))
    assert not d["force"].any() and np.array_equal(d["pot"], pot) and not d["virial"].any()
    e.close()


def test_list_statistics_in_pieces():
    """700 replicas of two or three neighbours: their list lengths take more room
    than the pinned memory of so few particles."""
    counts = np.array([2, 3] * 350)
    x = np.concatenate([1.0 + 0.4 * np.arange(n)[:, None] * [1.0, 0.0, 0.0] for n in counts])
    e = M.Engine(counts[:, None], [AR_MASS], [[5.0] * 3] * 700, force_mode="fp64_list")
    e.upload(x, np.zeros_like(x), [[5.0] * 3] * 700)
    e.update_force()
    st = e.stats()
    assert st["mean_list_len"] == (2 * 1 + 3 * 2) / 5 and st["max_list_len"] == 2
    e.close()


def test_no_jump_in_time():
    def best(n):
        e = engine(n)[0]
        t = []
        for _ in range(60):
            t0 = time.perf_counter()
            e.download()
            t.append(time.perf_counter() - t0)
        e.close()
        return min(t[10:])
    assert best(3375) < 1.7 * best(2744)
