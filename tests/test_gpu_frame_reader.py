"""State files parsed on the device (moldyn_amd/csrc/md_frames.hip k_line_*,
k_frame_parse): every number as Python's correctly rounded float() reads it, at
the edges of the parsing blocks, and texts the device leaves to the host."""
import os

import numpy as np
import pytest

import moldyn_amd as M
from moldyn_amd import _lib as L
from moldyn_amd.frames import FRAME_HEADER, StateToSave

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def context():
    yield M.Engine([8], [1.0], [5.0, 5.0, 5.0])  # the device reads for a process that drives it


def number(rng, kind):
    sign = "-" if rng.random() < 0.5 else ""
    if kind == 0:  # as the writer prints them
        return repr(float(np.round(rng.normal() * 10.0 ** rng.integers(-3, 8), 17))).replace("e+", "e")
    if kind == 1:  # any digits, any exponent of a normal number
        d = "".join(rng.choice(list("0123456789"), rng.integers(1, 20)))
        e = int(rng.integers(-290, 280))
        return f"{sign}{d}e{e}"
    if kind == 2:  # halves between neighbours, and one digit off
        u = int(rng.integers(1 << 52, 1 << 53))
        s = int(rng.integers(0, 10))
        return f"{sign}{2 * u + 1}{'' if s < 5 else '.0'}e{0 if s < 8 else -22}" if s else f"{sign}{(2 * u + 1) * 10 + 1}e-1"
    if kind == 3:  # subnormal, zero
        return f"{sign}{rng.integers(1, 999)}.5e-322" if rng.random() < 0.02 else f"{sign}0.0"
    return f"{sign}{rng.integers(0, 9)}.{rng.integers(0, 10 ** 9):09d}{rng.integers(0, 10 ** 9):09d}"


def write(tmp_path, lines, end="\n", last=True):
    os.makedirs(tmp_path / "data", exist_ok=True)
    with open(tmp_path / "data" / "0.csv", "w", newline="") as f:
        f.write(end.join([FRAME_HEADER] + lines) + (end if last else ""))
    with open(tmp_path / "bb.csv", "w") as f:
        f.write("x,y,z\n1.5,2.5,3.5\n")


def rows(n, seed):
    rng = np.random.default_rng(seed)
    ids = rng.integers(0, 65536, n)
    nums = [[number(rng, int(rng.integers(0, 5))) for _ in range(6)] for _ in range(n)]
    lines = [",".join([str(i)] + r) for i, r in zip(ids, nums)]
    return ids, np.array([[float(t) for t in r] for r in nums]), lines


def check(tmp_path, ids, vals):
    st = StateToSave.load_from_file(str(tmp_path), 0)
    assert np.array_equal(st.ids, ids)
    assert np.array_equal(st.x.view(np.uint64), np.ascontiguousarray(vals[:, :3]).view(np.uint64))
    assert np.array_equal(st.v.view(np.uint64), np.ascontiguousarray(vals[:, 3:]).view(np.uint64))
    assert np.array_equal(st.boundary_box, [1.5, 2.5, 3.5])


@pytest.mark.parametrize("n,last", [(4096, True), (4097, False), (4223, True), (20000, False)])
def test_numbers(context, tmp_path, n, last):
    ids, vals, lines = rows(n, n)
    write(tmp_path, lines, last=last)
    check(tmp_path, ids, vals)


@pytest.mark.parametrize("kind", ["crlf", "blank", "plus", "long", "short", "quoted"])
def test_left_to_the_host(context, tmp_path, kind):
    ids, vals, lines = rows(12000 if kind == "short" else 4200, 7)
    if kind == "short":
        vals[:] = 0.0
        ids[:] = 3
        lines = ["3,0.0,0.0,0.0,0.0,0.0,0.0"] * len(lines)
    elif kind == "blank":
        lines[4000] += "\n"
    elif kind == "plus":
        vals[77, 0] = 2.5
        lines[77] = ",".join(["%d" % ids[77], "+2.5"] + lines[77].split(",")[2:])
    elif kind == "long":  # more than 19 digits
        vals[78, 0] = float("0." + "123456789" * 60)
        lines[78] = ",".join(["%d" % ids[78], "0." + "123456789" * 60] + lines[78].split(",")[2:])
    elif kind == "quoted":
        lines[5] = '"%d",%s' % (ids[5], lines[5].split(",", 1)[1])
    write(tmp_path, lines, end="\r\n" if kind == "crlf" else "\n")
    check(tmp_path, ids, vals)


@pytest.mark.parametrize("bad", ["1,2,3", "70000,0.0,0.0,0.0,0.0,0.0,0.0", "1,0.0,0.0,x,0.0,0.0,0.0",
                                 "1,0.0,0.0,1e999,0.0,0.0,0.0", "1,0.0,0.0,,0.0,0.0,0.0", "1,0.0,0.0,0.0,0.0,0.0,0.0,"])
def test_bad_rows_are_refused_alike(context, tmp_path, bad):
    ids, vals, lines = rows(4200, 9)
    lines[4100] = bad
    write(tmp_path, lines)
    with pytest.raises(L.MdError, match="record 4102"):
        StateToSave.load_from_file(str(tmp_path), 0)
