"""The pair terms' shared reciprocal (md_common.h quotient): bit for bit the
division, over its stated range (CPU)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_quotient_is_the_division(tmp_path):
    from moldyn_amd.build import CSRC, HIPCC, ROOT
    if shutil.which(HIPCC) is None and not os.path.exists(HIPCC):
        pytest.skip("needs hipcc")
    exe = str(tmp_path / "quotient")
    r = subprocess.run([HIPCC, "--offload-host-only", "-O2", "-mfma", "-std=c++17", "-ffp-contract=off",
                        "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-x", "hip",
                        os.path.join(HERE, "quotient_check.cpp"), "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe, "2000000"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
    assert int(r.stdout.split()[0]) > 10_000_000
