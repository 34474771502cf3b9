"""The host side of the C ABI when device memory runs out (CPU): md_api.hip
built for the host alone under AddressSanitizer and linked with
host_runtime_mock.cpp, which stands in for the HIP runtime and the kernels."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    from moldyn_amd.build import CSRC, FLAGS, HIPCC, ROOT
    clang = os.path.join(os.path.dirname(HIPCC), "..", "llvm", "bin", "clang++")
    if shutil.which(HIPCC) is None or not os.path.exists(clang):
        pytest.skip("needs hipcc")
    out = tmp_path_factory.mktemp("host_runtime")
    objs = []
    for src in (os.path.join(CSRC, "md_api.hip"), os.path.join(HERE, "host_runtime_mock.cpp")):
        objs.append(str(out / (os.path.basename(src) + ".o")))
        r = subprocess.run([HIPCC, "--offload-host-only", "-O1", "-g", "-std=c++17", "-ffp-contract=off",
                            "-Xarch_host", "-fsanitize=address", "-fPIC", "-I" + os.path.join(ROOT, "include"),
                            "-I" + CSRC, "-x", "hip", "-c", src, "-o", objs[-1]], capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
    exe = str(out / "host_runtime")
    r = subprocess.run([clang, "-Xarch_host", "-fsanitize=address", "-o", exe] + objs, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


@pytest.mark.parametrize("case", ["lists", "layout", "staging", "footprint"])
def test_out_of_device_memory(program, case):
    r = subprocess.run([program, case], capture_output=True, text=True, timeout=120,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=1:abort_on_error=1"))
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip().splitlines()[-1] == f"{case} passed"
