"""The host checks that decide what the kernels are given (xt_bounds.hpp), built
with AddressSanitizer and UndefinedBehaviorSanitizer and run on the CPU at the
edges of what they accept (tests/integration/bounds_host.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    out = str(tmp_path_factory.mktemp("bounds") / "bounds_host")
    cmd = ["g++", "-std=c++17", "-O2", "-g", "-Wall", "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined",
           "-I" + os.path.join(ROOT, "xxtric_amd", "csrc"),
           os.path.join(ROOT, "tests", "integration", "bounds_host.cpp"), "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    return out


@pytest.mark.parametrize("group", ["offsets", "index32", "lists"])
def test_bounds(exe, group):
    r = subprocess.run([exe, group], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert group + " hold" in r.stdout
