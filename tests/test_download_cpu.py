"""Copies of results through the pinned ring (csrc/download.hpp), on the CPU with
the HIP calls stood in for (tests/native/download_check.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CLANG = shutil.which("amdclang++") or "/opt/rocm/bin/amdclang++"


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not os.path.exists(CLANG):
        pytest.skip("no compiler for HIP sources")
    d = tmp_path_factory.mktemp("download")
    subprocess.check_call([CLANG, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O1", "-fPIC",
                           "-I" + os.path.join(ROOT, "spatialpy_amd", "csrc"), "-c",
                           os.path.join(ROOT, "tests", "native", "download_check.cpp"), "-o", str(d / "check.o")])
    subprocess.check_call(["g++", str(d / "check.o"), "-o", str(d / "check"), "-lpthread"])
    return str(d / "check")


@pytest.mark.parametrize("what", ["sizes", "allocations"])
def test_download(program, what):
    r = subprocess.run([program, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout[-300:], r.stderr[-300:])
