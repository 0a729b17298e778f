"""Compiles tests/stage_check.cpp with g++ against the library's transfer
header and runs it: the header's HIP calls are defined by the program, so
that what it asks of the runtime, and what it does when the runtime refuses,
is seen without a GPU."""
import os
import subprocess

import pytest

import _pkg


@pytest.fixture(scope="module")
def stage_check(tmp_path_factory):
    src = os.path.join(_pkg.ROOT, "tests", "stage_check.cpp")
    inc = os.path.join(_pkg.PKG_DIR, "csrc")
    exe = str(tmp_path_factory.mktemp("stage") / "stage_check")
    subprocess.run(["g++", "-O2", "-std=c++20", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I", inc,
                    "-pthread", "-o", exe, src], check=True)
    return exe


@pytest.mark.parametrize("check", ["coherent", "refused", "beside", "crowd"])
def test_host_transfers(stage_check, check):
    out = subprocess.run([stage_check, check], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.strip() == "ok"
