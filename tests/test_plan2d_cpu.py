"""Compiles tests/plan2d_check.cpp with g++ against the library's 2-D planning
header and runs it."""
import os
import subprocess

import _pkg


def test_plans_cover_and_keep_limits(tmp_path):
    src = os.path.join(_pkg.ROOT, "tests", "plan2d_check.cpp")
    inc = os.path.join(_pkg.PKG_DIR, "csrc")
    exe = str(tmp_path / "plan2d_check")
    subprocess.run(["g++", "-O2", "-std=c++20", "-I", inc, "-o", exe, src], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.strip() == "ok"
