"""The trilinear sample's reciprocal quotients and 32-bit brick offsets give
the bits of the plain division and the general addresses
(tests/trilinear_driver.cpp, host build of terrain_math.hpp)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


def test_fast_paths_equal_the_plain_form(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not found")
    exe = tmp_path / "trilinear_driver"
    r = subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", str(ROOT / "tests" / "trilinear_driver.cpp"),
                        "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
