"""The totals of a level of the device kd build are exact beyond 31 bits, and a
level that its indices cannot hold is refused (tests/kd_level_driver.cpp, host
build of kdbuild.hpp)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


def test_level_totals_and_their_limits(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not found")
    exe = tmp_path / "kd_level_driver"
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", str(ROOT / "tests" / "kd_level_driver.cpp"), "-o",
                        str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
