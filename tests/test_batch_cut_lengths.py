"""The lengths of a batch's work items on the device: sphere-traced tiles are
cut into at most 1,024 items where the configuration allows, every ray is in
one item (tests/batch_cut_driver.cpp, host build of the plan)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


def test_items_of_each_kind(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not found")
    exe = tmp_path / "batch_cut_driver"
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", f"-I{ROOT / 'include'}",
                        str(ROOT / "tests" / "batch_cut_driver.cpp"),
                        *map(str, sorted((ROOT / "rayengine_amd" / "csrc" / "host").glob("*.cpp"))), "-fopenmp",
                        "-ffp-contract=off", "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr
