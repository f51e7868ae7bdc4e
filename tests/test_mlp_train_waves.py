"""The training kernel's waves are ordered by its barriers alone: the kernel's
source built as host code (tests/mlp_train_waves_driver.cpp) gives the same
bits for one block whichever of its waves run ahead to the next barrier, with
one to five rounds of its loop, whole and part-filled."""
import os
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
ROCM = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))


def test_no_result_depends_on_the_order_of_waves(tmp_path):
    clang = ROCM / "llvm" / "bin" / "clang++"
    if not clang.exists():
        pytest.skip("no clang++ of the ROCm toolchain")
    exe = tmp_path / "waves"
    r = subprocess.run([str(clang), "-x", "c++", "-std=c++17", "-O2", "-w", "-ffp-contract=off",
                        f"-I{ROCM / 'include'}", f"-I{ROOT / 'include'}",
                        str(ROOT / "tests" / "mlp_train_waves_driver.cpp"), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([str(exe), *map(str, range(1, 11))], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
