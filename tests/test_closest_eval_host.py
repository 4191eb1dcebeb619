"""Host check that the closest-point walk's upper bounds come only from triangles whose FP64
evaluation confirms them (rmagine_amd/csrc/rmh_closest_bounds.hpp, which the kernel compiles):
tests/cpp/closest_eval_check.cpp compares both over 6e6 random triangles, degenerate ones among
them.  A triangle whose first two vertices coincide has no FP64 distance for queries on the third
one's side (0 / 0), and must not keep the walk from the valid triangles farther away."""
import shutil
import subprocess
from pathlib import Path

import pytest

SRC = Path(__file__).resolve().parent / "cpp" / "closest_eval_check.cpp"


def test_upper_bounds_hold_for_the_evaluation(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = tmp_path / "closest_eval_check"
    n = 6_000_000
    subprocess.run([cxx, "-O2", "-std=c++17", "-ffp-contract=off", "-o", str(exe), str(SRC)], check=True)
    res = subprocess.run([str(exe), str(n)], capture_output=True, text=True, timeout=300)
    checked, finite, bad = map(int, res.stdout.split("\n")[-2].split())
    # of ordinary triangles (a fifth of all) most have a bound; sizes below the FP32 spacing have none
    assert checked == n and finite > n // 20
    assert bad == 0 and res.returncode == 0, res.stdout[-2000:]
