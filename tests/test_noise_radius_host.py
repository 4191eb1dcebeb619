"""Exhaustive host check of the radius of the Box-Muller draw (rmagine_amd/csrc/
rmh_noise_draw.hpp): tests/cpp/noise_radius_check.cpp evaluates it for all 2^24 draws against
sqrt(-2 log u) in long double, with reciprocals of FP32 precision and slightly worse."""
import shutil
import subprocess
from pathlib import Path

import pytest

SRC = Path(__file__).resolve().parent / "cpp" / "noise_radius_check.cpp"


@pytest.mark.parametrize("rough", ["1.0", "1.0000002"])
def test_radius_within_1e15_for_every_draw(tmp_path, rough):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = tmp_path / "noise_radius_check"
    subprocess.run([cxx, "-O2", "-std=c++17", "-ffp-contract=off", "-DRMH_DRAW_ROUGH=" + rough, "-o", str(exe), str(SRC)],
                   check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    n, worst, libm = res.stdout.split()
    assert res.returncode == 0 and int(n) == 1 << 24 and float(worst) < 1e-15, res.stdout
