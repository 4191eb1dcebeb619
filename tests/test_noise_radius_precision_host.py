"""Precision of the Box-Muller radius (rmagine_amd/csrc/rmh_noise_draw.hpp) over all 2^24 draws:
that of a logarithm and a root rounded once each.  The logarithm's half ulp counts half in the root
(2^-54 at most), the root's own is at most 2^-53, together 1.5 x 2^-53 = 1.665e-16 of the value;
the program's long double results are 2^-11 of that from exact."""
import shutil
import subprocess
from pathlib import Path

import pytest

SRC = Path(__file__).resolve().parent / "cpp" / "noise_radius_check.cpp"


@pytest.mark.parametrize("rough", ["1.0", "1.0000002", "0.9999998"])
def test_radius_is_rounded_like_log_and_root(tmp_path, rough):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = tmp_path / "noise_radius_check"
    subprocess.run([cxx, "-O2", "-std=c++17", "-ffp-contract=off", "-DRMH_DRAW_ROUGH=" + rough, "-o", str(exe), str(SRC)],
                   check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    n, worst, libm = res.stdout.split()
    assert int(n) == 1 << 24 and float(worst) < 1.5 * 2.0**-53 * (1 + 2.0**-9), res.stdout
