"""Host check of the FP32 bounds of the closest-point walk (rmagine_amd/csrc/
rmh_closest_bounds.hpp, which the kernel compiles): tests/cpp/tri_bound_check.cpp requires
that they enclose the FP64 squared distance of 4e6 random queries to triangles (slivers and
degenerate ones among them) and boxes.  Built without the margins it must find violations."""
import shutil
import subprocess
from pathlib import Path

import pytest

SRC = Path(__file__).resolve().parent / "cpp" / "tri_bound_check.cpp"


@pytest.mark.parametrize("defines,n,holds", [([], 4_000_000, True), (["-DRMH_CB_NO_MARGIN"], 500_000, False)])
def test_bounds_enclose_the_distance(tmp_path, defines, n, holds):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = tmp_path / "tri_bound_check"
    subprocess.run([cxx, "-O2", "-std=c++17", "-ffp-contract=off", *defines, "-o", str(exe), str(SRC)], check=True)
    res = subprocess.run([str(exe), str(n)], capture_output=True, text=True, timeout=300)
    checked, bad = map(int, res.stdout.split("\n")[-2].split())
    assert checked == n and (bad == 0) == holds and (res.returncode == 0) == holds, res.stdout[-2000:]
