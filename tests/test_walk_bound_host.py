"""Host check of the closest-point walk's box test as the kernel compiles it (rmagine_amd/csrc/
rmh_closest_bounds.hpp: box_d2 against walk_bound): tests/cpp/walk_bound_check.cpp requires that no
box within the bound is dropped, for 4e6 random queries and boxes (coordinates up to 1e19, gaps down
to one float).  With the bound not raised the same program must find dropped boxes."""
import shutil
import subprocess
from pathlib import Path

import pytest

SRC = Path(__file__).resolve().parent / "cpp" / "walk_bound_check.cpp"


@pytest.mark.parametrize("defines,holds", [([], True), (["-DWALK_BOUND_AS_GIVEN"], False)])
def test_no_box_within_the_bound_is_dropped(tmp_path, defines, holds):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = tmp_path / "walk_bound_check"
    subprocess.run([cxx, "-O2", "-std=c++17", "-ffp-contract=off", *defines, "-o", str(exe), str(SRC)], check=True)
    res = subprocess.run([str(exe), "4000000"], capture_output=True, text=True, timeout=120)
    n, dropped = map(int, res.stdout.split("\n")[-2].split())
    assert n == 4_000_000 and (dropped == 0) == holds and (res.returncode == 0) == holds, res.stdout[-2000:]
