"""Host check that a recorded batched launch replayed against a table cut into other tiles stays
within its entries (rmagine_amd/csrc/rmh_batch_tiles.hpp, which the kernel compiles).  With the
first tile kept from the table the launch was made for, the same program must find violations."""
import shutil
import subprocess
from pathlib import Path

import pytest

SRC = Path(__file__).resolve().parent / "cpp" / "batch_tiles_check.cpp"


@pytest.mark.parametrize("defines,holds", [([], True), (["-DBATCH_TILES_FIXED_BASE"], False)])
def test_launch_stays_in_its_entries(tmp_path, defines, holds):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = tmp_path / "batch_tiles_check"
    subprocess.run([cxx, "-O2", "-std=c++17", "-Wall", *defines, "-o", str(exe), str(SRC)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    launches, bad = map(int, res.stdout.split())
    assert launches == 600_000 and (bad == 0) == holds and (res.returncode == 0) == holds
