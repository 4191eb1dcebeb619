"""Host check of the slab test's set-up (rmagine_amd/csrc/rmh_slab.hpp, which the ray kernels
compile): no box is culled that a ray of a non-unit direction meets (ray lists take their directions
as given).  With reciprocals off by up to an ulp the same program must find culled boxes."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
SRC = ROOT / "tests" / "cpp" / "slab_length_check.cpp"


@pytest.mark.parametrize("defines,holds", [([], True), (["-DSLAB_RECIPROCAL_WITHIN_AN_ULP"], False)])
def test_no_box_culled_for_long_directions(tmp_path, defines, holds):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = tmp_path / "slab_length_check"
    subprocess.run([cxx, "-O2", "-std=c++17", "-ffp-contract=off", *defines, "-o", str(exe), str(SRC)], check=True)
    res = subprocess.run([str(exe), "8000000"], capture_output=True, text=True, timeout=200)
    n, culled = map(int, res.stdout.split())
    assert n == 8_000_000 and (culled == 0) == holds, res.stdout


def test_kernels_take_their_reciprocals_from_the_set_up():
    text = (ROOT / "rmagine_amd" / "csrc" / "rmh_trace.hpp").read_text()
    assert "make_slab_ray(" in text and "amdgcn_rcpf" not in text
