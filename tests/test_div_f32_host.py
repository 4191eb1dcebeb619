"""Host check of the shared-reciprocal division of the ray set-up (rmagine_amd/csrc/
rmh_trace.hpp, div_f32_f64): tests/cpp/div_f32_check.cpp requires the bits of the IEEE quotient
for 2e6 pairs of FP32 values and reciprocals up to two units in the last place off."""
import shutil
import subprocess
from pathlib import Path

import pytest

SRC = Path(__file__).resolve().parent / "cpp" / "div_f32_check.cpp"


def test_quotients_from_one_reciprocal_are_correctly_rounded(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = tmp_path / "div_f32_check"
    subprocess.run([cxx, "-O2", "-std=c++17", "-ffp-contract=off", "-o", str(exe), str(SRC)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout[-2000:]
