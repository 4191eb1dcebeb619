"""The device's treelet pass (k_treelet_nodes, one wave per treelet) against the serial
treelet_optimize() of the same header, run on the host by tests/cpp/treelet_check.cpp: with
single-triangle leaves the device reports the SAH cost of the refined tree itself, and the two
must agree to the printed digits (a different topology anywhere changes it)."""
import json
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

from rmagine_amd import scenes
from rmagine_amd.simulation import HipMap

pytestmark = pytest.mark.gpu
SRC = Path(__file__).resolve().parent / "cpp" / "treelet_check.cpp"


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = tmp_path_factory.mktemp("treelet") / "treelet_check"
    # no contraction, as the kernels are compiled
    subprocess.run([cxx, "-O2", "-std=c++17", "-ffp-contract=off", "-o", str(exe), str(SRC)], check=True)
    return exe


def _soup(n, seed, flat=False, same=False):
    """n triangles of random size and place; in one plane, or stacked on each other."""
    rng = np.random.default_rng(seed)
    c = np.zeros((n, 1, 3)) if same else rng.uniform(-50, 50, (n, 1, 3))
    V = c + rng.normal(size=(n, 3, 3)) * 10.0 ** rng.uniform(-2, 1, (n, 1, 1))
    if flat:
        V[..., 2] = 1.0
    return V.reshape(-1, 3).astype(np.float32), np.arange(3 * n, dtype=np.uint32).reshape(-1, 3)


CASES = {**{f"soup{n}": (lambda n=n: _soup(n, n)) for n in (7, 8, 9, 13, 64, 1000)},
         "flat": lambda: _soup(500, 1, flat=True), "stacked": lambda: _soup(300, 2, same=True),
         "sphere": scenes.genSphere, "room": lambda: scenes.room_with_boxes()[:2],
         "terrain": lambda: scenes.heightfield_mesh(scenes.terrain_heights(90), 0.1),
         "objects": lambda: scenes.objects_mesh(n_objects=200, n_ico=60)}


@pytest.mark.parametrize("name", CASES)
def test_tree_equals_the_serial_one(checker, tmp_path, name):
    V, F = CASES[name]()
    V, F = np.asarray(V, np.float32), np.asarray(F, np.uint32)
    p = tmp_path / "mesh.bin"
    with open(p, "wb") as f:
        np.array([len(V), len(F)], np.uint32).tofile(f)
        V.tofile(f)
        F.tofile(f)
    res = subprocess.run([str(checker), str(p), "3"], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout + res.stderr
    want = json.loads(res.stdout)["sah_treelets"]
    got = HipMap(V, F, max_leaf_size=1).info()["sah_cost"]
    # four printed digits; the last FP32 bits of the quotient
    assert abs(got - want) <= 5e-5 + 2e-7 * want, (name, got, want)
