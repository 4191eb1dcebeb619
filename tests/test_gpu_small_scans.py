"""Small casts put fewer rays into a wave and deal them to the XCDs differently from large
ones: a pose must give the same bytes whatever the number of poses it is cast with."""
import numpy as np
import pytest
import torch

from rmagine_amd import scenes
from rmagine_amd import types as T
from rmagine_amd.simulation import HipMap, simulator_for

pytestmark = pytest.mark.gpu

ATTRS = ("hits", "ranges", "points", "normals", "face_ids")


def _models():
    rng = np.random.default_rng(3)
    r = T.Interval(0.1, 60.0)
    sphere = T.SphericalModel(phi=T.DiscreteInterval(T.f32(-0.4), T.f32(0.07), 11),
                              theta=T.DiscreteInterval(T.f32(-3.0), T.f32(0.067), 93), range=r)
    line = T.SphericalModel(phi=T.DiscreteInterval(T.f32(-0.1), T.f32(0.07), 1),
                            theta=T.DiscreteInterval(T.f32(-3.0), T.f32(0.02), 301), range=r)
    pin = T.PinholeModel(61, 35, r, (30.0, 30.0), (30.0, 17.0))
    d = scenes.random_unit_dirs(1333, rng)
    o1 = T.O1DnModel(1333, 1, r, (0.0, 0.0, 0.05), d)
    on = T.OnDnModel(43, 31, r, rng.normal(scale=0.02, size=(1333, 3)).astype(np.float32), d)
    return {"sphere": sphere, "line": line, "pinhole": pin, "o1dn": o1, "ondn": on}


@pytest.fixture(scope="module")
def worlds():
    V, F, P = scenes.room_workload(n_sensors=2048)
    h = scenes.terrain_heights(300)  # 178,802 triangles: a deep map
    Vt, Ft = scenes.heightfield_mesh(h, 0.1)
    Pt = P.copy()
    Pt[:, 6] = scenes.terrain_height_at(h, 0.1, Pt[:, 4], Pt[:, 5]) + 1.0
    return {"room": (HipMap(V, F), torch.as_tensor(P, device="cuda")),
            "terrain": (HipMap(Vt, Ft), torch.as_tensor(Pt, device="cuda"))}


@pytest.mark.parametrize("name", ["sphere", "line", "pinhole", "o1dn", "ondn"])
@pytest.mark.parametrize("world", ["room", "terrain"])
def test_a_pose_gives_the_same_bytes_in_casts_of_any_size(worlds, world, name):
    hm, poses = worlds[world]
    sim = simulator_for(_models()[name], hm)
    ref = sim.simulate(poses, attrs=ATTRS)  # 64 rays per wave
    ref = {k: getattr(ref, k).reshape(len(poses), -1).clone() for k in ATTRS}
    for n in (1, 2, 7, 31, 63, 64, 150):  # down to 2 rays per wave
        got = sim.simulate(poses[:n].contiguous(), attrs=ATTRS)
        for k in ATTRS:
            a, b = getattr(got, k).reshape(n, -1), ref[k][:n]
            assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8)), (n, k)
