"""The chunk count of a batch counts its rays in tiles of 64, whatever the tiles a small batch is
cast in."""
import numpy as np
import pytest
import torch

from rmagine_amd import scenes
from rmagine_amd import types as T
from rmagine_amd.simulation import BatchSimulatorHip, HipMap

pytestmark = pytest.mark.gpu


def _chunks(W, H, poses, rows, chunk_rays, ray_list):
    if ray_list:
        W, H, rows = W * H, 1, 1
    th = 1
    while th * 2 <= rows and th * 2 <= H:
        th *= 2
    tw = 64 // th
    rays = poses * -(-W // tw) * -(-H // th) * 64
    return -(-rays // chunk_rays)


@pytest.mark.parametrize("n_poses", [1, 3, 120])
@pytest.mark.parametrize("params", [{}, {"chunk_rays": 64}, {"chunk_rays": 192, "tile_rows": 16}, {"tile_rows": 1, "launches": 2}])
def test_total_chunks(n_poses, params):
    V, F, P = scenes.room_workload(n_sensors=4)
    hm = HipMap(V, F)
    poses = torch.as_tensor(P, device="cuda").repeat(30, 1)[:n_poses].contiguous()
    r = T.Interval(0.1, 60.0)
    lidar = T.SphericalModel(phi=T.DiscreteInterval(T.f32(-0.2), T.f32(0.025), 16),
                             theta=T.DiscreteInterval(T.f32(-3.1), T.f32(0.0068), 900), range=r)
    camera = T.PinholeModel(61, 35, r, (30.0, 30.0), (30.0, 17.0))
    rays = T.O1DnModel(777, 1, r, (0.0, 0.0, 0.0), scenes.random_unit_dirs(777, np.random.default_rng(2)))
    batch = BatchSimulatorHip(hm, [{"model": m, "Tbm": poses} for m in (lidar, camera, rays)])
    batch.set_params(**params)
    chunk, rows = params.get("chunk_rays", 256), params.get("tile_rows", 4)
    want = (_chunks(900, 16, n_poses, rows, chunk, False) + _chunks(61, 35, n_poses, rows, chunk, False)
            + _chunks(777, 1, n_poses, rows, chunk, True))
    assert batch.params()["total_chunks"] == want
    assert batch.params()["total_rays"] == n_poses * (900 * 16 + 61 * 35 + 777)
