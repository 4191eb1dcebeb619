"""A recorded batched launch replayed after the batch was cut into more tiles: it casts the tiles
it has workgroups for, and every ray list whole."""
import numpy as np
import pytest
import torch

from rmagine_amd import scenes
from rmagine_amd import types as T
from rmagine_amd.simulation import BatchSimulatorHip, HipMap

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("launches", [1, 2])
@pytest.mark.parametrize("n_lists", [1, 3])
def test_captured_batch_after_a_recut_into_more_tiles(launches, n_lists):
    V, F, P = scenes.room_workload(n_sensors=2)
    hm = HipMap(V, F)
    poses = torch.as_tensor(P, device="cuda")
    rng = np.random.default_rng(9)
    lidar = T.SphericalModel(phi=T.DiscreteInterval(T.f32(-0.2), T.f32(0.025), 16),
                             theta=T.DiscreteInterval(T.f32(-3.1), T.f32(0.0068), 900), range=T.Interval(0.1, 60.0))
    lists = [T.O1DnModel(k, 1, T.Interval(0.1, 60.0), (0.0, 0.0, 0.0), scenes.random_unit_dirs(k, rng))
             for k in (700, 65, 1000)[:n_lists]]
    # enough poses for tiles of 64 rays: 900 x 16 is 228 tiles of 4 rows and 240 of 1 row
    many = poses.repeat(40, 1)
    entries = [{"model": lidar, "Tbm": many}] + [{"model": m, "Tbm": poses} for m in lists]
    batch = BatchSimulatorHip(hm, entries, tile_rows=4, launches=launches)
    ref = [b.ranges.clone() for b in batch.simulate()]
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        batch.simulate()
    batch.set_params(tile_rows=1)
    for _ in range(3):
        for b in batch.bundles:
            b.ranges.fill_(-1.0)
        g.replay()
        torch.cuda.synchronize()
        got = [b.ranges for b in batch.bundles]
        cast = got[0] != -1.0
        assert torch.equal(got[0][cast], ref[0][cast]) and cast.float().mean() > 0.9
        if launches == 2:
            assert all(torch.equal(x, y) for x, y in zip(got[1:], ref[1:]))
        # a launch made for the new tiles casts everything
        batch.simulate()
        assert all(torch.equal(x, y) for x, y in zip(got, ref))
