"""Batched casts where the table is searched in more than one step and the tiles do not divide
evenly: every entry must hold the bytes of its own simulate()."""
import numpy as np
import pytest
import torch

from rmagine_amd import scenes
from rmagine_amd import types as T
from rmagine_amd.simulation import BatchSimulatorHip, HipMap, simulator_for

pytestmark = pytest.mark.gpu


def _list_model(n, rng):
    return T.O1DnModel(n, 1, T.Interval(0.1, 60.0), (0.0, 0.0, 0.05), scenes.random_unit_dirs(n, rng))


def _camera(w, h):
    return T.PinholeModel(w, h, T.Interval(0.05, 80.0), (0.5 * w, 0.5 * w), (0.5 * (w - 1), 0.5 * (h - 1)))


@pytest.mark.parametrize("kinds", ["mixed", "images", "lists"])
@pytest.mark.parametrize("n", [1, 2, 64, 65, 130])
def test_batch_tables_of_many_entries(n, kinds):
    V, F, P = scenes.room_workload(n_sensors=4)
    hm = HipMap(V, F)
    poses = torch.as_tensor(P, device="cuda")
    rng = np.random.default_rng(n)
    images = [_camera(1, 1), _camera(17, 5), _camera(64, 3)]
    lists = [_list_model(k, rng) for k in (1, 63, 64, 65, 700)]
    models = {"mixed": images + lists, "images": images, "lists": lists}[kinds]
    picks = [models[i % len(models)] for i in range(n)]
    # entries without poses between those that have some: nothing to cast, no tile
    Tbm = [poses[: (i * 3 + 1) % 5] for i in range(n)]
    attrs = ("hits", "ranges", "face_ids", "points")
    entries = [{"model": m, "Tbm": t, "attrs": attrs} for m, t in zip(picks, Tbm)]
    batch = BatchSimulatorHip(hm, entries)
    sims = {id(m): simulator_for(m, hm) for m in models}
    ref = [sims[id(m)].simulate(t, attrs=attrs).to_numpy() if len(t) else None for m, t in zip(picks, Tbm)]
    for prm in ({}, {"chunk_rays": 64}, {"chunk_rays": 192, "waves_per_cu": 5}, {"launches": 2, "waves_per_cu": 1}):
        batch.set_params(**prm)
        for b in batch.bundles:
            for k in attrs:
                getattr(b, k).fill_(7)
        batch.simulate()
        for i, r in enumerate(ref):
            for k in attrs if r is not None else ():
                got = getattr(batch.bundles[i], k).cpu().numpy()
                np.testing.assert_array_equal(got.view(np.uint8), r[k].view(np.uint8), err_msg=f"{prm} entry {i} {k}")


def test_captured_batch_outlives_a_recut_table():
    """A recorded launch replayed after the batch was cut into fewer tiles runs past none of them."""
    V, F, P = scenes.room_workload(n_sensors=2)
    hm = HipMap(V, F)
    poses = torch.as_tensor(P, device="cuda")
    batch = BatchSimulatorHip(hm, [{"model": _camera(40, 64), "Tbm": poses}], tile_rows=1)
    ref = [b.ranges.clone() for b in batch.simulate()]
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        batch.simulate()
    batch.set_params(tile_rows=16)  # 64 x 1 tiles -> 10 x 4 of them: 64 -> 40 per pose
    for _ in range(3):
        batch.bundles[0].ranges.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(batch.bundles[0].ranges, ref[0])
