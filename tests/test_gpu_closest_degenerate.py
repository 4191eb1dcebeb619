"""Closest points beside isolated degenerate triangles: a triangle without an FP64 distance (its
first two vertices equal, the query on the third one's side) or with a rounded one (a sliver)
must not hide the valid triangles farther away."""
import numpy as np
import pytest
import torch

from oracle import closest as C
from rmagine_amd import scenes
from rmagine_amd.simulation import HipMap

pytestmark = pytest.mark.gpu

# vertices of one triangle relative to its place: two or three equal ones, collinear ones, a sliver
SHAPES = {
    "a=b": [[0, 0, 0], [0, 0, 0], [1, 1, 0]],
    "a=c": [[0, 0, 0], [1, 1, 0], [0, 0, 0]],
    "b=c": [[0, 0, 0], [1, 1, 0], [1, 1, 0]],
    "a=b=c": [[0, 0, 0], [0, 0, 0], [0, 0, 0]],
    "collinear": [[0, 0, 0], [1, 1, 0], [0.5, 0.5, 0]],
    "sliver": [[0, 0, 0], [1, 0, 0], [0.5, 1e-5, 0]],
    "a~b": [[0, 0, 0], [1e-6, 0, 0], [1, 1, 0]],
}


@pytest.mark.parametrize("max_distance", [C.FLT_MAX, 1.5])
@pytest.mark.parametrize("shape", SHAPES)
def test_queries_around_a_degenerate_triangle(shape, max_distance):
    V, F, _ = scenes.room_workload(n_sensors=1)
    V = np.asarray(V, np.float32)
    rng = np.random.default_rng(sorted(SHAPES).index(shape))
    at = rng.uniform([-6, -6, 2.0], [6, 6, 3.5], size=(5, 3))
    t = (np.asarray(SHAPES[shape])[None] + at[:, None]).reshape(-1, 3).astype(np.float32)
    F = np.concatenate([F, (np.arange(15).reshape(5, 3) + len(V)).astype(F.dtype)])
    V = np.concatenate([V, t])
    # along each triangle's diagonal, beyond both ends of it, near it and up to a metre off
    k = rng.integers(0, 5, 1500)
    Q = at[k] + rng.uniform(-0.5, 1.5, (1500, 1)) * [1, 1, 0] + rng.normal(size=(1500, 3)) * 10.0 ** rng.uniform(-5, 0, (1500, 1))
    Q = Q.astype(np.float32)
    r = HipMap(V, F).closest_points(torch.as_tensor(Q, device="cuda"), max_distance)
    dist, face = r["dist"].cpu().numpy(), r["face_ids"].cpu().numpy()
    corners = [V.astype(np.float64)[F[:, j].astype(np.int64)] for j in range(3)]
    limit = float(np.float32(max_distance)) ** 2
    for i, q in enumerate(Q.astype(np.float64)):
        d2 = ((C.closest_on_triangles(q, *corners) - q) ** 2).sum(1)  # NaN where a triangle has none
        least = np.nanmin(d2)
        if least >= limit:
            assert dist[i] == np.float32(C.FLT_MAX) and face[i] == -1
            continue
        np.testing.assert_allclose(dist[i], np.sqrt(least), rtol=2e-7, atol=1e-7)
        assert d2[face[i]] <= least * (1 + 1e-9) + 1e-14
