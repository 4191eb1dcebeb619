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


def test_meshes_of_thin_triangles():
    """Every triangle without FP32 bounds: a fan around a vertex and scattered needles."""
    rng = np.random.default_rng(12)
    a = np.linspace(0, 2 * np.pi, 2500, endpoint=False)
    fan = np.concatenate([[[0, 0, 0]], np.stack([5 * np.cos(a), 5 * np.sin(a), 0.01 * np.sin(7 * a)], 1)])
    i = np.arange(2500)
    Ff = np.stack([0 * i, i + 1, (i + 1) % 2500 + 1], 1)
    at, d = rng.uniform(-5, 5, (400, 1, 3)), rng.normal(size=(400, 1, 3))
    thin = at + np.array([0, 1, 0.5])[None, :, None] * d + np.array([0, 0, 2e-4])[None, :, None] * rng.normal(size=(400, 3, 3))
    V = np.concatenate([fan, thin.reshape(-1, 3)]).astype(np.float32)
    F = np.concatenate([Ff, np.arange(1200).reshape(-1, 3) + len(fan)]).astype(np.uint32)
    Q = rng.uniform(-6, 6, (400, 3)).astype(np.float32)
    Q[::4, 2] = 0.0
    r = HipMap(V, F).closest_points(torch.as_tensor(Q, device="cuda"))
    dist, face = r["dist"].cpu().numpy(), r["face_ids"].cpu().numpy()
    corners = [V.astype(np.float64)[F[:, j].astype(np.int64)] for j in range(3)]
    for k, q in enumerate(Q.astype(np.float64)):
        d2 = ((C.closest_on_triangles(q, *corners) - q) ** 2).sum(1)
        np.testing.assert_allclose(dist[k], np.sqrt(d2.min()), rtol=2e-7, atol=1e-7)
        assert d2[face[k]] <= d2.min() * (1 + 1e-9) + 1e-14
