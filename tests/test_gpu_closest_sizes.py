"""rmh_closest_points over its launch shapes: the queries per wave follow the batch size, and
neither they nor the order of the batch may change a result."""
import numpy as np
import pytest
import torch

from oracle import closest as C
from rmagine_amd import scenes
from rmagine_amd.simulation import HipMap

pytestmark = pytest.mark.gpu


def _queries(V, F, n, rng):
    """Points in the room, on its vertices, edge midpoints and faces, and far outside."""
    Q = rng.uniform([-12, -12, -1], [12, 12, 5], size=(n, 3))
    tri = V[F.astype(np.int64)].astype(np.float64)
    k = rng.integers(0, len(tri), n)
    w = rng.dirichlet([1, 1, 1], n)
    w[0::4] = np.eye(3)[rng.integers(0, 3, len(w[0::4]))]
    w[1::4, 2] = 0.0
    w[1::4, :2] = 0.5
    on = (tri[k] * w[:, :, None]).sum(1)
    pick = rng.integers(0, 3, n)
    Q[pick == 1] = on[pick == 1]
    Q[(pick == 2) & (np.arange(n) % 16 == 0)] *= 1e3
    return Q.astype(np.float32)


@pytest.fixture(scope="module")
def room():
    V, F, _ = scenes.room_workload(n_sensors=1)
    V = np.asarray(V, np.float32)
    # slivers and degenerate triangles beside the boxes
    s = np.array([[0, 0, 3], [4, 0, 3], [2, 1e-5, 3], [1, 1, 3.5], [1, 1, 3.5], [2, 2, 3.5]], np.float32)
    F = np.concatenate([F, np.array([[0, 1, 2], [3, 4, 5]], F.dtype) + len(V)])
    V = np.concatenate([V, s])
    rng = np.random.default_rng(31)
    Q = _queries(V, F, 200_000, rng)
    hm = HipMap(V, F)
    r = hm.closest_points(torch.as_tensor(Q, device="cuda"))
    return V, F, Q, hm, {k: v.cpu().numpy() for k, v in r.items()}


def test_large_batch_against_the_oracle(room):
    V, F, Q, _, r = room
    corners = [V.astype(np.float64)[F[:, k].astype(np.int64)] for k in range(3)]
    for i in range(600):
        q = Q[i].astype(np.float64)
        d2 = ((C.closest_on_triangles(q, *corners) - q) ** 2).sum(1)  # NaN for the degenerate triangle
        np.testing.assert_allclose(r["dist"][i], np.sqrt(np.nanmin(d2)), rtol=2e-7, atol=1e-7)
        # among ties the lowest face, up to the last bits of the two FP64 evaluations
        face = r["face_ids"][i]
        assert d2[face] <= np.nanmin(d2) * (1 + 1e-12) + 1e-300
        assert face == np.nanargmin(d2) or not np.array_equal(d2[face], np.nanmin(d2))


@pytest.mark.parametrize("n", [1, 63, 64, 65, 3072, 3073, 6144, 6145, 24577, 65535, 65536, 196609])
def test_results_do_not_depend_on_the_batch(room, n):
    _, _, Q, hm, r = room
    rng = np.random.default_rng(n)
    at = rng.permutation(len(Q))[:n]
    out = hm.closest_points(torch.as_tensor(Q[at], device="cuda"))
    for k, v in out.items():
        np.testing.assert_array_equal(v.cpu().numpy(), r[k][at], err_msg=k)


@pytest.mark.parametrize("max_distance", [0.0, 1e-4, 0.25, 1e19])
def test_max_distance_cuts_the_same_queries(room, max_distance):
    _, _, Q, hm, r = room
    out = hm.closest_points(torch.as_tensor(Q[:5000], device="cuda"), max_distance)
    near = r["dist"][:5000] < np.float32(max_distance)
    got = out["dist"].cpu().numpy()
    # the limit is compared in FP64: queries within one FP32 rounding of it may go either way
    edge = np.abs(r["dist"][:5000] - np.float32(max_distance)) <= 1e-7 * max(max_distance, 1e-30)
    np.testing.assert_array_equal((got != C.FLT_MAX)[~edge], near[~edge])
    np.testing.assert_array_equal(got[near & ~edge], r["dist"][:5000][near & ~edge])
