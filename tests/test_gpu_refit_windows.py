"""Refit of trees around the window sizes of its passes (one window, two, several passes,
long chains): rays through moved maps give the bytes of a fresh build, and a refit to the
vertices a map already has leaves boxes as tight as the build's."""
import numpy as np
import pytest
import torch

from rmagine_amd import types as T
from rmagine_amd.simulation import HipMap, simulator_for

pytestmark = pytest.mark.gpu


def _soup(n, layout, rng):
    """n small triangles: spread over a cube, or on a line with sizes and gaps that double
    (uneven trees, long chains of ancestors)."""
    if layout == "cube":
        c = rng.uniform(-20.0, 20.0, (n, 1, 3))
        d = rng.normal(scale=0.3, size=(n, 3, 3))
    else:
        s = 2.0 ** -(np.arange(n) % 24)[:, None, None]
        c = np.concatenate([20.0 * s, 0.0 * s, 0.0 * s], -1) + rng.normal(scale=1e-3, size=(n, 1, 3)) * s
        d = rng.normal(scale=0.2, size=(n, 3, 3)) * s
    return (c + d).reshape(-1, 3).astype(np.float32), np.arange(3 * n, dtype=np.uint32).reshape(n, 3)


def _model():
    return T.SphericalModel(phi=T.DiscreteInterval(T.f32(-1.2), T.f32(0.04), 60),
                            theta=T.DiscreteInterval(T.f32(-3.1), T.f32(0.03), 200), range=T.Interval(0.0, 100.0))


@pytest.mark.parametrize("layout", ["cube", "line"])
@pytest.mark.parametrize("n", [1, 2, 9, 512, 513, 514, 1025, 5000, 70000, 600000])
def test_refit_equals_rebuild(n, layout):
    rng = np.random.default_rng(n)
    V, F = _soup(n, layout, rng)
    hm = HipMap(V, F)
    sim = simulator_for(_model(), hm)
    poses = T.make_transforms([[0.0, 0.0, 0.0], [3.0, 1.0, -2.0]], [[0.0, 0.0, 0.0, 1.0]] * 2)
    P = torch.as_tensor(poses, device="cuda")
    if n > 8:  # boxes padded once more per level: at most a little wider than the build's
        before = sim.visit_stats(P)
        hm.refit(V)
        after = sim.visit_stats(P)
        visits = [s["vector_node_visits"] + s["scalar_node_visits"] for s in (before, after)]
        assert visits[0] > 0 and visits[1] <= 1.05 * visits[0], visits
    for step in range(2):
        V2 = (V + rng.normal(scale=0.05 if layout == "cube" else 1e-3, size=V.shape) + 0.5 * step).astype(np.float32)
        hm.refit(V2)
        a = sim.simulate(P, attrs=T.ATTRIBUTES).to_numpy()
        b = simulator_for(_model(), HipMap(V2, F)).simulate(P, attrs=T.ATTRIBUTES).to_numpy()
        for k in T.ATTRIBUTES:
            np.testing.assert_array_equal(a[k].view(np.uint8), b[k].view(np.uint8), err_msg=f"{step} {k}")
