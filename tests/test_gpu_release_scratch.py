"""The scratch memory kept between calls can be given back, and later calls work without it."""
import numpy as np
import pytest
import torch

from rmagine_amd import scenes
from rmagine_amd.simulation import HipMap, release_scratch

pytestmark = pytest.mark.gpu


def test_scratch_is_given_back():
    V, F, _ = scenes.room_workload(n_sensors=1)
    hm = HipMap(V, F)
    Q = torch.rand((8_000_000, 3), device="cuda") * 10 - 5  # sorted in 136 MB of scratch
    a = hm.closest_points(Q)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    release_scratch()
    after = torch.cuda.mem_get_info()[0]
    assert after - before >= 100e6
    b = hm.closest_points(Q)
    again = HipMap(V, F).closest_points(Q)
    torch.cuda.synchronize()
    for k in a:
        np.testing.assert_array_equal(a[k].cpu().numpy(), b[k].cpu().numpy(), err_msg=k)
        np.testing.assert_array_equal(a[k].cpu().numpy(), again[k].cpu().numpy(), err_msg=k)
