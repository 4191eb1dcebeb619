"""pose_range_loss on the device (rmh_pose_loss) against the same loss composed of perturb,
pose_grad and the SO(3) left Jacobian, over pose counts around the sums' block of four poses,
tile counts from one up, input types and layouts.  Both evaluate the same FP64 expressions;
the tiles are summed in one order, so only the last bits of the Jacobian may differ."""
import pytest
import torch

from rmagine_amd import adjoint as A
from rmagine_amd import scenes
from rmagine_amd import types as T
from rmagine_amd.simulation import HipMap, simulator_for

pytestmark = pytest.mark.gpu
dev = "cuda"


@pytest.fixture(scope="module")
def room():
    V, F, Tbm = scenes.room_workload(n_sensors=600)
    return HipMap(V, F), torch.as_tensor(Tbm, device=dev)


@pytest.mark.parametrize("w,h,n,dtype", [(1, 1, 1, torch.float64), (50, 1, 3, torch.float64), (64, 2, 4, torch.float32),
                                         (900, 16, 5, torch.float64), (33, 9, 257, torch.float32),
                                         (120, 7, 600, torch.float64)])
def test_loss_and_gradient_equal_the_composition(room, w, h, n, dtype):
    hm, poses = room
    model = T.SphericalModel(phi=T.DiscreteInterval(-0.2, 0.03, h), theta=T.DiscreteInterval(-3.0, 6.0 / w, w),
                             range=T.Interval(0.1, 100.0))
    sim = simulator_for(model, hm)
    g = torch.Generator(device=dev).manual_seed(n)
    T0 = poses[:n].contiguous()
    target = sim.simulate(T0, attrs=("ranges",)).ranges + 0.05 * torch.randn(n * w * h, generator=g, device=dev)
    xi = (0.1 * torch.randn((n, 6), generator=g, device=dev, dtype=torch.float64)).to(dtype)
    xi[0] = 0.0
    xi[n // 2, 3:] = torch.tensor([1e-7, -2e-7, 3e-8], device=dev, dtype=dtype)
    strided = torch.empty((6, n), dtype=dtype, device=dev).t()
    strided.copy_(xi)
    for x in (xi, strided):
        x = x.detach().requires_grad_(True)
        loss = A.pose_range_loss(x, T0, sim, target, huber_delta=0.05)
        (grad,) = torch.autograd.grad(loss.sum(), x)
        raw = A.pose_grad(sim, A.perturb(T0, xi), target, per_pose_targets=n > 1, huber_delta=0.05)
        J = A.so3_left_jacobian(xi.to(torch.float64)[:, 3:])
        want = torch.cat([raw[:, 1:4], (J * raw[:, 4:7, None]).sum(1)], 1)
        assert loss.dtype == torch.float64 and grad.dtype == dtype
        assert torch.equal(loss, raw[:, 0])
        eps = 1e-13 if dtype == torch.float64 else 2.0 ** -23
        assert (grad.double() - want).abs().max() <= eps * (raw.abs().max() + 1.0)


def test_argument_errors(room):
    hm, poses = room
    sim = simulator_for(scenes.vlp16_workload_model(), hm)
    xi, target = torch.zeros((2, 6), device=dev, dtype=torch.float64), torch.zeros(14400, device=dev)
    with pytest.raises(ValueError):
        A.pose_range_loss(xi, poses[:2].double(), sim, target)
    with pytest.raises(ValueError):
        A.pose_range_loss(xi, poses[:2], sim, target[:-1])
    with pytest.raises(ValueError):
        A.pose_range_loss(xi, poses[:2], sim, target.double())
    with pytest.raises(ValueError):
        A.pose_range_loss(xi, poses[:2], sim, target, target[:10].to(torch.uint8))
