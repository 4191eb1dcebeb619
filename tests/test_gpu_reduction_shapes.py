"""The segmented reductions over their launch shapes: four elements per lane where the arrays
are aligned, one where they are not, one to many blocks per segment.  Every form is compared
with an FP64 evaluation in torch; sums of n terms in another order differ by about n 2^-53 of
the sum of magnitudes at most, far less in practice: 1e-12 of it is allowed."""
import pytest
import torch

from rmagine_amd import math as M

pytestmark = pytest.mark.gpu
dev = "cuda"


def _shifted(x, by):
    """The same values at an address `by` elements into an allocation."""
    y = torch.empty((x.shape[0] + by, *x.shape[1:]), dtype=x.dtype, device=dev)[by:]
    y.copy_(x)
    return y


def _cloud(seg, nseg, shift, ids):
    g = torch.Generator(device=dev).manual_seed(seg * 7 + nseg)
    n = seg * nseg
    d = torch.randn((n, 3), generator=g, device=dev) * 5
    m = d + 0.3 * torch.randn((n, 3), generator=g, device=dev)
    nr = torch.nn.functional.normalize(torch.randn((n, 3), generator=g, device=dev), dim=1)
    mask = [(torch.rand(n, generator=g, device=dev) > 0.2).to(torch.uint8) * k for k in (255, 1)]
    i = torch.randint(0, 3, (n,), generator=g, device=dev, dtype=torch.int32) if ids else None
    q = torch.randn((nseg, 8), generator=g, device=dev) * 0.1
    q[:, 3], q[:, 7] = 1.0, 0.0
    q[:, :4] /= q[:, :4].norm(dim=1, keepdim=True)
    s = lambda x: None if x is None else _shifted(x, shift)
    return (q.contiguous(), M.PointCloudView(s(d), mask=s(mask[0]), ids=s(i)),
            M.PointCloudView(s(m), mask=s(mask[1]), normals=s(nr), ids=s(i)))


def _pairs(q, data, model, seg, nseg, prm, p2l):
    """FP64 moved dataset points, model points, normals, residuals and which count."""
    x, y, z, w = q[:, :4].double().unbind(1)
    R = torch.stack([w * w + x * x - y * y - z * z, 2 * (x * y - w * z), 2 * (x * z + w * y),
                     2 * (x * y + w * z), w * w - x * x + y * y - z * z, 2 * (y * z - w * x),
                     2 * (x * z - w * y), 2 * (y * z + w * x), w * w - x * x - y * y + z * z], 1).view(nseg, 3, 3)
    t = q[:, 4:7].double()
    d = data.points.double().view(nseg, seg, 3) @ R.transpose(1, 2).contiguous() + t[:, None]
    m, n = model.points.double().view(nseg, seg, 3), model.normals.double().view(nseg, seg, 3)
    keep = (data.mask.bool() & model.mask.bool()).view(nseg, seg)
    if data.ids is not None:
        keep &= ((data.ids == prm.dataset_id) & (model.ids == prm.model_id)).view(nseg, seg)
    r = ((d - m) * n).sum(-1)
    keep &= (r.abs() < prm.max_dist) if p2l else ((m - d).norm(dim=-1) < prm.max_dist)
    return d, m, n, r, keep


def _close(got, want, scale):
    assert (got - want).abs().max().item() <= 1e-12 * scale, ((got - want).abs().max().item(), scale)


SHAPES = [(1, 1), (3, 2), (4, 1), (5, 3), (1023, 1), (1024, 2), (1027, 5), (2049, 64), (4100, 9), (13, 3000),
          (300_002, 1), (2_100_001, 1), (8192, 2001)]


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("seg,nseg", SHAPES)
def test_reductions_over_shapes(seg, nseg, shift):
    ids = seg % 2 == 1
    q, data, model = _cloud(seg, nseg, shift, ids)
    prm = M.UmeyamaReductionConstraints(max_dist=0.6, dataset_id=1, model_id=1)
    for kind in (M.P2L, M.P2P):
        st = M.statistics(kind, q, data, model, prm, segment_size=seg, n_segments=nseg)
        d, m, n, r, keep = _pairs(q, data, model, seg, nseg, prm, kind == M.P2L)
        if kind == M.P2L:
            m = d - n * r[..., None]
        k = keep[..., None].double()
        cnt = k.sum(1)
        assert torch.equal(M.stats_n_meas(st).long(), cnt[:, 0].long())
        c = cnt.clamp(min=1)
        dm, mm = (d * k).sum(1) / c, (m * k).sum(1) / c
        cov = ((m - mm[:, None]) * k).transpose(1, 2).contiguous() @ ((d - dm[:, None]) * k) / c[..., None]
        _close(st[:, 0:3], dm, 100.0)
        _close(st[:, 3:6], mm, 100.0)
        _close(st[:, 6:15], cov.transpose(1, 2).reshape(nseg, 9), 1000.0)
    d, m, n, r, keep = _pairs(q, data, model, seg, nseg, prm, True)
    sys = M.linear_system_p2l(q, data, model, prm, kernel_scale=5.0, segment_size=seg, n_segments=nseg)
    w = torch.where(keep, 25.0 / (5.0 + r) ** 2, torch.zeros_like(r))
    J = torch.cat([torch.linalg.cross(d, n), n], -1)
    scale = 1000.0 * seg
    _close(sys[:, :36], ((J * w[..., None]).transpose(1, 2).contiguous() @ J).reshape(nseg, 36), scale)
    _close(sys[:, 36:42], (J * (w * r)[..., None]).sum(1), scale)
    _close(sys[:, 42], (w * r * r).sum(1), scale)
    mo = M.vec3_moments(data.points, model.points, data.mask, segment_size=seg, n_segments=nseg)
    k = data.mask.bool().view(nseg, seg, 1).double()
    a, b = data.points.double().view(nseg, seg, 3) * k, model.points.double().view(nseg, seg, 3) * k
    assert torch.equal(mo["count"].long(), k.sum((1, 2)).long())
    _close(mo["sum"], a.sum(1), 100.0 * seg)
    cov = b.transpose(1, 2).contiguous() @ a / k.sum(1).clamp(min=1)[..., None]
    _close(mo["cov"], cov.transpose(1, 2).reshape(nseg, 9), 1000.0)
