"""The vertex gathers read only triangles that won a pixel.

A double cone of many triangles around two poles (vertices of more corners than
the gathers keep in flight at once), half of it hidden, with an unused vertex,
an out-of-range corner's triangle and a triangle outside the image.  The
workspace's memory is filled with NaN first, so a partial that was not written
shows if it is read.  Gradients against the oracle: 1e-5 of scale for the
attributes (sums of a few hundred products), 1e-4 through the positions' chain.
"""
import math

import numpy as np
import pytest
import torch

import oracle
from diffrp_amd import nvdr

pytestmark = pytest.mark.gpu


def _cones(n, views):
    g = torch.Generator().manual_seed(n)
    a = 2 * math.pi * torch.arange(n) / n
    ring = torch.stack([0.8 * torch.cos(a), 0.7 * torch.sin(a), torch.zeros(n)], 1)
    pts = torch.cat([ring, torch.tensor([[0.1, 0.05, -0.6], [0.0, -0.1, 0.6], [3.0, 3.0, 0.0]])])
    i = torch.arange(n)
    j = (i + 1) % n
    front = torch.stack([i, j, torch.full((n,), n)], 1)
    back = torch.stack([j, i, torch.full((n,), n + 1)], 1)
    tri = torch.cat([front, back, torch.tensor([[0, 1, 999], [n + 2, n + 2, 0]])]).int()
    pos = []
    for v in range(views):
        w = 1.0 + 0.3 * torch.rand(len(pts), 1, generator=g)
        p = pts + torch.tensor([0.05 * v, -0.03 * v, 0.0])
        pos.append(torch.cat([p[:, :2] * w, (-1 if v % 2 else 1) * 0.5 * p[:, 2:] * w, w], 1))
    return torch.stack(pos).contiguous(), tri.contiguous(), g


def _close(a, b, rtol, what):
    a, b = a.detach().double().cpu().numpy(), np.asarray(b, np.float64)
    err = np.abs(a - b).max() / max(np.abs(b).max(), 1e-30)
    assert err <= rtol, f'{what}: {err:.3e} > {rtol}'


@pytest.mark.parametrize('n', [7, 40])
@pytest.mark.parametrize('views', [1, 5, 9])
@pytest.mark.parametrize('C', [1, 3, 4, 8, 16, 20])
def test_gradients_with_hidden_triangles(cuda, n, views, C):
    pos, tri, g = _cones(n, views)
    res = (45, 70)
    attr = torch.rand(pos.shape[1], C, generator=g)
    go = torch.randn(views, *res, C, generator=g)
    print(f'case: live triangles n={n} views={views} C={C}', flush=True)
    p, a, t = pos.cuda().requires_grad_(True), attr.cuda().requires_grad_(True), tri.cuda()
    rast, _ = nvdr.rasterize(nvdr.RasterizeCudaContext(), p, t, res, grad_db=False)
    out, _ = nvdr.interpolate(a, rast, t)
    poison = [torch.full((1 << k,), float('nan'), device='cuda') for k in range(10, 23)]
    del poison
    gp, ga = torch.autograd.grad(out, [p, a], go.cuda())
    r = rast.detach().cpu().numpy()
    oa, orr = oracle.interpolate_bwd(attr.numpy(), r, tri.numpy(), go.numpy())
    op = oracle.rasterize_bwd(pos.numpy(), tri.numpy(), r, orr)
    _close(ga, oa, 1e-5, 'grad attr')
    _close(gp, op, 1e-4, 'grad pos')


@pytest.mark.parametrize('views', [1, 9])
@pytest.mark.parametrize('C', [3, 8])
def test_accumulating_and_overwriting_calls(cuda, views, C):
    """The fused call adds to the gradients given; its overwriting form replaces them."""
    from diffrp_amd import _lib
    from diffrp_amd._lib import check, ptr, stream_of
    pos, tri, g = _cones(40, views)
    H, W = 45, 70
    V, F = pos.shape[1], tri.shape[0]
    p, t = pos.cuda().requires_grad_(True), tri.cuda()
    a, go = torch.rand(V, C, generator=g).cuda(), torch.randn(views, H, W, C, generator=g).cuda()
    rast, _ = nvdr.rasterize(nvdr.RasterizeCudaContext(), p, t, (H, W), grad_db=False)
    boxes, (off, inc), r, p = rast._drp_boxes[0], nvdr.incidence(t, V), rast.detach(), p.detach()
    L, vpg = _lib.lib(), nvdr._views_per_group(views, F)
    ws = torch.empty(L.drp_interpolate_rasterize_bwd_workspace_size(views, H, W, F, C, vpg), dtype=torch.uint8, device='cuda')

    def call(ga, gp, overwrite):
        args = [stream_of(a), ptr(a), views, V, C, ptr(r), H, W, ptr(t), F, ptr(p), 1, ptr(go), ptr(ga), None, ptr(gp),
                ptr(boxes), vpg, ptr(off), ptr(inc), ptr(ws), ws.numel()]
        if overwrite is None:
            check(L.drp_interpolate_rasterize_bwd(*args), 'add')
        else:
            check(L.drp_interpolate_rasterize_bwd_to(*args, overwrite), 'to')
        return ga, gp
    z, one = call(torch.zeros_like(a), torch.zeros_like(p), None), (torch.ones_like(a), torch.ones_like(p))
    nan = (torch.full_like(a, float('nan')), torch.full_like(p, float('nan')))
    assert z[0].abs().sum() > 0 and z[1].abs().sum() > 0
    for overwrite in (None, 0, 1, 2, 3):
        bits = overwrite or 0
        ga, gp = call((nan if bits & 1 else one)[0].clone(), (nan if bits & 2 else one)[1].clone(), overwrite)
        assert torch.equal(ga, z[0] if bits & 1 else z[0] + 1)
        assert torch.equal(gp, z[1] if bits & 2 else z[1] + 1)
