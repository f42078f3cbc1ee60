"""
The tile backward over its channel counts: every compiled width, passes over
wider attributes, rows that are not whole quads, and the gradients of the
screen-space derivatives, against the oracle on ragged images whose last tiles
are partly outside and whose corners hold empty tiles.

Tolerances are those the operators have elsewhere: 1e-5 of scale for sums of
products of float32 (hundreds of terms, each within a few 2^-24), 1e-4 through
the positions' chain.
"""
import numpy as np
import pytest
import torch

import oracle
from diffrp_amd import nvdr
from tests.scenes import noisy_clip

pytestmark = pytest.mark.gpu


def _close(a, b, rtol, what):
    a, b = a.detach().double().cpu().numpy(), np.asarray(b, np.float64)
    err = np.abs(a - b).max() / max(np.abs(b).max(), 1e-30)
    assert err <= rtol, f'{what}: {err:.3e} > {rtol}'


def _scene(C, views, res, seed, subdiv=4):
    pos, tri, _ = noisy_clip(subdiv, 0.01, res[0], views=views)
    g = torch.Generator().manual_seed(seed)
    return pos, tri, torch.rand(pos.shape[-2], C, generator=g), torch.randn(views, *res, C, generator=g), g


@pytest.mark.parametrize('C', [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 17, 19, 20, 21, 33, 48])
def test_attribute_backward_of_any_width(cuda, C):
    res = (83, 101)
    pos, tri, attr, go, _ = _scene(C, 3, res, C)
    rast, _ = nvdr.rasterize(nvdr.RasterizeCudaContext(), pos.cuda(), tri.cuda(), res, grad_db=False)
    a, r = attr.cuda().requires_grad_(True), rast.detach().requires_grad_(True)
    r._drp_boxes = rast._drp_boxes[:2] + (r._version, None)
    out, _ = nvdr.interpolate(a, r, tri.cuda())
    ga, gr = torch.autograd.grad(out, [a, r], go.cuda(), retain_graph=True)
    oa, orr = oracle.interpolate_bwd(attr.numpy(), rast.cpu().numpy(), tri.numpy(), go.numpy())
    _close(ga, oa, 1e-5, 'grad attr')
    _close(gr, orr, 1e-5, 'grad rast')
    again, _ = torch.autograd.grad(out, [a, r], go.cuda())
    assert torch.equal(ga, again)  # fixed summation order


@pytest.mark.parametrize('C', [1, 2, 3, 5, 6, 7, 9, 12, 13, 14, 15, 16])
@pytest.mark.parametrize('views', [1, 9])
def test_fused_backward_of_any_width_equals_the_separate_passes(cuda, C, views):
    res = (70, 53)
    pos, tri, attr, go, _ = _scene(C, views, res, 100 + C, subdiv=3)
    got = []
    for fused in (nvdr._FUSED_C, ()):
        saved, nvdr._FUSED_C = nvdr._FUSED_C, fused
        try:
            p, a = pos.cuda().requires_grad_(True), attr.cuda().requires_grad_(True)
            rast, _ = nvdr.rasterize(nvdr.RasterizeCudaContext(), p, tri.cuda(), res, grad_db=False)
            out, _ = nvdr.interpolate(a, rast, tri.cuda())
            got.append(torch.autograd.grad(out, [p, a], go.cuda()))
        finally:
            nvdr._FUSED_C = saved
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    assert got[0][0].abs().sum() > 0


@pytest.mark.parametrize('C,idx', [(2, 'all'), (1, [0]), (3, [2, 0]), (5, 'all'), (9, [8, 1, 1, 4]), (16, [0, 15]),
                                   (18, 'all')])
@pytest.mark.parametrize('batched', [False, True])
def test_derivative_gradients(cuda, C, idx, batched):
    res, views = (60, 77), 3
    pos, tri, attr, go, g = _scene(C, views, res, 200 + C)
    if batched:
        attr = torch.rand(views, pos.shape[-2], C, generator=g)
    ids = list(range(C)) if idx == 'all' else idx
    rast, db = nvdr.rasterize(nvdr.RasterizeCudaContext(), pos.cuda(), tri.cuda(), res)
    a, d = attr.cuda().requires_grad_(True), db.detach().requires_grad_(True)
    r = rast.detach().requires_grad_(True)
    r._drp_boxes = rast._drp_boxes[:2] + (r._version, None)
    out, da = nvdr.interpolate(a, r, tri.cuda(), rast_db=d, diff_attrs=idx)
    gda = torch.randn(da.shape, generator=g)
    ga, gr, gd = torch.autograd.grad([out, da], [a, r, d], [go.cuda(), gda.cuda()])
    oa, orr, od = oracle.interpolate_bwd(attr.numpy(), rast.cpu().numpy(), tri.numpy(), go.numpy(),
                                         rast_db=db.cpu().numpy(), diff_attrs=ids, grad_da=gda.numpy())
    _close(ga, oa, 1e-5, 'grad attr')
    _close(gr, orr, 1e-5, 'grad rast')
    _close(gd, od, 1e-5, 'grad db')
