"""The attribute backward of a large mesh in a small image, for channel counts
and derivative gradients that may go either by tile passes or by per-pixel
atomics: both routes give the same sums, and the rule takes the atomics only
where pixels are few beside triangles."""
import pytest
import torch

from diffrp_amd import nvdr
from tests.scenes import noisy_clip

pytestmark = pytest.mark.gpu


def _grads(p, t, attr, res, C, nd, position, route, monkeypatch):
    chosen = []
    rule = nvdr._pixel_atomics

    def spy(*a):
        chosen.append(rule(*a) if route is None else route)
        return chosen[-1]

    monkeypatch.setattr(nvdr, '_pixel_atomics', spy)
    pos, a = p.clone().requires_grad_(position), attr.clone().requires_grad_(True)
    rast, db = nvdr.rasterize(nvdr.RasterizeCudaContext(), pos, t, res)
    out, da = nvdr.interpolate(a, rast, t, *((db, 'all') if nd else ()))
    g = torch.Generator().manual_seed(C)
    ys = [out, da] if nd else [out]
    gs = [torch.randn(y.shape, generator=g).cuda() for y in ys]
    grads = torch.autograd.grad(ys, [a, pos] if position else [a], gs)
    monkeypatch.undo()
    return grads, chosen


@pytest.mark.parametrize('res,few', [((12, 40), True), ((300, 300), False)])
@pytest.mark.parametrize('C,nd', [(5, False), (12, False), (24, False), (3, True), (8, True)])
@pytest.mark.parametrize('views,position', [(1, False), (3, False), (1, True)])
def test_both_routes_agree(cuda, res, few, C, nd, views, position, monkeypatch):
    pos, tri, _ = noisy_clip(6, 0.002, res[0], seed=51, views=views)  # 81,920 triangles
    p, t = (pos[0] if views == 1 else pos).cuda().contiguous(), tri.cuda().int().contiguous()
    attr = torch.rand(p.shape[-2], C, generator=torch.Generator().manual_seed(52)).cuda()
    args = p, t, attr, res, C, nd, position
    print(f'case: {views} views {res} C={C} derivatives={nd} position={position}', flush=True)
    tiles, _ = _grads(*args, False, monkeypatch)
    atomics, _ = _grads(*args, True, monkeypatch)
    got, chosen = _grads(*args, None, monkeypatch)
    fused = position and not nd and C <= 16
    assert chosen == ([] if fused else [few])
    for x, y, z in zip(tiles, atomics, got):
        scale = float(x.abs().max())
        assert scale > 0
        # the same float32 terms, at most a few dozen to a sum, in another order (positions: a chain over grad_rast)
        assert float((y - x).abs().max()) <= 1e-5 * scale and float((z - x).abs().max()) <= 1e-5 * scale


def test_compiled_counts_keep_the_passes(cuda, monkeypatch):
    pos, tri, _ = noisy_clip(6, 0.002, 24, seed=53)
    p, t = pos.cuda().contiguous(), tri.cuda().int().contiguous()
    for C in (1, 2, 3, 4, 8, 16):
        attr = torch.rand(p.shape[-2], C, generator=torch.Generator().manual_seed(54)).cuda()
        first, chosen = _grads(p, t, attr, (24, 40), C, False, False, None, monkeypatch)
        again, _ = _grads(p, t, attr, (24, 40), C, False, False, None, monkeypatch)
        assert chosen == [] and torch.equal(first[0], again[0])
