"""The gradient of rast itself, which the fused interpolation backward leaves
out where nothing sees it: torch.autograd.grad of rast (alone, with the
positions), retain_grad with a second consumer, and hooks that read or block it
give what the separate passes give, for a uniform batch and for UnevenBatch."""
import pytest
import torch

from diffrp_amd import batch, nvdr
from tests.scenes import noisy_clip
from tests.test_gpu_batch import SMALL_RES, SMALL_S, _scene

pytestmark = pytest.mark.gpu


def _uniform(C, fused, monkeypatch):
    monkeypatch.setattr(nvdr, '_FUSED_C', tuple(range(1, 17)) if fused else ())
    pos, tri, _ = noisy_clip(4, 0.01, 72, seed=70, views=2)
    p, tri = pos.cuda().contiguous().requires_grad_(True), tri.cuda().int().contiguous()
    g = torch.Generator().manual_seed(71)
    a = torch.rand(p.shape[-2], C, generator=g).cuda().requires_grad_(True)
    rast, _ = nvdr.rasterize(nvdr.RasterizeCudaContext(), p, tri, (72, 104), grad_db=False)
    out, _ = nvdr.interpolate(a, rast, tri)
    img = nvdr.antialias(out, rast, p, tri)
    return p, a, rast, out, img


def _uneven(C, fused, monkeypatch):
    monkeypatch.setattr(batch, '_FUSED_C', (1, 2, 3, 4, 8, 16) if fused else ())
    pos, tri = _scene(SMALL_S, SMALL_RES, 0.02, 72)
    g = torch.Generator().manual_seed(73)
    ub = batch.UnevenBatch(nvdr.RasterizeCudaContext(), [t.cuda() for t in tri], [q.shape[0] for q in pos], SMALL_RES)
    p = torch.cat(pos).cuda().contiguous().requires_grad_(True)
    a = torch.rand(p.shape[0], C, generator=g).cuda().requires_grad_(True)
    rast, boxes = ub.rasterize(p)
    out = ub.interpolate(a, rast, boxes)
    return p, a, rast, out, ub.antialias(out, rast, p)


def _call(how, p, a, rast, out, img):
    g = torch.Generator().manual_seed(74)
    go = torch.randn(out.shape, generator=g).cuda()
    dw = torch.randn(rast.shape[:-1], generator=g).cuda()
    loss = (out * go).sum()
    if how == 'grad rast':
        return torch.autograd.grad(loss, [rast])
    if how == 'grad rast and pos':
        return torch.autograd.grad(loss, [rast, p, a])
    if how == 'antialiased':
        return torch.autograd.grad((img * go).sum(), [rast, p])
    if how == 'retain, two consumers':
        rast.retain_grad()
        (loss + (rast[..., 2] * dw).sum()).backward()
        return rast.grad, p.grad, a.grad
    if how == 'hook blocks':
        rast.register_hook(lambda x: x * 0)
        loss.backward()
        assert p.grad.abs().max() == 0
        return p.grad, a.grad
    seen = []
    rast.register_hook(lambda x: seen.append(x.clone()))
    loss.backward()
    return seen[0], p.grad, a.grad


@pytest.mark.parametrize('how', ['grad rast', 'grad rast and pos', 'antialiased', 'retain, two consumers',
                                 'hook blocks', 'hook reads'])
@pytest.mark.parametrize('C', [3, 8])
@pytest.mark.parametrize('scene', [_uniform, _uneven])
def test_gradient_of_rast(cuda, scene, C, how, monkeypatch):
    print(f'case: {scene.__name__} C={C} {how}', flush=True)
    want = _call(how, *scene(C, False, monkeypatch))
    got = _call(how, *scene(C, True, monkeypatch))
    assert len(got) == len(want)
    for x, y in zip(got, want):
        # the same kernels in the same order; two antialias or position gradients may be added in either order,
        # and the antialias sums its vertices with atomics
        scale = float(y.abs().max())
        if how == 'antialiased':
            assert float((x - y).abs().max()) <= 1e-5 * scale and scale > 0
        else:
            assert torch.equal(x, y)
            assert how == 'hook blocks' or scale > 0
