"""Backward passes with too little memory for the scratch of the route they
would take: the fused pass gives way to the separate ones, and channel counts
and derivative gradients without a need for the tile passes to the per-pixel
atomics, with the same gradients; a count that always has the passes raises."""
import pytest
import torch

from diffrp_amd import batch, nvdr
from tests.scenes import noisy_clip

pytestmark = pytest.mark.gpu


def _cap(monkeypatch, mib):
    """Allocations of scratch beyond mib MiB fail as the allocator's do."""
    new = nvdr._new_scratch

    def limited(nbytes, device):
        if nbytes > mib << 20:
            raise torch.OutOfMemoryError(f'no room for {nbytes} bytes')
        return new(nbytes, device)

    monkeypatch.setattr(nvdr, '_new_scratch', limited)


def _calls(monkeypatch, lib, names):
    seen = []
    for name in names:
        fn = getattr(lib, name)
        monkeypatch.setattr(lib, name, lambda *a, fn=fn, name=name: seen.append((name, a)) or fn(*a))
    return seen


# 8 views of 512^2.  Scratch in MiB: 5 channels 235 fused with the positions', 137 in the passes of its own, then 107
# in the rasterize backward's; 16 channels 492 and 394; 2 channels with derivatives 73; the limit is on each.
@pytest.mark.parametrize('C,nd,position,mib,want', [
    (5, False, True, 230, ['drp_interpolate_bwd', 'drp_rasterize_bwd']),
    (16, False, True, 460, ['drp_interpolate_bwd', 'drp_rasterize_bwd']),
    (5, False, False, 100, ['drp_interpolate_bwd']),
    (24, False, False, 300, ['drp_interpolate_bwd']),
    (2, True, False, 60, ['drp_interpolate_bwd'])])
def test_gradients_without_room(cuda, C, nd, position, mib, want, monkeypatch):
    pos, tri, _ = noisy_clip(4, 0.005, 512, seed=31, views=8)
    p = pos.cuda().contiguous().requires_grad_(position)
    t = tri.cuda().int().contiguous()
    a = torch.rand(p.shape[1], C, generator=torch.Generator().manual_seed(32)).cuda().requires_grad_(True)
    rast, db = nvdr.rasterize(nvdr.RasterizeCudaContext(), p, t, (512, 512), grad_db=nd)
    out, da = nvdr.interpolate(a, rast, t, *((db, 'all') if nd else ()))
    ys = [out, da] if nd else [out]
    g = torch.Generator(device='cuda').manual_seed(33)
    gs = [torch.randn(y.shape, generator=g, device='cuda') for y in ys]
    xs = [a, p] if position else [a]
    print(f'case: C={C} derivatives={nd} position={position} {mib} MiB', flush=True)
    seen = _calls(monkeypatch, nvdr._lib.lib(), ['drp_interpolate_rasterize_bwd_to', 'drp_interpolate_bwd',
                                                 'drp_rasterize_bwd'])
    _cap(monkeypatch, mib)
    got = torch.autograd.grad(ys, xs, gs, retain_graph=True)
    assert [name for name, _ in seen] == want
    monkeypatch.undo()
    full = torch.autograd.grad(ys, xs, gs)
    for x, y in zip(got, full):
        scale = float(y.abs().max())
        # sums of up to some thousand float32 terms of either sign in another order: sqrt(4096) 2^-24 = 4e-6
        assert scale > 0 and float((x - y).abs().max()) <= 2e-5 * scale


def test_compiled_count_without_room_raises(cuda, monkeypatch):
    pos, tri, _ = noisy_clip(4, 0.005, 512, seed=34, views=8)
    p, t = pos.cuda().contiguous(), tri.cuda().int().contiguous()
    a = torch.rand(p.shape[1], 8, generator=torch.Generator().manual_seed(35)).cuda().requires_grad_(True)
    rast, _ = nvdr.rasterize(nvdr.RasterizeCudaContext(), p, t, (512, 512), grad_db=False)
    out, _ = nvdr.interpolate(a, rast, t)
    go = torch.ones_like(out)
    _cap(monkeypatch, 100)
    with pytest.raises(torch.OutOfMemoryError):
        torch.autograd.grad(out, a, go, retain_graph=True)
    monkeypatch.undo()
    assert float(torch.autograd.grad(out, a, go)[0].abs().max()) > 0


def test_uneven_batch_without_room(cuda, monkeypatch):
    pos, tri, _ = noisy_clip(4, 0.005, 512, seed=36, views=8)
    ub = batch.UnevenBatch(nvdr.RasterizeCudaContext(), [tri.cuda().int()] * 8, [pos.shape[1]] * 8, [(512, 512)] * 8)
    p = pos.view(-1, 4).cuda().contiguous().requires_grad_(True)
    a = torch.rand(p.shape[0], 16, generator=torch.Generator().manual_seed(37)).cuda().requires_grad_(True)
    rast, boxes = ub.rasterize(p)
    out = ub.interpolate(a, rast, boxes)
    go = torch.randn(out.shape, generator=torch.Generator(device='cuda').manual_seed(38), device='cuda')
    seen = _calls(monkeypatch, nvdr._lib.lib(), ['drp_batch_interpolate_rasterize_bwd_to', 'drp_batch_interpolate_bwd',
                                                 'drp_batch_rasterize_bwd'])
    _cap(monkeypatch, 460)
    got = torch.autograd.grad(out, [p, a], go, retain_graph=True)
    assert [name for name, _ in seen] == ['drp_batch_interpolate_bwd', 'drp_batch_rasterize_bwd']
    full = torch.autograd.grad(out, [p, a], go)
    assert all(torch.equal(x, y) for x, y in zip(got, full)) and float(full[0].abs().max()) > 0
