"""The fused backward of a packed uneven batch at every channel count it takes,
against the two separate passes, over memory filled with NaN (its gradients are
written whole): small items, and a batch past 2^18 vertices (a thread per
vertex gathers both sums where the channels are whole quads) with an item that
no pixel sees and one without triangles."""
import pytest
import torch

from diffrp_amd import batch, nvdr
from diffrp_amd.geometry import noisy_icosphere
from tests.test_gpu_batch import SMALL_RES, SMALL_S, _scene

pytestmark = pytest.mark.gpu


def _poison():
    x = [torch.full((1 << k,), float('nan'), device='cuda') for k in range(8, 25)]
    del x


def _grads(pos, tri, res, C, antialias, fused, monkeypatch):
    monkeypatch.setattr(batch, '_FUSED_C', (1, 2, 3, 4, 8, 16) if fused else ())
    g = torch.Generator().manual_seed(60 + C)
    ub = batch.UnevenBatch(nvdr.RasterizeCudaContext(), [t.cuda() for t in tri], [p.shape[0] for p in pos], res)
    p = torch.cat(pos).cuda().contiguous().requires_grad_(True)
    a = torch.rand(p.shape[0], C, generator=g).cuda().requires_grad_(True)
    go = torch.randn(ub.n_pix, C, generator=g).cuda()
    rast, boxes = ub.rasterize(p)
    out = ub.interpolate(a, rast, boxes)
    if antialias:
        out = ub.antialias(out, rast, p)
    _poison()
    return torch.autograd.grad(out, [p, a], go)


@pytest.mark.parametrize('C', [1, 2, 3, 4, 8, 16])
@pytest.mark.parametrize('antialias', [False, True])
def test_fused_widths_equal_the_separate_passes(cuda, C, antialias, monkeypatch):
    print(f'case: 6 meshes s=2..5, C={C} antialias={antialias}', flush=True)
    pos, tri = _scene(SMALL_S, SMALL_RES, 0.02, 61)
    fp, fa = _grads(pos, tri, SMALL_RES, C, antialias, True, monkeypatch)
    sp, sa = _grads(pos, tri, SMALL_RES, C, antialias, False, monkeypatch)
    assert torch.equal(fa, sa) and float(sa.abs().max()) > 0 and float(sp.abs().max()) > 0
    if antialias:  # its position gradients are summed with float atomics
        assert float((fp - sp).abs().max()) <= 1e-5 * float(sp.abs().max())
    else:
        assert torch.equal(fp, sp)


def _clip(v, z):
    """Vertices around the origin, put at depth z with a perspective w."""
    w = z - v[:, 2:]
    return torch.cat([v[:, :2] * 2.0, (w - 1.0) * 1.01, w], 1)


@pytest.mark.parametrize('C', [1, 3, 4, 8, 16])
def test_large_batch_with_dead_items(cuda, C, monkeypatch):
    v, f = noisy_icosphere(7, 0.8, 0.01, seed=62)      # 163,842 vertices
    s, fs = noisy_icosphere(4, 0.8, 0.01, seed=63)
    pos = [_clip(v, 3.0), _clip(s, -3.0), _clip(s, 3.0), _clip(v, 4.0), s.new_ones(5, 4)]
    tri = [f, fs, fs, f, fs[:0]]                       # the second item lies behind the eye
    res = [(128, 160), (33, 47), (64, 64), (200, 96), (9, 9)]
    assert sum(p.shape[0] for p in pos) >= 1 << 18
    print(f'case: large uneven batch C={C}', flush=True)
    fp, fa = _grads(pos, tri, res, C, False, True, monkeypatch)
    sp, sa = _grads(pos, tri, res, C, False, False, monkeypatch)
    assert torch.equal(fp, sp) and torch.equal(fa, sa)
    at = [0]
    for p in pos:
        at.append(at[-1] + p.shape[0])
    for i, seen in enumerate([True, False, True, True, False]):
        assert bool((fa[at[i]:at[i + 1]] != 0).any()) == seen
