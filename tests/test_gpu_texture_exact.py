"""Texture gradients that float32 holds exactly, in any order of the sums: texel
indices and weights are short binary fractions and the output gradients small
integers, so the 2-D backward equals grid_sample in float64 to the last bit.
Image-shaped samples around the 16 x 16 blocks, and lists of points with one or
a few rows; footprints inside and beyond a block's LDS box, one texel for all
samples, reflected coordinates, masked backgrounds."""
import pytest
import torch

from oracle import glue
from diffrp_amd import texture

pytestmark = pytest.mark.gpu

W, H = 64, 32


def _index(kind, shape, steps, g):
    """Texel indices (x, y), multiples of 1 / steps, of samples [*shape]."""
    n, h, w = (1,) * (3 - len(shape)) + tuple(shape)
    if kind == 'point':
        at = torch.tensor([W // 3 + 0.5, H // 2 + 0.5]).expand(n, h, w, 2)
    else:
        y, x = torch.meshgrid(torch.arange(h) * (H / h), torch.arange(w) * (W / w), indexing='ij')
        at = torch.stack([x, y], -1).expand(n, h, w, 2)
        at = at * (0.15 if kind == 'magnified' else 1.3) + 2 * torch.rand(n, h, w, 2, generator=g) - 1.5
        if kind == 'seam':
            at = torch.where((torch.arange(w) % 7 < 3)[:, None], torch.tensor([W, H]) - at, at)
    return ((at * steps).round() / steps).reshape(*shape, 2)


@pytest.mark.parametrize('shape', [(1, 5, 15), (1, 16, 15), (2, 8, 16), (2, 7, 16), (1, 37, 17), (3, 70, 250), (1, 4000),
                                   (3, 1300), (16, 16), (15, 300), (2, 2, 2, 900)])
@pytest.mark.parametrize('kind', ['magnified', 'plain', 'seam', 'point'])
@pytest.mark.parametrize('C,mode', [(1, 'bilinear'), (3, 'bilinear'), (7, 'bilinear'), (4, 'nearest'), (2, 'bicubic')])
def test_texture_gradient_is_exact(cuda, shape, kind, C, mode):
    g = torch.Generator().manual_seed(sum(shape) * 31 + len(kind) * 7 + C)
    # bilinear: quarters, so weights in sixteenths; bicubic: halves, weights in 1/1024; nearest: texel centres
    steps, unit = {'bilinear': (4, 16), 'bicubic': (2, 1024), 'nearest': (1, 1)}[mode]
    if mode == 'nearest' and kind == 'point':
        kind = 'magnified'  # (the point is a tie)
    at = _index(kind, shape if len(shape) < 4 else (shape[0] * shape[1],) + shape[2:], steps, g).reshape(*shape, 2)
    uv = torch.stack([(at[..., 0] + 0.5) / W, 1 - (at[..., 1] + 0.5) / H], -1)
    assert uv.dtype == torch.float32
    tex = torch.randint(-3, 4, (H, W, C), generator=g).float()
    go = torch.randint(-1, 2, (*shape, C), generator=g).float()
    go[..., : shape[-1] * (3 if mode == 'bicubic' else 1) // 4, :] = 0.0  # a masked background
    sums = []
    for x in (go, go.abs()):
        t64 = tex.double().requires_grad_(True)
        u64 = uv.double()
        (glue.sample2d(t64, u64, 'reflection', mode) * x.double()).sum().backward()
        sums.append(t64.grad)
    want, terms = sums
    # every partial sum is a multiple of 1 / unit below 2^24 / unit (a bicubic weight's magnitude is at most
    # its absolute value's, and there are four signs to a sum: a factor of two covers them)
    assert 2 * float(go.abs().sum(tuple(range(len(shape)))).max()) * unit < 2 ** 24 or \
        4 * float(terms.abs().max()) * unit < 2 ** 24
    assert torch.equal(want * unit, (want * unit).round())
    t = tex.cuda().requires_grad_(True)
    (texture.sample2d(t, uv.cuda(), 'reflection', mode) * go.cuda()).sum().backward()
    assert float(want.abs().max()) > 0
    assert torch.equal(t.grad.cpu().double(), want)
