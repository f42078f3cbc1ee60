"""
Texture gradients of image-shaped samples (the 16 x 16 blocks of the 2-D
backward) against the oracle's grid_sample in float64: rows narrower than, equal
to and past a block, footprints inside and beyond the block's LDS box, every
sample on one texel, and masked backgrounds.

Tolerance: a texel's sum of m float32 contributions is off by at most
m 2^-24 of the sum of their magnitudes, and a bilinear weight by at most
8 max(H, W) 2^-23 (the float32 source index), so m max|g| times that again.
"""
import pytest
import torch

from oracle import glue
from diffrp_amd import texture

pytestmark = pytest.mark.gpu


def _uv(kind, n, h, w, g):
    """Coordinates of n images of h x w samples."""
    if kind == 'point':
        return torch.full((n, h, w, 2), 0.37)
    y, x = torch.meshgrid(torch.arange(h) / max(h, 2), torch.arange(w) / max(w, 2), indexing='ij')
    base = torch.stack([x, y], -1).float().expand(n, h, w, 2)
    scale = 0.2 if kind == 'magnified' else 1.0
    uv = base * scale + 0.05 + 0.002 * torch.rand(n, h, w, 2, generator=g)
    if kind == 'seam':  # half of the samples jump across the texture
        uv = torch.where((torch.arange(w) % 7 < 3)[:, None], 1.0 - uv, uv)
    return uv


@pytest.mark.parametrize('shape', [(1, 5, 15), (2, 16, 16), (1, 37, 17), (3, 70, 250)])
@pytest.mark.parametrize('kind', ['magnified', 'plain', 'seam', 'point'])
@pytest.mark.parametrize('C,mode', [(1, 'bilinear'), (3, 'bilinear'), (7, 'bilinear'), (4, 'nearest'), (2, 'bicubic')])
def test_texture_gradient_of_image_samples(cuda, shape, kind, C, mode):
    g = torch.Generator().manual_seed(hash_of(shape, kind, C))
    H, W = 61, 83
    tex = torch.rand(H, W, C, generator=g)
    uv = _uv(kind, *shape, g)
    if mode == 'nearest':  # texel centres: no rounding ties
        size = torch.tensor([W, H])
        uv = (torch.floor(uv * size).clamp(min=0) + 0.5) / size
    go = torch.randn(*shape, C, generator=g)
    go[:, shape[1] // 2:, : shape[2] // 2] = 0.0  # a masked background
    t64 = tex.double().requires_grad_(True)
    u64 = uv.double().requires_grad_(True)
    (glue.sample2d(t64, u64, 'reflection', mode) * go.double()).sum().backward()
    ta = tex.double().requires_grad_(True)
    (glue.sample2d(ta, uv.double(), 'reflection', mode) * go.double().abs()).sum().backward()
    t, u = tex.cuda().requires_grad_(True), uv.cuda().requires_grad_(True)
    (texture.sample2d(t, u, 'reflection', mode) * go.cuda()).sum().backward()
    m = 16 * shape[0] * shape[1] * shape[2]
    ew = 8 * max(H, W) * 2.0 ** -23
    per_texel = shape[0] * shape[1] * shape[2] if kind == 'point' else 4 * max(1, m // (H * W))
    tol = m * 2.0 ** -24 * (ta.grad.abs() + 1) + ew * per_texel * float(go.abs().max())
    assert bool(((t.grad.cpu().double() - t64.grad).abs() <= tol).all())
    if mode == 'bilinear':
        # the coordinate gradient is size * (difference of texels) * g, summed over the channels
        bound = 2 * max(H, W) * C * float(go.abs().max()) * (16 * 2.0 ** -23 + 2 * ew)
        # (it jumps where the source index crosses a texel centre or a reflected border: a float32
        # index within its own rounding of such a place may lie on either side)
        src = uv.double() * torch.tensor([W, H]) - 0.5
        sure = ((src - src.round()).abs() > max(H, W) * 2.0 ** -20).all(-1, keepdim=True)
        assert float(((u.grad.cpu().double() - u64.grad).abs() * sure).max()) <= bound
        assert float(sure.double().mean()) > 0.9


def hash_of(shape, kind, C):
    return sum(shape) * 31 + len(kind) * 7 + C
