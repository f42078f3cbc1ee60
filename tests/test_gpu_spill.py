"""
Spill lists with some bins full and others not: a tile whose bin is full must
see the triangles that met a full bin, a tile with room must not lose any, and
every tile must see the triangles too large to bin.  A dense blob in one corner
over sparse triangles elsewhere, with and without screen-filling triangles, bit
for bit against the oracle for every tile shape, whole and peeled.
"""
import numpy as np
import pytest
import torch

import oracle
from diffrp_amd import nvdr

pytestmark = pytest.mark.gpu

RES = (150, 260)


def _soup(large, seed):
    g = torch.Generator().manual_seed(seed)

    def tris(n, lo, hi, size, z):
        c = torch.rand(n, 1, 2, generator=g) * (torch.tensor(hi) - torch.tensor(lo)) + torch.tensor(lo)
        xy = c + size * (torch.rand(n, 3, 2, generator=g) - 0.5)
        return torch.cat([xy, z + 0.2 * torch.rand(n, 3, 1, generator=g), torch.ones(n, 3, 1)], -1)
    parts = [tris(3000, (-0.9, -0.9), (-0.5, -0.4), 0.15, 0.1), tris(400, (-1.0, -1.0), (1.0, 1.0), 0.2, 0.0)]
    if large:
        parts.append(tris(3, (-0.2, -0.2), (0.2, 0.2), 8.0, 0.05))
    p = torch.cat(parts)
    p = p[torch.randperm(len(p), generator=g)]
    return p.reshape(-1, 4).contiguous(), torch.arange(3 * len(p), dtype=torch.int32).reshape(-1, 3)


@pytest.mark.parametrize('large', [False, True])
@pytest.mark.parametrize('tile', [(8, 8), (16, 8), (16, 16), (32, 8)])
@pytest.mark.parametrize('cap', [16, 64])
def test_partly_full_bins(cuda, large, tile, cap):
    pos, tri = _soup(large, 5)
    ctx = nvdr.RasterizeCudaContext(tile=tile, bin_capacity=cap)
    prev = None
    with nvdr.DepthPeeler(ctx, pos.cuda(), tri.cuda(), RES, grad_db=False) as dp:
        for layer in range(3):
            r = dp.rasterize_next_layer()[0].cpu().numpy()
            o = oracle.rasterize(pos.numpy(), tri.numpy(), RES, prev=prev)
            assert np.array_equal(r.view(np.uint32), np.ascontiguousarray(o, np.float32).view(np.uint32)), layer
            assert (o[..., 3] > 0).any()
            prev = o
