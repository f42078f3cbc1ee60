"""Antialias at the edges of its 64 x 8 pixel blocks.

The forward evaluates the pairs that reach into a block from the column to its
left and the row below a second time and keeps a list of blending pairs per
block for the backward.  On triangle soups (every edge a silhouette, so nearly
every pair of differing pixels blends) at image sizes around the block's, for
every compiled channel count and general ones: the image equals the float32
oracle's bit for bit; the colour gradient agrees to 1e-5 of its scale (at most
nine float32 terms per value) and the position gradient to 1e-4 of its scale
(float32 sums in another order, a few hundred terms per vertex); a second
backward, which evaluates the pairs anew, gives the same colour gradient bit
for bit.  An uneven batch of the same sizes gives the same images and
gradients as one call per item."""
import numpy as np
import pytest
import torch

import oracle
from diffrp_amd import batch, nvdr
from tests.scenes import random_soup

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (1, 64), (8, 64), (7, 63), (9, 65), (8, 1), (17, 130), (24, 129)]


def _rel(a, b, rtol, what):
    b = b.astype(np.float64)
    scale = max(np.abs(b).max(), 1e-30)
    err = np.abs(a.detach().cpu().numpy().astype(np.float64) - b).max() / scale
    assert err <= rtol, f'{what}: {err:.3e} > {rtol}'


@pytest.mark.parametrize('C', [1, 2, 3, 4, 5, 6, 7, 8, 9, 12, 16])
def test_blocks(cuda, C):
    pos, tri = random_soup(40, 3)
    pos2, _ = random_soup(40, 4)
    P = torch.stack([torch.as_tensor(pos), torch.as_tensor(pos2)]).float()
    T = torch.as_tensor(tri).int()
    g = torch.Generator().manual_seed(C)
    for H, W in SIZES:
        print(f'case: antialias blocks C={C} {H}x{W}', flush=True)
        rast, _ = nvdr.rasterize(nvdr.RasterizeCudaContext(), P.cuda(), T.cuda(), (H, W), grad_db=False)
        col = torch.rand(2, H, W, C, generator=g)
        go = torch.randn(2, H, W, C, generator=g)
        c, p = col.cuda().requires_grad_(True), P.cuda().requires_grad_(True)
        out = nvdr.antialias(c, rast, p, T.cuda())
        r = rast.cpu().numpy()
        want = oracle.antialias(col.numpy(), r, P.numpy(), T.numpy())
        np.testing.assert_array_equal(out.detach().cpu().numpy().view(np.uint32), want.view(np.uint32))
        gc, gp = torch.autograd.grad(out, [c, p], go.cuda(), retain_graph=True)
        oc, op = oracle.antialias_bwd(col.numpy(), r, P.numpy(), T.numpy(), go.numpy())
        _rel(gc, oc, 1e-5, f'{H}x{W} colour gradient')
        _rel(gp, op, 1e-4, f'{H}x{W} position gradient')
        gc2, gp2 = torch.autograd.grad(out, [c, p], go.cuda())
        assert torch.equal(gc2, gc)
        _rel(gp2, op, 1e-4, f'{H}x{W} position gradient, pairs evaluated anew')


@pytest.mark.parametrize('C', [3, 5, 8])
def test_uneven_batch_of_block_edges(cuda, C):
    soups = [random_soup(30, 10 + i) for i in range(len(SIZES))]
    pos = [torch.as_tensor(s[0]).float().cuda() for s in soups]
    tri = [torch.as_tensor(s[1]).int().cuda() for s in soups]
    ub = batch.UnevenBatch(nvdr.RasterizeCudaContext(), tri, [q.shape[0] for q in pos], SIZES)
    P = torch.cat(pos).contiguous().requires_grad_(True)
    g = torch.Generator(device='cuda').manual_seed(C)
    col = torch.rand(ub.n_pix, C, generator=g, device='cuda').requires_grad_(True)
    go = torch.randn(ub.n_pix, C, generator=g, device='cuda')
    print(f'case: antialias blocks, uneven batch C={C}', flush=True)
    rast, _ = ub.rasterize(P.detach())
    out = ub.antialias(col, rast, P)
    gc, gp = torch.autograd.grad(out, [col, P], go)
    a = v = 0
    for q, t, (H, W) in zip(pos, tri, SIZES):
        b, w = a + H * W, v + q.shape[0]
        ri, _ = nvdr.rasterize(nvdr.RasterizeCudaContext(), q, t, (H, W), grad_db=False)
        ci, qi = col[a:b].detach().view(1, H, W, C).requires_grad_(True), q.clone().requires_grad_(True)
        oi = nvdr.antialias(ci, ri, qi, t)
        gci, gqi = torch.autograd.grad(oi, [ci, qi], go[a:b].view(1, H, W, C))
        assert torch.equal(out[a:b], oi.view(-1, C))
        assert torch.equal(gc[a:b], gci.view(-1, C))
        _rel(gp[v:w], gqi.cpu().numpy(), 1e-5, f'{H}x{W} position gradient')
        a, v = b, w
