"""The vertex gather of large meshes (a thread per vertex) against the separate
passes' gathers, bit for bit: the same sums in the same order.  A sheet of 270k
vertices with a vertex of many corners, a hidden half and one image."""
import pytest
import torch

from diffrp_amd import nvdr

pytestmark = pytest.mark.gpu


def _sheet(n):
    g = torch.Generator().manual_seed(n)
    y, x = torch.meshgrid(torch.linspace(-0.95, 0.95, n), torch.linspace(-0.95, 0.95, n), indexing='ij')
    z = torch.where(x > 0, 0.5, -0.2) + 0.01 * torch.rand(n, n, generator=g)
    pos = torch.stack([x, y, z, torch.ones(n, n)], -1).view(-1, 4)
    pos[:, :2] += 0.4 / n * torch.randn(n * n, 2, generator=g)
    i = torch.arange(n * n).view(n, n)
    a, b, c, d = i[:-1, :-1].reshape(-1), i[:-1, 1:].reshape(-1), i[1:, :-1].reshape(-1), i[1:, 1:].reshape(-1)
    tri = torch.cat([torch.stack([a, b, c], 1), torch.stack([d, c, b], 1)])
    cover = torch.tensor([[0.0, -1.0, 0.0, 1.0], [1.0, -1.0, 0.0, 1.0], [1.0, 1.0, 0.0, 1.0]])  # hides part of x > 0
    fan = torch.stack([torch.full((30,), n * n + 3), torch.arange(30) * 40, torch.arange(30) * 40 + 25], 1)
    pos = torch.cat([pos, cover, torch.tensor([[0.0, -0.99, -0.5, 1.0]])])
    tri = torch.cat([tri, n * n + torch.arange(3)[None], fan])
    return pos.contiguous(), tri.int().contiguous(), g


@pytest.mark.parametrize('C', [4, 8, 12, 16])
def test_large_mesh_gather_equals_the_separate_passes(cuda, C):
    pos, tri, g = _sheet(520)
    res = (300, 411)
    attr = torch.rand(pos.shape[0], C, generator=g)
    go = torch.randn(1, *res, C, generator=g)
    print(f'case: large mesh gather C={C}', flush=True)
    t = tri.cuda()
    got = []
    for fused in (nvdr._FUSED_C, ()):
        saved, nvdr._FUSED_C = nvdr._FUSED_C, fused
        try:
            p, a = pos.cuda().requires_grad_(True), attr.cuda().requires_grad_(True)
            rast, _ = nvdr.rasterize(nvdr.RasterizeCudaContext(), p, t, res, grad_db=False)
            out, _ = nvdr.interpolate(a, rast, t)
            poison = [torch.full((1 << k,), float('nan'), device='cuda') for k in range(16, 25)]
            del poison
            got.append(torch.autograd.grad(out, [p, a], go.cuda()))
        finally:
            nvdr._FUSED_C = saved
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    assert got[0][0].abs().sum() > 0 and torch.isfinite(got[0][1]).all()
