"""Calls whose work does not fit one launch's threads (2^32 in a dimension):
an image of 16-byte quads read by four lanes a pixel past 2^30 pixels, narrow
coordinate images past the 16 x 16 blocks of one launch, and a per-channel
vertex gather past 2^32 channels; and one that just fits, which the padding of
a grid must not push past."""
import pytest
import torch

from diffrp_amd import batch, nvdr, texture

pytestmark = pytest.mark.gpu


@pytest.fixture
def room(cuda):
    def need(gib):
        torch.cuda.empty_cache()
        if torch.cuda.mem_get_info()[0] < gib << 30:
            pytest.skip(f'needs {gib} GiB of device memory')
    yield need
    torch.cuda.empty_cache()


def test_interpolate_past_2_30_pixels(cuda, room):
    room(80)
    n, H, W, C = 65, 4096, 4096, 12
    print(f'case: interpolate {n} x {H} x {W} x {C}', flush=True)
    attr = torch.rand(5, C, generator=torch.Generator().manual_seed(90)).cuda()
    tri = torch.tensor([[0, 1, 2], [2, 3, 4]], dtype=torch.int32).cuda()
    rast = torch.zeros(n, H, W, 4, device='cuda')
    at = torch.tensor([0, 1, 2 ** 29 - 1, 2 ** 29, 2 ** 29 + 77, 2 ** 30 - 1, 2 ** 30, 2 ** 30 + 5, n * H * W - 1])
    frag = torch.rand(len(at), 4, generator=torch.Generator().manual_seed(91)) * 0.5
    frag[:, 3] = torch.arange(len(at)) % 2 + 1
    rast.view(-1, 4)[at.cuda()] = frag.cuda()
    out, _ = nvdr.interpolate(attr, rast, tri)
    del rast
    want, _ = nvdr.interpolate(attr, frag.cuda().view(1, 1, -1, 4), tri)
    assert torch.equal(out.view(-1, C)[at.cuda()], want.view(-1, C))
    assert sum(int(torch.count_nonzero(o)) for o in out) == int(torch.count_nonzero(want))


def test_narrow_coordinate_image_past_one_launch(cuda, room):
    room(100)
    rows, width = 140_000_000, 17  # two 16 x 16 blocks a row of blocks: 17.5M blocks
    print(f'case: sample2d {rows} x {width}', flush=True)
    tex = torch.rand(4, 4, 1, generator=torch.Generator().manual_seed(92)).cuda().requires_grad_(True)
    uv = torch.full((1, rows, width, 2), 0.125, device='cuda')
    flat = uv.view(-1, 2)
    at = torch.tensor([0, 2 ** 31 - 1, 2 ** 31, 2 ** 31 + 9, rows * width - 1]).cuda()
    flat[at] = torch.tensor([[0.375, 0.125], [0.625, 0.375], [0.875, 0.625], [0.125, 0.875], [0.625, 0.875]]).cuda()
    uv.requires_grad_(True)
    out = texture.sample2d(tex, uv, mode='nearest')
    t = tex.detach().view(4, 4)
    assert torch.equal(out.view(-1)[at], torch.stack([t[3, 1], t[2, 2], t[1, 3], t[0, 0], t[0, 2]]))
    go = torch.zeros_like(out)
    go.view(-1)[at] = torch.tensor([1.0, 2.0, 4.0, 8.0, 16.0], device='cuda')
    gt, guv = torch.autograd.grad(out, [tex, uv], go)
    want = torch.zeros(4, 4)
    for (r, c), x in zip([(3, 1), (2, 2), (1, 3), (0, 0), (0, 2)], [1, 2, 4, 8, 16]):
        want[r, c] = x
    assert torch.equal(gt.cpu().view(4, 4), want)
    assert int(torch.count_nonzero(guv)) == 0


def test_vertex_gather_past_one_launch(cuda, room):
    room(140)
    V, C = 1_440_000_000, 3  # 4.3e9 channels: 16.9M blocks
    print(f'case: interpolate backward V={V} C={C}', flush=True)
    tri = torch.tensor([[0, 1, V - 1], [V - 1, V - 2, 1]], dtype=torch.int32).cuda()
    corners = torch.tensor([0, 1, V - 2, V - 1]).cuda()
    xy = torch.tensor([[-0.8, -0.7, 0, 1.0], [0.9, -0.6, 0, 1.0], [0.7, 0.8, 0, 1.0], [-0.6, 0.9, 0, 1.0]]).cuda()
    va = torch.rand(4, C, generator=torch.Generator().manual_seed(93)).cuda()
    go = torch.randn(1, 32, 32, C, generator=torch.Generator().manual_seed(94)).cuda()

    def grads(pos, attr, tri):
        pos.requires_grad_(True)
        attr.requires_grad_(True)
        rast, _ = nvdr.rasterize(nvdr.RasterizeCudaContext(), pos, tri, (32, 32), grad_db=False)
        out, _ = nvdr.interpolate(attr, rast, tri)
        return torch.autograd.grad(out, [pos, attr], go)

    wp, wa = grads(xy.clone(), va.clone(), torch.tensor([[0, 1, 3], [3, 2, 1]], dtype=torch.int32).cuda())
    pos, attr = torch.zeros(V, 4, device='cuda'), torch.zeros(V, C, device='cuda')
    pos[corners], attr[corners] = xy, va
    gp, ga = grads(pos, attr, tri)
    del pos, attr
    assert torch.equal(gp[corners], wp) and torch.equal(ga[corners], wa) and float(wa.abs().max()) > 0
    for g, w in ((gp, wp), (ga, wa)):  # (in parts: the count's temporary is an image of the tensor)
        assert sum(int(torch.count_nonzero(x)) for x in g.split(1 << 28)) == int(torch.count_nonzero(w))


def test_uneven_batch_just_below_one_launch(cuda, room):
    room(150)
    # 16 x 16 tiles: 15 times 2^20, 2^20 - 1024 and 1000, 24 short of 2^24
    res = [(16384, 16384)] * 15 + [(16368, 16384), (16, 16000)]
    print('case: uneven batch of 2^24 - 24 tiles', flush=True)
    xy = torch.tensor([[-0.5, -0.5, 0.25, 1.0], [0.5, -0.5, 0.25, 1.0], [0.0, 0.75, 0.25, 1.0]]).cuda()
    small = xy * torch.tensor([2.0 ** -9, 2.0 ** -9, 1.0, 1.0], device='cuda')  # some 32 pixels across
    pos = torch.cat([small] * 16 + [xy])
    tri = torch.tensor([[0, 1, 2]], dtype=torch.int32).cuda()
    ctx = nvdr.RasterizeCudaContext(tile=(16, 16), bin_capacity=32)
    ub = batch.UnevenBatch(ctx, [tri] * 17, [3] * 17, res)
    poison = torch.full((ub.n_pix, 4), float('nan'), device='cuda')
    del poison  # (what rasterize does not write stays NaN)
    rast, _ = ub.rasterize(pos)
    first, last = rast[:16384 * 16384], rast[-16 * 16000:]
    for part, p, (h, w), i in ((first, small, res[0], 0), (last, xy, res[-1], 16)):
        want, _ = nvdr.rasterize(nvdr.RasterizeCudaContext(), p, tri, (h, w), grad_db=False)
        want = want.view(-1, 4)
        covered = want[:, 3] > 0
        assert int(covered.sum()) > 100
        assert torch.equal(part[:, :3], want[:, :3]) and torch.equal(part[:, 3], want[:, 3] * (i + 1))
        del want, covered
    assert not any(bool(torch.isnan(x).any()) for x in rast.split(1 << 27))
