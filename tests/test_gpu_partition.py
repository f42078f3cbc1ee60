"""The stencil partition of a layer: counted for few owners, sorted for many,
both against nonzero() per owner, with the fragments and indices that come with
it; and a session's images with and without the fragments path."""
import pytest
import torch

from diffrp_amd import deferred as dd, nvdr
from diffrp_amd.camera import PerspectiveCamera
from diffrp_amd.geometry import icosphere

pytestmark = pytest.mark.gpu


def _layer(H, W, F, seed):
    """Random ids (encoded as floats, some past F) with runs, as in an image."""
    g = torch.Generator().manual_seed(seed)
    ids = torch.randint(0, F + 3, (H * W,), generator=g)
    ids = torch.where(torch.rand(H * W, generator=g) < 0.6, ids.roll(1), ids).float()
    rast = torch.cat([torch.rand(H * W, 3, generator=g), ids[:, None]], 1)
    return rast.view(1, H, W, 4).cuda()


@pytest.mark.parametrize('H,W', [(1, 1), (7, 13), (64, 32), (33, 2049), (500, 513)])
@pytest.mark.parametrize('n_owner', [0, 1, 5, 63, 1023, 1024, 3000])
def test_partition_fragments(cuda, H, W, n_owner):
    F = 400
    rast = _layer(H, W, F, H + n_owner)
    g = torch.Generator().manual_seed(n_owner)
    st = torch.cat([torch.zeros(1), torch.randint(-1, n_owner + 2, (F,), generator=g).float()]).int().cuda()
    print(f'case: partition {H}x{W} owners {n_owner}', flush=True)
    order, runs, layer = dd._partition(rast, st, n_owner, True)
    order2, runs2 = dd.stencil_partition(rast, st, n_owner)
    ids = rast[..., 3].reshape(-1).long()
    owner = torch.where(ids <= F, st[ids.clamp(max=F)].long(), 0)
    owner = torch.where((owner < 0) | (owner > n_owner), 0, owner)
    want = torch.sort(owner, stable=True)[1]
    assert torch.equal(order.long(), want) and torch.equal(order2, order) and runs == runs2
    count = torch.bincount(owner, minlength=n_owner + 1)
    end = torch.cumsum(count, 0)
    for k, (c, e) in enumerate(zip(count.tolist(), end.tolist())):
        assert tuple(runs[k]) == ((e - c, e) if c else (0, 0)), k
    assert torch.equal(layer.frag[:H * W], rast.view(-1, 4)[want]) and not layer.frag[H * W:].any()
    assert torch.equal(layer.rows, want // W) and torch.equal(layer.cols, want % W)


class _NoNormal(dd.SurfaceMaterial):
    def shade(self, su, si):
        return dd.SurfaceOutputStandard(albedo=si.color[..., :3], emission=si.color[..., 1:4])


def _images(grad, empty):
    v, f = icosphere(3)
    v, f = torch.as_tensor(v).float().cuda(), torch.as_tensor(f).int().cuda()
    g = torch.Generator(device='cuda').manual_seed(5)
    scene = dd.Scene()
    for i, off in enumerate([(-0.4, 0.0), (0.4, 0.1), (50.0, 0.0) if empty else (0.0, 0.5), (0.0, -0.4)]):
        M = torch.eye(4, device='cuda')
        M[0, 0] = M[1, 1] = M[2, 2] = 0.5
        M[0, 3], M[1, 3] = off
        verts = v.clone().requires_grad_(grad)
        mat = _NoNormal() if i % 2 else dd.DefaultMaterial()
        scene.add_mesh_object(dd.MeshObject(mat, verts, f, v.clone(), M,
                                            color=torch.rand(len(v), 4, generator=g, device='cuda')))
    cam = PerspectiveCamera.looking_at_origin_from([1.0, 0.8, 2.5], h=301, w=157)
    rp = dd.SurfaceDeferredRenderSession(scene, cam)
    return [rp.albedo(), rp.emission(), rp.false_color_camera_space_normal(), rp.depth(), rp.world_position()]


@pytest.mark.parametrize('empty', [False, True])
def test_session_with_and_without_gradients(cuda, empty):
    for a, b in zip(_images(False, empty), _images(True, empty)):
        assert torch.equal(a, b.detach())
