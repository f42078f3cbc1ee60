"""A material may replace or change its interpolator's fragments and pixels:
the session gives what it gives with every object's fragments gathered on their
own (the path that keeps a gradient through rast), values and gradients."""
import pytest
import torch

from diffrp_amd import deferred as dd
from diffrp_amd.camera import PerspectiveCamera
from diffrp_amd.geometry import noisy_icosphere

pytestmark = pytest.mark.gpu


class _Plain(dd.SurfaceMaterial):
    def shade(self, su, si):
        return dd.SurfaceOutputStandard(albedo=si.color[..., :3], alpha=si.uv[..., :1])


class _Swapped(_Plain):
    def shade(self, su, si):  # u and v exchanged, in a new tensor
        si.interpolator.vi_data = si.interpolator.vi_data[:, [1, 0, 2, 3]].contiguous()
        return super().shade(su, si)


class _InPlace(_Plain):
    def shade(self, su, si):
        si.interpolator.vi_data[:, :2].mul_(0.5)
        return super().shade(su, si)


class _Cutout(_Plain):
    def shade(self, su, si):  # every other fragment discarded
        ip = si.interpolator
        ip.vi_data, ip.indices = ip.vi_data[::2].contiguous(), tuple(x[::2] for x in ip.indices)
        return super().shade(su, si)


class _Moved(_Plain):
    def shade(self, su, si):  # drawn at the object's own pixels in reverse order (each once: no pixel is written twice)
        si.interpolator.indices = tuple(x.flip(0) for x in si.interpolator.indices)
        return super().shade(su, si)


def _scene(materials, grad):
    scene = dd.Scene()
    leaves = []
    for i, m in enumerate(materials):
        v, f = noisy_icosphere(3, 0.5, 0.01, seed=20 + i)
        color = torch.rand(len(v), 4, generator=torch.Generator().manual_seed(30 + i)).cuda().requires_grad_(grad)
        M = torch.eye(4, device='cuda')
        M[0, 3] = 0.45 * (i - 1)
        leaves.append(color)
        scene.add_mesh_object(dd.MeshObject(m(), v.cuda(), f.cuda(), normals='smooth', M=M, color=color,
                                            uv=torch.rand(len(v), 2, generator=torch.Generator().manual_seed(i)).cuda()))
    return scene, leaves


def _images(scene, leaves, grad):
    rp = dd.SurfaceDeferredRenderSession(scene, PerspectiveCamera(h=144, w=120), opaque_only=False,
                                         options=dd.SurfaceDeferredRenderSessionOptions(max_layers=2))
    img, normal, depth = rp.albedo(), rp.world_space_normal(), rp.depth()
    if not grad:
        return [img, normal, depth]
    return [img.detach(), normal, depth] + list(torch.autograd.grad((img ** 2).sum(), leaves))


@pytest.mark.parametrize('grad', [False, True])
@pytest.mark.parametrize('materials', [(_Plain, _Swapped, _Plain), (_Plain, _InPlace, _InPlace),
                                       (_Cutout, _Plain, _Cutout), (_Plain, _Moved, _Plain), (_Plain, _Plain, _Plain)])
def test_materials_may_change_their_fragments(cuda, materials, grad, monkeypatch):
    scene, leaves = _scene(materials, grad)  # once: smooth normals are summed by atomics
    got = _images(scene, leaves, grad)
    partition = dd._partition
    monkeypatch.setattr(dd, '_partition', lambda rast, st, n, fragments: partition(rast, st, n, False))
    want = _images(scene, leaves, grad)
    for i, (x, y) in enumerate(zip(got, want)):
        assert float(y.abs().max()) > 0
        if i < 3:
            assert torch.equal(x, y)
        else:  # float atomics of the same terms in any order
            assert float((x - y).abs().max()) <= 1e-5 * float(y.abs().max())
