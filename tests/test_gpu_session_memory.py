"""What a session's interpolators hold: their objects' fragments and pixel
indices, at most twice that with the background between them, never the layer
of a mostly empty view."""
import pytest
import torch

from diffrp_amd import deferred as dd
from diffrp_amd.camera import PerspectiveCamera
from diffrp_amd.geometry import noisy_icosphere

pytestmark = pytest.mark.gpu


def _session(size, distance):
    scene = dd.Scene()
    for i in range(2):
        v, f = noisy_icosphere(3, 0.3, 0.01, seed=40 + i)
        M = torch.eye(4, device='cuda')
        M[0, 3] = 0.35 * (2 * i - 1)
        scene.add_mesh_object(dd.MeshObject(dd.DefaultMaterial(), v.cuda(), f.cuda(), M=M))
    return dd.SurfaceDeferredRenderSession(scene, PerspectiveCamera.looking_at_origin_from([0.0, 0.0, distance], h=size,
                                                                                           w=size))


@pytest.mark.parametrize('size,distance', [(512, 1.0), (512, 12.0), (257, 4.0), (64, 500.0)])
def test_interpolators_hold_their_objects_pixels(cuda, size, distance):
    rp = _session(size, distance)
    alpha = rp.albedo()[..., 3:]
    interps = [si.interpolator for mats in rp.layer_material() for si, _ in mats]
    pixels = sum(i.vi_data.shape[0] for i in interps)
    assert pixels == int((alpha > 0).sum())
    held = {}
    for i in interps:
        for t in (i.vi_data,) + tuple(i.indices):
            s = t.untyped_storage()
            held[s.data_ptr()] = s.nbytes()
        if i.run is not None:
            for t in (i.run.layer.frag, i.run.layer.rows, i.run.layer.cols):
                held[t.untyped_storage().data_ptr()] = t.untyped_storage().nbytes()
    # 16 bytes of fragment and 16 of row and column a pixel, and one padded row of fragments
    assert sum(held.values()) <= 2 * 32 * pixels + 16 * dd._FRAG_ROW + 8 * len(interps)
