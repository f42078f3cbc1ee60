"""The fused compositing step past the pixels of one launch: the library refuses
the size before it launches anything, and layers of it go through the operators
(tensors without memory: only the route is taken)."""
import os

import torch

from diffrp_amd import _lib, build_ext, layered


def test_library_refuses_more_than_one_launch():
    if not os.path.exists(build_ext.LIB_PATH):
        build_ext.build()
    L = _lib.lib()
    for n in ((1 << 31) + 1, 1 << 32, 1 << 38, -1):
        assert L.drp_compose_layer_fwd(None, 16, 16, None, None, n, 16, 16) < 0
        assert b'out of range' in L.drp_last_error()
        assert L.drp_compose_layer_bwd(None, 16, 16, None, n, None, None, 16, None) < 0
        assert b'out of range' in L.drp_last_error()


def test_larger_layers_go_through_the_operators():
    rgba = torch.empty(1, (1 << 16) + 1, 1 << 15, 4, device='meta')
    out, trans = layered._compose(rgba, torch.empty_like(rgba), None, None)
    assert out.shape[-1] == 3 and trans.shape[-1] == 1 and out.device.type == 'meta'
