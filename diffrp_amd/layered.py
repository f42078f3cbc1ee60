"""
Depth-peeled layers composited front to back, with the option of recomputing
each layer in the backward pass instead of keeping its buffers.

diffrp's session peels up to ``max_layers`` layers (surface_deferred.py:240-266),
builds a G-buffer per layer (``gbuffer_collect``, :299-346), blends the shaded
layers (``compose_layers``, :348-395) and antialiases the result against the
first layer (``nvdr_antialias``, :758-775).  ``render_layers`` runs that chain
for one mesh with per-vertex attributes and a caller-provided shading
function.  With ``recompute=True`` each layer's rasterize + interpolate + shade
runs under ``torch.utils.checkpoint``: autograd keeps only the layer's inputs
(the previous layer's rast, 16 bytes per pixel) and re-runs the layer in the
backward pass, so the per-layer G-buffers (4 C bytes per pixel) and shaded
colours are never held for the whole graph.
"""
from typing import Callable, List, Optional, Tuple

import torch
import torch.utils.checkpoint as ckpt

from . import _lib, nvdr
from ._lib import check, ptr, stream_of


def count_covered(rast: torch.Tensor) -> torch.Tensor:
    """Covered pixels per image of rast [n, H, W, 4] as a device int32 [n]
    (no host synchronisation)."""
    if rast.dim() != 4 or rast.shape[-1] != 4 or rast.dtype != torch.float32 or not rast.is_contiguous():
        raise ValueError('rast must be a contiguous float32 [n, H, W, 4] tensor')
    n, H, W = rast.shape[0], rast.shape[1], rast.shape[2]
    counts = torch.empty(n, dtype=torch.int32, device=rast.device)
    check(_lib.lib().drp_count_covered(stream_of(rast), ptr(rast), n, H, W, ptr(counts)), 'count_covered')
    return counts


def peel_layers(glctx: 'nvdr.RasterizeCudaContext', pos: torch.Tensor, tri: torch.Tensor,
                resolution: Tuple[int, int], max_layers: int, ranges: Optional[torch.Tensor] = None,
                grad_db: bool = False) -> List[torch.Tensor]:
    """The layers of diffrp's peeling loop (``surface_deferred.py:258-266``):
    layer i is kept unless it is empty and i < max_layers - 1; the loop stops at
    the first such empty layer.  Emptiness is counted on the device
    (``count_covered``) and copied to pinned host memory; the host reads layer
    i's count only after layer i + 1 has been queued, so the GPU never waits for
    the host (the one speculative layer behind an empty one is dropped)."""
    layers: List[torch.Tensor] = []
    pending = None  # (rast, pinned counts or None, event)
    with nvdr.DepthPeeler(glctx, pos, tri, resolution, ranges, grad_db=grad_db) as dp:
        for i in range(max_layers):
            rast, _ = dp.rasterize_next_layer()
            host, ev = None, None
            if i < max_layers - 1:
                cnt = count_covered(rast)
                host = torch.empty(cnt.shape, dtype=cnt.dtype, pin_memory=True)
                host.copy_(cnt, non_blocking=True)
                ev = torch.cuda.Event()
                ev.record()
            if pending is not None:
                prast, phost, pev = pending
                pev.synchronize()
                if int(phost.sum()) == 0:
                    return layers
                layers.append(prast)
            pending = (rast, host, ev)
    prast, phost, pev = pending
    if phost is not None:
        pev.synchronize()
        if int(phost.sum()) == 0:
            return layers
    layers.append(prast)
    return layers


def _blend(rgba, rast, out, trans):
    """One compositing step with torch operators: (out, transmittance) behind the layer."""
    rgba = rgba * (rast[..., 3:4] > 0).to(rgba.dtype)
    rgb, a = rgba[..., :3], rgba[..., 3:4]
    if out is None:
        return rgb * a, 1.0 - a
    return out + trans * a * rgb, trans * (1.0 - a)


class _Compose(torch.autograd.Function):
    """``_blend`` as one kernel forward and one backward (``drp_compose.hip``), the same values bit for bit."""

    @staticmethod
    def forward(fctx, rgba, rast, out, trans):
        o = torch.empty(rast.shape[:3] + (3,), dtype=torch.float32, device=rgba.device)
        t = torch.empty(rast.shape[:3] + (1,), dtype=torch.float32, device=rgba.device)
        check(_lib.lib().drp_compose_layer_fwd(stream_of(rgba), ptr(rgba), ptr(rast), ptr(out), ptr(trans), t.numel(),
                                               ptr(o), ptr(t)), 'compose')
        fctx.save_for_backward(rgba, rast, out, trans)
        fctx.set_materialize_grads(False)
        return o, t

    @staticmethod
    def backward(fctx, go, gt):
        rgba, rast, out, trans = fctx.saved_tensors
        if go is None and gt is None:
            return None, None, None, None
        if torch.is_grad_enabled():  # a differentiable backward: through the operators
            given = [x for x in (rgba, out, trans) if x is not None and x.requires_grad]
            res = [(y, g) for y, g in zip(_blend(rgba, rast, out, trans), (go, gt)) if g is not None]
            got = iter(torch.autograd.grad([y for y, _ in res], given, [g for _, g in res], create_graph=True,
                                           allow_unused=True))
            ga, gb, gc = (next(got) if x is not None and x.requires_grad else None for x in (rgba, out, trans))
            return ga, None, gb, gc
        go = None if go is None else go.contiguous()
        gt = None if gt is None else gt.contiguous()
        grgba = torch.empty(rast.shape, dtype=torch.float32, device=rgba.device)
        gtrans = torch.empty_like(trans) if trans is not None else None
        check(_lib.lib().drp_compose_layer_bwd(stream_of(rgba), ptr(rgba), ptr(rast), ptr(trans), rast.numel() // 4,
                                               ptr(go), ptr(gt), ptr(grgba), ptr(gtrans)), 'compose backward')
        return grgba, None, go if out is not None else None, gtrans


_COMPOSE_PIXELS = 1 << 31  # pixels of one launch


def _compose(rgba, rast, out, trans):
    # the kernel takes plain float32 buffers; what shade returns otherwise (another type or shape, a
    # subclass, a forward-mode dual) goes through the operators
    if (type(rgba) is torch.Tensor and rgba.dtype == torch.float32 and rgba.shape == rast.shape
            and rgba.device == rast.device and rast.is_contiguous() and rast.numel() <= 4 * _COMPOSE_PIXELS
            and (out is None or (out.dtype == torch.float32 and out.is_contiguous() and trans.is_contiguous()))
            and torch.autograd.forward_ad._current_level < 0):
        # kept for the backward: a copy, as the operators keep (shade may write to its buffer again, and a
        # slice would hold the whole of a wider one)
        kept = torch.is_grad_enabled() and (rgba.requires_grad or (trans is not None and trans.requires_grad))
        if kept or not rgba.is_contiguous() or rgba.data_ptr() % 16:
            rgba = rgba.clone(memory_format=torch.contiguous_format)
        return _Compose.apply(rgba, rast, out, trans)
    return _blend(rgba, rast, out, trans)


def _layer(ctx, pos, tri, attr, resolution, prev, shade):
    rast, _ = nvdr._rasterize_impl(ctx, pos, tri, resolution, None, False, prev)
    g, _ = nvdr.interpolate(attr, rast, tri)
    return rast, shade(g, rast)


def render_layers(ctx: 'nvdr.RasterizeCudaContext', pos: torch.Tensor, tri: torch.Tensor, attr: torch.Tensor,
                  resolution: Tuple[int, int], n_layers: int,
                  shade: Callable[[torch.Tensor, torch.Tensor], torch.Tensor], recompute: bool = True,
                  antialias: bool = True):
    """RGB [1, H, W, 3] of ``n_layers`` peeled layers composited front to back
    (premultiplied 'over'), antialiased against the first layer.

    pos [V, 4] clip space, tri [F, 3] int32, attr [V, C]; shade(g, rast) maps a
    layer's interpolated attributes [1, H, W, C] to RGBA [1, H, W, 4]
    (straight alpha).  Differentiable w.r.t. pos and attr.
    """
    out = None
    trans = None
    prev = None
    first = None
    for k in range(n_layers):
        if recompute and torch.is_grad_enabled():
            rast, rgba = ckpt.checkpoint(_layer, ctx, pos, tri, attr, resolution, prev, shade, use_reentrant=False)
        else:
            rast, rgba = _layer(ctx, pos, tri, attr, resolution, prev, shade)
        if first is None:
            first = rast
        prev = rast.detach()
        out, trans = _compose(rgba, prev, out, trans)
    if antialias:
        out = nvdr.antialias(out.contiguous(), first, pos, tri)
    return out
