"""render_layers with a shade that writes to the buffer it returned: each layer
is composited from what the buffer held then, forward and backward, as by the
torch operators."""
import pytest
import torch

from diffrp_amd import layered, nvdr
from tests.scenes import noisy_clip

pytestmark = pytest.mark.gpu


def _render(step, recompute, monkeypatch):
    monkeypatch.setattr(layered, '_compose', step)
    pos, tri, _ = noisy_clip(3, 0.01, 48, seed=80)
    p, tri = pos.cuda().contiguous().requires_grad_(True), tri.cuda().int().contiguous()
    a = torch.rand(p.shape[0], 4, generator=torch.Generator().manual_seed(81)).cuda().requires_grad_(True)
    last = []

    def shade(g, rast):
        rgba = g * 0.75
        if last:
            with torch.no_grad():
                last.pop().mul_(0.0)  # the layer before is composited; its buffer is free again
        last.append(rgba.detach())    # (the same memory)
        return rgba

    img = layered.render_layers(nvdr.RasterizeCudaContext(), p, tri, a, (48, 48), 3, shade, recompute=recompute)
    (img ** 2).sum().backward()
    return img.detach(), p.grad, a.grad


@pytest.mark.parametrize('recompute', [False, True])
def test_shade_may_reuse_its_buffer(cuda, recompute, monkeypatch):
    want = _render(layered._blend, recompute, monkeypatch)
    monkeypatch.undo()
    got = _render(layered._compose, recompute, monkeypatch)
    assert torch.equal(got[0], want[0]) and float(want[0].abs().max()) > 0
    for x, y in zip(got[1:], want[1:]):
        # the same float32 sums in another order (three products a pixel, atomics in the antialias)
        assert float((x - y).abs().max()) <= 1e-5 * float(y.abs().max())
        assert float(y.abs().max()) > 0
