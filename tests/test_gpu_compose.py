"""
The fused compositing step of peeled layers against the torch operators it
stands for: the same values bit for bit, gradients to 1e-6 of their scale
(three products summed in another order), from contiguous and sliced RGBA, at
sizes around a block, NaN under the mask included; what the kernel does not
take (another dtype, a forward-mode dual, a differentiable backward) goes
through the operators.
"""
import pytest
import torch

from diffrp_amd import layered

pytestmark = pytest.mark.gpu


def _inputs(h, w, layers, wide, seed):
    g = torch.Generator().manual_seed(seed)
    rgba = [torch.rand(1, h, w, 9 if wide else 4, generator=g).cuda().requires_grad_(True) for _ in range(layers)]
    rast = [torch.rand(1, h, w, 4, generator=g).cuda() for _ in range(layers)]
    for r in rast:
        r[..., 3] = (r[..., 3] * 5 - 2).clamp(min=0).ceil()
    return rgba, rast, torch.randn(1, h, w, 3, generator=g).cuda(), torch.randn(1, h, w, 1, generator=g).cuda()


def _chain(step, rgba, rast, wide):
    out = trans = None
    for x, r in zip(rgba, rast):
        out, trans = step(x[..., 2:6] if wide else x, r, out, trans)
    return out, trans


@pytest.mark.parametrize('size', [(1, 1), (3, 85), (16, 16), (37, 61)])
@pytest.mark.parametrize('wide', [False, True])
@pytest.mark.parametrize('layers', [1, 3])
@pytest.mark.parametrize('use', ['out', 'both', 'trans'])
def test_compose_equals_the_operators(cuda, size, wide, layers, use):
    rgba, rast, go, gt = _inputs(*size, layers, wide, 3)
    res = [_chain(step, rgba, rast, wide) for step in (layered._compose, layered._blend)]
    assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])
    assert 'Compose' in type(res[0][0].grad_fn).__name__ and 'Compose' not in type(res[1][0].grad_fn).__name__
    grads = []
    for out, trans in res:
        ys, gs = {'out': ([out], [go]), 'both': ([out, trans], [go, gt]), 'trans': ([trans], [gt])}[use]
        grads.append(torch.autograd.grad(ys, rgba, gs, allow_unused=True))
    for a, b in zip(*grads):
        assert float((a - b).abs().max()) <= 1e-6 * max(float(b.abs().max()), 1e-30)


def test_values_under_the_mask_stay_as_the_operators_have_them(cuda):
    rgba, rast, _, _ = _inputs(5, 7, 1, False, 4)
    with torch.no_grad():
        rgba[0][0, 0, 0] = float('nan')
        rast[0][0, 0, 0, 3] = 0.0
        a, b = (_chain(step, rgba, rast, False) for step in (layered._compose, layered._blend))
    assert torch.isnan(a[0][0, 0, 0]).all() and torch.equal(torch.isnan(a[0]), torch.isnan(b[0]))


def test_other_inputs_go_through_the_operators(cuda):
    rgba, rast, go, _ = _inputs(6, 9, 2, False, 5)
    half = [x.detach().half() for x in rgba]
    assert _chain(layered._compose, half, rast, False)[0].dtype == torch.float16
    with torch.autograd.forward_ad.dual_level():
        x = torch.autograd.forward_ad.make_dual(rgba[0].detach(), torch.ones_like(rgba[0]))
        out, _ = layered._compose(x, rast[0], None, None)
        assert torch.autograd.forward_ad.unpack_dual(out).tangent is not None


def test_second_derivatives(cuda):
    rgba, rast, go, gt = _inputs(6, 9, 3, False, 6)
    second = []
    for step in (layered._compose, layered._blend):
        out, trans = _chain(step, rgba, rast, False)
        first = torch.autograd.grad([out, trans], rgba, [go, gt], create_graph=True)
        second.append(torch.autograd.grad(sum((f ** 2).sum() for f in first), rgba))
    for a, b in zip(*second):
        assert b.abs().max() > 0
        assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max())
