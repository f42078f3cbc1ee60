"""_lib.grad_observed, the question a fused backward asks before it leaves out
the gradient of its intermediate: a function of the fused form (the gradient of
y = 2 x left out, that of x returned on a side input in its place) gives every
caller what the unfused one gives."""
import os

import pytest
import torch

from diffrp_amd import _lib, build_ext


@pytest.fixture(scope='module', autouse=True)
def built():
    if not os.path.exists(build_ext.AUTOGRAD_LIB_PATH):
        build_ext.build()


class _Double(torch.autograd.Function):
    @staticmethod
    def forward(fctx, x):
        fctx.set_materialize_grads(False)
        return 2 * x, x.new_zeros(3)

    @staticmethod
    def backward(fctx, g, _g2):
        return None if g is None else 2 * g


class _Times(torch.autograd.Function):
    """a y, y = 2 x: fused, y's gradient stays out and x's comes on the side input."""
    fuse, calls = True, []

    @staticmethod
    def forward(fctx, a, y, tag, x):
        fctx.save_for_backward(a, y)
        return a * y

    @staticmethod
    def backward(fctx, g):
        a, y = fctx.saved_tensors
        fused = _Times.fuse and not _lib.grad_observed(fctx, 1)
        _Times.calls.append(fused)
        return g * y, (None if fused else g * a), None, (2 * g * a if fused else None)


def _graph(a_grad=True):
    x = torch.tensor([1.0, -2.0, 3.0], requires_grad=True)
    a = torch.tensor([5.0, 7.0, 11.0], requires_grad=a_grad)
    x1 = x * 1.0
    y, z = _Double.apply(x1)
    return x, a, y, z, _Times.apply(a, y, 'tag', x1)


def _run(case, fuse):
    _Times.fuse, _Times.calls = fuse, []
    x, a, y, z, out = _graph(a_grad=case != 'fixed a')
    loss, kept = out.sum(), []
    if case == 'grad y':
        res = torch.autograd.grad(loss, y)
    elif case == 'grad y and x':
        res = torch.autograd.grad(loss, [y, x])
    elif case == 'grad x and a':
        res = torch.autograd.grad(loss, [x, a])
    elif case == 'grad y of two consumers':
        res = torch.autograd.grad(loss + (y * y).sum(), [y, x])
    elif case == 'inputs=y':
        loss.backward(inputs=[y])
        res = [y.grad]
    elif case == 'retain':
        y.retain_grad()
        (loss + (y * y).sum()).backward()
        res = [y.grad, x.grad, a.grad]
    elif case == 'hook that blocks':
        y.register_hook(lambda g: g * 0)
        loss.backward()
        res = [x.grad, a.grad]
    elif case == 'hook that reads':
        h = y.register_hook(lambda g: kept.append(g.clone()))
        loss.backward()
        res = kept + [x.grad]
        h.remove()
    elif case == 'hook of the node':
        y.grad_fn.register_prehook(lambda gs: (None if gs[0] is None else 3 * gs[0],) + gs[1:])
        loss.backward()
        res = [x.grad]
    elif case == 'hook behind the node':
        y.grad_fn.register_hook(lambda gi, go: (None if gi[0] is None else 3 * gi[0],))
        loss.backward()
        res = [x.grad]
    elif case == 'packed':  # saved tensors replaced by copies, and a hook
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t.clone(), lambda t: t):
            x, a, y, z, out = _graph()
        y.register_hook(lambda g: g * 0)
        out.sum().backward()
        res = [x.grad, a.grad]
    elif case == 'removed hook':
        y.register_hook(lambda g: g * 0).remove()
        loss.backward()
        res = [x.grad, a.grad]
    else:  # plain, fixed a
        loss.backward()
        res = [x.grad]
    return [r.clone() for r in res], list(_Times.calls)


OBSERVED = ['grad y', 'grad y and x', 'grad y of two consumers', 'inputs=y', 'retain', 'hook that blocks',
            'hook that reads', 'hook of the node', 'hook behind the node', 'packed']


@pytest.mark.parametrize('case', OBSERVED + ['grad x and a', 'plain', 'fixed a'])
def test_fused_form_gives_what_the_unfused_gives(case):
    want, _ = _run(case, False)
    got, fused = _run(case, True)
    assert len(got) == len(want) and all(torch.equal(g, w) for g, w in zip(got, want))
    assert fused == [case not in OBSERVED]


def test_a_removed_hook_gives_the_same():
    want, _ = _run('removed hook', False)
    got, _ = _run('removed hook', True)  # (fused or not: the emptied hook table may stay behind)
    assert all(torch.equal(g, w) for g, w in zip(got, want))


def test_a_second_pass_asks_again():
    _Times.fuse, _Times.calls = True, []
    x, a, y, z, out = _graph()
    loss = out.sum()
    gx, = torch.autograd.grad(loss, x, retain_graph=True)
    gy, = torch.autograd.grad(loss, y, retain_graph=True)
    gx2, = torch.autograd.grad(loss, x)
    assert _Times.calls == [True, False, True]
    assert torch.equal(gx, gx2) and torch.equal(gx, 2 * a.detach()) and torch.equal(gy, a.detach())


def test_outside_a_pass_and_without_a_gradient_it_is_observed():
    _Times.fuse = True
    x, a, y, z, out = _graph()
    assert _lib.grad_observed(out.grad_fn, 1)   # no pass is running
    assert _lib.grad_observed(out.grad_fn, 99) and _lib.grad_observed(object(), 0)


def test_missing_library_is_named(monkeypatch):
    monkeypatch.setattr(_lib, '_grad_observed', None)
    monkeypatch.setattr(_lib, 'AUTOGRAD_LIB_PATH', '/nonexistent/libdrp_autograd.so')
    with pytest.raises(RuntimeError, match='libdrp_autograd'):
        _lib.grad_observed(object(), 0)
