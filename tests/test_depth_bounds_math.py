"""
The upper depth bound that setup records carry beside the lower one (a peeled
layer skips the triangles that lie wholly in front of the previous layer), in
the kernel's float32 arithmetic: it is never below a computed depth of the box,
by brute force over every pixel centre on the triangles of the lower bound's
test, and its 27-bit form (the float's upper bits, rounded up) is never below
the bound.
"""
import numpy as np

from tests.test_depth_cull_math import F32, U, _cases, _check, _div, _eval, _fma, _mul, _pix, _rcp


def _upper(v, px0, px1, py0, py1, rng):
    """The kernel's upper bound on every computed depth in the box (None: no bound): the same margin above the
    corners' largest depth."""
    x, y, z, w = v
    MX = [max(abs(_fma(-w[k], px0, x[k])), abs(_fma(-w[k], px1, x[k]))) for k in range(3)]
    MY = [max(abs(_fma(-w[k], py0, y[k])), abs(_fma(-w[k], py1, y[k]))) for k in range(3)]
    ez = ew = F32(0)
    for k in range(3):
        i, j = (k + 1) % 3, (k + 2) % 3
        T = _fma(MX[i], MY[j], _mul(MX[j], MY[i]))
        ez = _fma(T, abs(z[k]), ez)
        ew = _fma(T, w[k], ew)
    ez, ew = _mul(ez, F32(8) * U), _mul(ew, F32(8) * U)
    q, w0 = [], F32(0)
    for c in range(4):
        zn, wn = _eval(v, px1 if c & 1 else px0, py1 if c & 2 else py0)
        if c == 0:
            w0 = F32(abs(wn) - ew)
        q.append(_mul(zn, _rcp(wn, rng)))
    if np.isnan(q).any():
        return None
    qmax, qa = max(q), max(abs(min(q)), abs(max(q)))
    if not (w0 > _mul(F32(3), ew)) or not (qa < np.inf):
        return None
    d = F32(w0 - ew)
    zb = _mul(F32(2), F32(_mul(qa, F32(1) + F32(5) * U) + _div(ez, d)))
    E = _div(F32(ez + _mul(zb, ew)), d)
    m = F32(F32(_mul(F32(2), E) + _mul(F32(8) * U, qa)) + _mul(F32(2) * U, F32(zb + E)))
    return F32(qmax + m)


def _packed(z):
    b = int(np.float32(z).view(np.uint32))
    if not b & 0x80000000:
        b += 31
    return np.uint32(b & ~31 & 0xffffffff).view(np.float32)


def test_upper_bound_is_above_every_computed_depth():
    rng = np.random.default_rng(11)
    used = 0
    for v, c0, c1, r0, r1, H, W, _ in _cases(rng, 4000):
        lo, zw = _check(v, c0, c1, r0, r1, H, W, rng)
        hi = _upper(v, _pix(c0, W), _pix(c1, W), _pix(r0, H), _pix(r1, H), rng)
        if hi is None or not np.isfinite(hi):
            continue
        assert float(hi) >= float(zw.max()), (float(hi), float(zw.max()), v, (c0, c1, r0, r1, H, W))
        assert lo is None or lo <= hi
        used += 1
    assert used > 2000


def test_packed_bound_rounds_up():
    rng = np.random.default_rng(12)
    z = np.concatenate([rng.normal(size=2000) * 10.0 ** rng.uniform(-6, 3, 2000), [0.0, 1.0, -1.0, np.inf]])
    for x in z.astype(F32):
        p = _packed(x)
        assert p >= x and (not np.isfinite(x) or p - x <= abs(x) * 2.0 ** -18 + 1e-43)
        assert int(np.float32(p).view(np.uint32)) & 31 == 0
