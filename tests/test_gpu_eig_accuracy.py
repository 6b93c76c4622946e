"""Accuracy of what the eigen solver's QR is made of, against long double: no
worse than the same quantities from ordinary double-precision arithmetic."""
import ctypes

import numpy as np
import pytest

from openrcwa_amd import _lib

pytestmark = pytest.mark.gpu


def _call(ctx, name, x, per_in, per_out):
    fn = getattr(_lib.load(), name)
    p = ctypes.POINTER(ctypes.c_double)
    fn.argtypes = [ctypes.c_void_p, ctypes.c_int, p, p]
    x = np.ascontiguousarray(x, dtype=complex)
    out = np.zeros((len(x), per_out), dtype=complex)
    assert x.shape[1:] == (per_in,)
    _lib.check(fn(ctx.handle, len(x), x.ctypes.data_as(p), out.ctypes.data_as(p)), name)
    return out


def _errors(x, c, s, r):
    """|c|^2 + |s|^2 - 1, and the error of (r, 0) relative to the pair."""
    x, c, s, r = (np.asarray(v, dtype=np.clongdouble) for v in (x, c, s, r))
    sq = lambda z: z.real * z.real + z.imag * z.imag
    unit = sq(c) + sq(s) - 1
    e0 = np.conj(c) * x[:, 0] + np.conj(s) * x[:, 1] - r
    e1 = c * x[:, 1] - s * x[:, 0]
    back = np.sqrt((sq(e0) + sq(e1)) / (sq(x[:, 0]) + sq(x[:, 1])))
    return np.abs(unit).astype(float), back.astype(float)


@pytest.mark.parametrize("spread", [0.1, 4.0, 20.0])
def test_rotations_as_accurate_as_root_and_division(gpu_ctx, spread):
    rng = np.random.default_rng(11)
    x = rng.uniform(-1, 1, (1 << 20, 2)) + 1j * rng.uniform(-1, 1, (1 << 20, 2))
    x[:, 1] *= np.exp(rng.uniform(-spread, spread, len(x)))
    out = _call(gpu_ctx, "orcwa_dbg_rotations", x, 2, 3)
    unit, back = _errors(x, out[:, 0], out[:, 1], out[:, 2])
    # x / |x| with one square root and one division, each rounded correctly
    norm = np.sqrt((x.real ** 2 + x.imag ** 2).sum(1))
    inv = 1.0 / norm
    unit0, back0 = _errors(x, inv * x[:, 0], inv * x[:, 1], norm)
    assert unit.max() <= unit0.max() and unit.std() <= unit0.std()
    # (maxima of 2^20 draws scatter by a few per cent)
    assert back.max() <= 1.05 * back0.max() and np.mean(back ** 2) <= np.mean(back0 ** 2)


@pytest.mark.parametrize("x0,x1", [(0, 0), (3 + 4j, 0), (0, 3 - 4j), (1e-160, 1), (1, 1e-160),
                                   (1e-75j, 2e-75), (1e75, 1e75j), (1e200j, -1e200), (1e-200, 1e-210)])
def test_rotations_at_the_ends_of_the_range(gpu_ctx, x0, x1):
    x = np.array([[x0, x1]], dtype=complex)
    c, s, r = _call(gpu_ctx, "orcwa_dbg_rotations", x, 2, 3)[0]
    scale = max(abs(x0), abs(x1)) or 1.0
    unit, back = _errors(x / scale, c[None], s[None], r[None] / scale)
    # a few roundings of 1.1e-16
    assert unit[0] <= 2e-15
    assert max(abs(x0), abs(x1)) == 0 or back[0] <= 2e-15


def _lapack_shift(a, c, b, d):
    """The eigenvalue of [[a, b], [c, d]] nearer to d as zlahqr forms it, in double."""
    l1 = lambda z: np.abs(z.real) + np.abs(z.imag)
    u, x = np.sqrt(b) * np.sqrt(c), 0.5 * (a - d)
    s = np.maximum(l1(u), l1(x))
    y = s * np.sqrt((x / s) ** 2 + (u / s) ** 2)
    y = np.where(x.real * y.real + x.imag * y.imag < 0, -y, y)
    return d - u * (u / (x + y))


@pytest.mark.parametrize("kind", ["dense", "graded", "near_double"])
def test_shifts_as_accurate_as_in_double(gpu_ctx, kind):
    rng = np.random.default_rng(5)
    m = rng.normal(size=(200000, 4)) + 1j * rng.normal(size=(200000, 4))
    if kind == "graded":
        m *= np.exp(rng.uniform(-12, 12, m.shape))
    if kind == "near_double":      # discriminant nearly zero
        h = 0.5 * (m[:, 0] - m[:, 3])
        m[:, 1] = -h * h / m[:, 2] * (1 + 1e-9 * rng.normal(size=len(m)))
    a, c, b, d = np.asarray(m.T, dtype=np.clongdouble)     # column-major
    l1 = lambda z: np.abs(z.real) + np.abs(z.imag)
    scale = np.maximum(l1(a - d) / 2, np.maximum(l1(b), l1(c)))

    def residual(sh):
        # of the characteristic equation, against its terms and the rounding of sh
        return (np.abs((a - sh) * (d - sh) - b * c) /
                (scale ** 2 + np.abs(sh) * (np.abs(a - sh) + np.abs(d - sh)))).astype(float)

    sh = _call(gpu_ctx, "orcwa_dbg_shifts", m, 4, 1)[:, 0]
    got, ref = residual(sh), residual(_lapack_shift(*m.T))
    assert np.mean(got ** 2) <= np.mean(ref ** 2)
    assert got.max() <= 1.2 * ref.max()      # (maxima of 2e5 draws scatter)
    # the eigenvalue nearer to d
    assert (np.abs(sh - d) <= np.abs(a - sh) * (1 + 1e-9) + 1e-9 * scale).all()
