"""The LU's pivots: the accuracy of their reciprocals against double precision."""
import ctypes

import numpy as np
import pytest

from openrcwa_amd import _lib
from .gpu_helpers import fortran_batch, from_fortran, zgesv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ratio", [1.0, 1e-3, 1e3])
def test_pivot_reciprocals_as_accurate_as_in_double(gpu_ctx, ratio):
    """[[z, 0], [1, 1]] x = (1, 0) has x_2 = -1 / z, every other operation being
    exact: the multiplier is 1 times the reciprocal of the pivot."""
    rng = np.random.default_rng(2)
    z = rng.uniform(1, 2, 40000) * np.exp(2j * np.pi * rng.uniform(size=40000))
    z = 4.0 * (z.real + 1j * ratio * z.imag) / min(1.0, ratio)     # |z| > 1: the pivot
    A = np.zeros((len(z), 2, 2), dtype=complex)
    A[:, 0, 0], A[:, 1, 0], A[:, 1, 1] = z, 1.0, 1.0
    B = np.zeros((len(z), 2, 1), dtype=complex)
    B[:, 0, 0] = 1.0
    X, info = zgesv(gpu_ctx, A, B)
    assert not info.any()
    w = np.asarray(z, dtype=np.clongdouble)
    error = lambda inv: np.abs(inv * w - 1).astype(float)
    got, ref = error(-X[:, 1, 0]), error(1.0 / z)        # numpy divides as Smith does
    # rms of 40000 draws: scatter below 1 %
    assert np.mean(got ** 2) <= 1.02 ** 2 * np.mean(ref ** 2)
    assert got.max() <= 1.1 * ref.max()


@pytest.mark.parametrize("n,batch", [(60, 300), (530, 66), (700, 66), (1040, 66)])
def test_same_solution_in_any_batch(gpu_ctx, n, batch):
    """A matrix is factored the same way whatever it is batched with, so a plan
    that runs in chunks agrees with one that does not."""
    rng = np.random.default_rng(n)
    A = rng.normal(size=(batch, n, n)) + 1j * rng.normal(size=(batch, n, n))
    B = rng.normal(size=(batch, n, 33)) + 1j * rng.normal(size=(batch, n, 33))
    X, info = zgesv(gpu_ctx, A, B)
    few, info2 = zgesv(gpu_ctx, A[:2], B[:2])
    assert not info.any() and not info2.any()
    assert np.array_equal(X[:2], few)


def zgetrf(ctx, A):
    fn = _lib.load().orcwa_dbg_zgetrf
    q = ctypes.POINTER(ctypes.c_int)
    fn.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.POINTER(ctypes.c_double), q, q,
                   ctypes.c_int]
    batch, n, _ = A.shape
    a = fortran_batch(A)
    ipiv, info = np.zeros((batch, n), dtype=np.int32), np.zeros(batch, dtype=np.int32)
    _lib.check(fn(ctx.handle, n, a.ctypes.data_as(ctypes.POINTER(ctypes.c_double)),
                  ipiv.ctypes.data_as(q), info.ctypes.data_as(q), batch), "orcwa_dbg_zgetrf")
    return from_fortran(a, n, n), ipiv, info


def eliminate(a):
    """LU with the lowest row of the largest |re| + |im| as the pivot; also the
    number of columns where more than one row has it."""
    a, n, ties = a.copy(), len(a), 0
    piv = np.zeros(n, dtype=np.int32)
    for k in range(n):
        m = np.abs(a[k:, k].real) + np.abs(a[k:, k].imag)
        ties += (m == m.max()).sum() > 1
        piv[k] = k + int(np.argmax(m))
        a[[k, piv[k]]] = a[[piv[k], k]]
        a[k + 1:, k] /= a[k, k]
        a[k + 1:, k + 1:] -= np.outer(a[k + 1:, k], a[k, k + 1:])
    return a, piv, ties


# one wave; all 512 rows; more rows than that in the first panels, 1024; more again
@pytest.mark.parametrize("blocks", [(64,), (32, 8), (512,), (512, 32, 32), (512, 256), (1024,),
                                    (1024, 64)])
def test_ties_take_the_lowest_row(gpu_ctx, blocks):
    """Hadamard blocks, their rows shuffled and turned by units: nearly every column
    has ties for its pivot, within a wave and across waves, and elimination is
    exact (every entry is a small multiple of a power of two)."""
    n = sum(blocks)
    rng = np.random.default_rng(n)
    mats = []
    for _ in range(2):
        a = np.zeros((n, n), dtype=complex)
        r = 0
        for m in blocks:
            h = np.ones((1, 1))
            while len(h) < m:
                h = np.block([[h, h], [h, -h]])
            a[r:r + m, r:r + m] = h
            r += m
        mats.append(np.array([1, 1j, -1, -1j])[rng.integers(0, 4, n), None] * a[rng.permutation(n)])
    lu, ipiv, info = zgetrf(gpu_ctx, np.array(mats))
    assert not info.any()
    for b in range(2):
        ref, piv, ties = eliminate(mats[b])
        assert ties > n // 4
        assert np.array_equal(ipiv[b], piv)
        assert np.array_equal(lu[b], ref)


@pytest.mark.parametrize("n", [40, 300, 600, 1030])
def test_a_matrix_that_is_not_finite(gpu_ctx, n):
    """It ends, its pivots are rows of the matrix, and the others of its batch are
    as without it."""
    rng = np.random.default_rng(n)
    a = rng.normal(size=(4, n, n)) + 1j * rng.normal(size=(4, n, n))
    ref = zgetrf(gpu_ctx, a)
    a[1][:, n // 2] = np.nan
    a[2][n // 3, n // 4] = np.inf
    lu, ipiv, info = zgetrf(gpu_ctx, a)
    assert ((ipiv >= np.arange(n)) & (ipiv < n)).all()
    for b in (0, 3):
        assert np.array_equal(lu[b], ref[0][b]) and np.array_equal(ipiv[b], ref[1][b])
        assert info[b] == 0
