"""The LU's pivots: the accuracy of their reciprocals against double precision."""
import numpy as np
import pytest

from .gpu_helpers import zgesv

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
