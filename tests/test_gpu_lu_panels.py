"""LU panels held in registers: 512 rows of 32 columns, 1024 rows of 16, and
taller ones in memory; sizes at the edges, ties between pivots, a singular
matrix, against numpy."""
import numpy as np
import pytest

from .gpu_helpers import zgesv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nrhs,batch", [(1, 3, 2), (33, 5, 3), (511, 70, 2), (513, 64, 1),
                                          (529, 300, 2), (1024, 7, 1), (1030, 65, 1)])
def test_solve_at_panel_edges(gpu_ctx, n, nrhs, batch):
    rng = np.random.default_rng(n)
    A = rng.normal(size=(batch, n, n)) + 1j * rng.normal(size=(batch, n, n))
    if batch > 1:
        # every column of a permuted small-integer matrix has ties for its pivot
        A[1] = rng.integers(-1, 2, size=(n, n)) + 2 * n * np.eye(n)[rng.permutation(n)]
    B = rng.normal(size=(batch, n, nrhs)) + 1j * rng.normal(size=(batch, n, nrhs))
    X, info = zgesv(gpu_ctx, A, B)
    assert not info.any()
    for b in range(batch):
        r = np.abs(A[b] @ X[b] - B[b]).sum(0).max()
        s = np.abs(A[b]).sum(1).max() * np.abs(X[b]).sum(0).max()
        # backward error n u times a pivot growth of up to n^(2/3)
        assert r <= n ** (5.0 / 3.0) * 2.3e-16 * s + 1e-15


@pytest.mark.parametrize("n", [40, 600])
def test_singular_is_flagged(gpu_ctx, n):
    rng = np.random.default_rng(n)
    A = rng.normal(size=(2, n, n)) + 0j
    A[1][:, n - 2] = 0.0
    _, info = zgesv(gpu_ctx, A, np.ones((2, n, 1), complex))
    assert info[0] == 0 and info[1] != 0
