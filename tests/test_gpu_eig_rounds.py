"""The QR iteration in rounds (few matrices of 128 rows or more; section 3c of
csrc/qr_ms.inc) against numpy: sizes at the edges of its 64-line strips and
48-row windows, with a batch small enough to take it."""
import numpy as np
import pytest

from .gpu_helpers import zgeev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,batch", [(128, 1), (129, 2), (191, 3), (192, 1), (257, 5), (338, 2)])
def test_rounds_match_numpy(gpu_ctx, n, batch):
    rng = np.random.default_rng(n)
    a = rng.normal(size=(batch, n, n)) + 1j * rng.normal(size=(batch, n, n))
    # a graded matrix and one that splits into two blocks, as well as dense ones
    if batch > 1:
        a[1] *= np.geomspace(1.0, 1e-3, n)[:, None]
    if batch > 2:
        a[2][n // 2:, :n // 2] = 0.0
    lam, W, resid, info = zgeev(gpu_ctx, a)
    assert not info.any()
    # backward error of a QR iteration: a small multiple of n u (2e-14 n here)
    assert resid.max() <= 2e-14 * n
    for b in range(batch):
        ref = np.linalg.eigvals(a[b])
        # condition numbers of these eigenvalues stay below 1e4
        tol = 1e4 * 2e-16 * n * np.linalg.norm(a[b], 2)
        d = np.abs(lam[b][:, None] - ref[None, :])
        assert d.min(1).max() <= tol and d.min(0).max() <= tol
        assert np.abs(np.linalg.norm(W[b], axis=0) - 1.0).max() <= 1e-12


@pytest.mark.parametrize("n,batch", [(130, 40), (162, 40), (242, 9), (242, 80), (338, 16), (450, 27)])
def test_same_matrix_in_any_batch(gpu_ctx, n, batch):
    """A matrix's eigenvalues, their order included, do not depend on the batch it
    is solved in (few matrices iterate in rounds, many in one kernel): a plan that
    runs in chunks, or inside a captured graph, agrees with one that does not."""
    rng = np.random.default_rng(n)
    a = rng.normal(size=(batch, n, n)) + 1j * rng.normal(size=(batch, n, n))
    lam, W, _, info = zgeev(gpu_ctx, a)
    few = zgeev(gpu_ctx, a[:2])
    assert not info.any() and not few[3].any()
    assert np.array_equal(lam[:2], few[0]) and np.array_equal(W[:2], few[1])
