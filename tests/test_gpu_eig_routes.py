"""The routes of the eigen solver's QR (rounds over the whole chip, one kernel, and
the one kernel going on from a state of the rounds): one result, and one way to
fail."""
import ctypes

import numpy as np
import pytest

from openrcwa_amd import _lib
from .gpu_helpers import fortran_batch, from_fortran

pytestmark = pytest.mark.gpu
NOCONV = _lib.STATUS_NOCONV


def zgeev(ctx, A, rounds=-1, maxsweep=0):
    fn = _lib.load().orcwa_dbg_zgeev_route
    p, q = ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_int)
    fn.argtypes = [ctypes.c_void_p, ctypes.c_int, p, p, p, p, q, ctypes.c_int, ctypes.c_int,
                   ctypes.c_int]
    batch, n, _ = A.shape
    a = fortran_batch(A)
    lam, w = np.zeros((batch, n), dtype=complex), np.zeros_like(a)
    resid, info = np.zeros(batch), np.zeros(batch, dtype=np.int32)
    _lib.check(fn(ctx.handle, n, a.ctypes.data_as(p), lam.ctypes.data_as(p), w.ctypes.data_as(p),
                  resid.ctypes.data_as(p), info.ctypes.data_as(q), batch, rounds, maxsweep),
               "orcwa_dbg_zgeev_route")
    return lam, from_fortran(w, n, n), info


def matrices(n, batch):
    """Dense ones, a graded one and one that splits into blocks."""
    rng = np.random.default_rng(n)
    a = rng.normal(size=(batch, n, n)) + 1j * rng.normal(size=(batch, n, n))
    a[1] *= np.geomspace(1.0, 1e-6, n)[:, None]
    if batch > 2:
        a[2][n // 3:, :n // 3] = 0.0
        a[2][2 * n // 3:, :2 * n // 3] = 0.0
    return a


# (no more sweeps than n / 4 are needed by any of these, and more than 3)
@pytest.mark.parametrize("n", [135, 191, 242, 338, 450])
def test_rounds_one_kernel_and_takeover_agree(gpu_ctx, n):
    a = matrices(n, 3)
    lam, W, info = zgeev(gpu_ctx, a, rounds=n)
    assert not info.any()
    for rounds in (0, 1, 3, n // 20):
        other = zgeev(gpu_ctx, a, rounds=rounds)
        assert not other[2].any()
        assert np.array_equal(lam, other[0]) and np.array_equal(W, other[1])
    other = zgeev(gpu_ctx, a)       # as dispatched
    assert np.array_equal(lam, other[0]) and np.array_equal(W, other[1])


@pytest.mark.parametrize("n,batch", [(338, 136), (450, 200)])
def test_dispatch_agrees_across_its_line(gpu_ctx, n, batch):
    """More matrices than the rounds take, and two of them."""
    a = matrices(n, batch)
    lam, W, info = zgeev(gpu_ctx, a)
    few = zgeev(gpu_ctx, a[:2])
    assert not info.any() and not few[2].any()
    assert np.array_equal(lam[:2], few[0]) and np.array_equal(W[:2], few[1])


@pytest.mark.parametrize("rounds", [0, 2, 160])
def test_too_few_sweeps_are_reported(gpu_ctx, rounds):
    """A matrix that is given up is flagged on each route; one that needs no sweep
    is not, and is right."""
    n = 160
    a = matrices(n, 3)
    a[1] = np.diag(np.arange(1.0, n + 1))
    lam, _, info = zgeev(gpu_ctx, a, rounds=rounds, maxsweep=4)
    assert info[0] & NOCONV
    assert info[1] == 0 and np.abs(np.sort(lam[1].real) - np.arange(1.0, n + 1)).max() < 1e-10 * n


@pytest.mark.parametrize("bad", [np.nan, np.inf, complex(1.0, np.nan)])
@pytest.mark.parametrize("rounds", [0, 2, 160])
def test_a_matrix_that_is_not_finite(gpu_ctx, rounds, bad):
    """It is given up and reported, and the others of its batch are as without it."""
    n = 160
    a = matrices(n, 3)
    ref = zgeev(gpu_ctx, a, rounds=0)
    assert not ref[2].any()
    a[1][n // 2, n // 3] = bad
    # (each sweep that finds only NaN solves its windows to the limit: the limit here
    # is what the other two need twice over)
    lam, W, info = zgeev(gpu_ctx, a, rounds=rounds, maxsweep=60)
    assert info[1] & NOCONV
    assert info[0] == 0 and info[2] == 0
    for b in (0, 2):
        assert np.array_equal(lam[b], ref[0][b]) and np.array_equal(W[b], ref[1][b])
