"""Diagonal-block Cholesky: block rows of one wave each.

Edges: one row, one block row and its neighbours, the four-wave form's limit
(128) and the eight-wave form's, sizes that end inside a 32-row tile, a leading
dimension and a start that are not 16-byte aligned, a bad pivot in every part.
"""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def potrf_block(h, T, lda):
    info = C.c_int(0)
    torch.cuda.synchronize()
    rc = h.lib.mpc_potrf_block(h.h, C.c_void_p(T.data_ptr()), T.shape[0], lda, C.byref(info))
    assert rc >= 0 and rc == info.value
    return rc


def graded_spd(n, seed):
    """SPD with rows and columns scaled over six decades."""
    g = np.random.default_rng(seed)
    B = g.standard_normal((n, n))
    A = B @ B.T / n + 0.1 * np.eye(n)
    d = 10.0 ** (-6.0 * np.arange(n) / n)
    A = (A * d[:, None] * d[None, :]).astype(np.float32)
    return np.tril(A) + np.tril(A, -1).T


def place(A, lda, off):
    """A in column-major device storage with leading dimension lda, off floats in."""
    n = A.shape[0]
    buf = torch.full((off + n * lda,), 7.0, dtype=torch.float32)
    buf[off:].view(n, lda)[:, :n] = torch.from_numpy(np.ascontiguousarray(A.T))
    buf = buf.cuda()
    return buf, buf[off:].view(n, lda).t()[:n]


@pytest.mark.parametrize("n", [1, 31, 32, 33, 64, 96, 97, 127, 128, 129, 160, 193, 224, 255, 256])
def test_block_sizes(handle, n):
    print("potrf sizes", n, flush=True)
    A = graded_spd(n, n)
    buf, T = place(A, n + 3, 1)
    assert potrf_block(handle, T, n + 3) == 0
    L = T.cpu().numpy().astype(np.float64)
    # strict upper triangle and everything outside the block untouched
    assert np.array_equal(np.triu(L, 1), np.triu(A.astype(np.float64), 1))
    pad = buf.cpu()[1:].view(n, n + 3)[:, n:]
    assert bool((pad == 7.0).all()) and float(buf[0]) == 7.0
    L = np.tril(L)
    # |L L^T - A|_ij <= gamma_(n+1) sum_k |l_ik l_jk| <= gamma_(n+1) sqrt(a_ii a_jj)
    # to first order; 4 more for the reciprocal square roots (about 1 ulp each)
    sc = np.sqrt(np.diag(A).astype(np.float64))
    err = np.abs(L @ L.T - A) / (sc[:, None] * sc[None, :])
    assert err.max() <= (n + 5) * U, err.max()


@pytest.mark.parametrize("n", [40, 128, 200, 256])
@pytest.mark.parametrize("where", [0, 0.3, 0.6, 1])
@pytest.mark.parametrize("value", [-1.0, 0.0, float("nan")])
def test_block_bad_pivot(handle, n, where, value):
    c = int(where * (n - 1))
    print("potrf bad pivot", n, c, value, flush=True)
    A = np.eye(n, dtype=np.float32) * 4.0
    A[c, c] = value
    buf, T = place(A, n, 0)
    assert potrf_block(handle, T, n) == c + 1
