"""The panel leaf (one leaf, 1 to 32 columns) against textbook unblocked LU
with partial pivoting in the same precision, at the edges of its row splits:
one workgroup of one row per thread (<= 512 rows), of three (<= 1536), up to
32 workgroups of one row per thread (<= 16384), three rows per thread above,
and the two ways of the pivot exchange (<= 32 workgroups, more).

Tolerance: every entry of the leaf is at most w multiply-subtracts and one
division away from the matrix, so with |l| <= 1 the two agree to about
w * eps * max|u|; 64 w eps leaves room for the growth of u."""
import numpy as np
import pytest

import rochpl_amd as rp

pytestmark = pytest.mark.gpu

ROWS = [3, 64, 511, 512, 513, 1536, 1537, 3100, 16384, 16385, 49152, 49153,
        90001]


def lu(A):
    """Unblocked LU; NaNs are never pivots while the column has a number."""
    A = A.copy()
    m, n = A.shape
    piv = np.empty(n, np.int32)
    for j in range(min(m, n)):
        a = np.abs(A[j:, j])
        a[np.isnan(a)] = -1
        p = j + int(np.argmax(a))  # the first of equal maxima
        piv[j] = p
        A[[j, p]] = A[[p, j]]
        if A[j, j] != 0:
            A[j + 1:, j] /= A[j, j]
        A[j + 1:, j + 1:] -= np.outer(A[j + 1:, j], A[j, j + 1:])
    return A, piv


def device_lu(ctx, A, jb):
    m, n = A.shape
    lda = m + 5
    buf = np.full((lda, n), 7.0, A.dtype, order="F")
    buf[:m] = A
    d, dp = ctx.alloc(buf.nbytes), ctx.alloc(4 * jb)
    d.upload(buf)
    f = ctx.pdfact if A.dtype == np.float64 else ctx.spdfact
    info = f(d.ptr, lda, m, jb, dp.ptr, nbmin=32)
    got = d.download((lda, n), A.dtype)
    assert np.all(got[m:] == 7.0)
    return got[:m], dp.download((jb,), np.int32), info


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m", ROWS)
def test_leaf_matches_unblocked_lu(ctx, m, dtype):
    for w in (1, 7, 8, 9, 31, 32):
        w = min(w, m)
        print("[gpu-case] leaf m=%d w=%d %s" % (m, w, dtype.__name__), flush=True)
        rng = np.random.default_rng(m * 37 + w)
        A = rng.uniform(-0.5, 0.5, (m, w)).astype(dtype)
        got, piv, info = device_lu(ctx, A, w)
        want, wpiv = lu(A)
        assert info == 0
        assert np.array_equal(piv, wpiv)
        tol = 64 * w * np.finfo(dtype).eps * np.abs(want).max()
        assert np.abs(got - want).max() <= tol


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m", [40, 700, 2000, 60000])
def test_leaf_ties_nans_and_zero_columns(ctx, m, dtype):
    """Exact ties (all entries +-1, +-2, ... of a few small integers), rows
    that hold NaNs, and an exactly zero column."""
    print("[gpu-case] leaf ties m=%d %s" % (m, dtype.__name__), flush=True)
    rng = np.random.default_rng(m)
    A = rng.integers(-2, 3, (m, 4)).astype(dtype)
    got, piv, info = device_lu(ctx, A, 4)
    want, wpiv = lu(A)
    assert np.array_equal(piv, wpiv)
    assert np.allclose(got, want, rtol=0, atol=64 * np.finfo(dtype).eps * 8)

    A = rng.uniform(-0.5, 0.5, (m, 9)).astype(dtype)
    A[m // 3, 0] = np.nan
    A[m - 1, 4] = np.nan
    got, piv, info = device_lu(ctx, A, 9)
    want, wpiv = lu(A)
    assert np.array_equal(piv, wpiv)
    assert np.array_equal(np.isnan(got), np.isnan(want))

    A = rng.uniform(-0.5, 0.5, (m, 5)).astype(dtype)
    A[:, 2] = 0
    got, piv, info = device_lu(ctx, A, 5)
    want, wpiv = lu(A)
    assert info == 3
    assert np.array_equal(piv, wpiv)
    assert np.all(got[:, 2] == 0)


@pytest.mark.parametrize("m,jb", [(1500, 96), (20000, 70)])
def test_leaf_moves_reach_the_other_columns(ctx, m, jb):
    """The interchanges of every leaf reach the panel's other columns: the
    pivots and factors of a panel of several leaves are unblocked LU's."""
    print("[gpu-case] panel m=%d jb=%d" % (m, jb), flush=True)
    rng = np.random.default_rng(m + jb)
    A = rng.uniform(-0.5, 0.5, (m, jb))
    got, piv, info = device_lu(ctx, A, jb)
    want, wpiv = lu(A)
    assert info == 0 and np.array_equal(piv, wpiv)
    assert np.abs(got - want).max() <= 64 * jb * 2.0 ** -52 * np.abs(want).max()
