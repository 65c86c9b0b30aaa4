"""The triangular solves of hplx_pdgetrs at the ends of what they take."""
import ctypes

import numpy as np
import pytest
import scipy.linalg as sl

import rochpl_amd as rp
from oracle import oracle as o

pytestmark = pytest.mark.gpu


def solve(ctx, mat, B, trans):
    n, nrhs = B.shape
    d = ctx.alloc(B.nbytes)
    try:
        d.upload(np.asfortranarray(B))
        ctx.pdgetrs(mat, trans, nrhs, d.ptr, n)
        return d.download((n, nrhs), np.float64)
    finally:
        d.free()


@pytest.mark.parametrize("nrhs", [1, 1000])
@pytest.mark.parametrize("nb", [501, 2000, 40000])
def test_panels_wider_than_the_matrix(ctx, nb, nrhs):
    """A caller's own hplx_pmat may state a panel wider than the matrix: one
    panel, the same bits as with nb = n."""
    n = 500
    print("[gpu-case] getrs n=%d nb=%d nrhs=%d" % (n, nb, nrhs), flush=True)
    mat = ctx.pmat_alloc(n, n)
    try:
        ctx.pdrandmat(n, n, n, mat.A, mat.ld)
        assert ctx.pdgetrf(rp.palg_default(), mat) == 0
        wide = rp.PMat.from_buffer_copy(mat)
        wide.nb = nb
        B = np.random.default_rng(nb).standard_normal((n, nrhs))
        for trans in (0, 1):
            assert np.array_equal(solve(ctx, wide, B, trans), solve(ctx, mat, B, trans))
    finally:
        ctx.pmat_free(mat)


@pytest.mark.parametrize("nb", [1025, 40000])
def test_panels_too_wide_are_refused(ctx, nb):
    n = 1500
    print("[gpu-case] getrs n=%d nb=%d refused" % (n, nb), flush=True)
    mat = ctx.pmat_alloc(n, 1024)
    try:
        wide = rp.PMat.from_buffer_copy(mat)
        wide.nb = nb
        for nrhs in (1, 1024):
            for trans in (0, 1):
                with pytest.raises(rp.HplxError) as e:
                    solve(ctx, wide, np.ones((n, nrhs)), trans)
                assert e.value.code == rp.HPLX_ERR_HIP
    finally:
        ctx.pmat_free(mat)


def test_no_rows(ctx):
    print("[gpu-case] getrs n=0", flush=True)
    mat = ctx.pmat_alloc(8, 8)
    try:
        none = rp.PMat.from_buffer_copy(mat)
        none.n = 0
        for trans in (0, 1):
            assert rp.lib().hplx_pdgetrs(ctx.h, ctypes.byref(none), trans, 3,
                                         ctypes.c_void_p(mat.X), 8) == rp.HPLX_SUCCESS
    finally:
        ctx.pmat_free(mat)


def upload(mat, A):
    hip = ctypes.CDLL("libamdhip64.so.7")
    full = np.zeros((mat.ld, A.shape[1]), order="F")
    full[:A.shape[0]] = A
    assert hip.hipMemcpy(ctypes.c_void_p(mat.A), full.ctypes.data_as(ctypes.c_void_p),
                         ctypes.c_size_t(full.nbytes), 1) == 0


@pytest.mark.parametrize("nrhs", [2, 40, 200])
@pytest.mark.parametrize("n,nb", [(90, 30), (250, 100), (500, 200), (129, 65), (700, 257)])
def test_infinities_spread_as_in_substitution(ctx, n, nb, nrhs):
    """Factors whose entries off U's diagonal are all negative turn one infinite
    right-hand side entry into +inf in every row, and nothing into NaN: the
    padding of a ragged panel takes no part."""
    print("[gpu-case] getrs inf n=%d nb=%d nrhs=%d" % (n, nb, nrhs), flush=True)
    L = np.tril(np.full((n, n), -0.5 / n), -1) + np.eye(n)
    U = np.triu(np.full((n, n), -0.5 / n), 1) + 4 * np.eye(n)
    mat = ctx.pmat_alloc(n, nb)
    try:
        upload(mat, L @ U)
        assert ctx.pdgetrf(rp.palg_default(), mat) == 0
        assert np.array_equal(ctx.download_vec(mat.ipiv, n, np.int32), np.arange(n))
        B = np.random.default_rng(3).standard_normal((n, nrhs))
        for trans in (0, 1):
            X = solve(ctx, mat, B, trans)
            for k in (0, 10, nb - 1, nb, n - 1):
                C = B.copy()
                C[k, 0] = np.inf
                Y = solve(ctx, mat, C, trans)
                assert np.all(Y[:, 0] == np.inf), (trans, k)
                assert np.array_equal(Y[:, 1:], X[:, 1:])
    finally:
        ctx.pmat_free(mat)


@pytest.mark.parametrize("n,nb,cols", [(60, 60, 8192), (128, 50, 8192), (129, 129, 4096),
                                       (300, 128, 2720), (700, 100, 1360), (1025, 300, 1024)])
def test_passes_of_right_hand_sides(ctx, n, nb, cols):
    """Up to the right-hand sides that one pass takes, and past them, against
    LAPACK with the same matrix (diagonally dominant, so that n eps is kept)."""
    A = o.matgen(n, n) + n * np.eye(n)
    lu = sl.lu_factor(A)
    mat = ctx.pmat_alloc(n, nb)
    try:
        ctx.pdrandmat(n, n, nb, mat.A, mat.ld, rp.HPL_ISEED, float(n))
        assert ctx.pdgetrf(rp.palg_default(), mat) == 0
        for nrhs in (cols - 15, cols, cols + 5):
            print("[gpu-case] getrs n=%d nb=%d nrhs=%d" % (n, nb, nrhs), flush=True)
            B = np.random.default_rng(nrhs).standard_normal((n, nrhs))
            for trans in (0, 1):
                X, R = solve(ctx, mat, B, trans), sl.lu_solve(lu, B, trans=trans)
                assert np.abs(X - R).max() <= 4 * n * 2.0 ** -52 * np.abs(R).max()
    finally:
        ctx.pmat_free(mat)


@pytest.mark.parametrize("n,nb,counts", [(4300, 32, (1, 9)), (8300, 64, (2,)),
                                         (16500, 512, (1, 64)), (11000, 256, (88,))])
def test_panels_and_chunks_prepared_more_than_once(ctx, n, nb, counts):
    """More than 128 panels of at most 128 rows are prepared in several runs, and U
    of more blocks than the exchange buffer holds (128 with few right-hand sides,
    85 with 84 to 96) is solved in several chunks: the residual stays within n eps
    of |A| |x| + |b| per row (A diagonally dominant)."""
    shift = float(n)
    A = o.matgen(n, n)
    A[np.arange(n), np.arange(n)] += shift
    norms = [np.abs(A).sum(1).max(), np.abs(A).sum(0).max()]
    mat = ctx.pmat_alloc(n, nb)
    try:
        ctx.pdrandmat(n, n, nb, mat.A, mat.ld, rp.HPL_ISEED, shift)
        assert ctx.pdgetrf(rp.palg_default(), mat) == 0
        for nrhs in counts:
            print("[gpu-case] getrs n=%d nb=%d nrhs=%d" % (n, nb, nrhs), flush=True)
            B = np.random.default_rng(nrhs).standard_normal((n, nrhs))
            for trans in (0, 1):
                X = solve(ctx, mat, B, trans)
                res = np.abs((A.T if trans else A) @ X - B).max()
                assert res <= n * 2.0 ** -52 * (norms[trans] * np.abs(X).max() +
                                                np.abs(B).max())
    finally:
        ctx.pmat_free(mat)
