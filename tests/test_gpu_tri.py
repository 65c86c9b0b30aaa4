"""The unit lower solve and the inverse of L11 at the edges of their chunks
(64 rows, 16 rows, 16 columns), bit for bit where L and the right-hand sides
are small integers, which every order of exact operations gives alike, and a
column that overflows beside finite ones."""
import numpy as np
import pytest

import rochpl_amd as rp

pytestmark = pytest.mark.gpu


def update(ctx, L, B):
    """U12 = L^-1 B by hplx_pdupdate with the identity as interchange."""
    jb, n = B.shape
    A = np.asfortranarray(np.hstack([np.tril(L, -1) + 7.0 * np.triu(np.ones((jb, jb))), B]))
    perm = np.concatenate([np.arange(jb), np.full(jb, -1)]).astype(np.int32)
    dA, dP, dW = ctx.alloc(A.nbytes), ctx.alloc(perm.nbytes), ctx.alloc(8 * (jb + 8) * (n + 8))
    dA.upload(A)
    dP.upload(perm)
    ctx.pdupdate(dA.ptr, jb, jb, jb, n, dP.ptr, dW.ptr)
    return dA.download(A.shape, np.float64)[:, jb:]


@pytest.mark.parametrize("jb", [1, 2, 15, 16, 17, 31, 33, 63, 64, 65, 127, 128, 129, 200,
                                511, 512, 513, 895, 1024])
def test_inverse_of_l11(ctx, jb):
    """L with entries in {-1, 0, 1} near the diagonal, so that L^-1 is whole
    and small: U12 = L^-1 B has to be exact."""
    print("[gpu-case] linv jb=%d" % jb, flush=True)
    rng = np.random.default_rng(jb)
    L = np.eye(jb)
    for i in range(1, jb):
        L[i, rng.integers(0, i)] = rng.integers(0, 2)
    X = rng.integers(-4, 5, (jb, 19)).astype(float)
    got = update(ctx, L, L @ X)
    assert np.array_equal(got, X)


@pytest.mark.parametrize("n,nb,ndiv,nbmin", [(70, 70, 2, 16), (300, 300, 2, 32), (520, 500, 2, 8),
                                             (1100, 1024, 2, 32)])
def test_panel_solves(ctx, n, nb, ndiv, nbmin):
    """The recursion's solves with every width from the leaf's to half the
    panel's: the factors' backward error."""
    print("[gpu-case] panel solves n=%d nb=%d" % (n, nb), flush=True)
    from oracle import oracle as o
    A = o.matgen(n, n)
    mat = ctx.pmat_alloc(n, nb)
    palg = rp.palg_default()
    palg.nbdiv, palg.nbmin = ndiv, nbmin
    try:
        ctx.pdrandmat(n, n, nb, mat.A, mat.ld, rp.HPL_ISEED)
        assert ctx.pdgetrf(palg, mat) == 0
        X = np.random.default_rng(n).standard_normal((n, 3))
        B = np.asfortranarray(A @ X)
        d = ctx.alloc(B.nbytes)
        d.upload(B)
        ctx.pdgetrs(mat, 0, 3, d.ptr, n)
        got = d.download(B.shape, np.float64)
        res = np.abs(A @ got - B).max()
        assert res <= 8 * n * 2.0 ** -52 * (np.abs(A).sum(1).max() * np.abs(got).max()
                                            + np.abs(B).max())
    finally:
        ctx.pmat_free(mat)


def test_a_column_that_overflows(ctx):
    """The panel's second 32 columns, whose first overflows half way down:
    U12 is what the substitution gives row by row, the others are untouched."""
    print("[gpu-case] trsm overflow", flush=True)
    w = 32
    L = np.eye(w) + np.tril(np.full((w, w), 0.5), -1)
    A = np.zeros((2 * w, 2 * w), order="F")
    A[:w, :w] = L
    B = np.random.default_rng(3).standard_normal((w, w))
    B[:, 0] = np.where(np.arange(w) % 2, 1.7e308, -1.7e308)
    A[:w, w:] = B
    A[w:, w:] = np.eye(w)
    U = B.copy()
    with np.errstate(all="ignore"):
        for j in range(w):
            for i in range(j + 1, w):
                U[i] -= L[i, j] * U[j]  # exact up to one rounding, as the FMA
    dA, dp = ctx.alloc(A.nbytes), ctx.alloc(4 * 2 * w)
    dA.upload(A)
    ctx.pdfact(dA.ptr, 2 * w, 2 * w, 2 * w, dp.ptr, nbmin=w)
    got = dA.download(A.shape, np.float64)[:w, w:]
    assert np.array_equal(np.isnan(got), np.isnan(U)) and not np.isfinite(U[:, 0]).all()
    assert np.array_equal(got[~np.isfinite(U)], U[~np.isfinite(U)], equal_nan=True)
    fin = np.isfinite(U)
    assert np.allclose(got[fin], U[fin], rtol=1e-13, atol=1e-13)


@pytest.mark.parametrize("jb", [1, 2, 64, 65, 1000, 1024])
@pytest.mark.parametrize("kind", ["none", "last", "one below", "few", "far"])
def test_interchanges_that_share_targets(ctx, jb, kind):
    """Composed interchanges where many steps have the same target."""
    from oracle import oracle as o
    print("[gpu-case] pipid jb=%d %s" % (jb, kind), flush=True)
    i = np.arange(jb)
    rng = np.random.default_rng(jb)
    ipiv = {"none": i, "last": np.full(jb, jb - 1), "one below": np.full(jb, jb),
            "few": np.maximum(i, rng.choice([jb // 2, jb - 1, jb + 3, 2 * jb], jb)),
            "far": jb + 2048 * rng.integers(1, 5, jb)}[kind].astype(np.int32)
    dp, dq = ctx.alloc(4 * jb), ctx.alloc(8 * jb)
    dp.upload(ipiv)
    ctx.pipid(jb, dp.ptr, dq.ptr)
    assert np.array_equal(dq.download(2 * jb, np.int32), o.pipid(ipiv))
