"""The triangular solves of hplx_pdgetrs at the edges of their blocks (128
rows, halves of 64), slices (4 or 16 right-hand sides) and of the split into
chain and product (192 right-hand sides), against LAPACK with the same
factors' matrix; non-finite right-hand sides; and captured replays."""
import ctypes

import numpy as np
import pytest
import scipy.linalg as sl

import rochpl_amd as rp
from oracle import oracle as o

pytestmark = pytest.mark.gpu


class Factored:
    def __init__(self, ctx, n, nb, shift=0.0):
        self.ctx, self.n = ctx, n
        self.mat = ctx.pmat_alloc(n, nb)
        ctx.pdrandmat(n, n, nb, self.mat.A, self.mat.ld, rp.HPL_ISEED, shift)
        assert ctx.pdgetrf(rp.palg_default(), self.mat) == 0

    def solve(self, B, trans):
        ldb = self.n + 3
        buf = np.full((ldb, B.shape[1]), 5.0, order="F")
        buf[:self.n] = B
        d = self.ctx.alloc(buf.nbytes)
        d.upload(buf)
        self.ctx.pdgetrs(self.mat, trans, B.shape[1], d.ptr, ldb)
        got = d.download(buf.shape, np.float64)
        assert np.all(got[self.n:] == 5.0)
        return got[:self.n]

    def free(self):
        self.ctx.pmat_free(self.mat)


@pytest.mark.parametrize("n,nb", [
    (1, 1), (2, 64), (63, 63), (64, 64), (65, 65), (127, 128), (128, 128),
    (129, 200), (193, 64), (256, 100), (320, 1000), (700, 130), (1023, 257),
    (1290, 640), (2500, 1024)])
def test_solves_match_lapack_at_block_edges(ctx, n, nb):
    nb = min(nb, n)
    A = o.matgen(n, n)
    lu = sl.lu_factor(A)
    tol = 1e-15 * np.linalg.cond(A, 1) * 10 * n ** 0.5
    s = Factored(ctx, n, nb)
    try:
        for nrhs in (1, 4, 5, 16, 17, 33, 191, 192):
            print("[gpu-case] getrs n=%d nb=%d nrhs=%d" % (n, nb, nrhs), flush=True)
            B = np.random.default_rng(n + nrhs).standard_normal((n, nrhs))
            for trans in (0, 1):
                X, R = s.solve(B, trans), sl.lu_solve(lu, B, trans=trans)
                assert np.linalg.norm(X - R) <= tol * np.linalg.norm(R)
    finally:
        s.free()


def test_wide_slices_and_many_blocks(ctx):
    """n x nrhs beyond the narrow slices' 512 workgroups, and more right-hand
    sides than one pass takes (1024)."""
    n, nb = 3000, 384
    A = o.matgen(n, n)
    lu = sl.lu_factor(A)
    tol = 1e-15 * np.linalg.cond(A, 1) * 10 * n ** 0.5
    s = Factored(ctx, n, nb)
    try:
        for nrhs in (84, 88, 90, 1030):
            print("[gpu-case] getrs n=%d nrhs=%d" % (n, nrhs), flush=True)
            B = np.random.default_rng(nrhs).standard_normal((n, nrhs))
            for trans in (0, 1):
                X, R = s.solve(B, trans), sl.lu_solve(lu, B, trans=trans)
                assert np.linalg.norm(X - R) <= tol * np.linalg.norm(R)
    finally:
        s.free()


@pytest.mark.parametrize("nrhs", [3, 40])
def test_non_finite_right_hand_sides_stay_in_their_columns(ctx, nrhs):
    """A NaN (of any payload, the exchange's own among them) or an infinity in
    one right-hand side ends the solve as usual and leaves the others alone."""
    n, nb = 900, 256
    print("[gpu-case] getrs non-finite nrhs=%d" % nrhs, flush=True)
    s = Factored(ctx, n, nb)
    try:
        B = np.random.default_rng(5).standard_normal((n, nrhs))
        C = np.asfortranarray(B)
        C[100, 0] = np.nan
        C[n - 1, 1] = np.inf
        C.view(np.uint64).T[2, 7] = 0x7ff8b10cffffb10c
        for trans in (0, 1):
            X, Y = s.solve(B, trans), s.solve(C, trans)
            assert np.all(np.isnan(Y[:, 0]).any() and ~np.isfinite(Y[:, 1]).all())
            assert np.isnan(Y[:, 2]).any()
            assert np.array_equal(X[:, 3:], Y[:, 3:])
    finally:
        s.free()


def test_captured_solves_replay(ctx):
    """hplx_pdgetrs_noalloc recorded into a graph: every replay, with eager
    solves between, gives the eager result bit for bit."""
    n, nb, nrhs = 1500, 256, 6
    print("[gpu-case] captured getrs_noalloc", flush=True)
    rp.lib()
    hip = ctypes.CDLL("libamdhip64.so.7")
    vp = ctypes.c_void_p
    s = Factored(ctx, n, nb)
    st, graph, ex = vp(), vp(), vp()
    assert hip.hipStreamCreate(ctypes.byref(st)) == 0
    try:
        d = ctx.alloc(8 * n * nrhs)

        def solve(trans):
            assert rp.lib().hplx_pdgetrs_noalloc(ctypes.byref(s.mat), trans, nrhs,
                                                 vp(d.ptr), n, st) == 0

        rng = np.random.default_rng(9)
        for trans in (0, 1):
            B0 = np.asfortranarray(rng.standard_normal((n, nrhs)))
            d.upload(B0)
            solve(trans)
            assert hip.hipStreamSynchronize(st) == 0
            assert hip.hipStreamBeginCapture(st, 1) == 0
            solve(trans)
            assert hip.hipStreamEndCapture(st, ctypes.byref(graph)) == 0
            assert hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None,
                                           ctypes.c_size_t(0)) == 0
            for rep in range(4):
                B = np.asfortranarray(rng.standard_normal((n, nrhs)))
                d.upload(B)
                solve(trans)
                assert hip.hipStreamSynchronize(st) == 0
                want = d.download((n, nrhs), np.float64)
                d.upload(B)
                assert hip.hipGraphLaunch(ex, st) == 0
                assert hip.hipStreamSynchronize(st) == 0
                assert np.array_equal(d.download((n, nrhs), np.float64), want)
            assert hip.hipGraphExecDestroy(ex) == 0
            assert hip.hipGraphDestroy(graph) == 0
    finally:
        hip.hipStreamDestroy(st)
        s.free()


def upload(mat, A):
    hip = ctypes.CDLL("libamdhip64.so.7")
    full = np.zeros((mat.ld, A.shape[1]), order="F")
    full[:A.shape[0]] = A
    assert hip.hipMemcpy(ctypes.c_void_p(mat.A), full.ctypes.data_as(ctypes.c_void_p),
                         ctypes.c_size_t(full.nbytes), 1) == 0


@pytest.mark.parametrize("kind", ["gauss", "tiny", "huge"])
def test_ill_conditioned_triangles_keep_a_small_residual(ctx, kind):
    """Diagonal blocks whose inverses are huge (a Gaussian kernel matrix), or
    whose diagonal is near the ends of the exponents' range: the residual stays
    within n eps of |A| |x| + |b| per row, as substitution promises (with the
    factors' own growth, taken as 8)."""
    n, nb, nrhs = 500, 128, 3
    i = np.arange(n)
    if kind == "gauss":
        A = np.exp(-((i[:, None] - i) / 8.0) ** 2) + 1e-10 * np.eye(n)
    else:
        A = o.matgen(n, n) + n * np.eye(n)
        A *= 2.0 ** (-1010 if kind == "tiny" else 1008)
    s = Factored(ctx, n, nb)
    try:
        upload(s.mat, A)
        assert ctx.pdgetrf(rp.palg_default(), s.mat) == 0
        for trans in (0, 1):
            print("[gpu-case] getrs %s trans=%d" % (kind, trans), flush=True)
            At = (A.T if trans else A).astype(np.longdouble)
            xt = np.random.default_rng(1).standard_normal((n, nrhs))
            B = (At @ xt).astype(np.float64)
            X = s.solve(B, trans)
            assert np.all(np.isfinite(X))
            res = np.abs(At @ X.astype(np.longdouble) - B).max(0)
            scale = np.abs(At).sum(1).max() * np.abs(X).max(0) + np.abs(B).max(0)
            assert np.all(res <= 8 * n * 2.0 ** -52 * scale)
    finally:
        s.free()
