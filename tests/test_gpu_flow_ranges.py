"""The triangular solves of hplx_pdgetrs at the ends of what they take."""
import ctypes

import numpy as np
import pytest

import rochpl_amd as rp

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
