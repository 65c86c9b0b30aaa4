"""The matrix-vector products of the mixed-precision solves at the edges of their
column runs (a wave has a quarter of the block's columns, in runs of 32, 4 and 1)
and of their 64-row workgroups: the residual of L U x = P b on the CPU in FP64,
with the downloaded factors.  A sum of n terms in the vectors' unit u is off by
n u at most, relative to the same sum of absolute values; the two triangles and
the inverses of their (diagonally dominant) blocks take twice two of these."""
import ctypes

import numpy as np
import pytest

import rochpl_amd as rp
from oracle import oracle as o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solve_fp64", [1, 0])
@pytest.mark.parametrize("storage", [rp.HPLX_STORE_FP32, rp.HPLX_STORE_FP16])
@pytest.mark.parametrize("n,nb", [(65, 64), (191, 124), (193, 128), (281, 150),
                                  (400, 132), (600, 280), (1100, 1024)])
def test_solve_products(ctx, n, nb, storage, solve_fp64):
    print("[gpu-case] mixed solve n=%d nb=%d storage=%d fp64=%d"
          % (n, nb, storage, solve_fp64), flush=True)
    mat = ctx.mxp_alloc(n, nb, storage)
    f16 = storage == rp.HPLX_STORE_FP16
    opts = rp.mxp_opts_default(rp.HPLX_UPDATE_BF16 if f16 else rp.HPLX_UPDATE_FP32, 2)
    opts.solve_fp64 = solve_fp64
    try:
        ctx.mxp_matgen(mat, rp.HPL_ISEED, float(n))
        assert ctx.mxp_pdgetrf(rp.palg_default(), opts, mat) == 0
        F = np.empty((mat.ld, n), dtype=np.float16 if f16 else np.float32, order="F")
        rp.lib().hplx_memcpy_d2h(ctx.h, F.ctypes.data_as(ctypes.c_void_p),
                                 ctypes.c_void_p(mat.A), F.nbytes)
        F = F[:n].astype(np.float64)
        assert np.array_equal(ctx.download_vec(mat.ipiv, n, np.int32), np.arange(n))
        b = o.matgen_tile(n, 0, n, n, 1)[:, 0]
        d = ctx.alloc(b.nbytes)
        d.upload(b)
        ctx.mxp_pdgetrs(mat, d.ptr)
        x = d.download((n,), np.float64)
    finally:
        ctx.mxp_free(mat)
    L, U = np.tril(F, -1) + np.eye(n), np.triu(F)
    u = 2.0 ** -53 if solve_fp64 else 2.0 ** -24
    bound = 4 * n * u * (np.abs(L) @ (np.abs(U) @ np.abs(x)) + np.abs(b))
    assert np.all(np.abs(L @ (U @ x) - b) <= bound)
