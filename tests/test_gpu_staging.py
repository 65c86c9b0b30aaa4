"""FP16 storage: the copies of panels and U rows to FP32 and back, at the edges of
their 8-row, 4-column groups and for columns that do not lie on 16 bytes.  The
first block column and block row of the factors depend on no low-precision
product, so they are those of an FP32 matrix with the same values, rounded."""
import ctypes

import numpy as np
import pytest

import rochpl_amd as rp

pytestmark = pytest.mark.gpu


def transfer(ctx, fn, dst, src, nbytes):
    assert fn(ctx.h, dst, src, nbytes) == 0


def factors(ctx, mat, opts, A=None):
    """Factors mat (with the values A, if given); the matrix before and after."""
    lib = rp.lib()
    dt = np.float16 if mat.storage == rp.HPLX_STORE_FP16 else np.float32
    dev = ctypes.c_void_p(mat.A)
    before = np.zeros((mat.ld, mat.n), dtype=dt, order="F")
    if A is None:
        ctx.mxp_matgen(mat, rp.HPL_ISEED, 0.0)
        transfer(ctx, lib.hplx_memcpy_d2h, before.ctypes.data_as(ctypes.c_void_p), dev,
                 before.nbytes)
    else:
        before[:mat.n] = A
        transfer(ctx, lib.hplx_memcpy_h2d, dev, before.ctypes.data_as(ctypes.c_void_p),
                 before.nbytes)
    assert ctx.mxp_pdgetrf(rp.palg_default(), opts, mat) == 0
    F = np.empty_like(before)
    transfer(ctx, lib.hplx_memcpy_d2h, F.ctypes.data_as(ctypes.c_void_p), dev, F.nbytes)
    return before[:mat.n], F[:mat.n], ctx.download_vec(mat.ipiv, mat.n, np.int32)


@pytest.mark.parametrize("n,nb", [(1, 8), (7, 8), (8, 8), (9, 16), (61, 64), (64, 64),
                                  (131, 64), (250, 36), (515, 128), (1022, 1024),
                                  (2051, 256)])
def test_fp16_panels_are_the_fp32_ones_rounded(ctx, n, nb):
    print("[gpu-case] staging n=%d nb=%d" % (n, nb), flush=True)
    opts = rp.mxp_opts_default(rp.HPLX_UPDATE_BF16, 3)
    half = ctx.mxp_alloc(n, nb, rp.HPLX_STORE_FP16)
    single = ctx.mxp_alloc(n, nb, rp.HPLX_STORE_FP32)
    try:
        A, F16, p16 = factors(ctx, half, opts)
        _, F32, p32 = factors(ctx, single, opts, A)
    finally:
        ctx.mxp_free(half)
        ctx.mxp_free(single)
    k = min(n, nb)
    assert np.array_equal(p16[:k], p32[:k])
    assert np.array_equal(F16[:, :k], F32[:, :k].astype(np.float16))
    assert np.array_equal(F16[:k], F32[:k].astype(np.float16))
