"""The residual check's pass at the edges of its column steps (8), of the chunks
(32 columns of one row a thread up to 2048, above it 256 of four rows) and of the
chunks wider than the 256 columns kept in LDS at once (from 46341), for a given x,
against the oracle's check.  Two orders of a sum of n terms differ by n eps of the
sum of their absolute values at most."""
import ctypes

import numpy as np
import pytest

import rochpl_amd as rp
from oracle import oracle as o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,shift", [
    (n, s) for n in (1, 7, 8, 9, 31, 32, 33, 63, 65, 255, 256, 257, 511, 513, 2047, 2048, 2049)
    for s in (0.0, 3.0)] + [(46400, 3.0)])
def test_check_matches_the_oracle(ctx, n, shift):
    print("[gpu-case] check n=%d shift=%g" % (n, shift), flush=True)
    x = np.random.default_rng(n).standard_normal(n)
    mat = ctx.pmat_alloc(n, min(n, 64))
    try:
        assert rp.lib().hplx_memcpy_h2d(ctx.h, ctypes.c_void_p(mat.X),
                                        x.ctypes.data_as(ctypes.c_void_p), x.nbytes) == 0
        got = ctx.pdtest_check(mat, diag_shift=shift)
    finally:
        ctx.pmat_free(mat)
    want = o.residual(n, x, diag_shift=shift)
    eps = n * 2.0 ** -52
    for k in ("AnormI", "Anorm1", "Xnorm1"):
        assert abs(got[k] - want[k]) <= eps * want[k], k
    assert got["XnormI"] == want["XnormI"] and got["BnormI"] == want["BnormI"]
    noise = eps * (want["AnormI"] * want["XnormI"] + want["BnormI"])
    for k in ("rnorm", "r0"):
        assert abs(got[k] - want[k]) <= noise, k
