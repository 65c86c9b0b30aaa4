"""The small tiles of the GEMM at their edges (32 and 64 rows and columns,
stages of 32 in k, odd extents) against NumPy, and bit for bit against the
128 x 128 kernel, which takes the operands with odd leading dimensions."""
import ctypes

import numpy as np
import pytest

import rochpl_amd as rp

pytestmark = pytest.mark.gpu


def product(ctx, A, B, C, pad, alpha, beta):
    """C after the call, with `pad` rows below A, B and C (checked for C)."""
    (m, k), n = A.shape, B.shape[1]
    dev = []
    for X in (A, B, C):
        full = np.full((X.shape[0] + pad[len(dev)], X.shape[1]), 3.0, order="F")
        full[:X.shape[0]] = X
        d = ctx.alloc(full.nbytes)
        d.upload(full)
        dev.append((d, full))
    (a, fa), (b, fb), (c, fc) = dev
    r = rp.lib().hplx_dgemm(ctx.h, m, n, k, ctypes.c_double(alpha),
                            ctypes.c_void_p(a.ptr), fa.shape[0],
                            ctypes.c_void_p(b.ptr), fb.shape[0],
                            ctypes.c_double(beta), ctypes.c_void_p(c.ptr), fc.shape[0])
    assert r == 0
    got = c.download(fc.shape, np.float64)
    assert np.all(got[m:] == 3.0)
    return got[:m]


@pytest.mark.parametrize("m,n,k", [
    (1, 1, 1), (2, 2, 2), (31, 33, 32), (32, 32, 33), (33, 31, 31), (64, 64, 64),
    (65, 63, 96), (500, 257, 100), (1023, 32, 32), (2049, 65, 30), (4096, 300, 64),
    (35001, 32, 31), (33000, 31, 2), (9001, 384, 37), (2600, 700, 65)])
@pytest.mark.parametrize("alpha,beta", [(-1.0, 1.0), (1.0, 0.0)])
def test_small_tiles(ctx, m, n, k, alpha, beta):
    print("[gpu-case] dgemm tiles m=%d n=%d k=%d beta=%g" % (m, n, k, beta), flush=True)
    rng = np.random.default_rng(m + n + k)
    A, B, C = (rng.standard_normal(s) for s in ((m, k), (k, n), (m, n)))
    even = [x % 2 for x in (m, k, m)]
    odd = [1 - x for x in even]
    got = product(ctx, A, B, C, even, alpha, beta)
    ref = alpha * (A @ B) + beta * C
    bound = 2.0 ** -52 * (k + 2) * (np.abs(A) @ np.abs(B) + np.abs(beta * C))
    assert np.all(np.abs(got - ref) <= bound)
    assert np.array_equal(got, product(ctx, A, B, C, odd, alpha, beta))
