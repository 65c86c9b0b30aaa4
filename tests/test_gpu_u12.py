"""U12 = L11^{-1} A12 at the edges of its row tiles (32, 64 and 128 rows, each with
its own K bound) and column tiles: the residual of L11 U12 = A12 in NumPy.  With
entries of at most 1 / (2 jb) below the diagonal, |L11| is 1.5 and |L11^{-1}| 1.65
at most (infinity norm), so the inverse (jb u |L^{-1}| |L| |L^{-1}|), its product
with A12 and the check itself stay within 20 jb u of max |A12|."""
import numpy as np
import pytest

import rochpl_amd as rp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("jb,n", [(32, 1), (64, 65), (96, 2049), (100, 4100), (129, 31),
                                  (200, 8200), (384, 5000), (640, 9300), (1000, 9001),
                                  (1024, 8193)])
def test_u12_tiles(ctx, jb, n):
    print("[gpu-case] u12 jb=%d n=%d" % (jb, n), flush=True)
    rng = np.random.default_rng(jb + n)
    lda = jb + 8 - jb % 8
    A = np.zeros((lda, jb + n), order="F")
    L = np.tril(rng.uniform(-0.5, 0.5, (jb, jb)) / jb, -1)
    A[:jb, :jb] = L + np.triu(rng.uniform(-0.5, 0.5, (jb, jb)))
    T = rng.uniform(-0.5, 0.5, (jb, n))
    A[:jb, jb:] = T
    perm = np.concatenate([np.arange(jb), np.full(jb, -1)]).astype(np.int32)
    dA, dP, dW = ctx.alloc(A.nbytes), ctx.alloc(perm.nbytes), ctx.alloc(8 * jb * (n + 4))
    dA.upload(A)
    dP.upload(perm)
    ctx.pdupdate(dA.ptr, lda, jb, jb, n, dP.ptr, dW.ptr)
    got = dA.download(A.shape, np.float64)
    assert np.array_equal(got[:, :jb], A[:, :jb])
    U = got[:jb, jb:]
    assert np.abs(U + L @ U - T).max() <= 20 * jb * 2.0 ** -53 * np.abs(T).max()
