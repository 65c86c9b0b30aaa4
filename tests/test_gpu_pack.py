"""The FP8 update's packed U rows: with columns on 16 bytes (four values a load) and
not, at the edges of its 128 x 128 tiles, the same bits, and each C[0, j] the exact
product of a first row of L that picks out one row of U."""
import numpy as np
import pytest

import rochpl_amd as rp

pytestmark = pytest.mark.gpu


def update(ctx, L, U, pad):
    (m, k), n = L.shape, U.shape[1]
    full = np.full((k + pad, n), np.float32(7e4), order="F")  # the padding is not read
    full[:k] = U
    C = np.zeros((m, n), np.float32, order="F")
    dev = []
    for X in (np.asfortranarray(L), full, C):
        dev.append(ctx.alloc(X.nbytes))
        dev[-1].upload(X)
    dL, dU, dC = dev
    ctx.mxp_update(rp.HPLX_UPDATE_FP8, 1, rp.HPLX_STORE_FP32, m, n, k, dL.ptr, m, dU.ptr,
                   k + pad, dC.ptr, m)
    out = dC.download((m, n), np.float32)
    for d in dev:
        d.free()
    return out


@pytest.mark.parametrize("k", [1, 3, 4, 127, 128, 130, 259])
@pytest.mark.parametrize("n", [1, 7, 128, 133])
def test_fp8_rows_of_u(ctx, n, k):
    print("[gpu-case] fp8 pack n=%d k=%d" % (n, k), flush=True)
    rng = np.random.default_rng(n + k)
    U = rng.choice(np.float32([-2, -1, -0.5, 0.25, 1, 1.5, 3]), (k, n))
    L = np.zeros((40, k), np.float32)
    rows = rng.integers(0, k, 40)
    L[np.arange(40), rows] = 1.0
    aligned = update(ctx, L, U, -k % 4 + 4)
    assert np.array_equal(aligned, -U[rows])
    assert np.array_equal(aligned, update(ctx, L, U, (-k % 4) + 1))
