"""The FP8 update's tile exponent over the range of FP32: the largest power of
two that keeps a tile within e4m3, against the oracle's, with L a row of ones'
places, so that each C[i, j] is one product (exact in FP32: an e4m3 value times a
power of two).  Infinite entries end the call as usual and stay in their tile."""
import numpy as np
import pytest

import rochpl_amd as rp
from oracle import mxp_oracle as mo

pytestmark = pytest.mark.gpu


def update(ctx, L, U):
    (m, k), n = L.shape, U.shape[1]
    dev = []
    for X in (L, U, np.zeros((m, n), np.float32)):
        X = np.asfortranarray(X)
        dev.append(ctx.alloc(X.nbytes))
        dev[-1].upload(X)
    ctx.mxp_update(rp.HPLX_UPDATE_FP8, 1, rp.HPLX_STORE_FP32, m, n, k, dev[0].ptr, m,
                   dev[1].ptr, k, dev[2].ptr, m)
    out = dev[2].download((m, n), np.float32)
    for d in dev:
        d.free()
    return out


@pytest.mark.parametrize("which", ["U", "L"])
def test_tile_exponents_match_the_oracle(ctx, which):
    print("[gpu-case] fp8 tile exponents of %s" % which, flush=True)
    tops = [np.float32(t) * s for s in np.float32(2.0) ** np.arange(-149, 120, 7, np.float32)
            for t in (1.0, 1.75, np.nextafter(np.float32(1.75), np.float32(2)), 1.999)]
    k, n = 3, 128 * len(tops)
    rng = np.random.default_rng(4)
    X = rng.uniform(-1, 1, (k, n)).astype(np.float32)
    for i, t in enumerate(tops):  # a tile per largest entry
        X[:, 128 * i:128 * (i + 1)] *= t
        X[1, 128 * i + 9] = t
    E = np.eye(k, dtype=np.float32)
    L, U = (E, X) if which == "U" else (np.ascontiguousarray(X.T), E)
    want = -mo.update_product(rp.HPLX_UPDATE_FP8, 1, L, U)
    got = update(ctx, L, U)
    # (the exponents end at -100: nothing is promised above 448 2^100)
    for i in (i for i, t in enumerate(tops) if t <= 448 * 2.0 ** 100):
        at = slice(128 * i, 128 * (i + 1))
        at = (slice(None), at) if which == "U" else at
        assert np.array_equal(got[at], want[at].astype(np.float32)), tops[i]


def test_infinite_entries_end_and_stay_in_their_tile(ctx):
    print("[gpu-case] fp8 update with infinite entries", flush=True)
    k, n = 130, 300
    U = np.random.default_rng(5).choice(np.float32([-1, 0.5, 2]), (k, n))
    L = np.eye(40, k, dtype=np.float32)
    want = -U[:40]
    U[3, 130], U[129, 131] = np.inf, -np.inf
    got = update(ctx, L, U)
    assert np.array_equal(got[:, :128], want[:, :128])
    assert np.array_equal(got[:, 256:], want[:, 256:])
