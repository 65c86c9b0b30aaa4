"""The residual check's one pass at the edges of its row blocks (1024), column
chunks (256) and steps (8), against NumPy on the same matrix."""
import numpy as np
import pytest

import rochpl_amd as rp
from oracle import oracle as o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [0.0, 3.0])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 255, 257, 1023, 1024, 1025, 1300, 2305])
def test_check_matches_numpy(ctx, n, shift):
    print("[gpu-case] check n=%d shift=%g" % (n, shift), flush=True)
    A = o.matgen(n, n + 1)
    b, A = A[:, n].copy(), A[:, :n] + shift * np.eye(n)
    mat = ctx.pmat_alloc(n, min(n, 64))
    try:
        ctx.pdrandmat(n, n + 1, min(n, 64), mat.A, mat.ld, rp.HPL_ISEED, shift)
        assert ctx.pdgesv(rp.palg_default(), mat) == 0
        got = ctx.pdtest_check(mat, diag_shift=shift)
        x = ctx.download_vec(mat.X, n)
    finally:
        ctx.pmat_free(mat)
    bound = 4 * n * 2.0 ** -53
    rows, cols = np.abs(A).sum(1), np.abs(A).sum(0)
    assert abs(got["AnormI"] - rows.max()) <= bound * rows.max()
    assert abs(got["Anorm1"] - cols.max()) <= bound * cols.max()
    assert got["BnormI"] == np.abs(b).max() and got["XnormI"] == np.abs(x).max()
    r = (b.astype(np.longdouble) - A.astype(np.longdouble) @ x).astype(float)
    noise = bound * (rows.max() * np.abs(x).max() + np.abs(b).max())
    assert abs(got["rnorm"] - np.abs(r).max()) <= noise
    assert abs(got["r0"] - abs(r[0])) <= noise
