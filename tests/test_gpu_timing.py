"""The times of the last FP64 solve outlive a mixed-precision solve."""
import pytest

import rochpl_amd as rp

pytestmark = pytest.mark.gpu


def test_fp64_times_outlive_a_mixed_solve(ctx):
    """hplx_swap_timing and hplx_panel_timing are those of the last hplx_pdgesv,
    also after a mixed solve of more panels."""
    print("[gpu-case] pdgesv n=500 nb=100, then mxp_pdgesv n=2000 nb=16", flush=True)
    with rp.Context(0) as c:
        mat, mx = c.pmat_alloc(500, 100), c.mxp_alloc(2000, 16)
        try:
            c.pdrandmat(500, 501, 100, mat.A, mat.ld)
            assert c.pdgesv(rp.palg_default(), mat) == 0
            swap, panel = c.swap_timing(), c.panel_timing()
            assert swap[1] == panel[1] == 5
            assert 0 < swap[0] < 100 and 0 < panel[0] < 100
            c.mxp_matgen(mx, rp.HPL_ISEED, 0.0)
            c.mxp_pdgesv(rp.palg_default(), rp.mxp_opts_default(), mx)
            assert c.update_stats()[1] == 124
            assert c.swap_timing() == swap and c.panel_timing() == panel
        finally:
            c.pmat_free(mat)
            c.mxp_free(mx)
