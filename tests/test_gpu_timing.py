"""The times of the last FP64 solve outlive a mixed-precision solve, and reading
them touches no other stream."""
import ctypes

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


def test_reading_times_does_not_wait_for_other_streams(ctx):
    """The queries work on the context's stream alone: copies that take a tenth
    of a second on another stream are still under way when they return."""
    print("[gpu-case] timing queries beside copies on another stream", flush=True)
    rp.lib()
    hip, vp, gib = ctypes.CDLL("libamdhip64.so.7"), ctypes.c_void_p, 1 << 30
    st = vp()
    with rp.Context(0) as c:
        mat, d = c.pmat_alloc(500, 100), c.alloc(2 * gib)
        assert hip.hipStreamCreate(ctypes.byref(st)) == 0
        try:
            c.pdrandmat(500, 501, 100, mat.A, mat.ld)
            assert c.pdgesv(rp.palg_default(), mat) == 0
            for query in (c.swap_timing, c.panel_timing, c.update_stats,
                          lambda: c.update_timing(1)):
                want = query()
                for _ in range(200):
                    assert hip.hipMemcpyAsync(vp(d.ptr), vp(d.ptr + gib), ctypes.c_size_t(gib),
                                              3, st) == 0
                got, busy = query(), hip.hipStreamQuery(st)
                assert hip.hipStreamSynchronize(st) == 0
                assert busy == 600 and got == want  # hipErrorNotReady
        finally:
            hip.hipStreamDestroy(st)
            d.free()
            c.pmat_free(mat)
