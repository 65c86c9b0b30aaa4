"""The waits of the triangular solves of hplx_pdgetrs: what a block reads of the
solved blocks does not depend on when their flags are raised, and a wait that
gives up makes the call fail."""
import ctypes

import numpy as np
import pytest

import rochpl_amd as rp

pytestmark = pytest.mark.gpu

ENQUEUE = "_ZN4hplx13getrs_enqueueEP12ihipStream_tPKdiiiPKiiiPdiRKNS_11FlowScratchE"
WORK, PERM, FLAGS = 1024 * 1024, 2 * 128 * 128, 2048


class Scratch(ctypes.Structure):
    """hplx::FlowScratch."""
    _fields_ = [("x", ctypes.c_void_p), ("work", ctypes.c_void_p),
                ("work_doubles", ctypes.c_size_t), ("perm", ctypes.c_void_p),
                ("flags", ctypes.c_void_p), ("raised", ctypes.c_int),
                ("err", ctypes.c_void_p), ("polls", ctypes.c_uint32)]


@pytest.mark.parametrize("n,nb,nrhs", [(1500, 1024, 1), (2500, 640, 17), (3000, 300, 90)])
def test_flags_are_only_hints(ctx, n, nb, nrhs):
    """With every flag raised from the start, blocks look for values long before
    they are there; they take none that is not, so the solutions are the same
    bits."""
    enqueue = getattr(rp.lib(), ENQUEUE)
    vp, i32 = ctypes.c_void_p, ctypes.c_int
    enqueue.argtypes = [vp, vp, i32, i32, i32, vp, i32, i32, vp, i32,
                        ctypes.POINTER(Scratch)]
    bufs = [ctx.alloc(8 * WORK), ctx.alloc(8 * WORK), ctx.alloc(4 * PERM),
            ctx.alloc(4 * FLAGS)]
    d = ctx.alloc(8 * n * nrhs)
    w = Scratch(bufs[0].ptr, bufs[1].ptr, WORK, bufs[2].ptr, bufs[3].ptr, 1,
                None, 1 << 22)
    B = np.asfortranarray(np.random.default_rng(n).standard_normal((n, nrhs)))
    mat = ctx.pmat_alloc(n, nb)
    hip = ctypes.CDLL("libamdhip64.so.7")
    try:
        ctx.pdrandmat(n, n, nb, mat.A, mat.ld, rp.HPL_ISEED, 0.0)
        assert ctx.pdgetrf(rp.palg_default(), mat) == 0
        for trans in (0, 1):
            print("[gpu-case] getrs, flags raised n=%d nrhs=%d trans=%d"
                  % (n, nrhs, trans), flush=True)
            d.upload(B)
            ctx.pdgetrs(mat, trans, nrhs, d.ptr, n)
            want = d.download((n, nrhs), np.float64)
            d.upload(B)
            assert enqueue(None, mat.A, n, nb, mat.ld, mat.ipiv, trans, nrhs, d.ptr, n,
                           ctypes.byref(w)) == 0
            assert hip.hipDeviceSynchronize() == 0
            assert np.array_equal(d.download((n, nrhs), np.float64), want)
    finally:
        ctx.pmat_free(mat)
        for b in bufs + [d]:
            b.free()


def test_a_wait_that_gives_up_is_an_error(ctx, monkeypatch):
    """With no failed poll allowed, every entry point that solves on the device
    reports it, with NaNs in the solution, and a solve of one block, which waits
    for nothing, still succeeds afterwards."""
    monkeypatch.setenv("HPLX_SOLVE_POLLS", "0")
    n, nb, nrhs = 1000, 128, 3
    with rp.Context(0) as c:
        mat, small = c.pmat_alloc(n, nb), c.pmat_alloc(64, 64)
        d = c.alloc(8 * n * nrhs)
        g = c.alloc(8 * n * nrhs)
        B = np.asfortranarray(np.random.default_rng(1).standard_normal((n, nrhs)))
        try:
            for m in (mat, small):
                c.pdrandmat(m.n, m.n + 1, m.nb, m.A, m.ld)
                assert c.pdgetrf(rp.palg_default(), m) == 0
            for what, call in (
                    ("getrs", lambda: c.pdgetrs(mat, 0, nrhs, d.ptr, n)),
                    ("getrs trans", lambda: c.pdgetrs(mat, 1, nrhs, d.ptr, n)),
                    ("adjoint", lambda: c.pdgesv_adjoint(mat, nrhs, d.ptr, n, d.ptr, n,
                                                         g.ptr, n, None, n)),
                    ("trsv", lambda: c.pdtrsv(n, nb, mat.A, mat.ld, d.ptr)),
                    ("gesv", lambda: (c.pdrandmat(n, n + 1, nb, mat.A, mat.ld),
                                      c.pdgesv(rp.palg_default(), mat)))):
                print("[gpu-case] no failed polls: " + what, flush=True)
                d.upload(B)
                with pytest.raises(rp.HplxError) as e:
                    call()
                assert e.value.code == rp.HPLX_ERR_HIP and "timed out" in str(e.value)
                if what.startswith("getrs"):
                    assert np.isnan(d.download((n, nrhs), np.float64)).any()
                d.upload(np.asfortranarray(B[:64]))
                c.pdgetrs(small, 0, nrhs, d.ptr, 64)
                assert np.all(np.isfinite(d.download((64, nrhs), np.float64)))
        finally:
            d.free()
            g.free()
            c.pmat_free(mat)
            c.pmat_free(small)
