"""Timed cases of rochpl_amd: what its users run, from the smallest solve to
the panels and updates of the full-size one.

Every case is one call (or one HPL test: generate, then solve) through the
public entry points of rochpl_amd, on inputs made from a seed.  Kinds:

  solve    an HPL test: pdrandmat, then pdgesv (FP64); x and the pivots
  getrf    pdrandmat, then pdgetrf: the factors and the pivots
  getrs    right-hand sides solved with stored factors (pdgetrs, or
           pdgetrs_noalloc as a serving loop calls it), A or A^T
  adjoint  the backward pass of a solve: pdgesv_adjoint, gradB and gradA
  mixed    hplx_mxp_pdgesv in the BF16 or the FP8 form: x and the pivots
  update   one trailing update of a factorisation (pdupdate)
  panel    one panel of a factorisation (pdfact)
  verify   the rest of an HPL test: the matrix, and the residual check of a x

torch is imported before rochpl_amd so that both use one HIP runtime.
"""
import ctypes
import math

import numpy as np
import torch

import rochpl_amd as rp

_DEV = "cuda:0"
_HPL = {}  # the program's context and stream, made at the first use


def _context():
    if not _HPL:
        torch.zeros(1, device=_DEV)
        stream = torch.cuda.Stream()
        ctx = rp.Context(0)
        ctx.set_stream(stream.cuda_stream)
        _HPL.update(ctx=ctx, stream=stream)
    return _HPL["ctx"], _HPL["stream"]


# ---- the cases --------------------------------------------------------------
def listed():
    return [
        # the smallest solves: one of HPL.dat's small sizes, where launches
        # and the latency of each pivot column count
        {"name": "solve_1000_nb64", "kind": "solve", "n": 1000, "nb": 64},
        # the sample input file: N = 4096, NB = 256
        {"name": "solve_4096_nb256", "kind": "solve", "n": 4096, "nb": 256},
        # an odd N whose last panel is ragged
        {"name": "solve_9001_nb384", "kind": "solve", "n": 9001, "nb": 384},
        # the largest factorisation that takes under a second, NB as in the
        # full-size run
        {"name": "getrf_32768_nb896", "kind": "getrf", "n": 32768, "nb": 896,
         "shift": 0.0},
        # the adjoint workload's forward and backward solves: N = 16384,
        # 64 right-hand sides, A = U(-0.5, 0.5) + 2 sqrt(N) I
        {"name": "getrs_16384_rhs64", "kind": "getrs", "n": 16384, "nb": 512,
         "nrhs": 64, "trans": 0, "noalloc": False, "shift": 256.0},
        {"name": "adjoint_16384_rhs64", "kind": "adjoint", "n": 16384,
         "nb": 512, "nrhs": 64, "grad_a": True, "shift": 256.0},
        # one right-hand side at a time, as a serving loop solves
        {"name": "serve_5000_rhs1", "kind": "getrs", "n": 5000, "nb": 128,
         "nrhs": 1, "trans": 0, "noalloc": True, "shift": 0.0},
        # the mixed forms: BF16 x 3 terms with FP32 factors, and FP8 with
        # FP16 factors on the diagonally dominant matrix
        {"name": "bf16_16384_nb512", "kind": "mixed", "form": "bf16",
         "n": 16384, "nb": 512, "shift": 0.0},
        {"name": "fp8_32768_nb1024", "kind": "mixed", "form": "fp8",
         "n": 32768, "nb": 1024, "shift": 8192.0},
        # one step of a large FP64 solve: its update and its panel
        {"name": "update_24576_nb896", "kind": "update", "m": 24576 + 896,
         "n": 24577, "jb": 896},
        {"name": "panel_131072_nb896", "kind": "panel", "m": 131072,
         "jb": 896},
        # what surrounds the solve in an HPL test
        {"name": "verify_20000", "kind": "verify", "n": 20000, "nb": 512},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "getrf", "getrs", "getrs", "adjoint",
                       "mixed", "mixed", "update", "panel", "verify"])
    c = {"kind": kind}
    if kind == "solve":
        c["n"] = _log_int(rng, 200, 9001)
        c["nb"] = min(c["n"], _log_int(rng, 16, 512))
    elif kind == "getrf":
        c.update(n=_log_int(rng, 6000, 28000), nb=rng.randint(128, 1024),
                 shift=0.0)
    elif kind == "getrs":
        c["n"] = _log_int(rng, 300, 16384)
        c.update(nb=_log_int(rng, 32, 1024), nrhs=_log_int(rng, 1, 128),
                 trans=rng.randint(0, 1), noalloc=rng.random() < 0.5,
                 # large unshifted matrices are too ill-conditioned for two
                 # orders of the same sums to agree to nine digits
                 shift=0.0 if c["n"] <= 5000 else round(2 * c["n"] ** 0.5, 3))
    elif kind == "adjoint":
        c["n"] = _log_int(rng, 500, 16384)
        c.update(nb=_log_int(rng, 32, 1024), nrhs=_log_int(rng, 1, 96),
                 grad_a=rng.random() < 0.7,
                 shift=round(2 * c["n"] ** 0.5, 3))
    elif kind == "mixed":
        c["form"] = rng.choice(["bf16", "fp8"])
        if c["form"] == "bf16":
            c.update(n=_log_int(rng, 2000, 16384), nb=rng.randint(64, 512),
                     shift=0.0)
        else:
            c.update(n=_log_int(rng, 3000, 32768), nb=rng.randint(128, 1024))
            c["shift"] = c["n"] / 4.0
    elif kind == "update":
        c.update(jb=rng.randint(48, 1024), n=_log_int(rng, 500, 24577))
        c["m"] = c["jb"] + _log_int(rng, 500, 24577)
    elif kind == "panel":
        c.update(m=_log_int(rng, 3000, 131072), jb=rng.randint(32, 896))
    else:
        c.update(n=_log_int(rng, 1000, 20000), nb=rng.randint(64, 1024))
    return c


def work(case):
    """Each input read once and each output written once; the operations of
    the usual counts (2/3 N^3 + 3/2 N^2 for a solve)."""
    k = case["kind"]
    if k in ("solve", "getrf", "mixed"):
        n = case["n"]
        es = 8 if k != "mixed" else 4 if case["form"] == "bf16" else 2
        return {"bytes": 2.0 * es * n * (n + 1),
                "flops": 2.0 / 3.0 * n ** 3 + 1.5 * n ** 2}
    if k == "getrs":
        n, r = case["n"], case["nrhs"]
        return {"bytes": 8.0 * n * n + 16.0 * n * r, "flops": 2.0 * n * n * r}
    if k == "adjoint":
        n, r, g = case["n"], case["nrhs"], case["grad_a"]
        return {"bytes": 8.0 * n * n * (2 if g else 1) + 24.0 * n * r,
                "flops": 2.0 * n * n * r * (2 if g else 1)}
    if k == "update":
        m, n, jb = case["m"], case["n"], case["jb"]
        return {"bytes": 16.0 * m * n + 8.0 * m * jb,
                "flops": 1.0 * jb * jb * n + 2.0 * (m - jb) * n * jb}
    if k == "panel":
        m, jb = case["m"], case["jb"]
        return {"bytes": 16.0 * m * jb, "flops": jb * jb * (m - jb / 3.0)}
    n = case["n"]  # verify: generate once, regenerate by rows and by columns
    return {"bytes": 8.0 * n * (n + 1), "flops": 3.0 * n * (n + 1)}


# ---- states -----------------------------------------------------------------
class _Matrix:
    """A matrix the library allocated, freed when nothing refers to it."""

    def __init__(self, ctx, mat, free):
        self.ctx, self.mat, self.free = ctx, mat, free

    def __del__(self):
        try:
            self.free(self.mat)
        except Exception:  # the interpreter is going down
            pass


class _Part:
    """Device memory of a _Matrix for torch, which holds this object, and so
    the matrix, for as long as a tensor refers to the memory."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape,
                                         "typestr": typestr, "version": 2,
                                         "strides": None}


def _view(owner, ptr, shape, typestr):
    return torch.as_tensor(_Part(owner, ptr, shape, typestr), device=_DEV)


class _State:
    """What the caller holds: a matrix of the library and torch tensors."""

    def __init__(self, case, seed):
        self.case, self.seed = case, int(seed) % (1 << 31)
        self.ctx, self.stream = _context()

    def matrix(self):
        m = self.mat = self.ctx.pmat_alloc(self.case["n"], self.case["nb"])
        own = self.owner = _Matrix(self.ctx, m, self.ctx.pmat_free)
        self.A = _view(own, m.A, (m.n + 1, m.ld), "<f8")  # row j: column j
        self.x = _view(own, m.X, (m.n,), "<f8")
        self.ipiv = _view(own, m.ipiv, (m.n,), "<i4")
        return m

    def mixed_matrix(self, storage):
        m = self.mat = self.ctx.mxp_alloc(self.case["n"], self.case["nb"],
                                          storage)
        own = self.owner = _Matrix(self.ctx, m, self.ctx.mxp_free)
        self.x = _view(own, m.X, (m.n,), "<f8")
        self.ipiv = _view(own, m.ipiv, (m.n,), "<i4")


def _gen(seed):
    return torch.Generator(device=_DEV).manual_seed(int(seed))


def _normal(rows, cols, seed):
    """rows x cols column-major: a (cols, rows) tensor."""
    return torch.randn(cols, rows, generator=_gen(seed), dtype=torch.float64,
                       device=_DEV)


def _uniform(rows, cols, ld, seed):
    a = torch.rand(cols, ld, generator=_gen(seed), dtype=torch.float64,
                   device=_DEV)
    return a.sub_(0.5)


def prepare(case, seed):
    s = _State(case, seed)
    ctx = s.ctx
    with torch.cuda.stream(s.stream):
        k = case["kind"]
        if k in ("solve", "getrf"):
            s.matrix()
        elif k in ("getrs", "adjoint"):
            n, r = case["n"], case["nrhs"]
            m = s.matrix()
            ctx.pdrandmat(n, n, m.nb, m.A, m.ld, s.seed, case["shift"])
            if ctx.pdgetrf(rp.palg_default(), m) != 0:
                raise RuntimeError("zero pivot")
            s.B = _normal(n, r, seed)
            s.X = torch.empty_like(s.B)
            if k == "adjoint":  # the forward pass: X, and its gradient G
                s.X.copy_(s.B)
                ctx.pdgetrs(m, 0, r, s.X.data_ptr(), n)
                s.G = _normal(n, r, seed + 1)
                s.gB = torch.empty_like(s.G)
                s.gA = torch.empty((n, n), dtype=torch.float64, device=_DEV) \
                    if case["grad_a"] else None
        elif k == "mixed":
            f16 = case["form"] == "fp8"
            s.mixed_matrix(rp.HPLX_STORE_FP16 if f16 else rp.HPLX_STORE_FP32)
            s.opts = rp.mxp_opts_default(
                rp.HPLX_UPDATE_FP8 if f16 else rp.HPLX_UPDATE_BF16,
                1 if f16 else 3)
        elif k == "update":
            m, n, jb = case["m"], case["n"], case["jb"]
            s.lda = rp.hpl_ld(m)
            s.A = _uniform(m, jb + n, s.lda, seed)
            ipiv = torch.empty(jb, dtype=torch.int32, device=_DEV)
            s.permU = torch.empty(2 * jb, dtype=torch.int32, device=_DEV)
            s.W = torch.empty(jb * (n + 4), dtype=torch.float64, device=_DEV)
            s.A0 = s.A[jb:].clone()
            ctx.pdfact(s.A.data_ptr(), s.lda, m, jb, ipiv.data_ptr())
            ctx.pipid(jb, ipiv.data_ptr(), s.permU.data_ptr())
        elif k == "panel":
            m, jb = case["m"], case["jb"]
            s.lda = rp.hpl_ld(m)
            s.P0 = _uniform(m, jb, s.lda, seed)
            s.P = torch.empty_like(s.P0)
            s.ipiv = torch.empty(jb, dtype=torch.int32, device=_DEV)
        else:
            m = s.matrix()
            s.x.copy_(_normal(m.n, 1, seed)[0])
    return s


def run(s):
    case, ctx = s.case, s.ctx
    k = case["kind"]
    with torch.cuda.stream(s.stream):
        if k == "solve":
            n, m = case["n"], s.mat
            ctx.pdrandmat(n, n + 1, m.nb, m.A, m.ld, s.seed)
            ctx.pdgesv(rp.palg_default(), m)
            return {"x": s.x, "ipiv": s.ipiv}
        if k == "getrf":
            n, m = case["n"], s.mat
            ctx.pdrandmat(n, n, m.nb, m.A, m.ld, s.seed, case["shift"])
            ctx.pdgetrf(rp.palg_default(), m)
            return {"lu": s.A[:n, :n], "ipiv": s.ipiv}
        if k == "getrs":
            n, r = case["n"], case["nrhs"]
            s.X.copy_(s.B)
            if case["noalloc"]:
                rc = rp.lib().hplx_pdgetrs_noalloc(
                    ctypes.byref(s.mat), case["trans"], r,
                    ctypes.c_void_p(s.X.data_ptr()), n,
                    ctypes.c_void_p(s.stream.cuda_stream))
                if rc != 0:
                    raise RuntimeError("pdgetrs_noalloc: %d" % rc)
            else:
                ctx.pdgetrs(s.mat, case["trans"], r, s.X.data_ptr(), n)
            return s.X
        if k == "adjoint":
            n, r = case["n"], case["nrhs"]
            ctx.pdgesv_adjoint(s.mat, r, s.X.data_ptr(), n, s.G.data_ptr(), n,
                               s.gB.data_ptr(), n,
                               s.gA.data_ptr() if case["grad_a"] else None, n)
            return {"gB": s.gB, "gA": s.gA} if case["grad_a"] else {"gB": s.gB}
        if k == "mixed":
            ctx.mxp_matgen(s.mat, s.seed, case["shift"])
            ctx.mxp_pdgesv(rp.palg_default(), s.opts, s.mat)
            return {"x": s.x, "ipiv": s.ipiv}
        if k == "update":
            m, n, jb = case["m"], case["n"], case["jb"]
            s.A[jb:].copy_(s.A0)  # in place: each pass updates fresh columns
            ctx.pdupdate(s.A.data_ptr(), s.lda, m, jb, n, s.permU.data_ptr(),
                         s.W.data_ptr())
            return s.A[jb:, :m]
        if k == "panel":
            s.P.copy_(s.P0)
            ctx.pdfact(s.P.data_ptr(), s.lda, case["m"], case["jb"],
                       s.ipiv.data_ptr())
            return {"lu": s.P[:, :case["m"]], "ipiv": s.ipiv}
        n, m = case["n"], s.mat
        ctx.pdrandmat(n, n + 1, m.nb, m.A, m.ld, s.seed)
        chk = ctx.pdtest_check(m, s.seed)
        return {"A": s.A[:, :n],
                "norms": np.array([chk[q] for q in (
                    "rnorm", "AnormI", "Anorm1", "XnormI", "Xnorm1",
                    "BnormI")])}


# ---- exact values -----------------------------------------------------------
_MULT, _MASK = 6364136223846793005, (1 << 64) - 1


def _jump(k):
    """(a, c) of k steps of the generator s -> MULT s + 1 mod 2^64."""
    a, c, pa, pc = 1, 0, _MULT, 1
    while k:
        if k & 1:
            a, c = pa * a & _MASK, (pa * c + pc) & _MASK
        pa, pc = pa * pa & _MASK, (pa * pc + pc) & _MASK
        k >>= 1
    return a, c


def _maps(step, count):
    """The maps of 0, step, 2 step, ... generator steps (numpy uint64)."""
    a, c = np.ones(1, np.uint64), np.zeros(1, np.uint64)
    while a.size < count:
        ja, jc = (np.uint64(v) for v in _jump(step * a.size))
        a, c = np.concatenate([a, a * ja]), np.concatenate([c, c * ja + jc])
    return a[:count], c[:count]


def _hpl_columns(seed, n, cols, shift=0.0):
    """Rows: the first `cols` columns of the n-row HPL matrix of this seed."""
    start = np.uint64((_MULT * seed + 1) & _MASK)
    ra, rc = (torch.from_numpy(v.view(np.int64)).to(_DEV) for v in _maps(1, n))
    ca, cc = _maps(n, cols)
    cs = torch.from_numpy((ca * start + cc).view(np.int64)).to(_DEV)
    out = torch.empty((cols, n), dtype=torch.float64, device=_DEV)
    for j in range(0, cols, 1024):
        s = cs[j:j + 1024, None] * ra + rc
        d = ((s >> 32) & 0xffffffff).double()
        d += (s & 0xffffffff).double() * 2.0 ** -32
        out[j:j + 1024] = 0.5 - d * 2.0 ** -32
    if shift:
        i = torch.arange(min(n, cols), device=_DEV)
        out[i, i] += shift
    return out


def _row_order(piv, m):
    """The row order that the interchanges i <-> piv[i] (0-based) give."""
    order = np.arange(m)
    for i, p in enumerate(piv):
        order[[i, p]] = order[[p, i]]
    return torch.from_numpy(order).to(_DEV)


def _lu(A, w=192):
    """A (n x n) factored in place by columns of w, their pivots found on the
    CPU (some library versions do not take the largest on the GPU)."""
    n, piv = A.shape[0], np.empty(A.shape[0], np.int64)
    for j in range(0, n, w):
        e = min(n, j + w)
        P, p = torch.linalg.lu_factor(A[j:, j:e].cpu())
        p = p.numpy() - 1
        piv[j:e] = p + j
        A[j:] = A[j:][_row_order(p, n - j)]
        A[j:, j:e] = P.to(A.device)
        if e < n:
            A[j:e, e:] = torch.linalg.solve_triangular(
                A[j:e, j:e], A[j:e, e:], upper=False, unitriangular=True)
            A[e:, e:] -= A[e:, j:e] @ A[j:e, e:]
    return A, piv


def exact(case, seed):
    k, hs = case["kind"], int(seed) % (1 << 31)
    if k == "solve" or (k == "mixed" and case["form"] == "bf16"):
        n = case["n"]
        Ab = _hpl_columns(hs, n, n + 1)
        return {"x": torch.linalg.solve(Ab[:n].t(), Ab[n]), "ipiv": None}
    if k == "mixed":  # diagonally dominant: the Jacobi iteration converges
        n = case["n"]
        Ab = _hpl_columns(hs, n, n + 1, case["shift"])
        A, b = Ab[:n].t(), Ab[n]
        d = A.diagonal().clone()
        x = b / d
        for _ in range(25):
            x = x + (b - A @ x) / d
        return {"x": x, "ipiv": None}
    if k == "getrf":
        n, nb = case["n"], case["nb"]
        LU, piv = _lu(_hpl_columns(hs, n, n, case["shift"]).t().contiguous())
        # HPL leaves each panel's multipliers where that panel put them: the
        # interchanges of the later panels are taken back
        order = np.arange(n)
        for j in range((n - 1) // nb * nb, -1, -nb):
            e = min(n, j + nb)
            LU[e:, j:e] = LU[torch.from_numpy(order[e:]).to(_DEV), j:e]
            for i in range(e - 1, j - 1, -1):
                order[[i, piv[i]]] = order[[piv[i], i]]
        return {"lu": LU.t().contiguous(), "ipiv": None}
    if k in ("getrs", "adjoint"):
        n, r = case["n"], case["nrhs"]
        A = _hpl_columns(hs, n, n, case["shift"]).t()
        B = _normal(n, r, seed).t()
        if k == "getrs":
            return torch.linalg.solve(A.t() if case["trans"] else A, B).t()
        X = torch.linalg.solve(A, B)
        gB = torch.linalg.solve(A.t(), _normal(n, r, seed + 1).t())
        out = {"gB": gB.t()}
        if case["grad_a"]:
            out["gA"] = -(X @ gB.t())
        return out
    if k == "update":
        m, n, jb = case["m"], case["n"], case["jb"]
        A = _uniform(m, jb + n, rp.hpl_ld(m), seed)[:, :m]
        LU, piv = torch.linalg.lu_factor(A[:jb].t())
        B = A[jb:].t()[_row_order(piv.cpu().numpy() - 1, m)]
        U = torch.linalg.solve_triangular(LU[:jb], B[:jb], upper=False,
                                          unitriangular=True)
        B[:jb] = U
        B[jb:] -= LU[jb:] @ U
        return B.t()
    if k == "panel":
        m, jb = case["m"], case["jb"]
        LU, _ = torch.linalg.lu_factor(
            _uniform(m, jb, rp.hpl_ld(m), seed)[:, :m].t())
        return {"lu": LU.t(), "ipiv": None}
    n = case["n"]
    Ab = _hpl_columns(hs, n, n + 1)
    x = _normal(n, 1, seed)[0]
    A = Ab[:n]
    return {"A": Ab,
            "norms": np.array([float(v) for v in (
                (Ab[n] - x @ A).abs().max(), A.abs().sum(0).max(),
                A.abs().sum(1).max(), x.abs().max(), x.abs().sum(),
                Ab[n].abs().max())])}
