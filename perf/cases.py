"""Performance cases of the library: what a program has it do, over the sizes,
data types and options that the public entry points are used with.

Every case runs on device-resident operands through the C entry points, on one
HIP stream that the program hands to the library once (calls are then
asynchronous on that stream, as a GPU program uses them). Matrices are
column-major: a matrix of r rows and c columns is a torch tensor of c rows of
`ld` elements, of which the first r are the column. "tight" leading dimensions
equal the rows; "pad8" ones are the rows rounded up to a multiple of 8.
"""
import ctypes as C
import math

import numpy as np
import torch

import blis_amd

TORCH = {"d": torch.float64, "s": torch.float32, "z": torch.complex128, "c": torch.complex64}
REAL = {"z": "d", "c": "s"}
CTYPE = {"d": C.c_double, "s": C.c_float}
TRANS = {"n": blis_amd.BLIS_NO_TRANSPOSE, "t": blis_amd.BLIS_TRANSPOSE,
         "c": blis_amd.BLIS_CONJ_TRANSPOSE}
BYTES = {"d": 8, "s": 4, "z": 16, "c": 8}


def listed():
    return [
        # The smallest call: one small product, where the launch is the cost.
        dict(name="dgemm_small", kind="gemm", dt="d", trans="nn", m=130, n=120, k=140, ld="tight"),
        # The small dense product of the plain-GEMM workload (512^3, beta 0.5).
        dict(name="dgemm_512", kind="gemm", dt="d", trans="nn", m=512, n=512, k=512, ld="tight"),
        # An ordinary product of odd sizes on tight storage: what comes out of
        # data whose dimensions nobody rounded.
        dict(name="dgemm_ragged_tn", kind="gemm", dt="d", trans="tn", m=1999, n=1501, k=1003,
             ld="tight"),
        # The large square product, the benchmark's headline.
        dict(name="dgemm_8192", kind="gemm", dt="d", trans="nn", m=8192, n=8192, k=8192,
             ld="tight"),
        # A rank-256 update of a large matrix, the trailing update of a blocked
        # factorisation, in single precision.
        dict(name="sgemm_8192_k256", kind="gemm", dt="s", trans="nt", m=8192, n=8192, k=256,
             ld="tight"),
        # Gram matrix X^T X of 30,000 samples of 500 features (normal equations).
        dict(name="dsyrk_gram", kind="syrk", dt="d", uplo="l", trans="t", n=500, k=30000,
             ld="tight"),
        # Triangular solve with many right-hand sides on a diagonally dominant
        # triangle, the benchmark's TRSM.
        dict(name="dtrsm_4096x1024", kind="trsm", dt="d", side="l", uplo="l", trans="n", diag="n",
             m=4096, n=1024, tri="dominant", ld="tight"),
        # The panel solve X L^T = B of a blocked Cholesky factorisation, odd
        # sizes, a factor that is not diagonally dominant.
        dict(name="strsm_panel", kind="trsm", dt="s", side="r", uplo="l", trans="t", diag="n",
             m=3001, n=515, tri="factor", ld="tight"),
        # The uneven batch: 10,000 products, dims log-uniform in [8, 512].
        dict(name="dbatch_10000", kind="batch", dt="d", count=10000, lo=8, hi=512, shapes=42),
        # A gradient step of least squares on a large dense matrix: gemv both
        # ways, dot and axpy, bound by memory.
        dict(name="dlsq_16384", kind="lsq", dt="d", m=16384, n=16384, ld="tight"),
        # Split-precision product on the INT8 units at the benchmark's size.
        dict(name="dsplit_8192", kind="split", dt="d", m=8192, n=8192, k=8192, sigma=0),
        # A complex product A B^H of odd sizes.
        dict(name="zgemm_ragged", kind="zgemm", dt="z", trans="nc", m=777, n=1030, k=641,
             ld="tight"),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["gemm", "gemm", "gemm", "syrk", "trsm", "batch", "lsq", "split", "zgemm"])
    dt = rng.choice("ds")
    ld = rng.choice(["tight", "pad8"])
    if kind == "gemm":
        return dict(kind=kind, dt=dt, trans=rng.choice(["nn", "nt", "tn", "tt"]),
                    m=size(64, 8192), n=size(64, 8192), k=size(64, 8192), ld=ld)
    if kind == "syrk":
        n = size(64, 4096)
        return dict(kind=kind, dt=dt, uplo=rng.choice("lu"), trans=rng.choice("nt"), n=n,
                    k=size(64, min(65536, (1 << 27) // n)), ld=ld)
    if kind == "trsm":
        return dict(kind=kind, dt=dt, side=rng.choice("lr"), uplo=rng.choice("lu"),
                    trans=rng.choice("nt"), diag=rng.choice("nu"), m=size(64, 4096),
                    n=size(64, 4096), tri=rng.choice(["dominant", "factor"]), ld=ld)
    if kind == "batch":
        return dict(kind=kind, dt=dt, count=size(100, 10000), lo=8, hi=size(32, 512),
                    shapes=rng.randrange(1 << 30))
    if kind == "lsq":
        return dict(kind=kind, dt=dt, m=size(256, 16384), n=size(256, 16384), ld=ld)
    if kind == "split":
        return dict(kind=kind, dt=dt, m=size(1024, 8192), n=size(1024, 8192), k=size(1024, 8192),
                    sigma=rng.choice([0, 4, 8]) if dt == "d" else 0)
    return dict(kind="zgemm", dt=rng.choice("zc"),
                trans=rng.choice("ntc") + rng.choice("ntc"), m=size(64, 2048), n=size(64, 2048),
                k=size(64, 2048), ld=ld)


# ---- storage ----------------------------------------------------------------

_stream = None


def _use_stream():
    """The program's one stream, handed to the library once."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
        blis_amd.lib().bli_amd_set_stream(_stream.cuda_stream, 0)
    return _stream


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _ld(rows, how):
    return rows if how == "tight" else (rows + 7) // 8 * 8


def _uniform(g, shape, dt):
    """Entries uniform in [-1, 1]."""
    if dt in REAL:
        re = torch.rand((*shape, 2), generator=g, device="cuda", dtype=TORCH[REAL[dt]])
        return torch.view_as_complex(re.mul_(2).sub_(1))
    return torch.rand(shape, generator=g, device="cuda", dtype=TORCH[dt]).mul_(2).sub_(1)


def _mat(g, rows, cols, dt, how):
    return _uniform(g, (cols, _ld(rows, how)), dt)


def _scalar(dt, v):
    if dt in REAL:
        return (CTYPE[REAL[dt]] * 2)(v, 0.0)
    return CTYPE[dt](v)


def _dims(t, r, c):
    """Stored rows and columns of an operand whose op() is r x c."""
    return (r, c) if t == "n" else (c, r)


def _op(buf, rows, t):
    """op(matrix) in 64 bits, from its column-major buffer."""
    x = buf[:, :rows].to(torch.complex128 if buf.is_complex() else torch.float64)
    x = x.T
    return x if t == "n" else (x.T if t == "t" else x.T.conj())


# ---- inputs -----------------------------------------------------------------

def _gemm_inputs(case, seed):
    g, dt = _gen(seed), case["dt"]
    m, n, k, (ta, tb) = case["m"], case["n"], case["k"], case["trans"]
    how = case.get("ld", "tight")
    return (_mat(g, *_dims(ta, m, k), dt, how), _mat(g, *_dims(tb, k, n), dt, how),
            _mat(g, m, n, dt, how))


def _syrk_inputs(case, seed):
    g = _gen(seed)
    return (_mat(g, *_dims(case["trans"], case["n"], case["k"]), case["dt"], case["ld"]),
            _mat(g, case["n"], case["n"], case["dt"], case["ld"]))


def _trsm_inputs(case, seed):
    """dominant: entries in [-1, 1], diagonal the order plus [0, 1] (entries
    scaled by the order under a unit diagonal); factor: a well-conditioned
    triangle with entries of about 1/sqrt(order) below a diagonal in [1, 2],
    like the Cholesky factor of a covariance, not diagonally dominant."""
    g, dt = _gen(seed), case["dt"]
    q = case["m"] if case["side"] == "l" else case["n"]
    a = _mat(g, q, q, dt, case["ld"])
    if case["tri"] == "factor":
        a.mul_(1.0 / math.sqrt(q))
    elif case["diag"] == "u":
        a.mul_(1.0 / q)
    d = a[:, :q].diagonal()
    d.copy_(torch.rand(q, generator=g, device="cuda", dtype=a.dtype).add_(
        q if case["tri"] == "dominant" else 1.0))
    return a, _mat(g, case["m"], case["n"], dt, case["ld"])


def _batch_shapes(case):
    """(m, n, k, ta, tb) of each problem, alpha and beta."""
    r = np.random.default_rng(case["shapes"])
    lo, hi, cnt = math.log(case["lo"]), math.log(case["hi"]), case["count"]
    dims = np.rint(np.exp(r.uniform(lo, hi, (3, cnt)))).astype(np.int64)
    tr = r.integers(0, 2, (2, cnt))
    return dims, tr, r.uniform(-1, 1, (2, cnt))


def _batch_layout(case):
    """Leading dimensions (multiples of 8) and offsets into one arena per operand."""
    (m, n, k), (ta, tb), _ = _batch_shapes(case)
    rows = [np.where(ta == 1, k, m), np.where(tb == 1, n, k), m]
    cols = [np.where(ta == 1, m, k), np.where(tb == 1, k, n), n]
    ld = [(r + 7) // 8 * 8 for r in rows]
    size = [a * b for a, b in zip(ld, cols)]
    off = [np.concatenate([[0], np.cumsum(s)]) for s in size]
    return rows, cols, ld, off


def _batch_inputs(case, seed):
    g = _gen(seed)
    _, _, _, off = _batch_layout(case)
    return [_uniform(g, (int(o[-1]),), case["dt"]) for o in off]


def _lsq_inputs(case, seed):
    g, dt = _gen(seed), case["dt"]
    return (_mat(g, case["m"], case["n"], dt, case["ld"]), _uniform(g, (case["n"],), dt),
            _uniform(g, (case["m"],), dt))


def _lsq_eta(case):
    """A step below 1/sigma_max(A)^2 for entries uniform in [-1, 1]."""
    return 1.5 / (math.sqrt(case["m"]) + math.sqrt(case["n"])) ** 2


def _split_inputs(case, seed):
    g, dt = _gen(seed), case["dt"]

    def spread(r, c):
        u = _uniform(g, (c, r), dt)
        if case["sigma"]:
            e = torch.randn((c, r), generator=g, device="cuda", dtype=torch.float32)
            u = torch.ldexp(u, e.mul_(case["sigma"]).round_().to(torch.int32))
        return u

    return (spread(case["m"], case["k"]), spread(case["k"], case["n"]),
            _uniform(g, (case["n"], case["m"]), dt))


# ---- preparation, one pass ----------------------------------------------------

def prepare(case, seed):
    _use_stream()
    return globals()["_prepare_" + case["kind"]](case, seed, blis_amd.lib())


def run(state):
    return state["run"](state)


def _call(state):
    for f, args in state["calls"]:
        f(*args)
    return state["out"]


def _prepare_gemm(case, seed, lib):
    a, b, c = _gemm_inputs(case, seed)
    dt, (ta, tb) = case["dt"], case["trans"]
    args = (TRANS[ta], TRANS[tb], case["m"], case["n"], case["k"], _scalar(dt, 1.0),
            a.data_ptr(), 1, a.shape[1], b.data_ptr(), 1, b.shape[1], _scalar(dt, 0.5),
            c.data_ptr(), 1, c.shape[1])
    return {"run": _call, "calls": [(getattr(lib, f"bli_{dt}gemm"), args)], "out": [c],
            "keep": (a, b)}


_prepare_zgemm = _prepare_gemm


def _prepare_syrk(case, seed, lib):
    a, c = _syrk_inputs(case, seed)
    dt = case["dt"]
    args = (blis_amd.BLIS_LOWER if case["uplo"] == "l" else blis_amd.BLIS_UPPER,
            TRANS[case["trans"]], case["n"], case["k"], _scalar(dt, 1.0), a.data_ptr(), 1,
            a.shape[1], _scalar(dt, 0.0), c.data_ptr(), 1, c.shape[1])
    return {"run": _call, "calls": [(getattr(lib, f"bli_{dt}syrk"), args)], "out": [c],
            "keep": (a,)}


def _run_trsm(state):
    # The solve overwrites its right-hand side, so each pass starts from a copy.
    with torch.cuda.stream(_stream):
        state["b"].copy_(state["b0"])
    return _call(state)


def _prepare_trsm(case, seed, lib):
    a, b0 = _trsm_inputs(case, seed)
    dt, b = case["dt"], torch.empty_like(b0)
    args = (blis_amd.BLIS_LEFT if case["side"] == "l" else blis_amd.BLIS_RIGHT,
            blis_amd.BLIS_LOWER if case["uplo"] == "l" else blis_amd.BLIS_UPPER,
            TRANS[case["trans"]],
            blis_amd.BLIS_UNIT_DIAG if case["diag"] == "u" else blis_amd.BLIS_NONUNIT_DIAG,
            case["m"], case["n"], _scalar(dt, 1.0), a.data_ptr(), 1, a.shape[1], b.data_ptr(), 1,
            b.shape[1])
    return {"run": _run_trsm, "calls": [(getattr(lib, f"bli_{dt}trsm"), args)], "out": [b],
            "b": b, "b0": b0, "keep": (a,)}


class _Plan:
    """A batch plan that is given back with the state that holds it."""

    def __init__(self, lib, handle):
        self.lib, self.handle = lib, handle

    def __del__(self):
        torch.cuda.synchronize()
        self.lib.bli_amd_gemm_batch_plan_destroy(self.handle)


def _prepare_batch(case, seed, lib):
    dt, cnt = case["dt"], case["count"]
    (m, n, k), tr, (alpha, beta) = _batch_shapes(case)
    _, _, ld, off = _batch_layout(case)
    bufs = _batch_inputs(case, seed)
    real = np.float64 if dt == "d" else np.float32
    ptrs = [np.ascontiguousarray(x.data_ptr() + o[:-1] * BYTES[dt]) for x, o in zip(bufs, off)]
    trans = [np.where(t == 1, blis_amd.BLIS_TRANSPOSE, 0).astype(np.int32) for t in tr]
    one = np.ones(cnt, np.int64)
    arrs = [trans[0], trans[1], m, n, k, alpha.astype(real), ptrs[0], one, ld[0], ptrs[1], one,
            ld[1], beta.astype(real), ptrs[2], one, ld[2]]
    arrs = [np.ascontiguousarray(x) for x in arrs]
    torch.cuda.synchronize()
    handle = getattr(lib, f"bli_amd_{dt}gemm_batch_plan_create")(
        *[x.ctypes.data for x in arrs], cnt, one.ctypes.data)
    plan = _Plan(lib, handle)
    return {"run": _call, "calls": [(lib.bli_amd_gemm_batch_plan_execute, (handle, 1))],
            "out": [bufs[2]], "keep": (bufs, plan)}


def _prepare_lsq(case, seed, lib):
    a, x, b = _lsq_inputs(case, seed)
    dt, m, n = case["dt"], case["m"], case["n"]
    r, g = torch.empty_like(b), torch.empty_like(x)
    rho = torch.empty(1, dtype=a.dtype, device="cuda")
    one, zero, eta = _scalar(dt, 1.0), _scalar(dt, 0.0), _scalar(dt, -_lsq_eta(case))
    minus = _scalar(dt, -1.0)
    gemv, axpyv = getattr(lib, f"bli_{dt}gemv"), getattr(lib, f"bli_{dt}axpyv")
    ap, lda = a.data_ptr(), a.shape[1]
    xp, bp, rp, gp = (t.data_ptr() for t in (x, b, r, g))
    calls = [
        (gemv, (0, 0, m, n, one, ap, 1, lda, xp, 1, zero, rp, 1)),              # r = A x
        (axpyv, (0, m, minus, bp, 1, rp, 1)),                                   # r -= b
        (gemv, (TRANS["t"], 0, m, n, one, ap, 1, lda, rp, 1, zero, gp, 1)),     # g = A^T r
        (getattr(lib, f"bli_{dt}dotv"), (0, 0, n, gp, 1, gp, 1, rho.data_ptr())),
        (axpyv, (0, n, eta, gp, 1, xp, 1)),                                     # x -= eta g
    ]
    return {"run": _call, "calls": calls, "out": [r, g, rho, x], "keep": (a, b)}


def _run_split(state):
    f, args = state["calls"][0]
    return [state["c"], f(*args)]


def _prepare_split(case, seed, lib):
    a, b, c = _split_inputs(case, seed)
    dt, bound = case["dt"], C.c_double(0.0)
    args = (0, 0, case["m"], case["n"], case["k"], _scalar(dt, 1.0), a.data_ptr(), 1, a.shape[1],
            b.data_ptr(), 1, b.shape[1], _scalar(dt, 0.5), c.data_ptr(), 1, c.shape[1], 0,
            C.byref(bound))
    return {"run": _run_split, "calls": [(getattr(lib, f"bli_amd_{dt}gemm_split"), args)], "c": c,
            "keep": (a, b, bound)}


# ---- work and exact results -----------------------------------------------------

def work(case):
    kind, e = case["kind"], BYTES[case["dt"]]
    if kind in ("gemm", "zgemm", "split"):
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": e * (m * k + k * n + 2 * m * n),
                "flops": (8 if kind == "zgemm" else 2) * m * n * k}
    if kind == "syrk":
        n, k = case["n"], case["k"]
        return {"bytes": e * (n * k + n * (n + 1) // 2), "flops": n * (n + 1) * k}
    if kind == "trsm":
        m, n = case["m"], case["n"]
        q, r = (m, n) if case["side"] == "l" else (n, m)
        return {"bytes": e * (q * (q + 1) // 2 + 2 * m * n), "flops": q * q * r}
    if kind == "batch":
        (m, n, k), _, _ = _batch_shapes(case)
        return {"bytes": e * int(np.sum(m * k + k * n + 2 * m * n)),
                "flops": int(np.sum(2 * m * n * k))}
    m, n = case["m"], case["n"]
    # r and the gradient both need all of A; vectors read and written once per use.
    return {"bytes": e * (2 * m * n + 4 * m + 6 * n), "flops": 4 * m * n + 2 * m + 4 * n}


def exact(case, seed):
    return globals()["_exact_" + case["kind"]](case, seed)


def _exact_gemm(case, seed):
    a, b, c = _gemm_inputs(case, seed)
    m, n, k, (ta, tb) = case["m"], case["n"], case["k"], case["trans"]
    out = c.to(torch.complex128 if c.is_complex() else torch.float64)
    # (op(A) op(B))^T on the transposed storage.
    p = _op(b, _dims(tb, k, n)[0], tb).T.contiguous() @ _op(a, _dims(ta, m, k)[0], ta).T.contiguous()
    out[:, :m] = p + 0.5 * out[:, :m]
    return [out]


_exact_zgemm = _exact_gemm


def _exact_syrk(case, seed):
    a, c = _syrk_inputs(case, seed)
    n, k = case["n"], case["k"]
    x = _op(a, _dims(case["trans"], n, k)[0], case["trans"]).contiguous()
    p = x @ x.T.contiguous()
    out = c.double()
    # out[j, i] is element (i, j); lower keeps i >= j.
    i = torch.arange(n, device="cuda")
    keep = i[None, :] >= i[:, None] if case["uplo"] == "l" else i[None, :] <= i[:, None]
    out[:, :n] = torch.where(keep, p, out[:, :n])
    return [out]


def _exact_trsm(case, seed):
    a, b = _trsm_inputs(case, seed)
    q = case["m"] if case["side"] == "l" else case["n"]
    t = a[:, :q].double().T                       # element (i, j)
    upper = case["uplo"] == "u"
    if case["trans"] == "t":
        t, upper = t.T, not upper
    out = b.double()
    rhs = out[:, :case["m"]].T
    x = torch.linalg.solve_triangular(t.contiguous(), rhs.contiguous(), upper=upper,
                                      left=case["side"] == "l", unitriangular=case["diag"] == "u")
    out[:, :case["m"]] = x.T
    return [out]


def _exact_batch(case, seed):
    a, b, c = [x.double() for x in _batch_inputs(case, seed)]
    rows, cols, ld, off = _batch_layout(case)
    _, (ta, tb), ab = _batch_shapes(case)
    if case["dt"] == "s":
        ab = ab.astype(np.float32).astype(np.float64)

    def part(buf, q, i):
        o = int(off[q][i])
        return buf[o:o + int(ld[q][i] * cols[q][i])].view(int(cols[q][i]), int(ld[q][i]))[
            :, :int(rows[q][i])]

    for i in range(case["count"]):
        x, y, z = part(a, 0, i), part(b, 1, i), part(c, 2, i)    # stored transposed
        x = x.T if ta[i] else x
        y = y.T if tb[i] else y
        z.copy_(float(ab[0, i]) * (y @ x) + float(ab[1, i]) * z)
    return [c]


def _exact_lsq(case, seed):
    a, x, b = _lsq_inputs(case, seed)
    m = case["m"]
    at, x = a.double()[:, :m], x.double()          # A^T
    r = at.T @ x - b.double()
    g = at @ r
    eta = np.float64(-_lsq_eta(case)) if case["dt"] == "d" else np.float64(
        np.float32(-_lsq_eta(case)))
    return [r, g, (g @ g).reshape(1), x + float(eta) * g]


def _exact_split(case, seed):
    a, b, c = _split_inputs(case, seed)
    p = b.double() @ a.double()
    return [p.add_(c.double(), alpha=0.5), None]
