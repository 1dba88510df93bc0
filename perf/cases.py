"""The calls whose speed this library is measured by, through its public Python entry points.

What a user of the library has it do: one triangular solve or multiply at a time, from the few rows of a
small factor to a full 8192 x 8192 problem; back-substitution with a handful of right-hand sides; thousands
of uneven systems in one plan; the FP64-accurate refined solve; and the factorization-side callers of the
same kernels (LU with partial pivoting, U*U^T, the block reflector of a QR).

Every entry point works in place.  A program that keeps its right-hand side (or the matrix that it factors)
copies it into a work array first; `run` does the same, so that it computes the same result on each call.
"""
import math
import os
import random
import sys

import numpy as np
import torch

_PKG = os.path.abspath("nextla.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import nextla_amd as nla  # noqa: E402
from nextla_amd.batch import BatchPlan  # noqa: E402
from nextla_amd.mixed import rectrxm_mixed_, workspace_bytes  # noqa: E402

DTYPES = {"f64": torch.float64, "f32": torch.float32}


def listed():
    return [
        # A tile's worth of work: the call of a blocked factorization on one of its small diagonal blocks.
        {"name": "trsm_small_f64", "kind": "rect", "func": "S", "dtype": "f64", "side": "L", "uplo": "L",
         "trans": "N", "n": 100, "m": 13, "alpha": 1.0},
        # The reference's own 512 x 512 problem with 64 right-hand sides.
        {"name": "trsm_512x64_f64", "kind": "rect", "func": "S", "dtype": "f64", "side": "L", "uplo": "L",
         "trans": "N", "n": 512, "m": 64, "alpha": 1.5},
        # Back-substitution with a handful of right-hand sides after a factorization: A is read once and little else.
        {"name": "trsm_few_rhs_f64", "kind": "rect", "func": "S", "dtype": "f64", "side": "L", "uplo": "U",
         "trans": "N", "n": 4096, "m": 8, "alpha": 1.0},
        # An ordinary ragged single-precision solve from the right with the transpose (the update of a Cholesky).
        {"name": "trsm_ragged_f32", "kind": "rect", "func": "S", "dtype": "f32", "side": "R", "uplo": "L",
         "trans": "T", "n": 1999, "m": 1531, "alpha": 1.0},
        # The full-size drop-in solve.
        {"name": "trsm_8192_f64", "kind": "rect", "func": "S", "dtype": "f64", "side": "L", "uplo": "L",
         "trans": "N", "n": 8192, "m": 8192, "alpha": 1.0},
        # A large single-precision multiply from the right.
        {"name": "trmm_4096_f32", "kind": "rect", "func": "M", "dtype": "f32", "side": "R", "uplo": "U",
         "trans": "N", "n": 4096, "m": 6000, "alpha": -0.75},
        # The FP64-accurate refined solve at its benchmark size, condition about 1e4.
        {"name": "refined_16384_f64", "kind": "refined", "uplo": "L", "trans": "N", "n": 16384, "m": 4096,
         "spread": 3000.0},
        # The batch of 10,000 uneven lower systems (n log-uniform in 16..1024, right-hand sides in 1..256), replayed
        # from its graph.
        {"name": "batch_10000_f64", "kind": "batch", "func": "S", "dtype": "f64", "count": 10000, "mix": 0},
        # LU with partial pivoting: a full-size square matrix and a small ragged tall one.
        {"name": "lu_8192_f64", "kind": "lu", "m": 8192, "n": 8192},
        {"name": "lu_1000x700_f64", "kind": "lu", "m": 1000, "n": 700},
        # U*U^T (the second half of an inverse from a Cholesky factor).
        {"name": "lauum_4096_f64", "kind": "lauum", "dtype": "f64", "uplo": "U", "n": 4096},
        # Q^T C with one block of 64 reflectors (a QR's trailing update).
        {"name": "larfb_4096_f64", "kind": "larfb", "dtype": "f64", "side": "L", "trans": "T", "m": 4096, "n": 4096,
         "k": 64},
    ]


def _log_int(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]; whole multiples of 64 and odd sizes both occur."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if v >= 256 and rng.random() < 0.3:
        v -= v % 64
    return max(lo, min(hi, v))


def draw(rng: random.Random):
    kind = rng.choice(["rect", "rect", "rect", "few", "refined", "batch", "lu", "lu", "lauum", "larfb"])
    if kind in ("rect", "few"):
        few = kind == "few"
        return {"kind": "rect", "func": rng.choice("SSM"), "dtype": rng.choice(["f64", "f64", "f32"]),
                "side": rng.choice("LR"), "uplo": rng.choice("LU"), "trans": rng.choice("NT"),
                "n": _log_int(rng, 512, 8192) if few else _log_int(rng, 32, 8192),
                "m": rng.randint(1, 32) if few else _log_int(rng, 4, 8192), "alpha": rng.choice([1.0, 1.5, -0.75])}
    if kind == "refined":
        return {"kind": "refined", "uplo": rng.choice("LU"), "trans": rng.choice("NT"),
                "n": _log_int(rng, 2048, 16384), "m": _log_int(rng, 128, 4096), "spread": rng.choice([30.0, 3000.0])}
    if kind == "batch":
        return {"kind": "batch", "func": rng.choice("SSM"), "dtype": rng.choice(["f64", "f32"]),
                "count": _log_int(rng, 100, 10000), "mix": rng.randint(1, 1 << 20)}
    if kind == "lu":
        m = _log_int(rng, 64, 8192)
        return {"kind": "lu", "m": m, "n": m if rng.random() < 0.5 else _log_int(rng, 32, m)}
    if kind == "lauum":
        return {"kind": "lauum", "dtype": rng.choice(["f64", "f64", "f32"]), "uplo": rng.choice("LU"),
                "n": _log_int(rng, 128, 8192)}
    return {"kind": "larfb", "dtype": rng.choice(["f64", "f64", "f32"]), "side": rng.choice("LR"),
            "trans": rng.choice("NT"), "m": _log_int(rng, 512, 8192), "n": _log_int(rng, 512, 8192),
            "k": rng.choice([16, 32, 48, 64, 100, 128, 256])}


# ---- inputs ---------------------------------------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _matrix(rows, cols, dtype):
    """An uninitialised column-major matrix, the layout of Julia's Matrix."""
    return torch.empty((cols, rows), dtype=dtype, device="cuda").t()


def _triangle(n, uplo, dtype, g):
    """Off-diagonals U(-1,1)/sqrt(n), diagonal 2 + U(0,1), zero outside the triangle."""
    a = _matrix(n, n, dtype)
    a.uniform_(-1.0, 1.0, generator=g).mul_(1.0 / math.sqrt(n))
    a.copy_(torch.tril(a) if uplo == "L" else torch.triu(a))
    a.diagonal().uniform_(2.0, 3.0, generator=g)
    return a


def _rect_inputs(case, seed):
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    n, m = case["n"], case["m"]
    a = _triangle(n, case["uplo"], dt, g)
    b = _matrix(*((n, m) if case["side"] == "L" else (m, n)), dt)
    return a, b.normal_(generator=g)


def _refined_inputs(case, seed):
    """A triangle whose diagonal runs from 2 to 2 * spread on a logarithmic scale."""
    g = _gen(seed)
    n, m = case["n"], case["m"]
    a = _triangle(n, case["uplo"], torch.float64, g)
    a.diagonal().copy_(2.0 * case["spread"] ** (torch.arange(n, dtype=torch.float64, device="cuda") / max(n - 1, 1)))
    return a, _matrix(n, m, torch.float64).normal_(generator=g)


def _batch_sizes(case):
    rng = np.random.default_rng(case["mix"])
    ns = np.exp(rng.uniform(np.log(16), np.log(1025), case["count"])).astype(int)
    ms = np.exp(rng.uniform(np.log(1), np.log(257), case["count"])).astype(int)
    return [int(v) for v in ns], [int(v) for v in ms]


def _batch_inputs(case, seed):
    """All systems' A in one array and all right-hand sides in another, each matrix column-major."""
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    ns, ms = _batch_sizes(case)
    abuf = torch.empty(sum(n * n for n in ns), dtype=dt, device="cuda").uniform_(-1.0, 1.0, generator=g)
    bbuf = torch.empty(sum(n * m for n, m in zip(ns, ms)), dtype=dt, device="cuda").normal_(generator=g)
    As, o = [], 0
    for n in ns:
        a = abuf[o:o + n * n].view(n, n).t()
        a.mul_(1.0 / n)
        a.diagonal().add_(1.5)
        As.append(a)
        o += n * n
    return As, bbuf, ns, ms


def _batch_views(buf, ns, ms):
    out, o = [], 0
    for n, m in zip(ns, ms):
        out.append(buf[o:o + n * m].view(m, n).t())
        o += n * m
    return out


def _lu_inputs(case, seed):
    return _matrix(case["m"], case["n"], torch.float64).normal_(generator=_gen(seed))


def _lauum_inputs(case, seed):
    """A whole matrix: the triangle that is not the factor's holds something else, and stays as it is."""
    g, n = _gen(seed), case["n"]
    a = _matrix(n, n, DTYPES[case["dtype"]]).normal_(generator=g)
    a.mul_(1.0 / math.sqrt(n))
    return a


def _larfb_inputs(case, seed):
    """V (its unit-lower part the reflectors, the rest an R that is not read), T with H = I - V T V^T orthogonal
    (T^-1 is the upper triangle of V^T V with its diagonal halved), and C."""
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    m, n, k = case["m"], case["n"], case["k"]
    q = m if case["side"] == "L" else n
    v = _matrix(q, k, torch.float64).normal_(generator=g)
    v.mul_(1.0 / math.sqrt(q))
    v = v.to(dt)
    v1 = torch.tril(v.double(), -1)
    v1.diagonal().fill_(1.0)
    gram = v1.t() @ v1
    tinv = torch.triu(gram, 1) + torch.diag(gram.diagonal() * 0.5)
    t = torch.linalg.solve_triangular(tinv, torch.eye(k, dtype=torch.float64, device="cuda"), upper=True)
    c = _matrix(m, n, dt).normal_(generator=g)
    return v.t().contiguous().t(), torch.triu(t).to(dt).t().contiguous().t(), c


def prepare(case, seed):
    kind = case["kind"]
    if kind == "rect":
        a, b = _rect_inputs(case, seed)
        return {"case": case, "a": a, "b": b, "x": torch.empty_like(b)}
    if kind == "refined":
        a, b = _refined_inputs(case, seed)
        ws = torch.empty(workspace_bytes("L", case["n"], case["m"]) + 256, dtype=torch.uint8, device="cuda")
        return {"case": case, "a": a, "b": b, "x": torch.empty_like(b), "ws": ws}
    if kind == "batch":
        As, bbuf, ns, ms = _batch_inputs(case, seed)
        xbuf = torch.empty_like(bbuf)
        plan = BatchPlan("L", "L", "N", case["func"], As, _batch_views(xbuf, ns, ms), 1.0)
        return {"case": case, "plan": plan, "b": bbuf, "x": xbuf}
    if kind == "lu":
        a = _lu_inputs(case, seed)
        return {"case": case, "a": a, "x": torch.empty_like(a)}
    if kind == "lauum":
        a = _lauum_inputs(case, seed)
        code = nla.NLA_F64 if case["dtype"] == "f64" else nla.NLA_F32
        ws = torch.empty(max(1, nla.load().nla_lauum_workspace_bytes(code, case["n"])), dtype=torch.uint8, device="cuda")
        return {"case": case, "a": a, "x": torch.empty_like(a), "ws": ws}
    v, t, c = _larfb_inputs(case, seed)
    wr = case["n"] if case["side"] == "L" else case["m"]
    return {"case": case, "v": v, "t": t, "c": c, "x": torch.empty_like(c), "ws": _matrix(wr, case["k"], c.dtype)}


def run(state):
    case = state["case"]
    kind = case["kind"]
    x = state["x"]
    if kind == "rect":
        x.copy_(state["b"])
        return nla.unified_rectrxm_(case["side"], case["uplo"], case["trans"], case["alpha"], case["func"], state["a"], x)
    if kind == "refined":
        x.copy_(state["b"])
        return rectrxm_mixed_("L", case["uplo"], case["trans"], 1.0, state["a"], x, precision="auto", tol=1e-14,
                              workspace=state["ws"])[0]
    if kind == "batch":
        x.copy_(state["b"])
        state["plan"].execute(use_graph=True)
        return x
    if kind == "lu":
        x.copy_(state["a"])
        lu, ipiv, info = nla.getrf2_(x)
        return {"lu": lu, "ipiv": ipiv, "info": info}
    if kind == "lauum":
        x.copy_(state["a"])
        return nla.lauum_(case["uplo"], case["n"], x, workspace=state["ws"])
    x.copy_(state["c"])
    return nla.larfb_(case["side"], case["trans"], "F", "C", state["v"], state["t"], x, work=state["ws"])


def work(case):
    kind = case["kind"]
    s = 4 if case.get("dtype") == "f32" else 8
    if kind in ("rect", "refined"):
        n, m = case["n"], case["m"]
        return {"bytes": (n * (n + 1) // 2 + 2 * n * m) * s, "flops": n * n * m}
    if kind == "batch":
        ns, ms = _batch_sizes(case)
        return {"bytes": sum(n * (n + 1) // 2 + 2 * n * m for n, m in zip(ns, ms)) * s,
                "flops": sum(n * n * m for n, m in zip(ns, ms))}
    if kind == "lu":
        m, n = case["m"], case["n"]
        return {"bytes": (2 * m * n + min(m, n)) * 8, "flops": m * n * n - n ** 3 // 3}
    if kind == "lauum":
        n = case["n"]
        return {"bytes": n * (n + 1) * s, "flops": n ** 3 // 3}
    m, n, k = case["m"], case["n"], case["k"]
    q = m if case["side"] == "L" else n
    return {"bytes": (2 * m * n + q * k + k * (k + 1) // 2) * s, "flops": 4 * m * n * k}


# ---- the same results in 64 bits, from torch alone --------------------------------------------------------------


def _tri_exact(func, side, uplo, trans, alpha, a, b):
    """unified_rectrxm! in 64 bits: op(A) X = alpha B, X op(A) = alpha B, or the products."""
    a = (torch.tril(a.double()) if uplo == "L" else torch.triu(a.double()))
    b = b.double() * alpha
    upper = uplo == "U"
    if trans == "T":
        a, upper = a.t(), not upper
    if func == "M":
        return a @ b if side == "L" else b @ a
    return torch.linalg.solve_triangular(a, b, upper=upper, left=side == "L")


def exact(case, seed):
    kind = case["kind"]
    if kind == "rect":
        a, b = _rect_inputs(case, seed)
        return _tri_exact(case["func"], case["side"], case["uplo"], case["trans"], case["alpha"], a, b)
    if kind == "refined":
        a, b = _refined_inputs(case, seed)
        return _tri_exact("S", "L", case["uplo"], case["trans"], 1.0, a, b)
    if kind == "batch":
        As, bbuf, ns, ms = _batch_inputs(case, seed)
        out = torch.empty_like(bbuf, dtype=torch.float64)
        for a, b, x in zip(As, _batch_views(bbuf, ns, ms), _batch_views(out, ns, ms)):
            x.copy_(_tri_exact(case["func"], "L", "L", "N", 1.0, a, b))
        return out
    if kind == "lu":
        lu, _ = torch.linalg.lu_factor(_lu_inputs(case, seed).cpu())
        return {"lu": lu, "ipiv": None, "info": None}
    if kind == "lauum":
        a = _lauum_inputs(case, seed).double()
        if case["uplo"] == "U":
            u = torch.triu(a)
            return torch.triu(u @ u.t()) + torch.tril(a, -1)
        low = torch.tril(a)
        return torch.tril(low.t() @ low) + torch.triu(a, 1)
    v, t, c = (z.double() for z in _larfb_inputs(case, seed))
    v = torch.tril(v, -1)
    v.diagonal().fill_(1.0)
    t = torch.triu(t)
    if case["trans"] == "T":
        t = t.t()
    if case["side"] == "L":
        return c - v @ (t @ (v.t() @ c))
    return c - (c @ v) @ t @ v.t()
