"""The calls whose speed counts: the batched SPD path through its C entry
points, as a Python program calls them (kblas-gpu_amd/pykblas.py).

One case is one kind of call ("kind") with its precision ("prec": d FP64, s
FP32), batch layout ("layout": strided or pointers), side, sizes and the excess
of the leading dimension over the order ("pad").  Matrices are column-major, so
a torch tensor T[b][c][r] holds element (r, c) of matrix b.

POTRF and POSV overwrite their operands.  A program that solves again keeps the
assembled matrix and works on a copy, so their passes begin with that copy (one
torch copy per operand into buffers that the program keeps).  The other kinds
need none: POTRS and TRSM solve in place of the vectors of the last pass, SYRK
accumulates, POTI inverts the inverse back, and the mixed POSV reads A and B
only.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "kblas-gpu_amd"))
import pykblas  # noqa: E402

DEV = "cuda"


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # The smallest call: new right-hand sides for a few kept factors, where
        # launch latency and the serial chain of one small solve count.
        dict(name="potrs_n24_small", kind="potrs", prec="d", layout="strided", side="R", n=24, nrhs=1, batch=48, pad=0),
        # The benchmark's uniform factorization: order 32, 10,000 matrices.
        dict(name="potrf_n32", kind="potrf", prec="d", layout="strided", side="R", n=32, nrhs=0, batch=10000, pad=0),
        # The benchmark's uniform solve of very small systems, 1 right-hand side.
        dict(name="posv_n16", kind="posv", prec="d", layout="strided", side="R", n=16, nrhs=1, batch=100000, pad=0),
        # Single precision, LAPACK's layout (A X = B), pointer arrays, an order
        # that fills no tile and a leading dimension above it.
        dict(name="sposv_n50_pointers", kind="posv", prec="s", layout="pointers", side="L", n=50, nrhs=5, batch=20000,
             pad=2),
        # The headline benchmark: mixed precision with refinement, order 64, 4
        # right-hand sides, condition 1e2..1e6.
        dict(name="dsposv_n64", kind="dsposv", prec="d", layout="strided", side="R", n=64, nrhs=4, batch=50000, pad=0),
        # The benchmark's non-uniform solve, orders 8..256 in one call.
        dict(name="posv_vbatch", kind="posv_vbatch", prec="d", layout="pointers", side="R", n=256, n_lo=8, nrhs=4,
             batch=20000, pad=0),
        # The benchmark's non-uniform mixed solve, orders 128..512, 64
        # right-hand sides, condition 1e2..1e4.
        dict(name="dsposv_vbatch", kind="dsposv_vbatch", prec="d", layout="pointers", side="R", n=512, n_lo=128,
             nrhs=64, batch=2000, pad=0),
        # The largest order of the reference's published DPOSV chart, nrhs = n.
        dict(name="posv_n256_square", kind="posv", prec="d", layout="strided", side="R", n=256, nrhs=256, batch=4096,
             pad=0),
        # Factorization above the one-wavefront orders: pointer arrays of a
        # block-sparse code, an odd order, padded columns.
        dict(name="potrf_n200_pointers", kind="potrf", prec="d", layout="pointers", side="R", n=200, nrhs=0, batch=2000,
             pad=8),
        # Triangular solves of the published DTRSM chart.
        dict(name="trsm_n128", kind="trsm", prec="d", layout="strided", side="L", n=128, nrhs=128, batch=4096, pad=0),
        # Rank-k updates of the same chart's trailing matrices.
        dict(name="syrk_n256", kind="syrk", prec="d", layout="strided", side="R", n=256, nrhs=256, batch=2048, pad=0),
        # The benchmark's SPD inverse: order 32, 10,000 matrices.
        dict(name="poti_n32", kind="poti", prec="d", layout="strided", side="R", n=32, nrhs=0, batch=10000, pad=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["potrs", "potrf", "potrf", "posv", "posv", "posv", "dsposv", "posv_vbatch", "dsposv_vbatch",
                       "trsm", "syrk", "poti"])
    c = dict(kind=kind, prec=rng.choice("dds"), layout=rng.choice(["strided", "pointers"]), side=rng.choice("LR"),
             pad=rng.choice([0, 0, 1, 8]))
    if kind == "potrs":
        c.update(n=_log_int(rng, 4, 256), nrhs=_log_int(rng, 1, 16), batch=_log_int(rng, 16, 2000))
    elif kind in ("potrf", "poti"):
        n = _log_int(rng, 8, 256 if kind == "potrf" else 64)
        c.update(n=n, nrhs=0, batch=max(64, _log_int(rng, 1e6, 1e8) // (n * n)))
    elif kind == "posv":
        n = _log_int(rng, 8, 256)
        c.update(n=n, nrhs=rng.choice([1, 2, 4, _log_int(rng, 1, n)]), batch=max(64, _log_int(rng, 1e6, 1e8) // (n * n)))
    elif kind == "dsposv":
        c.update(prec="d", n=_log_int(rng, 8, 64), nrhs=rng.randint(1, 8), batch=_log_int(rng, 2000, 40000))
    elif kind == "posv_vbatch":
        c.update(prec="d", layout="pointers", n_lo=_log_int(rng, 8, 32), n=_log_int(rng, 48, 256),
                 nrhs=_log_int(rng, 1, 16), batch=_log_int(rng, 1000, 10000), pad=0)
    elif kind == "dsposv_vbatch":
        c.update(prec="d", layout="pointers", side="R", n_lo=_log_int(rng, 64, 160), n=_log_int(rng, 192, 512),
                 nrhs=_log_int(rng, 8, 64), batch=_log_int(rng, 200, 1500), pad=0)
    else:
        n = _log_int(rng, 16, 256)
        c.update(n=n, nrhs=_log_int(rng, 16, 256), batch=max(64, _log_int(rng, 1e6, 1e8) // (n * n)))
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _dtype(case):
    return torch.float64 if case["prec"] == "d" else torch.float32


def _orders(case):
    """The orders of a non-uniform batch: part of the case, not of the seed."""
    r = np.random.RandomState(1000 * case["n"] + case["n_lo"])
    return r.randint(case["n_lo"], case["n"] + 1, size=case["batch"])


def _gram(g, batch, n):
    """B B^T + n I with B uniform in (-1, 1)."""
    b = torch.rand((batch, n, n), generator=g, device=DEV, dtype=torch.float64).mul_(2.0).sub_(1.0)
    a = torch.bmm(b, b.transpose(1, 2).contiguous())
    a.diagonal(dim1=1, dim2=2).add_(float(n))
    return 0.5 * (a + a.transpose(1, 2))


def _cond(g, batch, n, lk_lo, lk_hi):
    """Q diag(s) Q^T with cond = 10^U[lk_lo, lk_hi], s log-uniform with both
    ends taken, Q a cosine transform between random sign matrices, twice."""
    i = torch.arange(n, device=DEV, dtype=torch.float64)
    cos = torch.cos(math.pi / n * (i[:, None] + 0.5) * i[None, :]) * math.sqrt(2.0 / n)
    cos[:, 0] /= math.sqrt(2.0)
    sign = torch.randint(0, 2, (3, batch, n), generator=g, device=DEV).double().mul_(2.0).sub_(1.0)
    q = torch.matmul(sign[0].unsqueeze(2) * cos * sign[1].unsqueeze(1), cos) * sign[2].unsqueeze(1)
    lk = lk_lo + (lk_hi - lk_lo) * torch.rand((batch, 1), generator=g, device=DEV, dtype=torch.float64)
    t = torch.rand((batch, n), generator=g, device=DEV, dtype=torch.float64)
    t[:, 0] = 0.0
    t[:, n - 1] = 1.0
    s = torch.pow(10.0, -lk * t)
    a = torch.bmm(q * s.unsqueeze(1), q.transpose(1, 2).contiguous())
    return 0.5 * (a + a.transpose(1, 2))


def _triangle(g, batch, n):
    """Lower triangles with a diagonal in (1, 2) and off-diagonals O(1/n)."""
    t = torch.rand((batch, n, n), generator=g, device=DEV, dtype=torch.float64).mul_(2.0).sub_(1.0).div_(n)
    t = torch.triu(t, 1)  # T[b][c][r]: the lower triangle has r > c
    t.diagonal(dim1=1, dim2=2).copy_(1.0 + torch.rand((batch, n), generator=g, device=DEV, dtype=torch.float64))
    return t


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float64)


def _padded(t, pad):
    """t[b][c][r] in columns of pad more rows (the padding is zero)."""
    if not pad:
        return t.contiguous()
    out = torch.zeros((t.shape[0], t.shape[1], t.shape[2] + pad), device=DEV, dtype=t.dtype)
    out[:, :, : t.shape[2]] = t
    return out


def _rhs_shape(case, n):
    """B is nrhs x n for side R (X A = B) and n x nrhs for side L (A X = B)."""
    return (n, case["nrhs"]) if case["side"] == "R" else (case["nrhs"], n)


def _inputs(case, seed):
    """The operands in `_dtype`, without padding: A and, where there is one, B,
    as [batch][columns][rows]; for non-uniform batches lists over the orders."""
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * int(seed) + 17)
    kind, n, batch, dt = case["kind"], case["n"], case["batch"], _dtype(case)
    if kind.endswith("vbatch"):
        got = []
        for order, count in zip(*np.unique(_orders(case), return_counts=True)):
            order, count = int(order), int(count)
            a = _gram(g, count, order) if kind == "posv_vbatch" else _cond(g, count, order, 2.0, 4.0)
            got.append((a, _normal(g, count, *_rhs_shape(case, order))))
        return got
    if kind == "dsposv":
        return _cond(g, batch, n, 2.0, 6.0), _normal(g, batch, *_rhs_shape(case, n))
    if kind == "trsm":
        return _triangle(g, batch, n).to(dt), _normal(g, batch, *_rhs_shape(case, n)).to(dt)
    if kind == "syrk":  # A is n x nrhs, C is n x n
        return _normal(g, batch, case["nrhs"], n).to(dt), _normal(g, batch, n, n).to(dt)
    a = _gram(g, batch, n).to(dt)
    if kind == "poti":
        return a, None
    if kind == "potrf":
        return a, None
    b = _normal(g, batch, *_rhs_shape(case, n)).to(dt)
    if kind == "potrs":  # the kept factor
        low = torch.linalg.cholesky(a.double())
        return low.transpose(1, 2).contiguous().to(dt), b
    return a, b


def _pointers(t):
    """Device array of the device addresses of t's matrices."""
    step = t.stride(0) * t.element_size()
    return torch.arange(t.shape[0], device=DEV, dtype=torch.int64).mul_(step).add_(t.data_ptr())


class _State:
    """What the program holds between calls."""


def prepare(case, seed):
    s = _State()
    s.case = case
    s.h = pykblas.Handle(torch.cuda.current_stream().cuda_stream)
    s.lib, batch = s.h.lib, case["batch"]
    s.info = torch.zeros(batch, dtype=torch.int32, device=DEV)
    s.side = case["side"].encode()
    if case["kind"].endswith("vbatch"):
        _prepare_vbatch(s, case, seed)
        return s
    a, b = _inputs(case, seed)
    a = _padded(a, case["pad"])
    b = None if b is None else _padded(b, case["pad"])
    s.a0, s.b0 = a, b
    overwrites = case["kind"] in ("potrf", "posv")
    s.a = torch.empty_like(a) if overwrites else a
    s.b = torch.empty_like(b) if overwrites and b is not None else b
    if case["kind"] == "dsposv":
        s.x = torch.zeros_like(b)
        s.iters = torch.zeros(batch, dtype=torch.int32, device=DEV)
    if case["layout"] == "pointers":
        s.pa = _pointers(s.a)
        s.pb = None if s.b is None else _pointers(s.b)
        s.px = _pointers(s.x) if case["kind"] == "dsposv" else None
    return s


def _prepare_vbatch(s, case, seed):
    batch, parts = case["batch"], _inputs(case, seed)
    ns = _orders(case)
    s.a0 = torch.cat([a.reshape(-1) for a, _ in parts])
    s.b0 = torch.cat([b.reshape(-1) for _, b in parts])
    del parts
    rank = np.empty(batch, dtype=np.int64)  # the matrices lie sorted by order
    order = np.argsort(ns, kind="stable")
    rank[order] = np.arange(batch)
    sa = np.concatenate(([0], np.cumsum(ns[order].astype(np.int64) ** 2)))[rank]
    sb = np.concatenate(([0], np.cumsum(ns[order].astype(np.int64) * case["nrhs"])))[rank]
    s.n = torch.from_numpy(ns.astype(np.int32)).to(DEV)
    s.nrhs = torch.full_like(s.n, case["nrhs"])
    right = case["side"] == "R"
    s.m_arg, s.n_arg = (s.nrhs, s.n) if right else (s.n, s.nrhs)
    s.max_m, s.max_n = (case["nrhs"], case["n"]) if right else (case["n"], case["nrhs"])
    s.ldb = s.m_arg
    off = lambda t, o: torch.from_numpy(o * 8).to(DEV) + t.data_ptr()  # noqa: E731
    if case["kind"] == "posv_vbatch":
        s.a, s.b = torch.empty_like(s.a0), torch.empty_like(s.b0)
        s.pa, s.pb = off(s.a, sa), off(s.b, sb)
        s.lib.kblas_posv_vbatch_wsquery(s.h.h, case["n"], batch)
    else:
        s.x = torch.zeros_like(s.b0)
        s.iters = torch.zeros(batch, dtype=torch.int32, device=DEV)
        s.pa, s.pb, s.px = off(s.a0, sa), off(s.b0, sb), off(s.x, sb)
        s.lib.kblas_sposv_vbatch_wsquery(s.h.h, case["nrhs"], case["n"], batch)
    _check(s.lib.kblasAllocateWorkspace(s.h.h))


def _check(status):
    if status != pykblas.KBLAS_Success:
        raise RuntimeError("the call returned %d" % status)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    return _RUN[s.case["kind"]](s, s.case)


def _operands(s, t, ptrs):
    """The arguments of one operand: address, leading dimension, stride."""
    if s.case["layout"] == "strided":
        return t.data_ptr(), t.shape[2], t.stride(0)
    return ptrs.data_ptr(), t.shape[2]


def _call(s, name):
    prec = s.case["prec"].upper() if not name.startswith("sposv") else "D"
    return getattr(s.lib, "kblas%s%s_batch%s" % (prec, name, "_strided" if s.case["layout"] == "strided" else ""))


def _rhs_sizes(case):
    return (case["nrhs"], case["n"]) if case["side"] == "R" else (case["n"], case["nrhs"])


def _run_potrf(s, c):
    s.a.copy_(s.a0)
    _check(_call(s, "potrf")(s.h.h, b"L", c["n"], *_operands(s, s.a, getattr(s, "pa", None)), c["batch"],
                             s.info.data_ptr()))
    return {"l": s.a, "info": s.info}


def _run_posv(s, c):
    s.a.copy_(s.a0)
    s.b.copy_(s.b0)
    m, n = _rhs_sizes(c)
    _check(_call(s, "posv")(s.h.h, s.side, b"L", m, n, *_operands(s, s.a, getattr(s, "pa", None)),
                            *_operands(s, s.b, getattr(s, "pb", None)), c["batch"], s.info.data_ptr()))
    return {"l": s.a, "x": s.b, "info": s.info}


def _run_potrs(s, c):
    m, n = _rhs_sizes(c)
    _check(_call(s, "potrs")(s.h.h, s.side, b"L", m, n, *_operands(s, s.a, getattr(s, "pa", None)),
                             *_operands(s, s.b, getattr(s, "pb", None)), c["batch"]))
    return {"x": s.b}


def _run_dsposv(s, c):
    m, n = _rhs_sizes(c)
    f = s.lib.kblasDsposv_batch_strided if c["layout"] == "strided" else s.lib.kblasDsposv_batch
    _check(f(s.h.h, s.side, b"L", m, n, *_operands(s, s.a, getattr(s, "pa", None)),
             *_operands(s, s.b, getattr(s, "pb", None)), *_operands(s, s.x, getattr(s, "px", None)), c["batch"],
             s.info.data_ptr(), s.iters.data_ptr()))
    return {"x": s.x, "info": s.info, "iter": s.iters}


def _run_posv_vbatch(s, c):
    s.a.copy_(s.a0)
    s.b.copy_(s.b0)
    _check(s.lib.kblasDposv_vbatch(s.h.h, s.side, b"L", s.m_arg.data_ptr(), s.n_arg.data_ptr(), s.max_m, s.max_n,
                                   s.pa.data_ptr(), s.n.data_ptr(), s.pb.data_ptr(), s.ldb.data_ptr(), c["batch"],
                                   s.info.data_ptr()))
    return {"l": s.a, "x": s.b, "info": s.info}


def _run_dsposv_vbatch(s, c):
    _check(s.lib.kblasDsposv_vbatch(s.h.h, s.side, b"L", s.m_arg.data_ptr(), s.n_arg.data_ptr(), s.max_m, s.max_n,
                                    s.pa.data_ptr(), s.n.data_ptr(), s.pb.data_ptr(), s.ldb.data_ptr(),
                                    s.px.data_ptr(), s.ldb.data_ptr(), c["batch"], s.info.data_ptr(),
                                    s.iters.data_ptr()))
    return {"x": s.x, "info": s.info, "iter": s.iters}


def _run_trsm(s, c):
    m, n = _rhs_sizes(c)
    _check(_call(s, "trsm")(s.h.h, s.side, b"L", b"N", b"N", m, n, 1.0, *_operands(s, s.a, getattr(s, "pa", None)),
                            *_operands(s, s.b, getattr(s, "pb", None)), c["batch"]))
    return {"x": s.b}


def _run_syrk(s, c):
    _check(_call(s, "syrk")(s.h.h, b"L", b"N", c["n"], c["nrhs"], -1.0, *_operands(s, s.a, getattr(s, "pa", None)),
                            1.0, *_operands(s, s.b, getattr(s, "pb", None)), c["batch"]))
    return {"c": s.b}


def _run_poti(s, c):
    _check(_call(s, "poti")(s.h.h, b"L", c["n"], *_operands(s, s.a, getattr(s, "pa", None)), c["batch"],
                            s.info.data_ptr()))
    return {"inverse": s.a, "info": s.info}


_RUN = {"potrf": _run_potrf, "posv": _run_posv, "potrs": _run_potrs, "dsposv": _run_dsposv,
        "posv_vbatch": _run_posv_vbatch, "dsposv_vbatch": _run_dsposv_vbatch, "trsm": _run_trsm, "syrk": _run_syrk,
        "poti": _run_poti}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    """One triangle of a symmetric or triangular matrix read (and written where
    it is an output), every vector read and written once, info written; for
    POTRF and POSV also the copy that begins a pass, one read and one write of
    the kept matrices.  Additions and multiplications of the textbook
    algorithms; the mixed solve is counted as the FP64 one."""
    kind, w = case["kind"], 8 if case["prec"] == "d" else 4
    ns = _orders(case).astype(np.float64) if kind.endswith("vbatch") else np.full(1, float(case["n"]))
    times = 1 if kind.endswith("vbatch") else case["batch"]
    r = float(case["nrhs"])
    tri, vec = ns * (ns + 1) / 2, ns * r
    factor, solve = ns ** 3 / 3 + ns ** 2 / 2 + ns / 6, 2 * ns ** 2 * r
    if kind == "potrf":
        b, f = 2 * w * tri + 2 * w * ns * ns + 4, factor
    elif kind in ("posv", "posv_vbatch"):
        b, f = 2 * w * (tri + vec) + 2 * w * (ns * ns + vec) + 4, factor + solve
    elif kind == "potrs":
        b, f = w * tri + 2 * w * vec, solve
    elif kind in ("dsposv", "dsposv_vbatch"):
        b, f = w * tri + 2 * w * vec + 8, factor + solve
    elif kind == "trsm":
        b, f = w * tri + 2 * w * vec, ns ** 2 * r
    elif kind == "syrk":
        b, f = w * vec + 2 * w * tri, r * ns * (ns + 1)
    else:
        b, f = 2 * w * tri + 4, ns ** 3
    return {"bytes": float(b.sum()) * times, "flops": float(f.sum()) * times}


# ---------------------------------------------------------------------------
# 64-bit results
# ---------------------------------------------------------------------------
def _factor(a):
    """The buffer after POTRF: the factor in the lower triangle, A's strict
    upper triangle as it was, as T[b][c][r]."""
    low = torch.linalg.cholesky(a)
    return torch.triu(low.transpose(1, 2)) + torch.tril(a, -1), low


def _tri(t, b, upper):
    """T^-1 B by halves down to order 64, a few hundred matrices at a time (the
    library's scratch memory is bounded)."""
    n = t.shape[1]
    if n <= 64:
        return torch.cat([torch.linalg.solve_triangular(t[i:i + 512].contiguous(), b[i:i + 512].contiguous(),
                                                        upper=upper) for i in range(0, t.shape[0], 512)])
    h = n // 2
    one, two = (slice(h, n), slice(0, h)) if upper else (slice(0, h), slice(h, n))
    x1 = _tri(t[:, one, one], b[:, one], upper)
    x2 = _tri(t[:, two, two], b[:, two] - torch.bmm(t[:, two, one].contiguous(), x1), upper)
    return torch.cat((x2, x1) if upper else (x1, x2), dim=1)


def _solve(low, b, side):
    """The X of the stored B[b][c][r]."""
    rows = b.transpose(1, 2) if side == "L" else b  # columns of A X = B, either way
    x = _tri(low.transpose(1, 2), _tri(low, rows, False), True)
    return (x.transpose(1, 2) if side == "L" else x).contiguous()


def exact(case, seed):
    kind, pad = case["kind"], case["pad"]
    if kind.endswith("vbatch"):
        ls, xs = [], []
        for a, b in _inputs(case, seed):
            stored, low = _factor(a)
            ls.append(stored.reshape(-1))
            xs.append(_solve(low, b, case["side"]).reshape(-1))
        out = {"x": torch.cat(xs), "info": None}
        out.update({"l": torch.cat(ls)} if kind == "posv_vbatch" else {"iter": None})
        return out
    a, b = _inputs(case, seed)
    a = a.double()
    b = None if b is None else b.double()
    if kind == "potrf":
        return {"l": _padded(_factor(a)[0], pad), "info": None}
    if kind == "posv":
        stored, low = _factor(a)
        return {"l": _padded(stored, pad), "x": _padded(_solve(low, b, case["side"]), pad), "info": None}
    if kind == "dsposv":
        return {"x": _padded(_solve(torch.linalg.cholesky(a), b, case["side"]), pad), "info": None, "iter": None}
    if kind == "potrs":
        return {"x": _padded(_solve(a.transpose(1, 2).contiguous(), b, case["side"]), pad)}
    if kind == "trsm":
        low = a.transpose(1, 2).contiguous()
        if case["side"] == "L":  # A X = B
            x = _tri(low, b.transpose(1, 2), False).transpose(1, 2)
        else:  # X A = B, so A^T X^T = B^T
            x = _tri(a, b, True)
        return {"x": _padded(x.contiguous(), pad)}
    if kind == "syrk":
        prod = b - torch.bmm(a.transpose(1, 2).contiguous(), a).transpose(1, 2)
        return {"c": _padded(torch.triu(prod) + torch.tril(b, -1), pad)}
    low = torch.linalg.cholesky(a)
    eye = torch.eye(case["n"], device=DEV, dtype=torch.float64).expand_as(a).contiguous()
    half = _tri(low, eye, False)
    inv = torch.bmm(half.transpose(1, 2).contiguous(), half)
    return {"inverse": _padded(torch.triu(inv.transpose(1, 2)) + torch.tril(a, -1), pad), "info": None}
