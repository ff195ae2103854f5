"""Timed cases of the batched factor-and-solve calls.

Each case is one call (or the factor call and its solve call) of the C API on a
batch that is already on the GPU, as an application makes it: device pointer
arrays, pivots, info and a queue are set up once and kept.  The sizes are those
of the benchmark's workloads (bench.py), plus the smallest calls and odd orders.

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) inputs, buffers and the queue
    run(state)          one pass; returns the outputs
    work(case)          bytes and flops that one pass cannot do without
    exact(case, seed)   the outputs as torch's LAPACK gives them in FP64

The factorizations overwrite their matrix, so a pass first puts the matrix into
the work buffer: the program's own assembly of the next system, or the copy it
takes because it needs the matrix afterwards.  That copy is in the time and not
in work().
"""
import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

import magma_amd as ma
from magma_amd import gen

# What magma_amd_autotune picks on an MI355X (family -> variant per size class),
# set as a program sets the table that it has saved.
TUNED = {0: (-1, -1, -1, -1, 3, 0, 2, -1, -1, -1),        # LU
         1: (-1, -1, -1, -1, 4, 4, 0, -1, -1, -1),        # mixed precision
         2: (1, 1, 1, 3, 3, 3, -1, -1, -1, 3)}            # GEMM


def listed():
    return [
        # latency: the few small systems of one time step (a chemistry cell, a control loop)
        {"name": "gesv_n8_x100", "op": "gesv", "n": 8, "count": 100, "nrhs": 1},
        # many small general systems, the benchmark's lu32_gesv
        {"name": "gesv_n32_x10000", "op": "gesv", "n": 32, "count": 10000, "nrhs": 1},
        # many small SPD systems with a few right-hand sides, the benchmark's chol64_posv
        {"name": "posv_n64_x20000", "op": "posv", "n": 64, "count": 20000, "nrhs": 4, "upper": False},
        # SPD blocks of an odd order with a panel of right-hand sides (a block preconditioner, a Kalman update)
        {"name": "chol_n149_x2000", "op": "chol", "n": 149, "count": 2000, "nrhs": 16, "upper": False},
        # FP64 factor and solve at the order and batch of the benchmark's default workload
        {"name": "lu_n256_x8192", "op": "lu", "n": 256, "count": 8192, "nrhs": 1, "trans": False},
        # few systems at the top of the serving range, an odd order, several right-hand sides
        {"name": "lu_n500_x256", "op": "lu", "n": 500, "count": 256, "nrhs": 7, "trans": False},
        # the benchmark's default workload: FP32 factorization, FP64 refinement
        {"name": "mixed_n256_x8192", "op": "mixed", "n": 256, "count": 8192, "nrhs": 1, "spd": False},
        # uneven sizes in one call, the factorizations of the benchmark's vbatch_lu_gemm
        {"name": "getrf_v256_x50000", "op": "getrf_v", "n": 256, "count": 50000},
        # and its matrix products
        {"name": "gemm_v256_x50000", "op": "gemm_v", "n": 256, "count": 50000, "ta": False, "tb": False, "beta": 0.0},
        # triangular solves with a panel of vectors, from the benchmark's blas_batched
        {"name": "trsm_n64_x20000", "op": "trsm", "n": 64, "count": 20000, "nrhs": 16, "left": True, "upper": False,
         "trans": False, "unit": False},
        # QR of many small matrices (least squares, orthogonalization), from extras_batched
        {"name": "geqrf_n64_x20000", "op": "geqrf", "m": 64, "n": 64, "count": 20000},
        # explicit inverses from the factors (block Jacobi), from extras_batched
        {"name": "getri_n64_x20000", "op": "getri", "n": 64, "count": 20000},
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], its logarithm spread evenly."""
    return min(hi, max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    op = rng.choice(("gesv", "posv", "chol", "lu", "mixed", "getrf_v", "gemm_v", "trsm", "geqrf", "getri"))
    coin = lambda: rng.random() < 0.5      # noqa: E731
    if op in ("gesv", "posv"):
        c = {"op": op, "n": _log_int(rng, 2, 64), "nrhs": _log_int(rng, 1, 8)}
    elif op in ("lu", "chol"):
        c = {"op": op, "n": _log_int(rng, 65, 512), "nrhs": _log_int(rng, 1, 16)}
    elif op == "mixed":
        c = {"op": op, "n": _log_int(rng, 16, 512), "nrhs": _log_int(rng, 1, 16), "spd": coin()}
    elif op in ("getrf_v", "gemm_v"):
        c = {"op": op, "n": _log_int(rng, 16, 256)}
    elif op == "geqrf":
        n = _log_int(rng, 4, 128)
        c = {"op": op, "m": rng.randint(n, 128), "n": n}
    elif op == "trsm":
        c = {"op": op, "n": _log_int(rng, 4, 128), "nrhs": _log_int(rng, 1, 64)}
    else:
        c = {"op": op, "n": _log_int(rng, 4, 128)}
    if op in ("posv", "chol"):
        c["upper"] = rng.random() < 0.25
    elif op == "lu":
        c["trans"] = rng.random() < 0.25
    elif op == "gemm_v":
        c.update(ta=coin(), tb=coin(), beta=rng.choice((0.0, 1.0)))
    elif op == "trsm":
        c.update(left=coin(), upper=coin(), trans=coin(), unit=coin())
    # from a handful of matrices to 20,000, within about 1 GB of matrices
    order = max(c["n"], c.get("m", 0))
    c["count"] = _log_int(rng, 16, max(64, min(20000, int(1.2e8 / order ** 2))))
    return c


# ---- inputs -------------------------------------------------------------------

def _sizes(case):
    """The orders of a variable-size batch: log-uniform in [8, n]."""
    return gen.vbatch_sizes(2, case["count"], 8, case["n"]).astype(np.int64)


def _offsets(sizes):
    return np.concatenate([[0], np.cumsum(sizes)[:-1]]).astype(np.int64)


def _inputs(case, seed):
    """The operands on the GPU, column-major storage (count, cols, rows)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    uni = lambda *shape: torch.rand(*shape, generator=g, dtype=torch.float64, device="cuda").mul_(2.0).sub_(1.0)  # noqa: E731
    op, n, count = case["op"], case["n"], case["count"]
    if op in ("getrf_v", "gemm_v"):
        total = int((_sizes(case) ** 2).sum())
        return [uni(total)] if op == "getrf_v" else [uni(total), uni(total), uni(total)]
    if op == "geqrf":
        return [uni(count, n, case["m"])]
    if op == "getri":
        return [uni(count, n, n)]
    nrhs = case["nrhs"]
    if op in ("posv", "chol") or case.get("spd"):
        A = torch.empty(count, n, n, dtype=torch.float64, device="cuda")
        step = max(1, (1 << 24) // (n * n))
        for c0 in range(0, count, step):
            k = min(step, count - c0)
            F = torch.randn(k, n, n, generator=g, dtype=torch.float64, device="cuda")
            A[c0:c0 + k] = torch.bmm(F, F.transpose(1, 2).contiguous())
        A.diagonal(dim1=1, dim2=2).add_(float(n))
        return [A, uni(count, nrhs, n)]
    if op == "mixed":
        A, _ = gen.cond_batch_torch(seed % (1 << 20), count, n, "cuda")
        return [A, uni(count, nrhs, n)]
    A = uni(count, n, n)
    if op == "trsm":
        A.div_(max(1.0, n / 8.0))
        A.diagonal(dim1=1, dim2=2).uniform_(1.0, 2.0, generator=g)
        rows, cols = (n, nrhs) if case["left"] else (nrhs, n)
        return [A, uni(count, cols, rows)]
    return [A, uni(count, nrhs, n)]


def prepare(case, seed):
    L = ma.load()
    for family, row in TUNED.items():
        for size_class, variant in enumerate(row):
            L.magma_amd_tune_set(family, size_class, variant)
    op, n, count = case["op"], case["n"], case["count"]
    s = {"case": case, "L": L, "q": ma.Queue(0), "info": torch.zeros(count + 1, dtype=torch.int32, device="cuda")}

    def batch(name, t):
        s[name] = t
        s["p_" + name] = ma.ptr_array(t, t.shape[0], t[0].numel())

    ops = _inputs(case, seed)
    if op in ("getrf_v", "gemm_v"):
        sizes = _sizes(case)
        offs = _offsets(sizes ** 2)
        s["d_n"] = ma.dev_ints(sizes)
        if op == "getrf_v":
            s["A0"], s["A"] = ops[0], torch.empty_like(ops[0])
            s["ipiv"] = ma.VarInts(sizes)
            names = ("A",)
        else:
            s["A"], s["B"], s["C0"] = ops
            s["C"] = torch.zeros_like(s["C0"])
            names = ("A", "B", "C")
        for name in names:
            s["p_" + name] = torch.from_numpy(s[name].data_ptr() + offs * 8).cuda()
        return s
    if op in ("trsm", "mixed"):            # A is read only
        batch("A", ops[0])
    else:
        s["A0"] = ops[0]
        batch("A", torch.empty_like(ops[0]))
    if len(ops) > 1:
        s["B0"] = ops[1]
        batch("B", ops[1] if op == "mixed" else torch.empty_like(ops[1]))
    if op in ("gesv", "lu", "mixed", "getri"):
        s["ipiv"] = ma.IntBatch(count, n)
    if op == "mixed":
        batch("X", torch.zeros_like(ops[1]))
        s["iter"] = torch.zeros(count, dtype=torch.int32, device="cuda")
    elif op == "geqrf":
        batch("tau", torch.zeros(count, n, dtype=torch.float64, device="cuda"))
    elif op == "getri":                    # the factors are in hand, the call under test inverts
        batch("inv", torch.zeros_like(ops[0]))
        s["A"].copy_(s["A0"])
        L.magma_dgetrf_batched(n, n, s["p_A"].data_ptr(), n, s["ipiv"].ptr, s["info"].data_ptr(), count,
                               s["q"].handle)
    return s


# ---- one pass -------------------------------------------------------------------

def _uplo(case):
    return ma.MagmaUpper if case["upper"] else ma.MagmaLower


def _trans(flag):
    return ma.MagmaTrans if flag else ma.MagmaNoTrans


def run(s):
    c, L, q = s["case"], s["L"], s["q"].handle
    op, n, count, info = c["op"], c["n"], c["count"], s["info"]
    p = lambda name: s["p_" + name].data_ptr()      # noqa: E731
    if op == "mixed":
        if c["spd"]:
            L.magma_dsposv_batched(ma.MagmaLower, n, c["nrhs"], p("A"), n, p("B"), n, p("X"), n, info.data_ptr(),
                                   s["iter"].data_ptr(), count, q)
            return {"x": s["X"], "info": info[:count], "iter": s["iter"]}
        L.magma_dsgesv_batched(n, c["nrhs"], p("A"), n, s["ipiv"].ptr, p("B"), n, p("X"), n, info.data_ptr(),
                               s["iter"].data_ptr(), count, q)
        return {"x": s["X"], "ipiv": s["ipiv"].t, "info": info[:count], "iter": s["iter"]}
    if op == "trsm":
        s["B"].copy_(s["B0"])
        rows, cols = (n, c["nrhs"]) if c["left"] else (c["nrhs"], n)
        L.magmablas_dtrsm_batched(ma.MagmaLeft if c["left"] else ma.MagmaRight, _uplo(c), _trans(c["trans"]),
                                  ma.MagmaUnit if c["unit"] else ma.MagmaNonUnit, rows, cols, 1.0, p("A"), n, p("B"),
                                  rows, count, q)
        return {"x": s["B"]}
    if op == "gemm_v":
        d_n = s["d_n"].data_ptr()
        if c["beta"] != 0.0:
            s["C"].copy_(s["C0"])
        L.magmablas_dgemm_vbatched_max_nocheck(_trans(c["ta"]), _trans(c["tb"]), d_n, d_n, d_n, 1.0, p("A"), d_n,
                                               p("B"), d_n, c["beta"], p("C"), d_n, count, n, n, n, q)
        return {"c": s["C"]}
    if op == "getri":
        L.magma_dgetri_outofplace_batched(n, p("A"), n, s["ipiv"].ptr, p("inv"), n, info.data_ptr(), count, q)
        return {"inv": s["inv"], "info": info[:count]}
    s["A"].copy_(s["A0"])
    if op == "geqrf":
        L.magma_dgeqrf_batched(c["m"], n, p("A"), c["m"], p("tau"), info.data_ptr(), count, q)
        return {"qr": s["A"], "tau": s["tau"], "info": info[:count]}
    if op == "getrf_v":
        d_n = s["d_n"].data_ptr()
        L.magma_dgetrf_vbatched_max_nocheck(d_n, d_n, n, p("A"), d_n, s["ipiv"].ptr, info.data_ptr(), count, q)
        return {"lu": s["A"], "ipiv": s["ipiv"].t, "info": info[:count]}
    s["B"].copy_(s["B0"])
    nrhs = c["nrhs"]
    if op == "gesv":
        L.magma_dgesv_batched(n, nrhs, p("A"), n, s["ipiv"].ptr, p("B"), n, info.data_ptr(), count, q)
    elif op == "posv":
        L.magma_dposv_batched(_uplo(c), n, nrhs, p("A"), n, p("B"), n, info.data_ptr(), count, q)
    elif op == "lu":
        L.magma_dgetrf_batched(n, n, p("A"), n, s["ipiv"].ptr, info.data_ptr(), count, q)
        L.magma_dgetrs_batched(_trans(c["trans"]), n, nrhs, p("A"), n, s["ipiv"].ptr, p("B"), n, count, q)
    else:
        L.magma_dpotrf_batched(_uplo(c), n, p("A"), n, info.data_ptr(), count, q)
        L.magma_dpotrs_batched(_uplo(c), n, nrhs, p("A"), n, p("B"), n, count, q)
    out = {"factor": s["A"], "x": s["B"], "info": info[:count]}
    if op in ("gesv", "lu"):
        out["ipiv"] = s["ipiv"].t
    return out


# ---- what a pass cannot do without ------------------------------------------------

def work(case):
    """Each operand read once and each result written once; LAPACK's operation counts."""
    op, n, count = case["op"], case["n"], case["count"]
    lu_f = lambda k: 2.0 * k ** 3 / 3 - k ** 2 / 2 + 5.0 * k / 6      # noqa: E731
    if op == "getrf_v":
        k = _sizes(case).astype(np.float64)
        return {"bytes": float((16 * k * k + 4 * k + 4).sum()), "flops": float(lu_f(k).sum())}
    if op == "gemm_v":
        k = _sizes(case).astype(np.float64)
        return {"bytes": float(((24 if case["beta"] == 0.0 else 32) * k * k).sum()), "flops": float((2 * k ** 3).sum())}
    if op == "geqrf":
        m = case["m"]
        return {"bytes": count * (16.0 * m * n + 8 * n), "flops": count * 2.0 * n * n * (m - n / 3.0)}
    if op == "getri":
        return {"bytes": count * (16.0 * n * n + 4 * n), "flops": count * (4.0 / 3) * n ** 3}
    r = case["nrhs"]
    rhs, solve = 16.0 * n * r, 2.0 * n * n * r
    if op == "trsm":
        return {"bytes": count * (4.0 * n * (n + 1) + rhs), "flops": count * solve / 2}
    if op == "mixed":
        factor = n ** 3 / 3 if case["spd"] else 2 * n ** 3 / 3
        return {"bytes": count * (8.0 * n * n + rhs + 8), "flops": count * (factor + solve)}
    if op in ("posv", "chol"):
        return {"bytes": count * (8.0 * n * (n + 1) + rhs + 4), "flops": count * (n ** 3 / 3 + solve)}
    return {"bytes": count * (16.0 * n * n + rhs + 4 * n + 4), "flops": count * (lu_f(n) + solve)}


# ---- the same results from torch's LAPACK on the host -------------------------------

def _on_host(fn, count, *operands):
    """fn on slices of the host batches in `operands`, one slice a thread; its results joined."""
    threads = torch.get_num_threads()
    torch.set_num_threads(1)
    try:
        step = -(-count // 64)
        with ThreadPoolExecutor(max(1, threads)) as pool:
            parts = list(pool.map(lambda i: fn(*(t[i:i + step] for t in operands)), range(0, count, step)))
    finally:
        torch.set_num_threads(threads)
    return [torch.cat(p) for p in zip(*parts)]


def _lu(A):
    """Column-major storage in, column-major factors, row-order pivots."""
    LU, piv = torch.linalg.lu_factor(A.transpose(1, 2))
    return LU, piv


def _store(t):
    return t.transpose(1, 2).contiguous()


def exact(case, seed):
    op, n, count = case["op"], case["n"], case["count"]
    host = [t.cpu() for t in _inputs(case, seed)]
    if op in ("getrf_v", "gemm_v"):
        sizes = _sizes(case)
        offs = _offsets(sizes ** 2)
        out = host[0].clone() if op == "getrf_v" else host[2].clone()
        for k in np.unique(sizes):
            k = int(k)
            at = torch.from_numpy(offs[sizes == k]).view(-1, 1) + torch.arange(k * k).view(1, -1)
            take = lambda t: t[at].view(-1, k, k)      # noqa: E731
            if op == "getrf_v":
                out[at] = _on_host(lambda a: (_store(_lu(a)[0]),), at.shape[0], take(host[0]))[0].view(-1, k * k)
            else:                          # storage is the transpose: C' = op(B)' op(A)'
                a, b = take(host[0]), take(host[1])
                a = a.transpose(1, 2) if case["ta"] else a
                b = b.transpose(1, 2) if case["tb"] else b
                c = torch.bmm(b.contiguous(), a.contiguous()).view(-1, k * k)
                out[at] = c if case["beta"] == 0.0 else c + case["beta"] * out[at]
        return {"lu": out, "ipiv": None, "info": None} if op == "getrf_v" else {"c": out}
    if op == "geqrf":
        def qr(a):
            f, tau = torch.geqrf(a.transpose(1, 2))
            return _store(f), tau
        f, tau = _on_host(qr, count, *host)
        return {"qr": f, "tau": tau, "info": None}
    if op == "getri":
        return {"inv": _on_host(lambda a: (_store(torch.linalg.inv(a.transpose(1, 2))),), count, *host)[0], "info": None}
    if op == "trsm":
        def tri(a, b):
            t = a.transpose(1, 2)
            t = torch.triu(t) if case["upper"] else torch.tril(t)
            upper = case["upper"] != case["trans"]
            t = t.transpose(1, 2) if case["trans"] else t
            x = torch.linalg.solve_triangular(t, b.transpose(1, 2), upper=upper, left=case["left"],
                                              unitriangular=case["unit"])
            return (_store(x),)
        return {"x": _on_host(tri, count, *host)[0]}
    if op in ("posv", "chol"):
        def chol(a, b):
            l = torch.linalg.cholesky(a)
            x = torch.cholesky_solve(b.transpose(1, 2), l)
            # the triangle that is not referenced keeps what it held; a is symmetric
            keep = torch.tril(a, -1).transpose(1, 2) if not case["upper"] else torch.tril(a, -1)
            f = torch.tril(l)                  # L, row i column j
            return _store(f + keep if not case["upper"] else f.transpose(1, 2) + keep), _store(x)
        f, x = _on_host(chol, count, *host)
        return {"factor": f, "x": x, "info": None}

    def general(a, b):
        LU, piv = _lu(a)
        x = torch.linalg.lu_solve(LU, piv, b.transpose(1, 2), adjoint=bool(case.get("trans")))
        return (_store(LU), _store(x))

    f, x = _on_host(general, count, *host)
    if op == "mixed":
        return {"x": x, "info": None, "iter": None} if case["spd"] else {"x": x, "ipiv": None, "info": None, "iter": None}
    return {"factor": f, "x": x, "info": None, "ipiv": None}
