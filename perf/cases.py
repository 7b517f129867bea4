"""Performance cases of the tiled Cholesky solver: the calls a program makes, from one tile to the largest
matrix of the benchmark, each through the Python front of the C-ABI.

Kinds of case (the key "kind"):
  gemm   one C := C - A B^T (or its SYRK form) on caller-owned device arrays, FP64 / FP32 / BF16 / BF16x3
  trsm   one X L^T = B on caller-owned device arrays
  potrf  one LAPACK-shaped factorization of a caller-owned device array
  factor a dense device matrix into tiles, the tiled Cholesky, and the factor back out as a dense array
  posv   the mixed-precision solver on a resident tiled matrix (FP64 refinement to 1e-12)
  solve  new right-hand sides with a kept FP64 factor (two triangular sweeps)
  refine new right-hand sides with a kept FP32 factor, refined in FP64 to 1e-12
  serve  a burst of SPD solve requests of uneven sizes through the serving loop

Matrices are A = B B^T / n + delta I with B iid N(0, 1) rounded to a grid of 2^-8, so
that every product sum is exact in FP64 whatever the order it is formed in, and a matrix depends on its seed alone.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import tasktorrent_amd as tt

_CTX = None


def _ctx():
    """The program's one device context."""
    global _CTX
    if _CTX is None:
        _CTX = tt.Context(0)
    return _CTX


def _gen(seed: int):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _randn(shape, g, dtype=torch.float64):
    return torch.randn(shape, dtype=dtype, device="cuda", generator=g)


def _spd(n: int, seed: int, delta: float = 1.0):
    """A = B B^T / n + delta I. Symmetric, so row-major and column-major storage are the same."""
    g = _gen(seed)
    B = _randn((n, n), g)
    B.mul_(256.0).round_().div_(256.0)
    A = torch.matmul(B, B.t())
    del B
    A.div_(n)
    A.diagonal().add_(delta)
    return A


def _lower(n: int, g, dtype):
    """A lower-triangular factor as Cholesky leaves it: diagonal near 1.4, entries of order 1/sqrt(n) below."""
    L = torch.tril(_randn((n, n), g) * (0.7 / math.sqrt(n)), -1)
    L.diagonal().copy_(1.2 + 0.4 * torch.rand((n,), dtype=torch.float64, device="cuda", generator=g))
    return L.to(dtype)


def _colmajor(M, ld: int):
    """Column-major copy of M (m x n) with leading dimension ld, as a torch (n, ld) tensor."""
    m, n = M.shape
    out = torch.zeros((n, ld), dtype=M.dtype, device="cuda")
    out[:, :m].copy_(M.t())
    return out


def _tiled(ctx, A, n: int, tile: int):
    M = tt.TiledMatrix.uniform(ctx, n, tile, "f64")
    M.set(A)
    return M


_DT = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.float32, "bf16x3": torch.float32}


def listed():
    return [
        # one tile update of a graph of small tiles: launch and latency count
        {"name": "gemm_f64_256", "kind": "gemm", "prec": "f64", "m": 256, "n": 256, "k": 256, "pad": 0, "syrk": False},
        # a ragged symmetric update with a leading dimension of its own, FP32
        {"name": "syrk_f32_1000", "kind": "gemm", "prec": "f32", "m": 1000, "n": 1000, "k": 300, "pad": 3,
         "syrk": True},
        # the trailing update of the mixed solver as a caller's own call, ragged edges
        {"name": "gemm_bf16x3_5000", "kind": "gemm", "prec": "bf16x3", "m": 5000, "n": 3000, "k": 512, "pad": 0,
         "syrk": False},
        # the FP64 trailing update of a large matrix
        {"name": "gemm_f64_8192", "kind": "gemm", "prec": "f64", "m": 8192, "n": 8192, "k": 512, "pad": 0,
         "syrk": False},
        # the panel below a 512-column diagonal tile
        {"name": "trsm_f64_8000x512", "kind": "trsm", "prec": "f64", "m": 8000, "n": 512, "pad": 0},
        # one diagonal tile through the LAPACK-shaped call
        {"name": "potrf_f64_512", "kind": "potrf", "prec": "f64", "n": 512, "pad": 0},
        # a small dense system's factorization, the drop-in's own configuration (8 x 8 tiles of 256)
        {"name": "factor_f64_2048", "kind": "factor", "n": 2048, "tile": 256},
        # a large FP64 factorization (32 x 32 tiles of 512)
        {"name": "factor_f64_16384", "kind": "factor", "n": 16384, "tile": 512},
        # an ordinary mixed-precision solve of odd size, few right-hand sides
        {"name": "posv_f32_3000", "kind": "posv", "prec": "f32", "n": 3000, "tile": 256, "nrhs": 5, "delta": 1.0},
        # the headline solve: n = 32768, 16 right-hand sides, condition about 400
        {"name": "posv_bf16x3_32768", "kind": "posv", "prec": "bf16x3", "n": 32768, "tile": 512, "nrhs": 16,
         "delta": 1e-2},
        # more right-hand sides for a factor that the program kept in FP64
        {"name": "solve_f64_8192", "kind": "solve", "n": 8192, "tile": 512, "nrhs": 16},
        # serving: a burst of requests of uneven sizes, 1-8 right-hand sides each
        {"name": "serve_256", "kind": "serve", "requests": 256, "n_max": 4096, "prec": "bf16x3"},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the same ranges (rng: random.Random)."""
    kind = rng.choice(["gemm", "gemm", "trsm", "potrf", "factor", "posv", "posv", "solve", "refine", "serve"])
    if kind == "gemm":
        prec = rng.choice(["f64", "f32", "bf16", "bf16x3"])
        syrk = rng.random() < 0.3
        m = _log_int(rng, 64, 8192)
        n = m if syrk else _log_int(rng, 64, 8192)
        return {"kind": kind, "prec": prec, "m": m, "n": n, "k": _log_int(rng, 64, 1024),
                "pad": rng.choice([0, 0, 1, 6]), "syrk": syrk}
    if kind == "trsm":
        return {"kind": kind, "prec": rng.choice(["f64", "f64", "f32"]), "m": _log_int(rng, 64, 16384),
                "n": _log_int(rng, 64, 1024), "pad": rng.choice([0, 0, 1, 6])}
    if kind == "potrf":
        return {"kind": kind, "prec": rng.choice(["f64", "f64", "f32"]), "n": _log_int(rng, 64, 1024),
                "pad": rng.choice([0, 0, 1, 6])}
    if kind == "serve":
        return {"kind": kind, "requests": _log_int(rng, 32, 256), "n_max": rng.choice([1024, 2048, 4096]),
                "prec": rng.choice(["bf16x3", "f32"])}
    hi = {"factor": 16384, "posv": 32768, "solve": 16384, "refine": 16384}[kind]
    n = _log_int(rng, 256, hi)
    # tiles of 512 pay from a few thousand rows on; smaller matrices are cut finer
    tile = 512 if n >= 4096 else rng.choice([128, 256]) if n < 1024 else 256
    if kind == "factor":
        return {"kind": kind, "n": n, "tile": tile}
    nrhs = rng.choice([1, 2, 5, 8, 16, 16])
    if kind == "posv":
        return {"kind": kind, "prec": rng.choice(["bf16x3", "bf16x3", "f32", "f64"]), "n": n, "tile": tile,
                "nrhs": nrhs, "delta": 1.0}
    return {"kind": kind, "n": n, "tile": tile, "nrhs": nrhs}


def _serve_requests(case, seed):
    """Sizes n = 64 round(exp(U(ln 64, ln n_max)) / 64) and 1-8 right-hand sides per request. The numbers of rows
    and right-hand sides belong to the case; the matrices and right-hand sides to the seed."""
    rng = np.random.default_rng(1234)
    out = []
    for q in range(case["requests"]):
        n = int(64 * round(math.exp(rng.uniform(math.log(64), math.log(case["n_max"]))) / 64))
        out.append((max(64, min(case["n_max"], n)), int(rng.integers(1, 9)), int(seed) * 1009 + 7 * q + 1))
    return out


def _serve_rhs(n, nrhs, rseed):
    return np.asfortranarray(np.random.default_rng(rseed).standard_normal((n, nrhs)))


def _inputs(case, seed):
    """The dense inputs of a case, from the seed alone."""
    kind = case["kind"]
    if kind == "gemm":
        g, dt = _gen(seed), _DT[case["prec"]]
        m, n, k = case["m"], case["n"], case["k"]
        A = _randn((m, k), g, dt)
        B = A if case["syrk"] else _randn((n, k), g, dt)
        return A, B, _randn((m, n), g, dt)
    if kind == "trsm":
        g, dt = _gen(seed), _DT[case["prec"]]
        L = _lower(case["n"], g, dt)
        return L, _randn((case["m"], case["n"]), g, dt)
    if kind == "potrf":
        return _spd(case["n"], seed).to(_DT[case["prec"]])
    if kind == "factor":
        return _spd(case["n"], seed)
    A = _spd(case["n"], seed, case.get("delta", 1.0))
    return A, _randn((case["nrhs"], case["n"]), _gen(seed + 1))  # right-hand sides column-major


def prepare(case, seed):
    ctx = _ctx()
    kind = case["kind"]
    st = {"case": case, "ctx": ctx}
    if kind == "gemm":
        A, B, C = _inputs(case, seed)
        m, n, pad = case["m"], case["n"], case["pad"]
        st["A"] = _colmajor(A, m + pad)
        st["B"] = st["A"] if case["syrk"] else _colmajor(B, n + pad)
        st["C"] = _colmajor(C, m + pad)
        st["out"] = torch.empty_like(st["C"])
    elif kind == "trsm":
        L, B = _inputs(case, seed)
        st["L"] = _colmajor(L, case["n"] + case["pad"])
        st["B"] = _colmajor(B, case["m"] + case["pad"])
        st["out"] = torch.empty_like(st["B"])
    elif kind == "potrf":
        st["A"] = _colmajor(_inputs(case, seed), case["n"] + case["pad"])
        st["out"] = torch.empty_like(st["A"])
    elif kind == "factor":
        st["A"] = _inputs(case, seed)
        st["M"] = tt.TiledMatrix.uniform(ctx, case["n"], case["tile"], "f64")
        st["out"] = torch.empty_like(st["A"])
    elif kind == "serve":
        st["reqs"] = []
        for n, nrhs, rseed in _serve_requests(case, seed):
            A = _spd(n, rseed)
            M = _tiled(ctx, A, n, 256)
            torch.cuda.synchronize()
            st["reqs"].append((M, _serve_rhs(n, nrhs, rseed)))
        st["X"] = np.empty(sum(B.size for _, B in st["reqs"]))
    else:
        A, B = _inputs(case, seed)
        n, tile = case["n"], case["tile"]
        st["A"] = _tiled(ctx, A, n, tile)
        st["B"], st["X"] = B, torch.zeros_like(B)
        if kind == "solve":  # the factor that the program kept
            st["L"] = tt.TiledMatrix.uniform(ctx, n, tile, "f64")
            st["L"].copy_from(st["A"])
            assert ctx.potrf_tiled(st["L"], prec="f64") == 0
        elif kind == "refine":
            st["L"] = tt.TiledMatrix.uniform(ctx, n, tile, "f32")
            st["L"].copy_from(st["A"])
            assert ctx.potrf_tiled(st["L"], prio_kind=4, prec="bf16x3") == 0
    torch.cuda.synchronize()
    return st


def run(st):
    case, ctx = st["case"], st["ctx"]
    kind = case["kind"]
    if kind == "gemm":  # the update is in place: the program keeps its C in another array
        m, n, k, pad = case["m"], case["n"], case["k"], case["pad"]
        st["out"].copy_(st["C"])
        if case["prec"] in ("bf16", "bf16x3"):
            ctx.gemm_bf16(m, n, k, -1.0, st["A"], m + pad, st["B"], n + pad, 1.0, st["out"], m + pad,
                          syrk=case["syrk"], split=case["prec"] == "bf16x3")
        elif case["syrk"]:
            ctx.syrk(n, k, -1.0, st["A"], m + pad, 1.0, st["out"], m + pad)
        else:
            ctx.gemm(m, n, k, -1.0, st["A"], m + pad, st["B"], n + pad, 1.0, st["out"], m + pad)
        return st["out"]
    if kind == "trsm":
        m, n, pad = case["m"], case["n"], case["pad"]
        st["out"].copy_(st["B"])
        ctx.trsm(m, n, st["L"], n + pad, st["out"], m + pad)
        return st["out"]
    if kind == "potrf":
        st["out"].copy_(st["A"])
        info = ctx.potrf(st["out"], case["n"], case["n"] + case["pad"])
        return {"L": st["out"], "info": info}
    if kind == "factor":
        M = st["M"]
        M.set(st["A"])
        info = ctx.potrf_tiled(M, tt.TTAD_SCHED_PERSISTENT, 2, "f64")
        return {"L": M.get(st["out"]), "info": info}
    if kind == "posv":
        r = ctx.posv_mixed(st["A"], case["prec"], case["nrhs"], st["B"], st["X"], tol=1e-12)
        return {"X": st["X"], "rc": r["rc"]}
    if kind == "solve":
        ctx.solve(st["L"], case["nrhs"], st["B"], st["X"])
        return {"X": st["X"]}
    if kind == "refine":
        r = ctx.solve_ir(st["A"], st["L"], case["nrhs"], st["B"], st["X"], tol=1e-12)
        return {"X": st["X"], "rc": r["rc"]}
    # serve: the loop holds the device while it runs, so a program that has other work for the GPU opens it for a
    # burst and closes it
    srv = tt.Server(ctx, hbm_budget=8 << 30, max_tasks=1 << 20, max_requests=1024)
    try:
        ids = [srv.submit(M, B, prec=case["prec"])[0] for M, B in st["reqs"]]
        got = srv.wait_all(ids)
    finally:
        srv.close()
    off = 0
    for i in ids:  # the program's own array of all solutions, request after request, column-major
        X = got[i]["X"]
        st["X"][off:off + X.size] = X.ravel(order="F")
        off += X.size
    return {"X": st["X"], "status": np.array([got[i]["status"] for i in ids])}


def work(case):
    """Bytes and operations one pass cannot do without."""
    kind = case["kind"]
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        es = 8 if case["prec"] == "f64" else 4
        if case["syrk"]:
            return {"bytes": es * (m * k + m * (m + 1)), "flops": 1.0 * m * (m + 1) * k}
        return {"bytes": es * (m * k + n * k + 2 * m * n), "flops": 2.0 * m * n * k}
    if kind == "trsm":
        m, n = case["m"], case["n"]
        es = 8 if case["prec"] == "f64" else 4
        return {"bytes": es * (n * (n + 1) // 2 + 2 * m * n), "flops": 1.0 * m * n * n}
    if kind == "potrf":
        n = case["n"]
        es = 8 if case["prec"] == "f64" else 4
        return {"bytes": es * n * (n + 1), "flops": n ** 3 / 3.0}
    if kind == "factor":
        n = case["n"]
        return {"bytes": 8 * (n * (n + 1) // 2 + n * n), "flops": n ** 3 / 3.0}
    if kind == "serve":
        b = f = 0
        for n, nrhs, _ in _serve_requests(case, 0):
            b += 8 * (n * (n + 1) // 2 + 2 * n * nrhs)
            f += n ** 3 / 3.0 + 4.0 * n * n * nrhs  # solve and the residual that accepts it
        return {"bytes": b, "flops": f}
    n, nrhs = case["n"], case["nrhs"]
    vec = 8 * 2 * n * nrhs
    if kind == "posv":
        return {"bytes": 8 * (n * (n + 1) // 2) + vec, "flops": n ** 3 / 3.0 + 4.0 * n * n * nrhs}
    if kind == "solve":
        return {"bytes": 8 * (n * (n + 1) // 2) + vec, "flops": 2.0 * n * n * nrhs}
    return {"bytes": 12 * (n * (n + 1) // 2) + vec, "flops": 4.0 * n * n * nrhs}  # refine: A in FP64, L in FP32


def _chol_solve(A, Bt):
    """X^T of A X = B from B^T (rows are right-hand sides), FP64, corrected once."""
    L = torch.linalg.cholesky(A)
    B = Bt.t().contiguous()
    X = torch.cholesky_solve(B, L)
    X = X + torch.cholesky_solve(B - A @ X, L)
    return X.t().contiguous()


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemm":
        A, B, C = (t.double() for t in _inputs(case, seed))
        full = C - A @ B.t()
        if case["syrk"]:  # the strict upper triangle is not written
            full = torch.tril(full) + torch.triu(C, 1)
        return _colmajor(full, case["m"] + case["pad"])
    if kind == "trsm":
        L, B = (t.double() for t in _inputs(case, seed))
        X = torch.linalg.solve_triangular(L, B.t().contiguous(), upper=False)  # L X^T = B^T
        return _colmajor(X.t(), case["m"] + case["pad"])
    if kind == "potrf":
        A = _inputs(case, seed).double()
        L = torch.linalg.cholesky(A)
        return {"L": _colmajor(torch.tril(L) + torch.triu(A, 1), case["n"] + case["pad"]), "info": None}
    if kind == "factor":
        L = torch.linalg.cholesky(_inputs(case, seed))
        return {"L": L.t().contiguous(), "info": None}  # column-major
    if kind == "serve":
        X = []
        for n, nrhs, rseed in _serve_requests(case, seed):
            B = torch.from_numpy(_serve_rhs(n, nrhs, rseed)).cuda()
            X.append(_chol_solve(_spd(n, rseed), B.t()).cpu().numpy().ravel())
        return {"X": np.concatenate(X), "status": None}
    A, B = _inputs(case, seed)
    X = _chol_solve(A, B)
    return {"X": X} if kind == "solve" else {"X": X, "rc": None}
