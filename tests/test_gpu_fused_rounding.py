"""Rounding of updates of several steps in one task, on random SPD matrices of partitions that fuse (ragged ones among
them). FP32 and BF16 items subtract step by step in registers, so the factor is the host-sequenced schedule's to the last
bit. FP64 and bf16x3 items sum the steps' products first. FP64 is held to the oracle at the bounds of the other FP64
factorizations. For bf16x3, splitting an operand into two bf16 leaves about 2^-17 of it, and FP32 sums of 1024 products about
2^-24 sqrt(1024) = 2^-19: in quadrature 1.03 times the residual of single steps; 1.25 is allowed."""
import functools

import numpy as np
import pytest

import tasktorrent_amd as tt

pytestmark = pytest.mark.gpu

PARTITIONS = {
    "64": [64] * 26 + [5],
    "128": [128] * 24 + [37],
    "192": [192] * 15 + [130],
    "mixed": [64] * 9 + [128] * 8 + [96] * 3 + [64] * 6 + [1, 64, 64, 64],
    "64 large": [64] * 59 + [17],
    "256 large": [256] * 30 + [100],
}


@functools.lru_cache(maxsize=1)
def problem(name):
    from oracle import oracle as o
    n = sum(PARTITIONS[name])
    return PARTITIONS[name], np.asfortranarray(o.spd_bbt(n, n))


def factor(ctx, sizes, A, sched, prec):
    M = tt.TiledMatrix(ctx, sizes, "f64" if prec == "f64" else "f32")
    M.set(A)
    assert ctx.potrf_tiled(M, sched, 2, prec) == 0
    return M


@pytest.mark.parametrize("name,prec", [(p, q) for p in PARTITIONS for q in ("f32", "bf16")])
def test_register_sums_equal_single_steps(ctx, oracle, name, prec):
    sizes, A = problem(name)
    out = []
    for sched in (tt.TTAD_SCHED_STREAM, tt.TTAD_SCHED_PERSISTENT):
        M = factor(ctx, sizes, A, sched, prec)
        out.append(M.get())
        M.close()
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("name", PARTITIONS)
def test_fp64_sums_match_oracle(ctx, oracle, name):
    sizes, A = problem(name)
    M = factor(ctx, sizes, A, tt.TTAD_SCHED_PERSISTENT, "f64")
    L = M.get()
    M.close()
    Lref, st = oracle.cholesky(A, sizes=sizes, n_threads=4)
    assert st["info"] == 0
    assert np.linalg.norm(L - Lref) / np.linalg.norm(Lref) < 1e-12
    assert oracle.factor_residual(A, L) < 1e-14


@pytest.mark.parametrize("name", PARTITIONS)
def test_bf16x3_sums_are_as_accurate_as_single_steps(ctx, oracle, name):
    sizes, A = problem(name)
    A0 = tt.TiledMatrix(ctx, sizes, "f64")
    A0.set(A)
    r = []
    for sched in (tt.TTAD_SCHED_STREAM, tt.TTAD_SCHED_PERSISTENT):
        M = factor(ctx, sizes, A, sched, "bf16x3")
        r.append(ctx.factor_residual(A0, M))
        M.close()
    A0.close()
    assert r[1] <= 1.25 * r[0], r
