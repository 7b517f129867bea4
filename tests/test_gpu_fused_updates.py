"""Updates of several steps in one task (large tiled factorizations). The matrices are L L^T of integer factors with unit
diagonal tiles, so every product, sum and solve is exact in every precision and the factor must be L to the last bit."""
import functools

import numpy as np
import pytest

import tasktorrent_amd as tt

pytestmark = pytest.mark.gpu

# more than 8 items per CU (512 columns a sum) but the last two, beyond 128 (2048 columns, all steps that a task may hold);
# ragged last tiles, widths that change along the matrix, widths that are no multiple of 64, a group cut short
PARTITIONS = {
    "64": [64] * 25 + [5],
    "128": [128] * 24 + [37],
    "192": [192] * 15 + [130],
    "96": [96] * 25,
    "mixed": [64] * 9 + [128] * 8 + [96] * 3 + [64] * 6 + [1, 64, 64, 64],
    "64 large": [64] * 59 + [17],
    "128 large": [128] * 60,
}


@functools.lru_cache(maxsize=1)
def problem(name):
    sizes = PARTITIONS[name]
    n = sum(sizes)
    rng = np.random.default_rng(n)
    L = np.tril(rng.integers(-2, 3, (n, n)).astype(np.float32))
    at = 0
    for b in sizes:
        L[at:at + b, at:at + b] = np.eye(b)
        at += b
    return sizes, L.astype(np.float64), (L @ L.T).astype(np.float64)  # |entries| < 2^24


@pytest.mark.parametrize("name,prec", [(p, q) for p in PARTITIONS for q in ("f64", "f32", "bf16", "bf16x3")])
def test_integer_factor_exact(ctx, name, prec):
    sizes, L, A = problem(name)
    M = tt.TiledMatrix(ctx, sizes, "f64" if prec == "f64" else "f32")
    for prio in (2, 0):
        M.set(A)
        assert ctx.potrf_tiled(M, tt.TTAD_SCHED_PERSISTENT, prio, prec) == 0
        assert np.array_equal(M.get(), L)
    M.close()
