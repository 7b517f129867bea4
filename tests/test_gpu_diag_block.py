"""Edges of the 64x64 diagonal blocks of POTRF and TRSM, which are factored and inverted in 16-column panels: sizes
around a panel's and a block's end, and a non-positive pivot at the first and last column of each. FP64 against the
oracle at the 1e-13 of the other FP64 tile tests."""
import numpy as np
import pytest

from gpu_util import from_dev, rel, to_dev

pytestmark = pytest.mark.gpu

EDGES = [1, 2, 15, 16, 17, 31, 33, 47, 48, 49, 63, 64, 65, 79, 81, 127, 128, 129, 191, 193]


@pytest.mark.parametrize("n", EDGES)
def test_potrf_trsm_edges(ctx, oracle, n):
    A = oracle.spd_bbt(n, 500 + n)
    dA = to_dev(A)
    assert ctx.potrf(dA, n, n) == 0
    ref = A.copy(order="F")
    assert oracle.dpotrf(ref) == 0
    assert rel(np.tril(from_dev(dA)), np.tril(ref)) < 1e-13
    L = np.asfortranarray(np.tril(ref))
    B = np.asfortranarray(np.random.default_rng(n).standard_normal((37, n)))
    dB = to_dev(B)
    ctx.trsm(37, n, to_dev(L), n, dB, 37)
    want = B.copy(order="F")
    oracle.dtrsm_rltn(L, want)
    assert rel(from_dev(dB), want) < 1e-13


@pytest.mark.parametrize("col", [0, 1, 15, 16, 31, 32, 47, 48, 62, 63, 64, 69])
def test_bad_pivot_column(ctx, oracle, col):
    n = 70
    A = oracle.spd_bbt(n, 9)
    A[col, col] = -1.0
    ref = A.copy(order="F")
    info = ctx.potrf(to_dev(A), n, n)
    assert info == oracle.dpotrf(ref) == col + 1
