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


@pytest.mark.parametrize("n", [255, 256, 257, 320, 449, 513, 1030])
@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_potrf_block_items(ctx, oracle, n, dtype):
    # tiles of several 64-row blocks with a ragged last one, leading dimension above n, twice on the same flags
    import torch
    A = oracle.spd_bbt(n, 40 + n)
    ref = A.copy(order="F")
    assert oracle.dpotrf(ref) == 0
    ld = n + 3
    for _ in range(2):
        buf = torch.zeros((n, ld), dtype=torch.float64)
        buf[:, :n] = torch.from_numpy(np.ascontiguousarray(A.T))
        d = buf.to(torch.float32 if dtype == "f32" else torch.float64).cuda()
        assert ctx.potrf(d, n, ld) == 0
        out = from_dev(d)[:n]
        assert rel(np.tril(out), np.tril(ref)) < (2e-6 if dtype == "f32" else 1e-13)
        assert np.array_equal(np.triu(out, 1), np.triu(A.astype(np.float32) if dtype == "f32" else A, 1))


@pytest.mark.parametrize("m,n", [(1, 64), (15, 65), (16, 127), (17, 192), (33, 448), (31, 511), (65, 512), (40, 513)])
@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_trsm_strips(ctx, m, n, dtype):
    # strips of X in LDS (up to 512 columns) and beside them the form for wider L, odd leading dimensions
    import torch
    rng = np.random.default_rng(m * n)
    L = np.tril(rng.standard_normal((n, n)) * (0.7 / np.sqrt(n)), -1) + np.diag(rng.uniform(1.2, 1.6, n))
    B = rng.standard_normal((m, n))
    dt = torch.float64 if dtype == "f64" else torch.float32
    dL = torch.zeros((n, n + 1), dtype=torch.float64)
    dL[:, :n] = torch.from_numpy(np.ascontiguousarray(L.T))
    dB = torch.full((n, m + 3), 5.0, dtype=torch.float64)
    dB[:, :m] = torch.from_numpy(np.ascontiguousarray(B.T))
    dL, dB = dL.to(dt).cuda(), dB.to(dt).cuda()
    Lr, Br = from_dev(dL)[:n], from_dev(dB)[:m]
    ctx.trsm(m, n, dL, n + 1, dB, m + 3)
    out = from_dev(dB)
    want = np.linalg.solve(Lr, Br.T).T
    assert rel(out[:m], want) < (2e-6 if dtype == "f32" else 1e-13)
    assert (out[m:] == 5.0).all()
