"""64x64 GEMM/SYRK items (small products and the small steps of a factorization) at the edges of their tiles and
K-chunks, against FP64 products. Tolerances: FP64 1e-13 relative; FP32 and bf16x3 by their own exactness on integer
data; the tiled factorization bitwise against the host-sequenced schedule, which runs 128x128 items."""
import numpy as np
import pytest

import tasktorrent_amd as tt
from gpu_util import from_dev, rel, to_dev

pytestmark = pytest.mark.gpu

SHAPES = [(64, 64, 64), (63, 65, 31), (128, 64, 32), (129, 200, 33), (1, 1, 1), (257, 190, 65), (1500, 1400, 96)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("prec", ["f64", "f32", "bf16", "bf16x3"])
def test_small_items_integer_exact(ctx, m, n, k, prec):
    import torch
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    lda, ldb, ldc = m + 1, n + 2, m + 3
    A, B, C = (np.asfortranarray(rng.integers(-4, 5, s).astype(np.float64)) for s in ((lda, k), (ldb, k), (ldc, n)))
    dt = torch.float64 if prec == "f64" else torch.float32
    dA, dB, dC = to_dev(A, dt), to_dev(B, dt), to_dev(C, dt)
    if prec in ("f64", "f32"):
        ctx.gemm(m, n, k, -1.0, dA, lda, dB, ldb, 1.0, dC, ldc)
    else:
        ctx.gemm_bf16(m, n, k, -1.0, dA, lda, dB, ldb, 1.0, dC, ldc, split=prec == "bf16x3")
    want = C.copy()
    want[:m] -= A[:m] @ B[:n].T
    assert np.array_equal(from_dev(dC), want)


@pytest.mark.parametrize("n,k", [(64, 32), (65, 33), (200, 70), (700, 300)])
def test_small_items_syrk(ctx, n, k):
    rng = np.random.default_rng(n + k)
    A = np.asfortranarray(rng.standard_normal((n, k)))
    C = np.asfortranarray(rng.standard_normal((n, n)))
    dA, dC = to_dev(A), to_dev(C)
    ctx.syrk(n, k, -1.0, dA, n, 1.0, dC, n)
    out, want = from_dev(dC), C - A @ A.T
    assert rel(np.tril(out), np.tril(want)) < 1e-13
    assert np.array_equal(np.triu(out, 1), np.triu(C, 1))


@pytest.mark.parametrize("n,b", [(300, 128), (705, 192), (1100, 256)])
@pytest.mark.parametrize("prec", ["f64", "f32", "bf16", "bf16x3"])
def test_small_steps_bitwise_equal_to_stream_schedule(ctx, oracle, n, b, prec):
    A = oracle.spd_bbt(n, n)
    st = "f64" if prec == "f64" else "f32"
    out = []
    for sched in (tt.TTAD_SCHED_STREAM, tt.TTAD_SCHED_PERSISTENT):
        M = tt.TiledMatrix.uniform(ctx, n, b, st)
        M.set(A)
        assert ctx.potrf_tiled(M, sched, 2, prec) == 0
        out.append(M.get())
        M.close()
    assert np.array_equal(out[0], out[1])
