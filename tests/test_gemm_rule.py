"""Which items a raw GEMM takes: the faster ones of the two at sizes where both were timed (1 = 64x64), and on the GPU exact
products on both sides of the lines."""
import numpy as np
import pytest

import host_rules

F64, F32, BF16, BF16X3 = range(4)
# (precision, m, n, k, syrk) -> 64x64 items
MEASURED = {
    (F64, 256, 256, 256, 0): 1, (F64, 1000, 1000, 300, 0): 1, (F64, 1408, 1408, 16, 0): 1, (F64, 1536, 1536, 16, 0): 0,
    (F64, 1536, 1536, 64, 0): 1, (F64, 2048, 1536, 512, 0): 1, (F64, 2048, 2048, 512, 0): 0, (F64, 2048, 2048, 64, 1): 1,
    (F32, 1408, 1408, 24, 0): 1, (F32, 1536, 1536, 48, 0): 0, (F32, 1664, 1664, 64, 0): 1, (F32, 2816, 2816, 512, 0): 0,
    (BF16, 2048, 2048, 512, 0): 1, (BF16, 2048, 2048, 4096, 0): 0, (BF16, 1792, 1792, 3072, 0): 0,
    (BF16, 1700, 1700, 4096, 0): 1, (BF16, 1536, 1536, 4096, 0): 1, (BF16, 2816, 2816, 512, 0): 0,
    (BF16X3, 2048, 2048, 4096, 0): 1, (BF16X3, 2816, 2816, 512, 0): 0,
}


def test_faster_items(tmp_path):
    args = [v for k in MEASURED for v in k]
    out = host_rules.run(host_rules.build("gemm_rule", tmp_path), *args).split("\n")
    assert {tuple(map(int, line.split()[:5])): int(line.split()[5]) for line in out if line} == MEASURED


@pytest.mark.gpu
@pytest.mark.parametrize("prec,m,n,k", [("f64", 1410, 1409, 17), ("f64", 1537, 1500, 63), ("f64", 1537, 1500, 64),
                                        ("f32", 1410, 1409, 17), ("f32", 1537, 1500, 63), ("bf16", 1793, 1791, 1024),
                                        ("bf16", 1793, 1791, 1056)])
def test_integer_exact_on_both_sides(ctx, prec, m, n, k):
    import torch
    from gpu_util import from_dev, to_dev
    rng = np.random.default_rng(m + k)
    A, B, C = (rng.integers(-4, 5, s).astype(np.float64) for s in ((m, k), (n, k), (m, n)))
    dt = torch.float64 if prec == "f64" else torch.float32
    dC = to_dev(C, dt)
    if prec == "bf16":
        ctx.gemm_bf16(m, n, k, -1.0, to_dev(A, dt), m, to_dev(B, dt), n, 1.0, dC, m, split=False)
    else:
        ctx.gemm(m, n, k, -1.0, to_dev(A, dt), m, to_dev(B, dt), n, 1.0, dC, m)
    assert np.array_equal(from_dev(dC), C - A @ B.T)  # sums stay below 2^24
