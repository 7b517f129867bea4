"""Which form a raw TRSM takes: the faster one of the two at sizes where both were timed (1 = strips with X in LDS), and
on the GPU equal results on both sides of the line."""
import numpy as np
import pytest

import host_rules

# (element bytes, m, n) -> form
MEASURED = {
    (8, 256, 512): 1, (8, 8192, 512): 1, (8, 14000, 512): 1, (8, 16384, 512): 0, (8, 262144, 512): 0,
    (8, 4096, 256): 1, (8, 16384, 256): 0, (8, 65536, 256): 0, (8, 4096, 128): 1, (8, 16384, 128): 0,
    (8, 16384, 64): 0, (8, 262144, 64): 0, (8, 4096, 513): 0,
    (4, 16384, 512): 1, (4, 40000, 512): 1, (4, 262144, 512): 1, (4, 16384, 256): 1, (4, 40000, 256): 1,
    (4, 16384, 128): 1, (4, 32768, 128): 0, (4, 32768, 64): 0, (4, 262144, 64): 0,
}


def test_faster_form(tmp_path):
    args = [v for k in MEASURED for v in k]
    out = host_rules.run(host_rules.build("trsm_rule", tmp_path), *args).split("\n")
    assert {tuple(map(int, line.split()[:3])): int(line.split()[3]) for line in out if line} == MEASURED


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,n,m", [("f64", 64, 8192), ("f64", 100, 8192), ("f32", 100, 16384)])
def test_same_bits_on_both_sides(ctx, dtype, n, m):
    # the first m rows of a call just past the line are solved as by the call at the line
    import torch
    dt = torch.float64 if dtype == "f64" else torch.float32
    g = torch.Generator(device="cuda").manual_seed(n)
    L = torch.tril(torch.randn((n, n), dtype=dt, device="cuda", generator=g) * (0.7 / n ** 0.5), -1)
    L.diagonal().fill_(1.4)
    L = L.t().contiguous()  # column-major
    B = torch.randn((n, m + 64), dtype=dt, device="cuda", generator=g)
    one, two = B[:, :m].contiguous(), B.clone()
    ctx.trsm(m, n, L, n, one, m)
    ctx.trsm(m + 64, n, L, n, two, m + 64)
    assert np.array_equal(one.cpu().numpy(), two[:, :m].cpu().numpy())
