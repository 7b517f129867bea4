"""Leading dimensions of TRSM at which 64 columns pass 4 GB: the items that keep X in LDS address it by 32-bit lane
offsets behind a 64-bit base. The address rule on the CPU, and one such call on the GPU."""
import numpy as np
import pytest

import host_rules


def test_lane_offsets_match_64_bit_arithmetic(tmp_path):
    assert int(host_rules.run(host_rules.build("trsm_offsets", tmp_path))) > 0


@pytest.mark.gpu
@pytest.mark.parametrize("n", [63, 64])
def test_trsm_large_leading_dimension(ctx, oracle, n):
    # 63 columns of 8.53 M rows of FP64 are more than 2^32 bytes apart; only the first m rows are used
    import torch
    from gpu_util import rel, to_dev
    m, ldb = 33, 8_530_000
    A = oracle.spd_bbt(n, 77)
    assert oracle.dpotrf(A) == 0
    L = np.asfortranarray(np.tril(A))
    B = np.asfortranarray(np.random.default_rng(n).standard_normal((m, n)))
    dB = torch.empty((n, ldb), dtype=torch.float64, device="cuda")
    dB[:, :m].copy_(torch.from_numpy(np.ascontiguousarray(B.T)))
    ctx.trsm(m, n, to_dev(L), n, dB, ldb)
    got = np.asfortranarray(dB[:, :m].cpu().numpy().T)
    oracle.dtrsm_rltn(L, B)
    assert rel(got, B) < 1e-13  # as the other FP64 tile tests
