"""Matrix slots of a graph: any of 0 .. 65535, with gaps; only bound ones are reset before a run and reported after it."""
import numpy as np
import pytest

import tasktorrent_amd as tt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slots", [[0], [65535], [3, 700, 40000], [5, 6, 7]])
def test_slots_with_gaps(ctx, oracle, slots):
    n, b = 200, 64
    t0, indeg, prio, op, oi = tt.cholesky_dag(4, 2)
    seed = [tt.task_name(t) for t in t0].index("POTRF_0")
    tasks, ind, pr, optr, oidx = [], [], [], [0], []
    for s in slots:
        base = len(tasks)
        tasks += [(k, 0, s, i, j, kk) for (k, _, _, i, j, kk) in t0]
        ind, pr = ind + list(indeg), pr + list(prio)
        for t in range(len(t0)):
            oidx += [base + int(x) for x in oi[op[t]:op[t + 1]]]
            optr.append(len(oidx))
    G = tt.Graph(ctx, tasks, ind, optr, oidx, pr)
    M = [tt.TiledMatrix.uniform(ctx, n, b, "f64") for _ in slots]
    for q, s in enumerate(slots):
        G.bind(s, M[q])
        G.seed(q * len(t0) + seed)
    good = [np.asfortranarray(oracle.spd_bbt(n, s % 97)) for s in slots]
    bad = good[-1].copy(order="F")
    bad[150, 150] = -1.0
    for last, want_rc in ((good[-1], 0), (bad, 3), (good[-1], 0)):  # a bad pivot in the last slot, then none again
        for m, A in zip(M, good[:-1] + [last]):
            m.set(A)
        G.launch()
        rc, st = G.wait(30.0)
        assert rc == want_rc and st["items_done"] == st["items_total"]
        if rc == 0:
            for m, A in zip(M, good):
                L, _ = oracle.cholesky(A, b, n_threads=1)
                assert np.linalg.norm(m.get() - L) / np.linalg.norm(L) < 1e-12
    G.close()
    for m in M:
        m.close()
