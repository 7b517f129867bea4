"""Graphs in which many tasks are on a longest path (independent tasks, many matrices in one graph): the small items, which
take a longest path's updates off each other's way, are for paths that leave CUs idle. Which items a task has shows in
the number of a run's items; either form gives the same bits."""
import numpy as np
import pytest

import tasktorrent_amd as tt

pytestmark = pytest.mark.gpu


def updates(ctx, M, nt, last, prec):
    """The updates of step 0 of block columns 1 .. last - 1, below the diagonal, without an edge between them."""
    tasks = [(tt.TTAD_GEMM, prec, 0, i, j, 0) for j in range(1, last) for i in range(j + 1, nt)]
    n = len(tasks)
    G = tt.Graph(ctx, tasks, [1] * n, [0] * (n + 1), [])
    G.bind(0, M)
    for t in range(n):
        G.seed(t)
    G.launch()
    rc, st = G.wait(60.0)
    G.close()
    assert rc == 0
    return n, st["items_total"]


@pytest.mark.parametrize("storage,prec", [("f64", 0), ("f32", 1), ("f32", 3)])
def test_items_of_independent_updates(ctx, storage, prec):
    b, nt = 512, 12
    A = np.asfortranarray(np.tril(np.random.default_rng(3).integers(-3, 4, (b * nt, b * nt)).astype(np.float64)))
    M = tt.TiledMatrix.uniform(ctx, b * nt, b, storage)
    for last, per_task in ((2, 64), (nt, 16)):  # 10 tasks: 160 items of 128, small ones; 55 tasks: 880
        M.set(A)
        n, items = updates(ctx, M, nt, last, prec)
        assert items == n * per_task
        want = A.copy()
        for j in range(1, last):
            c = slice(j * b, j * b + b)
            want[c.stop:, c] -= A[c.stop:, :b] @ A[c, :b].T
        assert np.array_equal(M.get(), want)
    M.close()


@pytest.mark.parametrize("n,b,count,small", [(768, 256, 3, True), (768, 256, 90, False)])
def test_many_matrices_in_one_graph(ctx, oracle, n, b, count, small):
    # the updates of one level: 2 x 4 + 3 items per matrix at step 0, 3 at step 1
    t0, indeg, prio, op, oi = tt.cholesky_dag(n // b, 2)
    names = [tt.task_name(t) for t in t0]
    A = [np.asfortranarray(oracle.spd_bbt(n, 50 + q)) for q in range(3)]
    tasks, ind, pr, optr, oidx, M = [], [], [], [0], [], []
    for q in range(count):
        base = len(tasks)
        tasks += [(k, 0, q, i, j, kk) for (k, _, _, i, j, kk) in t0]
        ind, pr = ind + list(indeg), pr + list(prio)
        for t in range(len(t0)):
            oidx += [base + int(x) for x in oi[op[t]:op[t + 1]]]
            optr.append(len(oidx))
        M.append(tt.TiledMatrix.uniform(ctx, n, b, "f64"))
        M[q].set(A[q % 3])
    G = tt.Graph(ctx, tasks, ind, optr, oidx, pr)
    for q in range(count):
        G.bind(q, M[q])
        G.seed(q * len(t0) + names.index("POTRF_0"))
    G.launch()
    rc, st = G.wait(60.0)
    G.close()
    assert rc == 0
    # per matrix: 3 POTRF of 7 items, 3 TRSM of 16 strips or 8, updates: 3 SYRK of 10 items or 3, 1 GEMM of 16 or 4
    alone = 3 * 7 + 3 * 16 + 3 * 10 + 16
    assert (st["items_total"] == count * alone) == small and st["items_total"] <= count * alone
    for q in range(3):
        W = tt.TiledMatrix.uniform(ctx, n, b, "f64")
        W.set(A[q])
        assert ctx.potrf_tiled(W, tt.TTAD_SCHED_STREAM, 2, "f64") == 0
        want = W.get()
        W.close()
        for m in M[q::3]:
            assert np.array_equal(m.get(), want)
    for m in M:
        m.close()
