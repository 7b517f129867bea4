"""CPU model of the POTRF items of a diagonal tile (item_potrf in tasktorrent_amd/csrc/tile_ops.hpp), with the item
numbering compiled from the library's own header.

A block item (r, q) waits for flags (r, j) and (q, j), j < q, and for (q, q), and publishes (r, q); a row's tail item does
the same for (r, r-1) and then factors (r, r) and publishes it. The items run as generators in random interleavings, at
most `workers` at a time, started in the order of their numbers. A flag is a relaxed store: it is in flight until the
memory delivers it, in any order among stores of different items. The last item to count itself finished clears the flags.
Checked: no interleaving deadlocks, the factor is the Cholesky factor (numpy), and a second tile on the same flags is
right too, so they were left at zero."""
import random

import numpy as np
import pytest

import host_rules

DB = 64
SIZES = [1, 63, 64, 65, 128, 200, 320, 512]


@pytest.fixture(scope="module")
def tables(tmp_path_factory):
    """n -> (items, flags, fin, [(r, q, tail, flag(r, r), flag(r, q))])"""
    out = host_rules.run(host_rules.build("potrf_items", tmp_path_factory.mktemp("host")), *SIZES, 4096).split("\n")
    t, pos = {}, 0
    while pos < len(out) and out[pos]:
        n, items, flags, fin = map(int, out[pos].split())
        t[n] = items, flags, fin, [tuple(map(int, out[pos + 1 + i].split())) for i in range(items)]
        pos += 1 + items
    return t


@pytest.mark.parametrize("n", SIZES + [4096])
def test_numbering(tables, n):
    items, flags, fin, own = tables[n]
    nb = (n + DB - 1) // DB
    assert items == 1 + nb * (nb - 1) // 2 and fin == flags - 1
    setter = {}
    for it, (r, q, tail, frr, frq) in enumerate(own):
        if q >= 0:
            setter[r, q] = it, frq
        if tail:
            setter[r, r] = it, frr
    assert set(setter) == {(r, q) for r in range(nb) for q in range(r + 1)}
    assert sorted(f for _, f in setter.values()) == list(range(fin))
    for it, (r, q, tail, _, _) in enumerate(own):  # every wait is on a lower-numbered item
        waits = [(r, j) for j in range(q)] + [(q, j) for j in range(q)] + ([(q, q)] if q >= 0 else [])
        assert all(setter[w][0] < it for w in waits)


class Memory:
    """The flags: a store is in flight until delivered; those of one item to one flag stay in order."""

    def __init__(self, size):
        self.val, self.flight = [0] * size, []

    def store(self, item, idx, v):
        self.flight.append((item, idx, v))

    def pending(self, item):
        return any(f[0] == item for f in self.flight)

    def deliver(self, rnd=None):
        k = rnd.randrange(len(self.flight)) if rnd else 0
        item, idx, _ = self.flight[k]
        k = next(j for j, f in enumerate(self.flight) if f[:2] == (item, idx))
        _, idx, v = self.flight.pop(k)
        self.val[idx] = v


def _run_tile(table, n, A0, mem, rnd, workers, stores_waited):
    items, flags, fin, own = table
    flag = {}
    for r, q, tail, frr, frq in own:
        if q >= 0:
            flag[r, q] = frq
        if tail:
            flag[r, r] = frr
    A, inv, count = np.tril(A0).copy(), {}, [0]
    blk = lambda r: slice(r * DB, min(n, r * DB + DB))  # noqa: E731

    def seen(i, j):
        return mem.val[flag[i, j]] != 0

    def item(it):
        r, q, tail, frr, frq = own[it]
        if q >= 0:
            acc = A[blk(r), blk(q)].copy()
            accd = np.tril(A[blk(r), blk(r)]) if tail else None
            for j in range(q):
                while not (seen(r, j) and seen(q, j)):
                    yield
                acc -= A[blk(r), blk(j)] @ A[blk(q), blk(j)].T
                if tail:
                    accd -= np.tril(A[blk(r), blk(j)] @ A[blk(r), blk(j)].T)
            while not seen(q, q):
                yield
            A[blk(r), blk(q)] = acc @ inv[q].T
            if tail:
                accd -= np.tril(A[blk(r), blk(q)] @ A[blk(r), blk(q)].T)
            mem.store(it, frq, 1)
            yield
        else:
            accd = np.tril(A[blk(r), blk(r)])
        if tail:
            while mem.pending(it):  # every wave waits for its stores before the diagonal block is announced
                yield
            L = np.linalg.cholesky(accd + np.tril(accd, -1).T)
            A[blk(r), blk(r)], inv[r] = L, np.linalg.inv(L)
            mem.store(it, frr, 1)
            yield
        while stores_waited and mem.pending(it):
            yield
        count[0] += 1
        if count[0] == items:
            for f in range(flags):
                mem.store(it, f, 0)
        yield

    live, nxt, idle = {}, 0, 0
    while nxt < items or live:
        while nxt < items and len(live) < workers:
            live[nxt] = item(nxt)
            nxt += 1
        if mem.flight and rnd.random() < 0.3:
            mem.deliver(rnd)
        it = rnd.choice(sorted(live))
        try:
            next(live[it])
        except StopIteration:
            del live[it]
            idle = 0
        idle += 1
        assert idle < 200000, "the schedule deadlocked"
    while mem.flight:  # the end of the launch waits for every store, those of different items in any order
        mem.deliver(rnd)
    return np.abs(np.tril(A) - np.linalg.cholesky(A0)).max()


def _two_tiles(tables, n, seed, workers, stores_waited):
    rnd, rng = random.Random(seed), np.random.default_rng(seed)
    mem = Memory(tables[n][1])
    worst = 0.0
    for _ in range(2):
        B = rng.standard_normal((n, n))
        worst = max(worst, _run_tile(tables[n], n, B @ B.T / n + np.eye(n), mem, rnd, workers, stores_waited))
        if any(mem.val):
            return None
    return worst


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("workers", [1, 3, 1000])
def test_any_interleaving_gives_the_factor(tables, n, workers):
    assert _two_tiles(tables, n, n + workers, workers, True) < 1e-13


def _source():
    import re
    from pathlib import Path
    src = (Path(__file__).resolve().parent.parent / "tasktorrent_amd" / "csrc" / "tile_ops.hpp").read_text()
    src = re.sub(r"//[^\n]*", "", src)
    a = src.index("item_potrf(TS*")
    return src[a:src.index("\ntemplate <", a)]


def test_flag_stores_are_waited_for_before_the_item_counts_itself(tables):
    import re
    src = _source()
    end = src[src.rindex("publish(r, r)"):src.index("potrf_fin(n)")]
    assert re.search(r"if \(tid == 0\) \{\s*stores_done\(\);\s*if \(__hip_atomic_fetch_add\(flags \+ $", end)
    # without this wait, an item's flag can land behind the clearing of the last one: the model finds it
    assert any(_two_tiles(tables, 128, seed, 1000, False) is None for seed in range(200))


def _first_bad_pivot(seed, report_first, nb=4):
    """The chain of diagonal blocks, each of which fails once an earlier one has (its inverse holds NaN): block r is
    entered when block r - 1 has been published, and reports a bad pivot into the one word that keeps the first."""
    rnd = random.Random(seed)
    published, info = set(), [0]

    def block(r):
        while r > 0 and r - 1 not in published:
            yield
        for step in (("report", "publish") if report_first else ("publish", "report")):
            if step == "publish":
                published.add(r)
            elif info[0] == 0:
                info[0] = r + 1
            yield

    live = {r: block(r) for r in range(nb)}
    while live:
        r = rnd.choice(sorted(live))
        try:
            next(live[r])
        except StopIteration:
            del live[r]
    return info[0]


def test_bad_pivot_is_reported_before_the_block_is_published():
    src = _source()
    assert src.index("atomicCAS(info") < src.index("publish(r, r);")
    assert all(_first_bad_pivot(seed, True) == 1 for seed in range(100))
    assert any(_first_bad_pivot(seed, False) != 1 for seed in range(100))


@pytest.mark.parametrize("n", SIZES + [4096])
def test_benchmark_reports_the_item_count(tables, n):
    import bench
    assert bench.potrf_items(n) == tables[n][0]
