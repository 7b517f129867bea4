"""Releases of a whole workgroup's stores. __syncthreads orders the waves of a workgroup but does not wait for their
stores (gfx950: s_barrier has no vmcnt wait in front of it), and the write-back that one thread issues behind it waits
for that thread's wave alone. So every wave has to wait for its own stores in front of the barrier behind which one
thread announces them. The first test reads this order off the sources; the model shows what is lost without the wait."""
import random
import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "tasktorrent_amd" / "csrc"
WAIT = r"(stores_done\(\);|__builtin_amdgcn_s_waitcnt\(0x0F70\);)"
# a barrier with the one thread's release behind it
RELEASE = re.compile(r"__syncthreads\(\);\s*if \((threadIdx\.x|tid) == \w+\) \{\s*release_agent\(\);")


def _source(name):
    return re.sub(r"//[^\n]*", "", (CSRC / name).read_text())


def _unwaited(name):
    """Offsets of the releases in `name` whose barrier has no store wait right in front of it."""
    src = _source(name)
    return [m.start() for m in RELEASE.finditer(src) if not re.search(WAIT + r"\s*$", src[:m.start()])]


@pytest.mark.parametrize("name,sites", [("solve_ops.hpp", 1), ("tile_ops.hpp", 1), ("server.hip", 1)])
def test_stores_are_waited_for_in_front_of_the_barrier(name, sites):
    assert len(RELEASE.findall(_source(name))) == sites
    assert _unwaited(name) == []


def _run(seed, wait, waves=4):
    """Each wave of a workgroup stores and meets the barrier; wave 0 then writes the L2 back and announces. A store is
    in flight until the memory delivers it into the L2. Returns whether the announcement found every store written back."""
    rnd = random.Random(seed)
    in_flight, l2, memory = set(), set(), set()
    at_barrier = set()

    def wave(w):
        in_flight.add(w)
        yield
        while wait and w in in_flight:
            yield
        at_barrier.add(w)
        while len(at_barrier) < waves:
            yield
        if w == 0:
            while w in in_flight:  # release_agent waits for its own wave
                yield
            memory.update(l2)
            yield

    live = {w: wave(w) for w in range(waves)}
    while 0 in live:
        if in_flight and rnd.random() < 0.2:
            w = rnd.choice(sorted(in_flight))
            in_flight.discard(w)
            l2.add(w)
        w = rnd.choice(sorted(live))
        try:
            next(live[w])
        except StopIteration:
            del live[w]
    return memory == set(range(waves))


def test_model_loses_stores_without_the_wait():
    assert all(_run(seed, True) for seed in range(200))
    assert not all(_run(seed, False) for seed in range(200))
