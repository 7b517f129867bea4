"""The end of a graph run: every item is claimed and the last ones still run. Workers that find nothing leave; the
watchdog (5 s without finding work) is for runs in which items are left that nobody can claim."""
import pytest

import tasktorrent_amd as tt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tail", [1, 3])
def test_last_tasks_longer_than_the_watchdog(ctx, tail):
    # a short task, then `tail` tasks of 5.5 s side by side (tasks of up to 10 s are accepted)
    us = 5_500_000
    G = tt.Graph(ctx, [(tt.TTAD_SPIN, 0, 0, 0, 0, 100)] + [(tt.TTAD_SPIN, 0, 0, 1 + t, 0, us) for t in range(tail)],
                 [1] * (1 + tail), [0] + [tail] * (1 + tail), list(range(1, 1 + tail)))
    G.seed(0)
    G.launch()
    rc, st = G.wait(30.0)
    G.close()
    assert rc == 0 and st["abort_code"] == 0
    assert st["items_done"] == st["items_total"] == 1 + tail
    assert st["elapsed_s"] > 5.0  # the tail outlasted the watchdog
