"""A graph launched on a stream of the caller's that is destroyed while the graph runs (the runtime finishes the work that
the stream holds): waiting for the graph and destroying it need the run's events and its report, not the stream."""
import ctypes

import pytest

import tasktorrent_amd as tt

pytestmark = pytest.mark.gpu


def _hip():
    import torch  # noqa: F401  (the runtime that the process has loaded)
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    return ctypes.CDLL(path)


@pytest.mark.parametrize("wait", [True, False])
def test_stream_destroyed_during_the_run(ctx, wait):
    hip = _hip()
    s = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(s)) == 0
    G = tt.Graph(ctx, [(tt.TTAD_SPIN, 0, 0, t, 0, 20000) for t in range(3)], [1, 1, 1], [0, 1, 2, 2], [1, 2])
    G.seed(0)
    G.launch(stream=s)
    assert hip.hipStreamDestroy(s) == 0
    if wait:
        rc, st = G.wait(30.0)
        assert rc == 0 and st["items_done"] == 3
    G.close()
    # its report slot serves the next graph
    H = tt.Graph(ctx, [(tt.TTAD_SPIN, 0, 0, 0, 0, 10)], [1], [0, 0], [])
    H.seed(0)
    H.launch()
    rc, st = H.wait(30.0)
    assert rc == 0 and st["items_done"] == 1
    H.close()
