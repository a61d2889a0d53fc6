"""Device memory that closed graphs leave with the process goes back to the device when asked for."""
import ctypes

import pytest

from eggpu_amd import native

pytestmark = pytest.mark.gpu

MB = 1 << 20


def _free_bytes():
    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_trim_returns_what_closed_graphs_left(gpu_ready):
    print("device trim", flush=True)

    def life():
        with native.DeviceGraph.rmat(20, 16, seed=3, weighted=True, wseed=4) as g:
            g.pagerank(max_iter=2, tol=0.0)
            g.ppr([[0]], max_iter=2, tol=0.0)
            native.device_trim()  # with a graph open: its own memory stays
            return g.pagerank(max_iter=2, tol=0.0)[0]

    first = life()  # what the process makes once (streams, chunks, code) is there
    native.device_trim()
    before = _free_bytes()
    again = life()
    assert (first == again).all()
    assert before - _free_bytes() > 100 * MB  # kept for the next graph
    native.device_trim()
    assert before - _free_bytes() < 16 * MB
