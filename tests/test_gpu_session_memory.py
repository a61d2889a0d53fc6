"""Device memory of a batch session: two iterates, the teleport slots and one packed result of 4 bytes a node."""
import ctypes

import numpy as np
import pytest

from eggpu_amd import native

pytestmark = pytest.mark.gpu


def _free_bytes():
    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_a_session_holds_one_packed_result(gpu_ready):
    print("session memory", flush=True)
    n = 1 << 23  # blocks of these sizes are not rounded up
    with native.DeviceGraph.er(n, 4 * n, seed=5) as g:
        with g.batch() as b:  # what the graph keeps for its sessions is there
            b.assign(0, [3], max_iter=3, tol=0.0)
            b.run(3)
            want = b.result(0)
        native.device_trim()
        before = _free_bytes()
        with g.batch() as b:
            b.assign(0, [3], max_iter=3, tol=0.0)
            b.run(3)
            used = before - _free_bytes()
            got = b.result(0)
    print(f"session memory: {used / n:.1f} bytes a node", flush=True)
    assert np.array_equal(got, want)
    assert used < n * (2 * 8 * 4 + 4 + 8)  # eight columns; the partial sums fit in what is left of 8 bytes
