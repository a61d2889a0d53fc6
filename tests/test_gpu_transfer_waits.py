"""A result that is fetched behind a long solve: one thread waits for it, not the transfer's helpers."""
import time

import numpy as np
import pytest

from eggpu_amd import native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tol", [0.0, 1e-300])
@pytest.mark.parametrize("precision", [native.PRECISION_FP32, native.PRECISION_FP64])
def test_one_thread_waits_for_a_solve(gpu_ready, precision, tol):
    """4.2M nodes, 300 iterations of 0.1 to 0.4 ms: the process's CPU time stays below two cores (one that waits, and
    all of them for the 3 ms that the values take; eight that waited used 7.9 at tol 0)."""
    print(f"waiting threads precision={precision} tol={tol}", flush=True)
    with native.DeviceGraph.rmat(22, 16, seed=2) as g:
        first, _, _ = g.pagerank(max_iter=300, tol=tol, precision=precision)
        wall, cpu = time.perf_counter(), time.process_time()
        again, _, _ = g.pagerank(max_iter=300, tol=tol, precision=precision)
        wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
        assert np.array_equal(again, first)
        print(f"waiting threads: {wall * 1e3:.1f} ms, {cpu / wall:.2f} cores", flush=True)
        assert cpu < 2.0 * wall + 0.004
