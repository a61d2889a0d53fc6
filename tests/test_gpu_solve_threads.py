"""Solves that may stop early, from several threads that share one core: a thread that waits for the device lets the
others go on, so they take no longer than on cores of their own."""
import os
import threading
import time

import numpy as np
import pytest

from eggpu_amd import native

pytestmark = pytest.mark.gpu


def test_waiting_solves_share_a_core(gpu_ready):
    print("solves that share a core", flush=True)
    graphs = [native.DeviceGraph.rmat(scale, 16, seed=k) for k, scale in enumerate((14, 18, 18, 20))]
    first = [g.pagerank(max_iter=50, tol=1e-300) for g in graphs]
    cores = os.sched_getaffinity(0)
    wrong = []

    def solve(k, use):
        os.sched_setaffinity(0, use)  # of this thread
        for _ in range(20):
            ranks, it, _ = graphs[k].pagerank(max_iter=50, tol=1e-300)
            if it != first[k][1] or not np.array_equal(ranks, first[k][0]):
                wrong.append(k)

    def seconds(use):
        best = 1e9
        for _ in range(4):
            ts = [threading.Thread(target=solve, args=(k, use)) for k in range(len(graphs))]
            t = time.perf_counter()
            for th in ts:
                th.start()
            for th in ts:
                th.join()
            best = min(best, time.perf_counter() - t)
        return best

    apart, together = seconds(cores), seconds({min(cores)})
    print(f"solves that share a core: {together * 1e3:.1f} ms, on their own {apart * 1e3:.1f} ms", flush=True)
    for g in graphs:
        g.close()
    assert not wrong
    assert together < 1.2 * apart
