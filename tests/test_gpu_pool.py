"""Device blocks that one object released and another reuses: builds, solves and batch sessions that come and
go, on one thread and on several, must give the results of the first ones."""
import threading

import numpy as np
import pytest

from eggpu_amd import native
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _csr(seed, n, m):
    rng = np.random.default_rng(seed)
    src = np.sort(rng.integers(0, n, m))
    V = np.zeros(n + 1, np.int32)
    V[1:] = np.cumsum(np.bincount(src, minlength=n))
    return V, rng.integers(0, n, m).astype(np.int32), rng.uniform(0.1, 2.0, m)


def _life(V, E, W):
    """One graph's whole life: the pull CSC, a solve, a batch, a re-bin."""
    with native.DeviceGraph.from_csr(V, E, W) as g:
        csc = g.download_csc()
        pr, it, _ = g.pagerank(max_iter=30, tol=0.0)
        cols, _, _ = g.ppr([[0], [1, 2], []], max_iter=10, tol=0.0)
        g.set_bins(blocked=1, tile_sort=1)
        pb, _, _ = g.pagerank(max_iter=30, tol=0.0)
    return csc, pr, it, cols, pb


GRAPHS = [(1, 900, 7000), (2, 5000, 90000), (3, 4999, 91000), (4, 60000, 300000)]


@pytest.mark.parametrize("threads", [1, 4])
def test_reused_blocks_give_the_same_results(gpu_ready, threads):
    print(f"pool threads={threads}", flush=True)
    graphs = [_csr(*g) for g in GRAPHS]
    first = [_life(*g) for g in graphs]
    for (V, E, W), f in zip(graphs, first):
        r = O.build_inbound(V, E, W, 0.85)
        assert all(np.array_equal(a, b) for a, b in zip(f[0], r[:4]))
    wrong = []

    def work(k):
        for i in range(6):
            j = (i + k) % len(graphs)
            got = _life(*graphs[j])
            same = all(np.array_equal(a, b) for a, b in zip(got[0], first[j][0])) and got[2] == first[j][2]
            if not (same and all(np.array_equal(got[q], first[j][q]) for q in (1, 3, 4))):
                wrong.append((k, i))
            if i == 3 and k == 0:
                native.cache_reset()  # gives idle blocks back while the others run

    ts = [threading.Thread(target=work, args=(k,)) for k in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not wrong
