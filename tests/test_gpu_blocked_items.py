"""Item sizes of the blocked layout: one round of scatter items or several, whole and cut sub-bins, shared launches.  However
the work is cut, the iterate is the one of the pull layout."""
import numpy as np
import pytest

from eggpu_amd import native

pytestmark = pytest.mark.gpu


# one chunk; a few; one round of the largest items and just above it; 1,024 sub-bins
@pytest.mark.parametrize("n,factor", [(30000, 4), (32769, 60), (300007, 20), (1000003, 8), (1 << 20, 16), (1 << 20, 18),
                                      (1 << 21, 4)])
@pytest.mark.parametrize("weighted", [False, True])
def test_item_sizes_do_not_change_the_iterate(gpu_ready, n, factor, weighted):
    print(f"blocked items n={n} factor={factor} weighted={weighted}", flush=True)
    with native.DeviceGraph.rmat_n(n, factor * n, seed=3, weighted=weighted, wseed=4) as g:
        g.set_bins(blocked=0)
        want, it, _ = g.pagerank(max_iter=10, tol=0.0)
        for shared in (0, 1):
            g.set_bins(blocked=1, blocked_shared=shared)
            got, its, _ = g.pagerank(max_iter=10, tol=0.0)
            assert its == it
            # terms and iterates round to FP32 (2^-24 each) in both layouts, and the map contracts by 0.85
            assert np.abs(got - want).sum() <= 4 * 2.0 ** -24 / (1 - 0.85)
            (many,), _, _ = native.multi_pagerank([g], max_iter=10, tol=0.0)
            assert np.array_equal(many, got)


# scatter items as they are, joined in twos, and in threes (75 and 130 million slots over 256 compute units)
@pytest.mark.parametrize("count,factor", [(1, 4), (3, 26), (5, 28)])
@pytest.mark.parametrize("weighted", [False, True])
def test_joined_items_in_shared_launches(gpu_ready, count, factor, weighted):
    print(f"joined items count={count} factor={factor} weighted={weighted}", flush=True)
    n = 1000003
    graphs = [native.DeviceGraph.rmat_n(n, factor * n, seed=5 + k, weighted=weighted, wseed=4) for k in range(count)]
    try:
        for g in graphs:
            g.set_bins(blocked=1, blocked_shared=1)
        ranks, its, _ = native.multi_pagerank(graphs, max_iter=4, tol=0.0)
        for g, r, it in zip(graphs, ranks, its):
            want, w_it, _ = g.pagerank(max_iter=4, tol=0.0)
            assert it == w_it and np.array_equal(r, want)
    finally:
        for g in graphs:
            g.close()
