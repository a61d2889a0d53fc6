"""Results of a set of graphs, fetched together: vectors that share a chunk, fill one, or run over several."""
import numpy as np
import pytest

from eggpu_amd import native

pytestmark = pytest.mark.gpu

SETS = {
    "tiny": [2, 3, 2],
    "around_an_inline_copy": [65535, 2, 65537],
    "vectors_over_chunks": [70001, 600011, 33, 1500007, 2],
}


@pytest.mark.parametrize("name", sorted(SETS))
@pytest.mark.parametrize("precision", [native.PRECISION_FP32, native.PRECISION_FP64])
@pytest.mark.parametrize("tol", [0.0, 1e-6])
def test_each_graph_gets_its_own_values(gpu_ready, name, precision, tol):
    print(f"multi results {name} precision={precision} tol={tol}", flush=True)
    graphs = [native.DeviceGraph.er(n, 4 * n, seed=n) for n in SETS[name]]
    try:
        ranks, its, _ = native.multi_pagerank(graphs, max_iter=20, tol=tol, precision=precision)
        for g, r, it in zip(graphs, ranks, its):
            want, w_it, _ = g.pagerank(max_iter=20, tol=tol, precision=precision)
            assert it == w_it and np.array_equal(r, want)
    finally:
        for g in graphs:
            g.close()
