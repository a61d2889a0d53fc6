"""Row sums of the pull SpMV at the edges of its tiles and of the lane / wavefront split of a tile's rows."""
import numpy as np
import pytest

from eggpu_amd import native

pytestmark = pytest.mark.gpu


def _graph(in_lengths, seed, weighted):
    """In-degrees as given, sources at random."""
    rng = np.random.default_rng(seed)
    n = len(in_lengths)
    dst = np.repeat(np.arange(n), in_lengths)
    src = rng.integers(0, n, len(dst))
    order = np.lexsort((dst, src))
    src, dst = src[order], dst[order]
    V = np.zeros(n + 1, np.int32)
    V[1:] = np.cumsum(np.bincount(src, minlength=n))
    W = rng.uniform(0.1, 2.0, len(dst)).astype(np.float32).astype(np.float64) if weighted else None
    return V, dst.astype(np.int32), W, src


def _pagerank(n, src, dst, w, iters, alpha=0.85):
    w = np.ones(len(src)) if w is None else w
    out = np.bincount(src, weights=w, minlength=n)
    live = out > 0
    x = np.full(n, 1.0 / n)
    for _ in range(iters):
        t = np.zeros(n)
        t[live] = x[live] / out[live]
        x = alpha * np.bincount(dst, weights=w * t[src], minlength=n) + ((1 - alpha) + alpha * x[~live].sum()) / n
    return x / x.sum()


# lanes take rows of up to 48 arcs; wavefronts 64 at a time; hub rows start above 2048; tiles of 256, 1024 and more
CASES = {
    "one": [1],
    "lane_edge": [0, 47, 48, 49, 63, 64, 65, 0, 127, 128, 129, 1, 0],
    "all_long": [49] * 300,
    "long_among_short": ([3] * 63 + [500]) * 9 + [2047, 2048, 2049, 0, 4097],
    "empty_rows": [0] * 5000 + [60] + [0] * 5000,
    "many_tiles": list(np.random.default_rng(1).integers(0, 120, 40000)),
    "mid": list(np.minimum(np.random.default_rng(2).zipf(1.6, 300000), 3000)),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("bins", [dict(), dict(thread_row_max=1), dict(thread_row_max=2000, tile_items=7424, wave_row_max=512),
                                  dict(tile_sort=1), dict(tile_items=300, hub_segment=300)],
                         ids=["default", "wave", "lane", "sorted", "small"])
def test_row_sums(gpu_ready, name, weighted, bins):
    print(f"tiles {name} weighted={weighted} {bins}", flush=True)
    V, E, W, src = _graph(np.array(CASES[name]), 3, weighted)
    want = _pagerank(len(V) - 1, src, E, W, 4)
    with native.DeviceGraph.from_csr(V, E, W) as g:
        if bins:
            g.set_bins(blocked=0, **bins)
        # unweighted FP64: order of the sums only; weighted: arc values are FP32
        got, it, _ = g.pagerank(max_iter=4, tol=0.0, precision=native.PRECISION_FP64)
        assert it == 4 and np.max(np.abs(got - want) / want) <= (1e-6 if weighted else 1e-12)
        got, it, _ = g.pagerank(max_iter=4, tol=0.0)
        assert it == 4 and np.max(np.abs(got - want) / want) <= 2e-6
        inf = g.info()
        assert inf["rows_thread"] + inf["rows_wave"] + inf["rows_hub"] == len(V) - 1
