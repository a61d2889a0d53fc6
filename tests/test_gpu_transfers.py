"""Arrays to and from the device in pinned chunks (4 MiB, up to 12 per call): sizes at the one-chunk limit
(256 KiB), at a chunk's edges and past a whole ring, both directions, several callers at once."""
import threading

import numpy as np
import pytest

from eggpu_amd import native

pytestmark = pytest.mark.gpu


def _graph(n, m, seed):
    rng = np.random.default_rng(seed)
    src = np.sort(rng.integers(0, n, m))
    V = np.zeros(n + 1, np.int32)
    V[1:] = np.cumsum(np.bincount(src, minlength=n))
    return V, rng.integers(0, n, m).astype(np.int32), rng.uniform(0.1, 2.0, m), src


def _pagerank(n, src, dst, w, iters, alpha=0.85):
    out = np.bincount(src, weights=w, minlength=n)
    live = out > 0
    inv = np.zeros(n)
    inv[live] = 1.0 / out[live]
    x = np.full(n, 1.0 / n)
    for _ in range(iters):
        x = alpha * np.bincount(dst, weights=w * (x * inv)[src], minlength=n) + (
            (1.0 - alpha) + alpha * x[~live].sum()) / n
    return x / x.sum()


# packed floats: inline up to 65536, an eighth each up to 8388608, chunks of 1048576, a ring of 12582912; doubles half of that
SIZES = [(65535, 40000), (65537, 131073), (524289, 524287), (1048575, 300000), (1048577, 1048577),
         (4194305, 4194303), (6400001, 3000000), (12600001, 12600001)]


@pytest.mark.parametrize("n,m", SIZES)
def test_arrays_cross_whole(gpu_ready, n, m):
    print(f"transfers n={n} m={m}", flush=True)
    V, E, W, src = _graph(n, m, n)
    with native.DeviceGraph.from_csr(V, E, W, keep_csr=True) as g:
        v2, e2, w2 = g.download_csr()
        assert np.array_equal(v2, V) and np.array_equal(e2, E) and np.array_equal(w2, W)
        want = _pagerank(n, src, E, W, 4)
        for precision, bar in ((native.PRECISION_FP32, 1e-6), (native.PRECISION_FP64, 1e-6)):  # arc values are FP32
            got, it, _ = g.pagerank(max_iter=4, tol=0.0, precision=precision)
            assert it == 4 and np.max(np.abs(got - want) / want) <= bar
        if n < 4000000:
            cols, _, _ = g.ppr([[], [], []], max_iter=4, tol=0.0)
            assert np.max(np.abs(cols - want) / want) <= 1e-6
            assert np.array_equal(cols[0], cols[2])


def test_several_callers_at_once(gpu_ready):
    print("transfers from 6 threads", flush=True)
    graphs = [_graph(400000 + 7 * k, 900000, k) for k in range(6)]
    first, wrong = {}, []

    def life(k):
        V, E, W, _ = graphs[k]
        with native.DeviceGraph.from_csr(V, E, W) as g:
            return g.pagerank(max_iter=3, tol=0.0)[0]

    for k in range(6):
        first[k] = life(k)

    def work(k):
        for _ in range(4):
            if not np.array_equal(life(k), first[k]):
                wrong.append(k)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not wrong
