"""Large graphs that may stop early fold each iteration's sums in a launch of their own (2^24 arcs and more with pull
iterations, 2^26 with blocked ones).  Stops after several iterations must give the iterate and the count of a solve of
that many iterations that never looks at a tolerance, launched, polled and replayed; Katz and eigenvector centrality
those of plain numpy."""
import numpy as np
import pytest

from eggpu_amd import native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("blocked", [0, 1])
def test_stops_equal_fixed_lengths(gpu_ready, blocked, weighted):
    print(f"prefold blocked={blocked} weighted={weighted}", flush=True)
    scale, factor, least = (23, 10, 1 << 26) if blocked else (21, 16, 1 << 24)
    with native.DeviceGraph.rmat(scale, factor, seed=7, weighted=weighted, wseed=3) as g:
        g.set_bins(blocked=blocked)
        info = g.info()
        assert info["m"] >= least and info["blocked"] == blocked and info["n_dangling"] > 0 and info["rows_hub"] > 0
        precisions = [native.PRECISION_FP32] + ([] if blocked else [native.PRECISION_FP64])
        for precision in precisions:
            counts = []
            for tol, max_iter in ((3e-9, 60), (1e-10, 60), (1e-10, 5), (1.0, 60)):
                got, it, _ = g.pagerank(max_iter=max_iter, tol=tol, precision=precision)
                want, _, _ = g.pagerank(max_iter=it, tol=0.0, precision=precision)
                assert np.array_equal(got, want), (tol, max_iter, it)
                counts.append(it)
                for check, replay in ((1, False), (4, True), (3, True)):
                    again, st = g.pagerank_stats(max_iter=max_iter, tol=tol, precision=precision, download=True,
                                                 time_each_launch=False, hip_graph=replay, check_every=check)
                    assert st["iterations"] == it and np.array_equal(again, want), (tol, check, replay)
            assert counts[3] == 1 and counts[2] == 5 < counts[1] and 3 <= counts[0] < counts[1] < 60
            print(f"prefold: {counts} iterations", flush=True)
        nodes = [5, 77, 1 << 20]
        got, it, _ = g.ppr_single(nodes, max_iter=60, tol=1e-9)
        want, _, _ = g.ppr_single(nodes, max_iter=it, tol=0.0)
        assert 3 <= it < 60 and np.array_equal(got, want)


def _csr(n, m, seed):
    rng = np.random.default_rng(seed)
    src = np.sort(rng.integers(0, n, m))
    V = np.zeros(n + 1, np.int32)
    V[1:] = np.cumsum(np.bincount(src, minlength=n))
    return V, rng.integers(0, n, m).astype(np.int32), src


def test_katz_and_eigenvector_equal_numpy(gpu_ready):
    """Rows of at most 64 terms and a dozen iterations in FP64: relative differences stay below 64 * 12 * 2^-52 < 1e-12."""
    n, m = 1_100_000, 17_500_000
    print("prefold katz", flush=True)
    V, E, src = _csr(n, m, 4)
    alpha = 0.5 / int(np.diff(V).max())
    got, it, converged, _ = native.katz_csr(V, E, alpha=alpha, normalized=False)
    x = np.ones(n)
    for count in range(1, 100):
        y = alpha * np.bincount(src, weights=x[E], minlength=n) + 1.0
        if np.abs(y - x).sum() < 1e-6:
            break
        x = y
    assert converged and it == count > 3 and np.max(np.abs(got - x) / x) < 1e-12
    print(f"prefold eigenvector (katz {it} iterations)", flush=True)
    got, it, stop, _ = native.eigenvector_csr(V, E, tol=1e-4)
    x = np.full(n, 1.0 / n)
    for count in range(1, 100):
        y = np.bincount(E, weights=x[src], minlength=n)
        y /= np.linalg.norm(y)
        done = np.linalg.norm(y - x) < 1e-4
        x = y
        if done:
            break
    assert stop == native.EIG_CONVERGED and it == count > 3
    assert np.max(np.abs(got - x)) < 1e-12 * np.max(x)
