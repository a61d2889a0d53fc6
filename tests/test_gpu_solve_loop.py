"""The solve loop's ways to launch and to stop: every check interval, replayed or not, must give the iterate and the
iteration count of the plain call, on grids that are folded directly (small), reduced (split hub rows) and blocked."""
import numpy as np
import pytest

from eggpu_amd import native

pytestmark = pytest.mark.gpu

GRAPHS = {
    "direct": (dict(scale=11, edge_factor=8), dict()),
    "reduced": (dict(scale=16, edge_factor=16), dict(wave_row_max=256, hub_segment=256)),
    "blocked": (dict(scale=16, edge_factor=16), dict(blocked=1)),
}


@pytest.mark.parametrize("name", list(GRAPHS))
@pytest.mark.parametrize("weighted", [False, True])
def test_check_intervals_and_replays_agree(gpu_ready, name, weighted):
    rmat, bins = GRAPHS[name]
    print(f"solve loop {name} weighted={weighted}", flush=True)
    with native.DeviceGraph.rmat(seed=9, weighted=weighted, wseed=4, **rmat) as g:
        if bins:
            g.set_bins(**bins)
        for precision in (native.PRECISION_FP32, native.PRECISION_FP64):
            for tol, max_iter in ((1e-9, 100), (1e-4, 100), (0.0, 7), (1e-12, 5), (1.0, 9)):
                want, it, _ = g.pagerank(max_iter=max_iter, tol=tol, precision=precision)
                assert it == max_iter or tol > 0.0
                for check in (1, 2, 3, 4, 7, 64):
                    for replay in (False, True):
                        got, st = g.pagerank_stats(max_iter=max_iter, tol=tol, precision=precision, download=True,
                                                   time_each_launch=False, hip_graph=replay, check_every=check)
                        assert st["iterations"] == it, (tol, check, replay)
                        assert np.array_equal(got, want), (tol, check, replay)
                got, st = g.pagerank_stats(max_iter=max_iter, tol=tol, precision=precision, download=True)
                assert st["iterations"] == it and np.array_equal(got, want)
            many, its, _ = native.multi_pagerank([g], max_iter=100, tol=1e-9, precision=precision)
            want, it, _ = g.pagerank(max_iter=100, tol=1e-9, precision=precision)
            assert its[0] == it and np.array_equal(many[0], want)
