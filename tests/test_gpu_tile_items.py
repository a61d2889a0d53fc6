"""tile_items: every value that is asked for runs as it is, and egx_graph_info reports the size that runs."""
import numpy as np
import pytest

from eggpu_amd import native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3000, 60000, 500000])
def test_tiles_have_the_size_asked_for(gpu_ready, n):
    print(f"tile items n={n}", flush=True)
    with native.DeviceGraph.er(n, 8 * n, seed=2) as g:  # no hub rows
        def tiles():
            info = g.info()
            assert info["rows_hub"] == 0 and info["tiles"] == -(-(info["m"] + n) // info["tile_items"])
            return info["tile_items"]

        own = tiles()
        assert own != 5888
        want, _, _ = g.pagerank(max_iter=5, tol=0.0)
        for asked in (5888, 300, 4096, 5888):
            g.set_bins(tile_items=asked)
            assert tiles() == asked
            got, _, _ = g.pagerank(max_iter=5, tol=0.0)
            assert np.max(np.abs(got - want)) <= 1e-9
        for keep in (0, -1):
            g.set_bins(tile_items=keep)
            assert tiles() == 5888
        g.set_bins(tile_items=native.TILE_ITEMS_AUTO)
        assert tiles() == own
        g.set_bins(tile_items=native.TILE_ITEMS_AUTO, wave_row_max=7000)
        assert tiles() == min(own, 936)  # what the hub threshold leaves of a tile's LDS
        g.set_bins(wave_row_max=2048)
        assert tiles() == own


def test_the_tuner_starts_from_the_graph_s_own_size(gpu_ready):
    print("tile items, tuner", flush=True)
    from eggpu_amd import autotune

    with native.DeviceGraph.er(60000, 480000, seed=2) as g:
        own = g.info()["tile_items"]
        g.set_bins(tile_items=5888)
        cfg, _, _ = autotune.tune(g, space={"tile_sort": [0, 1]}, passes=1, iters=2)
        assert cfg["tile_items"] == own == g.info()["tile_items"]
