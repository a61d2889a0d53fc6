"""Batched solves over the sizes where their reduce and their split over wavefronts change: one workgroup or parts, few or
many hub rows, one wavefront or thousands.  A column has the same bits at every width and agrees with the oracle."""
import numpy as np
import pytest

from eggpu_amd import native
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# nodes 2^scale, arcs a node, hub rows above this in-degree (None: the default)
LAYOUTS = [(1, 2, None), (6, 4, None), (10, 8, None), (11, 8, None), (11, 16, 64), (14, 16, None), (14, 16, 64),
           (17, 8, 64)]


@pytest.mark.parametrize("scale,deg,hub", LAYOUTS)
def test_columns_over_reduce_layouts(gpu_ready, scale, deg, hub):
    print(f"spmm reduce scale={scale} deg={deg} hub={hub}", flush=True)
    V, E = (np.array([0, 1, 2], np.int32), np.array([1, 0], np.int32)) if scale == 1 else O.rmat_csr(scale, deg, seed=3)
    W = O.edge_weights(V, E, 8)
    n = len(V) - 1
    src, dst = O.csr_rows(V, E)
    rng = np.random.default_rng(scale)
    sets = [[]] + [sorted(rng.choice(n, min(n, 1 + j % 5), replace=False).tolist()) for j in range(63)]
    with native.DeviceGraph.from_csr(V, E, W) as g:
        if hub:
            g.set_bins(wave_row_max=hub)
        wide, its, _ = g.ppr(sets, alpha=0.85, max_iter=12, tol=0.0)
        assert all(int(i) == 12 for i in its)
        for k in (1, 8, 16, 32):
            some, _, _ = g.ppr(sets[:k], alpha=0.85, max_iter=12, tol=0.0)
            assert np.array_equal(some, wide[:k]), k
    for j in (0, 1, 31, 63):
        p = np.zeros(n)
        p[sets[j] or range(n)] = 1.0 / (len(sets[j]) or n)
        ref, _, _ = O.ppr_rows(n, src, dst, W, p, 0.85, 12, 0.0)
        # values and weights are rounded to FP32 (2^-24) every iteration and the map contracts by 0.85
        assert np.abs(wide[j] - ref).sum() <= 2.0 ** -24 * 3 / (1 - 0.85), j
