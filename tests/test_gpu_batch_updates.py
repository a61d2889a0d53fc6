"""Updates of a batch session as they land on the device: long lists, entries written twice in one update, and layouts that
narrow and widen between steps.  Every column must keep the bits it has when it runs alone."""
import numpy as np
import pytest

from eggpu_amd import native
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seeds", [1, 16, 300])
def test_updates_keep_columns_apart(gpu_ready, seeds):
    print(f"batch updates seeds={seeds}", flush=True)
    V, E = O.rmat_csr(10, 8, seed=6)
    n = len(V) - 1
    rng = np.random.default_rng(seeds)
    pool = [sorted(rng.choice(n, seeds, replace=False).tolist()) for _ in range(3)]
    sets = [pool[j % 3] for j in range(64)]  # rows shared by columns, so slots are freed and used again
    with native.DeviceGraph.from_csr(V, E) as g, native.DeviceGraph.from_csr(V, E) as h:
        alone = [h.ppr([p], max_iter=9, tol=0.0)[0][0] for p in pool]
        for k in (64, 1, 8, 9, 64, 3, 33, 2):  # 64 -> 1 -> 8: same buffers, 9: another width
            got, its, _ = g.ppr(sets[:k], max_iter=9, tol=0.0)
            assert all(int(i) == 9 for i in its)
            for j in range(k):
                assert np.array_equal(got[j], alone[j % 3]), (k, j)
            pool = pool[1:] + pool[:1]  # the next call's columns drop these seeds and take others
            alone = alone[1:] + alone[:1]
            sets = [pool[j % 3] for j in range(64)]
