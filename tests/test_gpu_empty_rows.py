"""Builds of graphs whose nodes mostly have no arcs, in long stretches between the ones that do: the rows are shared
out like the others (bit for bit against the oracle), so that a stretch costs no more than its nodes."""
import numpy as np
import pytest

from eggpu_amd import native
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _csr(n, lengths_at, weighted, seed=3):
    """Rows of the given lengths at the given nodes, no arcs elsewhere."""
    rng = np.random.default_rng(seed)
    cnt = np.zeros(n, np.int64)
    for at, lengths in lengths_at:
        cnt[at:at + len(lengths)] = lengths
    V = np.zeros(n + 1, np.int32)
    V[1:] = np.cumsum(cnt)
    m = int(V[-1])
    return V, rng.integers(0, n, m).astype(np.int32), rng.uniform(0.1, 2.0, m) if weighted else None


def _ones(k, length=10):
    return np.full(k, length)


# stretches at both ends and in the middle, around a tile of 4,096 rows and arcs and a run's 65,536 rows
SHAPES = [
    (5000, [(0, [3])]),
    (5000, [(4999, [5])]),
    (4096 * 3, [(0, [4095]), (4096 * 2, [1, 300, 2])]),
    (70000, [(0, _ones(40)), (65576, _ones(40))]),   # 65,536 rows between
    (70000, [(0, _ones(40)), (65577, _ones(40))]),   # one more
    (300000, [(0, [257, 1, 256]), (150000, _ones(500, 9)), (299990, [0, 7, 255, 4097])]),
]


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("k", range(len(SHAPES)))
def test_sparse_rows_build_as_the_oracle(gpu_ready, k, weighted):
    n, at = SHAPES[k]
    print(f"empty rows {k} weighted={weighted}", flush=True)
    V, E, W = _csr(n, at, weighted)
    with native.DeviceGraph.from_csr(V, E, W) as g:
        got = g.download_csc()
    want = O.build_inbound(V, E, W, 0.85)
    assert all(np.array_equal(a, b) for a, b in zip(got, want[:4]))


def _build_seconds(V, E, W):
    best = 1.0
    for _ in range(4):
        with native.DeviceGraph.from_csr(V, E, W) as g:
            best = min(best, g.info()["build_seconds"])
    return best


def test_a_stretch_costs_no_more_than_its_nodes(gpu_ready):
    """16M nodes: the arcs' weights and the place of the rows that have arcs must not multiply the build's time
    (when the arcs alone shared the rows out, 16 arcs took 37 ms with weights and 12 without, and 1M arcs at both ends
    of the ids 36 and 15; now about 1 each)."""
    n = 16_000_000
    print("empty rows, time", flush=True)
    few = _csr(n, [(0, _ones(16, 1))], True)
    plain = _build_seconds(few[0], few[1], None)
    assert _build_seconds(*few) < 3 * plain
    half = _ones(50000)
    near = _csr(n, [(0, half), (50000, half)], True)
    far = _csr(n, [(0, half), (n - 50000, half)], True)
    base = _build_seconds(near[0], near[1], None)
    times = [_build_seconds(far[0], far[1], None), _build_seconds(*near), _build_seconds(*far)]
    print(f"empty rows: 16 arcs {plain * 1e3:.2f} ms, 1M arcs {base * 1e3:.2f} ms, far / weighted / both "
          + " ".join(f"{t * 1e3:.2f}" for t in times), flush=True)
    assert max(times) < 3 * base
