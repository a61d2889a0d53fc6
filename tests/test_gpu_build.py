"""Device build at the edges of its kernels' row and tile sizes, bit for bit against the oracle."""
import numpy as np
import pytest

from eggpu_amd import native
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# out-degrees around the long-row limit (256) and the long rows' staging chunk (1024)
OUT_LENGTHS = [0, 1, 7, 8, 9, 15, 16, 17, 255, 256, 257, 1023, 1024, 1025, 2047, 2048, 2049, 5000]


def _weights(rng, kind, m):
    if kind == "float32":  # every partial sum exact
        return rng.uniform(0.1, 1.0, m).astype(np.float32).astype(np.float64)
    if kind == "wide":  # exponents too far apart for exact sums
        return np.ldexp(rng.uniform(0.5, 1.0, m), rng.integers(-60, 60, m))
    if kind == "subnormal":
        return rng.integers(1, 1 << 20, m) * 5e-324
    w = rng.uniform(0.1, 2.0, m)
    if kind == "bad":
        idx = rng.choice(m, m // 5, replace=False)
        w[idx] = rng.choice([-1.0, np.nan, np.inf, -np.inf, 0.0, -0.0], len(idx))
    return w


@pytest.mark.parametrize("kind", ["float32", "double", "wide", "subnormal", "bad"])
@pytest.mark.parametrize("invalid", [False, True])
def test_out_weight_sums_bit_exact(gpu_ready, kind, invalid):
    print(f"out weights {kind} invalid={invalid}", flush=True)
    rng = np.random.default_rng(5)
    lengths = np.array(OUT_LENGTHS * 3)
    n = len(lengths)
    V = np.zeros(n + 1, np.int32)
    V[1:] = np.cumsum(lengths)
    m = int(V[-1])
    E = rng.integers(0, n, m).astype(np.int32)
    if invalid:
        E[rng.choice(m, m // 7, replace=False)] = n + 3
    W = _weights(rng, kind, m)
    with native.DeviceGraph.from_csr(V, E, W, alpha=0.85) as g:
        got = g.download_csc()
    want = O.build_inbound(V, E, W, 0.85)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    assert np.array_equal(got[2].view(np.uint32), want[2].view(np.uint32))
    assert np.array_equal(got[3], want[3])


# rows against the 4096-arc tiles: a row of the limit that starts at a tile's last arc, empty rows on an edge and at the
# end, whole tiles without a row's start, an arc count of whole tiles
OUT_TILES = {
    "over_the_edge": [255] * 16 + [15, 256, 256, 1, 0, 0, 3],
    "empty_on_the_edge": [256] * 16 + [0] * 700 + [256] * 16 + [0] * 300,
    "tile_without_a_start": [4095, 9000, 2, 257, 256, 0],
    "long_first": [300, 0, 5],
    "one_arc": [0, 1, 0],
}


@pytest.mark.parametrize("name", sorted(OUT_TILES))
@pytest.mark.parametrize("invalid", [False, True])
def test_out_weight_tiles_bit_exact(gpu_ready, name, invalid):
    print(f"out weight tiles {name} invalid={invalid}", flush=True)
    rng = np.random.default_rng(8)
    lengths = np.array(OUT_TILES[name])
    n = len(lengths)
    V = np.zeros(n + 1, np.int32)
    V[1:] = np.cumsum(lengths)
    m = int(V[-1])
    E = rng.integers(0, n, m).astype(np.int32)
    if invalid:
        E[rng.choice(m, (m + 6) // 7, replace=False)] = -1
    for W in (_weights(rng, "double", m), np.ones(m)):
        with native.DeviceGraph.from_csr(V, E, W, alpha=0.85) as g:
            got = g.download_csc()
        want = O.build_inbound(V, E, W, 0.85)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        assert np.array_equal(got[2].view(np.uint32), want[2].view(np.uint32))
        assert np.array_equal(got[3], want[3])


@pytest.mark.parametrize("n,m", [(1, 3), (2, 2), (255, 1000), (257, 4096), (65537, 200001)])
def test_katz_transposes_and_normalises_on_the_device(gpu_ready, n, m):
    """Unsorted rows with duplicates; sums differ from the oracle's in FP64 order only."""
    print(f"katz n={n} m={m}", flush=True)
    rng = np.random.default_rng(n)
    src = np.sort(rng.integers(0, n, m))
    E = rng.integers(0, n, m).astype(np.int32)
    V = np.zeros(n + 1, np.int32)
    V[1:] = np.cumsum(np.bincount(src, minlength=n))
    beta = rng.uniform(0.5, 1.5, n)
    alpha = 0.5 / np.diff(V).max()
    for normalized in (True, False):
        got, it, converged, _ = native.katz_csr(V, E, alpha=alpha, beta=beta, normalized=normalized)
        want, it_ref = O.katz_rows(n, src, E, alpha=alpha, beta=beta, normalized=normalized)
        assert converged and it == it_ref
        assert np.abs(got - want).max() <= 1e-12 * np.abs(want).max()


@pytest.mark.parametrize("bad", [-1, 300])
@pytest.mark.parametrize("at", [0, 4999])
def test_bad_arcs_are_refused(gpu_ready, bad, at):
    print(f"bad arcs {bad} at {at}", flush=True)
    rng = np.random.default_rng(3)
    V = np.linspace(0, 5000, 301).astype(np.int32)
    E = rng.integers(0, 300, 5000).astype(np.int32)
    W = rng.uniform(0.1, 1.0, 5000)
    broken = E.copy()
    broken[at] = bad
    for call in (lambda: native.katz_csr(V, broken), lambda: native.eigenvector_csr(V, broken, W),
                 lambda: native.eigenvector_csr(V, broken, None, max_iter=0)):
        with pytest.raises(native.EgxError, match="outside"):
            call()
    for w in (-1.0, np.nan, np.inf):
        bad_w = W.copy()
        bad_w[at] = w
        with pytest.raises(native.EgxError, match="non-negative weights"):
            native.eigenvector_csr(V, E, bad_w)


# arcs around the sort's tiles (2048 keys up to 128 tiles, 8192 above) and key widths of one to three passes
@pytest.mark.parametrize("n,m", [(1, 1), (2, 2047), (3, 2048), (511, 2049), (512, 4097), (513, 8191), (70000, 262144),
                                 (131072, 262145), (262143, 270337), (300001, 999999)])
def test_sorted_build_bit_exact(gpu_ready, n, m):
    print(f"sort n={n} m={m}", flush=True)
    rng = np.random.default_rng(m)
    src = np.sort(rng.integers(0, n, m))
    E = np.minimum(rng.integers(0, n, m), rng.integers(0, n, m)).astype(np.int32)  # skewed heads
    V = np.zeros(n + 1, np.int32)
    V[1:] = np.cumsum(np.bincount(src, minlength=n))
    with native.DeviceGraph.from_csr(V, E) as g:
        got = g.download_csc()
    want = O.build_inbound(V, E, None, 0.85)
    assert all(np.array_equal(a, b) for a, b in zip(got, want[:4]))


# rows against the scans of their arc counts: one tile (2,048), the last size of one launch (16 tiles) and of two (1,024)
@pytest.mark.parametrize("n", [2046, 2047, 2048, 32766, 32767, 32768, 2097150, 2097152])
def test_row_offsets_at_scan_sizes(gpu_ready, n):
    print(f"scan sizes n={n}", flush=True)
    rng = np.random.default_rng(n)
    m = 3 * n
    src = np.sort(rng.integers(0, n, m))
    E = (rng.integers(0, n, m) ** 2 // n).astype(np.int32)  # low heads more often
    V = np.zeros(n + 1, np.int32)
    V[1:] = np.cumsum(np.bincount(src, minlength=n))
    with native.DeviceGraph.from_csr(V, E) as g:
        got, it, _ = g.pagerank(max_iter=3, tol=0.0, precision=native.PRECISION_FP64)
    out = np.bincount(src, minlength=n)
    x = np.full(n, 1.0 / n)
    for _ in range(3):
        s = np.divide(x, out, out=np.zeros(n), where=out > 0)
        x = 0.85 * np.bincount(E, weights=s[src], minlength=n) + (0.15 + 0.85 * x[out == 0].sum()) / n
    assert it == 3 and np.max(np.abs(got - x / x.sum()) / x) <= 1e-10  # sums of up to m terms of 2^-53 each


# hub rows against the 1,024 threads that list them; rows of one segment, of several, and of 7 and more
@pytest.mark.parametrize("hubs", [0, 1, 1023, 1024, 1025, 2100])
def test_hub_row_lists(gpu_ready, hubs):
    print(f"hub rows {hubs}", flush=True)
    n = 2200
    rng = np.random.default_rng(hubs)
    indeg = rng.integers(0, 65, n)
    indeg[rng.choice(n, hubs, replace=False)] = rng.choice([65, 255, 256, 257, 512, 513, 1536, 1537, 1800], hubs)
    dst = np.repeat(np.arange(n), indeg)
    src = rng.integers(0, n, len(dst))
    order = np.lexsort((dst, src))
    src, dst = src[order], dst[order].astype(np.int32)
    V = np.zeros(n + 1, np.int32)
    V[1:] = np.cumsum(np.bincount(src, minlength=n))
    out = np.bincount(src, minlength=n)
    x = np.full(n, 1.0 / n)
    for _ in range(3):
        s = np.divide(x, out, out=np.zeros(n), where=out > 0)
        x = 0.85 * np.bincount(dst, weights=s[src], minlength=n) + (0.15 + 0.85 * x[out == 0].sum()) / n
    with native.DeviceGraph.from_csr(V, dst) as g:
        for seg in (256, 512, 8192):
            g.set_bins(wave_row_max=64, hub_segment=seg)
            assert g.info()["rows_hub"] == hubs
            got, it, _ = g.pagerank(max_iter=3, tol=0.0, precision=native.PRECISION_FP64)
            assert it == 3 and np.max(np.abs(got - x / x.sum()) / x) <= 1e-11  # sums of at most 1,800 terms of 2^-53 each
