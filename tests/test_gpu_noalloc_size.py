"""egx_graph_pagerank_noalloc at the edge of its array: graphs whose iterates fit and whose partial sums may not are
solved all the same (the sums then wait in the result's place), bit for bit as by egx_graph_pagerank."""
import ctypes

import numpy as np
import pytest

from eggpu_amd import native

pytestmark = pytest.mark.gpu


# FP32 iterates of 4,192,000 nodes leave 36 KB of the 64 MiB, of 4,100,000 nodes 1.5 MB; FP64 half of that
@pytest.mark.parametrize("n,deg,precision", [(4100000, 16, native.PRECISION_FP32), (4171000, 16, native.PRECISION_FP32),
                                             (4174000, 16, native.PRECISION_FP32), (4192000, 4, native.PRECISION_FP32),
                                             (2087000, 16, native.PRECISION_FP64)])
def test_iterates_that_fit_are_solved(gpu_ready, n, deg, precision):
    print(f"noalloc n={n} precision={precision}", flush=True)
    hip = ctypes.CDLL("libamdhip64.so")
    with native.DeviceGraph.er(n, deg * n, seed=3) as g:
        ptr = ctypes.c_void_p()
        assert hip.hipMalloc(ctypes.byref(ptr), ctypes.c_size_t(8 * n)) == 0
        try:
            for tol in (0.0, 1e-12):
                it = ctypes.c_int32(-1)
                o = native.SolveOpts(0.85, 7, tol, precision, 0)
                native._check(native.lib().egx_graph_pagerank_noalloc(g.handle, ctypes.byref(o), ptr, ctypes.byref(it)))
                got = np.empty(n)
                assert hip.hipMemcpy(got.ctypes.data_as(ctypes.c_void_p), ptr, ctypes.c_size_t(8 * n), 2) == 0
                want, it_want, _ = g.pagerank(0.85, 7, tol, precision=precision)
                assert it.value == it_want and np.array_equal(got, want)
        finally:
            hip.hipFree(ptr)
