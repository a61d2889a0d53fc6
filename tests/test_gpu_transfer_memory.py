"""Transfers that run out of host memory on the way give their pinned chunks back.  A child process makes `new[]`
fail (a library loaded before the package's defines it); its runtime's log shows whether later transfers still have
chunks: without them values come by pageable copies."""
import os
import re
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
FAILING_NEW = """
#include <cstdlib>
#include <new>
static thread_local bool fail = false;
extern "C" void fail_next(int on) { fail = on != 0; }
void* operator new[](std::size_t n) {
    if (fail) {
        fail = false;
        throw std::bad_alloc();
    }
    void* p = std::malloc(n);
    if (!p) throw std::bad_alloc();
    return p;
}
"""
CHILD = """
import ctypes, sys
import numpy as np
failing = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
from eggpu_amd import native
with native.DeviceGraph.rmat(18, 8, seed=2) as g:
    want, _, _ = g.pagerank(max_iter=3, tol=0.0)
    failed = 0
    for _ in range(30):  # the process keeps 24 chunks
        failing.fail_next(1)
        try:
            g.pagerank(max_iter=3, tol=0.0)
        except native.EgxError:
            failed += 1
    failing.fail_next(0)
    assert failed == 30, failed
    print("after failures", file=sys.stderr, flush=True)
    got, _, _ = g.pagerank(max_iter=3, tol=0.0)
    assert np.array_equal(got, want)
    print("end", file=sys.stderr, flush=True)
"""


def test_chunks_come_back_after_a_failed_allocation(gpu_ready, tmp_path):
    print("chunks after failed allocations", flush=True)
    src, lib = tmp_path / "failing.cpp", tmp_path / "failing.so"
    src.write_text(FAILING_NEW)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", str(src), "-o", str(lib)], check=True)
    env = dict(os.environ, AMD_LOG_LEVEL="3", AMD_LOG_MASK="1")
    r = subprocess.run([sys.executable, "-c", CHILD, str(lib)], cwd=ROOT, env=env, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    after = r.stderr[r.stderr.index("after failures"):]
    assert not re.search(r"hipMemcpyWithStream \(", after)
