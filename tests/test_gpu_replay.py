"""EGX_SOLVE_HIP_GRAPH replays captured runs at every check interval, odd ones too: counted in the runtime's own log
of a child process, whose results are compared with plain calls."""
import os
import re
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHILD = """
import sys
import numpy as np
from eggpu_amd import native
with native.DeviceGraph.rmat(11, 8, seed=9) as g:
    for check, max_iter in ((1, 6), (3, 12), (4, 12), (7, 20)):
        want, it, _ = g.pagerank(max_iter=max_iter, tol=1e-300)
        print("solve", check, file=sys.stderr, flush=True)
        got, st = g.pagerank_stats(max_iter=max_iter, tol=1e-300, download=True, time_each_launch=False,
                                   hip_graph=True, check_every=check)
        assert st["iterations"] == it == max_iter and np.array_equal(got, want)
print("solve done", file=sys.stderr, flush=True)
"""


def test_every_check_interval_is_replayed(gpu_ready):
    print("replays by check interval", flush=True)
    env = dict(os.environ, AMD_LOG_LEVEL="3", AMD_LOG_MASK="1")
    r = subprocess.run([sys.executable, "-c", CHILD], cwd=ROOT, env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    parts = re.split(r"^solve (\w+)$", r.stderr, flags=re.M)
    launched = {parts[i]: len(re.findall(r"hipGraphLaunch \(", parts[i + 1])) for i in range(1, len(parts) - 1, 2)}
    assert {k: launched[k] for k in ("1", "3", "4", "7")} == {"1": 6, "3": 4, "4": 3, "7": 2}
