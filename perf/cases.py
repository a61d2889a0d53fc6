"""Performance cases of the PageRank library: what its users have it do, through its public entry points.

Every case is one dict of plain values; ``kind`` names the call:

  api     ``eggpu_amd.pagerank(G)`` on a dict-based DiGraph whose device graph is already cached
  csr     a graph that has just arrived as host CSR arrays: device build, one solve, the ranks back on the host
  solve   global PageRank on a device-resident graph (FP32 or FP64 iterates), a fixed number of iterations
  ppr1    one personalised vector on a device-resident graph
  batch   a batch of 1 to 64 personalised vectors on a device-resident graph
  multi   many device-resident graphs solved in shared launches
  serve   a burst of global and personalised requests against a pool of resident graphs
  katz    Katz centrality of a host CSR graph
  eigen   eigenvector centrality of a host CSR graph

Graphs are R-MAT (a=0.57, b=c=0.19) with 16 draws per node, self-loops and duplicates removed, as in
the benchmark's configurations; the sets of many graphs alternate with Erdos-Renyi graphs.  They are drawn with
torch from the seed, so no part of the library makes its own inputs.
"""
import os

import numpy as np
import torch

os.environ["EASYGRAPH_ENABLE_GPU"] = "TRUE"
os.environ["EASYGRAPH_GPU_STRICT_ERRORS"] = "TRUE"

import eggpu_amd  # noqa: E402
from eggpu_amd import native  # noqa: E402

ALPHA = 0.85
DRAW_CHUNK = 1 << 26


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # a script that asks for the ranks of a small Python graph again and again: latency only
        {"name": "api_small", "kind": "api", "n": 1000, "deg": 8},
        # a small graph that is new on every call (the CPU-runnable configuration, R-MAT 14): build and solve
        {"name": "csr_small", "kind": "csr", "n": 1 << 14, "deg": 16, "weighted": False},
        # a weighted edge list of ordinary size, new on every call, odd node count
        {"name": "csr_weighted", "kind": "csr", "n": 700001, "deg": 16, "weighted": True},
        # repeated solves on a resident graph of ordinary size
        {"name": "solve_mid", "kind": "solve", "n": 1 << 20, "deg": 16, "weighted": False, "fp64": False, "iters": 20},
        # the headline configuration: R-MAT 24, 20 iterations, and the ranks on the host
        {"name": "solve_large", "kind": "solve", "n": 1 << 24, "deg": 16, "weighted": False, "fp64": False,
         "iters": 20},
        # the same engine in double precision
        {"name": "solve_fp64", "kind": "solve", "n": 1 << 21, "deg": 16, "weighted": False, "fp64": True,
         "iters": 20},
        # one user's personalised ranks on a weighted graph, odd node count
        {"name": "ppr_weighted", "kind": "ppr1", "n": 3000017, "deg": 16, "weighted": True, "seeds": 8, "iters": 20},
        # personalised ranks of 64 users in one call
        {"name": "ppr_batch", "kind": "batch", "n": 300007, "deg": 16, "weighted": True, "columns": 64, "iters": 20},
        # a set of unlike graphs, half R-MAT and half Erdos-Renyi
        {"name": "multi_set", "kind": "multi", "graphs": 48, "n_lo": 1000, "n_hi": 300000, "iters": 20},
        # a burst of requests against a resident pool, each stopping on its own
        {"name": "serve_burst", "kind": "serve", "graphs": 8, "m_lo": 10000, "m_hi": 5000000, "requests": 64},
        # the other two centralities of the engine, on graphs that arrive as CSR arrays
        {"name": "katz_csr", "kind": "katz", "n": 500009, "deg": 16},
        {"name": "eigen_csr", "kind": "eigen", "n": 300007, "deg": 16, "weighted": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["api", "csr", "csr", "solve", "solve", "solve", "ppr1", "batch", "batch", "multi", "serve",
                       "katz", "eigen"])
    if kind == "api":
        return {"kind": kind, "n": _log_int(rng, 200, 4000), "deg": rng.randint(4, 16)}
    if kind == "csr":
        return {"kind": kind, "n": _log_int(rng, 2000, 1000000), "deg": rng.randint(4, 24),
                "weighted": rng.random() < 0.5}
    if kind == "solve":
        return {"kind": kind, "n": _log_int(rng, 1000, 12000000), "deg": rng.randint(4, 20),
                "weighted": rng.random() < 0.3, "fp64": rng.random() < 0.3, "iters": rng.randint(5, 20)}
    if kind == "ppr1":
        return {"kind": kind, "n": _log_int(rng, 1000, 4000000), "deg": rng.randint(4, 16),
                "weighted": rng.random() < 0.5, "seeds": rng.randint(1, 16), "iters": rng.randint(5, 20)}
    if kind == "batch":
        return {"kind": kind, "n": _log_int(rng, 2000, 300000), "deg": rng.randint(4, 16),
                "weighted": rng.random() < 0.5, "columns": _log_int(rng, 1, 64), "iters": rng.randint(5, 20)}
    if kind == "multi":
        return {"kind": kind, "graphs": rng.randint(4, 48), "n_lo": 1000, "n_hi": _log_int(rng, 5000, 300000),
                "iters": rng.randint(5, 20)}
    if kind == "serve":
        return {"kind": kind, "graphs": rng.randint(1, 8), "m_lo": 10000, "m_hi": _log_int(rng, 50000, 5000000),
                "requests": rng.randint(8, 64)}
    if kind == "katz":
        return {"kind": kind, "n": _log_int(rng, 2000, 500000), "deg": rng.randint(4, 16)}
    return {"kind": kind, "n": _log_int(rng, 2000, 300000), "deg": rng.randint(4, 16),
            "weighted": rng.random() < 0.5}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _pairs(kind, n, draws, gen, device):
    """Sorted distinct (u * n + v) of the draws, without self-loops."""
    levels = max(1, (n - 1).bit_length())
    parts = []
    for at in range(0, draws, DRAW_CHUNK):
        k = min(DRAW_CHUNK, draws - at)
        if kind == "er":
            u = torch.randint(n, (k,), generator=gen, device=device)
            v = torch.randint(n, (k,), generator=gen, device=device)
        else:
            u = torch.zeros(k, dtype=torch.int32, device=device)
            v = torch.zeros(k, dtype=torch.int32, device=device)
            for _ in range(levels):
                r = torch.rand(k, generator=gen, device=device)
                # quadrants (0,0) 0.57, (0,1) 0.19, (1,0) 0.19, (1,1) 0.05
                down = r >= 0.76
                right = ((r >= 0.57) & ~down) | (r >= 0.95)
                u.mul_(2).add_(down)
                v.mul_(2).add_(right)
            u, v = u.long(), v.long()
        keep = (u < n) & (v < n) & (u != v)
        parts.append((u * n + v)[keep])
    key = torch.cat(parts) if len(parts) > 1 else parts[0]
    del parts
    return torch.unique(key)


def _csr(n, draws, seed, weighted, kind="rmat"):
    """Host out-CSR arrays (V, E, W or None)."""
    device = "cuda" if torch.cuda.is_available() else "cpu"
    gen = torch.Generator(device=device)
    gen.manual_seed(int(seed))
    key = _pairs(kind, n, draws, gen, device)
    u = torch.div(key, n, rounding_mode="floor")
    E = (key - u * n).to(torch.int32)
    V = torch.zeros(n + 1, dtype=torch.int64, device=device)
    V[1:] = torch.cumsum(torch.bincount(u, minlength=n), 0)
    W = None
    if weighted:
        W = (0.1 + 0.9 * torch.rand(E.numel(), generator=gen, device=device)).double().cpu().numpy()
    return V.to(torch.int32).cpu().numpy(), E.cpu().numpy(), W


def _case_csr(case, seed):
    return _csr(case["n"], case["n"] * case["deg"], seed * 1000 + 7, case.get("weighted", False))


def _seed_nodes(rng, n, count):
    return sorted(int(v) for v in rng.choice(n, size=min(count, n), replace=False))


def _set_specs(case, seed):
    """(kind, n, draws, seed) of a set of unlike graphs; the sizes are the case's, the arcs the seed's."""
    rng = np.random.default_rng(case["graphs"] + case["n_hi"])
    specs = []
    for i in range(case["graphs"]):
        n = int(round(case["n_lo"] * (case["n_hi"] / case["n_lo"]) ** rng.random()))
        specs.append(("er" if i % 2 == 0 else "rmat", n, int(n * rng.uniform(4, 32)), seed * 1000 + i))
    return specs


def _serve_plan(case, seed):
    """Pool ((n, draws, weighted, seed) per graph) and requests ((graph, seed nodes) each); the pool's sizes and
    which graph each request asks are the case's, the arcs and the seed nodes the seed's."""
    rng = np.random.default_rng(case["graphs"] + case["m_hi"])
    pool = []
    for i in range(case["graphs"]):
        m = int(round(case["m_lo"] * (case["m_hi"] / case["m_lo"]) ** rng.random()))
        pool.append((max(m // 16, 2), m, i % 2 == 1, seed * 1000 + i))
    asked = rng.integers(case["graphs"], size=case["requests"])
    rng = np.random.default_rng(seed + 13)
    requests = []
    for g in asked.tolist():
        requests.append((g, [] if rng.random() < 0.25 else _seed_nodes(rng, pool[g][0], int(rng.integers(1, 17)))))
    return pool, requests


def _batch_seeds(case, seed):
    rng = np.random.default_rng(seed + 17)
    return [_seed_nodes(rng, case["n"], int(rng.integers(1, 17))) for _ in range(case["columns"])]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "api":
        V, E, _ = _case_csr(case, seed)
        G = eggpu_amd.DiGraph()
        G.add_nodes_from(range(case["n"]))
        G.add_edges_from(zip(np.repeat(np.arange(case["n"]), np.diff(V)).tolist(), E.tolist()))
        eggpu_amd.pagerank(G)  # the program's first call, which makes the cached device graph
        return {"kind": kind, "G": G}
    if kind in ("csr", "katz", "eigen"):
        V, E, W = _case_csr(case, seed)
        state = {"kind": kind, "V": V, "E": E, "W": W}
        if kind == "katz":
            state["alpha"] = 0.5 / max(1, int(np.diff(V).max()))
        return state
    if kind in ("solve", "ppr1", "batch"):
        V, E, W = _case_csr(case, seed)
        state = dict(case, g=native.DeviceGraph.from_csr(V, E, W, alpha=ALPHA))
        if kind == "ppr1":
            state["nodes"] = _seed_nodes(np.random.default_rng(seed + 17), case["n"], case["seeds"])
        if kind == "batch":
            state["sets"] = _batch_seeds(case, seed)
        return state
    if kind == "multi":
        graphs = []
        for spec, n, draws, s in _set_specs(case, seed):
            V, E, _ = _csr(n, draws, s, False, spec)
            g = native.DeviceGraph.from_csr(V, E, None, alpha=ALPHA)
            g.set_bins(blocked=1, blocked_shared=1)  # as the library's own benchmark lays a set out
            graphs.append(g)
        return dict(case, gs=graphs)
    pool, requests = _serve_plan(case, seed)
    graphs = []
    for n, draws, weighted, s in pool:
        V, E, W = _csr(n, draws, s, weighted)
        graphs.append(native.DeviceGraph.from_csr(V, E, W, alpha=ALPHA))
    return {"kind": kind, "gs": graphs, "server": native.Server(graphs), "requests": requests}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "api":
        ranks = eggpu_amd.pagerank(state["G"])
        return np.array(list(ranks.values()))
    if kind == "csr":
        with native.DeviceGraph.from_csr(state["V"], state["E"], state["W"], alpha=ALPHA) as g:
            ranks, iters, _ = g.pagerank(alpha=ALPHA)
        return ranks, iters
    if kind == "solve":
        ranks, iters, _ = state["g"].pagerank(
            alpha=ALPHA, max_iter=state["iters"], tol=0.0,
            precision=native.PRECISION_FP64 if state["fp64"] else native.PRECISION_FP32)
        return ranks, iters
    if kind == "ppr1":
        ranks, iters, _ = state["g"].ppr_single(state["nodes"], alpha=ALPHA, max_iter=state["iters"], tol=0.0)
        return ranks, iters
    if kind == "batch":
        ranks, iters, _ = state["g"].ppr(state["sets"], alpha=ALPHA, max_iter=state["iters"], tol=0.0)
        return ranks, iters
    if kind == "multi":
        ranks, iters, _ = native.multi_pagerank(state["gs"], alpha=ALPHA, max_iter=state["iters"], tol=0.0)
        return ranks, iters
    if kind == "serve":
        s = state["server"]
        ids = [s.submit(g, nodes) for g, nodes in state["requests"]]
        done = [s.wait(i) for i in ids]
        return [ranks for ranks, _ in done]
    if kind == "katz":
        x, iters, converged, _ = native.katz_csr(state["V"], state["E"], alpha=state["alpha"])
        return x, iters, converged
    x, iters, stop, _ = native.eigenvector_csr(state["V"], state["E"], state["W"])
    return x, iters, stop


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _sweep(n, m, weighted, fp64=False, columns=1):
    """One iteration: every arc's index (and weight), row offsets, degrees, and the iterate in and out."""
    return m * (8 if weighted else 4) + n * 8 + columns * n * (16 if fp64 else 8)


def work(case):
    kind = case["kind"]
    if kind in ("api", "csr"):
        n, m, w = case["n"], case["n"] * case["deg"], case.get("weighted", False)
        arrays = 0 if kind == "api" else 4 * n + m * (12 if w else 4)  # the CSR arrays, read once
        return {"bytes": arrays + _sweep(n, m, w) + 8 * n, "flops": 2 * m}
    if kind in ("solve", "ppr1", "batch"):
        n, m, w = case["n"], case["n"] * case["deg"], case["weighted"]
        c = case.get("columns", 1)
        return {"bytes": case["iters"] * _sweep(n, m, w, case.get("fp64", False), c) + 8 * n * c,
                "flops": 2 * m * c * case["iters"]}
    if kind == "multi":
        specs = _set_specs(case, 1)
        nodes, arcs = sum(s[1] for s in specs), sum(s[2] for s in specs)
        return {"bytes": case["iters"] * _sweep(nodes, arcs, False) + 8 * nodes, "flops": 2 * arcs * case["iters"]}
    if kind == "serve":
        pool, requests = _serve_plan(case, 1)
        cols = [0] * len(pool)
        for g, _ in requests:
            cols[g] += 1
        total = flops = 0
        for (n, m, w, _), c in zip(pool, cols):
            if c:  # at least one shared sweep, and every result written
                total += _sweep(n, m, w, False, c) + 8 * n * c
                flops += 2 * m * c
        return {"bytes": total, "flops": flops}
    n, m, w = case["n"], case["n"] * case["deg"], case.get("weighted", False)
    return {"bytes": 4 * n + m * (12 if w else 4) + _sweep(n, m, w, True) + 8 * n, "flops": 2 * m}


# ---------------------------------------------------------------------------
# the same in plain torch, 64 bits
# ---------------------------------------------------------------------------
class _Arcs:
    """pull(x)[v] = sum over arcs u -> v of x[u] * value in float64; with rows=True, sum over arcs v -> u of x[u]."""

    STEP = 1 << 21  # rows per reduction

    def __init__(self, V, E, W, device, rows=False):
        self.n = n = len(V) - 1
        deg = torch.from_numpy(np.diff(V).astype(np.int64)).to(device)
        col = torch.from_numpy(E).to(device)
        w = None if W is None else torch.from_numpy(W).to(device)
        self.out = deg.double() if w is None else self._sums(w, deg)
        if not rows:  # order the arcs by head
            src = torch.repeat_interleave(torch.arange(n, dtype=torch.int32, device=device), deg)
            deg = torch.bincount(col, minlength=n)
            order = torch.sort(col, stable=True)[1]
            col, w = src[order], (None if w is None else w[order])
        self.col, self.w, self.deg = col, w, deg

    def _sums(self, t, lengths):
        parts, at = [], 0
        for r in range(0, self.n, self.STEP):
            part = lengths[r:r + self.STEP]
            size = int(part.sum())
            parts.append(torch.segment_reduce(t[at:at + size], "sum", lengths=part, unsafe=True, initial=0.0))
            at += size
        return torch.cat(parts)

    def pull(self, x):
        t = x[self.col]
        return self._sums(t if self.w is None else t * self.w, self.deg)


def _pagerank(a, max_iter, tol, nodes=()):
    out = a.out
    live = out > 0
    inv = torch.where(live, 1.0 / torch.where(live, out, torch.ones_like(out)), torch.zeros_like(out))
    p = torch.full((a.n,), 1.0 / a.n, dtype=torch.float64, device=out.device)
    x = p.clone()
    if len(nodes):
        p.zero_()
        p[torch.tensor(nodes, device=p.device)] = 1.0 / len(nodes)
    for _ in range(max_iter):
        y = ALPHA * a.pull(x * inv) + ((1.0 - ALPHA) + ALPHA * x[~live].sum()) * p
        err = float((y - x).abs().sum())
        x = y
        if err < tol * a.n:
            break
    return (x / x.sum()).cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    device = "cuda" if torch.cuda.is_available() else "cpu"
    if kind == "multi":
        ranks = []
        for spec, n, draws, s in _set_specs(case, seed):
            ranks.append(_pagerank(_Arcs(*_csr(n, draws, s, False, spec), device), case["iters"], 0.0))
        return ranks, None
    if kind == "serve":
        pool, requests = _serve_plan(case, seed)
        arcs = [_Arcs(*_csr(n, draws, s, weighted), device) for n, draws, weighted, s in pool]
        return [_pagerank(arcs[g], 100, 1e-6, nodes) for g, nodes in requests]
    V, E, W = _case_csr(case, seed)
    if kind == "katz":
        rows = _Arcs(V, E, None, device, rows=True)
        alpha = 0.5 / max(1, int(np.diff(V).max()))
        x = torch.ones(case["n"], dtype=torch.float64, device=device)
        for _ in range(1000):
            y = alpha * rows.pull(x) + 1.0
            if float((y - x).abs().sum()) < 1e-6:
                break
            x = y
        return (x / x.norm()).cpu().numpy(), None, None
    a = _Arcs(V, E, W, device)
    if kind == "eigen":
        x = torch.full((case["n"],), 1.0 / case["n"], dtype=torch.float64, device=device)
        for _ in range(100):
            y = a.pull(x)
            y = y / y.norm()
            done = float((y - x).norm()) < 1e-6
            x = y
            if done:
                break
        return x.cpu().numpy(), None, None
    if kind == "api":
        return _pagerank(a, 200, 1e-6)
    if kind == "csr":
        return _pagerank(a, 200, 1e-6), None
    if kind == "batch":
        return np.stack([_pagerank(a, case["iters"], 0.0, nodes) for nodes in _batch_seeds(case, seed)]), None
    nodes = _seed_nodes(np.random.default_rng(seed + 17), case["n"], case["seeds"]) if kind == "ppr1" else ()
    return _pagerank(a, case["iters"], 0.0, nodes), None
