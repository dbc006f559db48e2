"""Workloads of the traversal engine: what its users run, from the smallest
call to the largest graph, each through the public entry points.

A case names an application, a graph and the options of the call:

  app        bfs, sssp, pagerank, cc, bfs_multi, sssp_multi or serve
  graph      rmat (scale, ef: the generator's edge factor; symmetric),
             grid (rows x cols, 4 neighbours; road-like, high diameter) or
             directed (V vertices, about E edges, skewed degrees, loaded from
             host arrays as a program with a CSR of its own does)
  wmax       weights 1..wmax (0: unweighted)
  sources    traversals of one pass (bfs, sssp), queries of a batch or of a
             served load
  resident   share of the edges that stays in HBM (1: all; below 1 the capped
             placement, the rest in pinned host memory)

A program keeps its context, its graph, the workspaces the library caches
with the graph, and (for large results) pinned result buffers; the graph and
the sources are what a new input changes.
"""
import ctypes as C

import numpy as np
import torch

import grus_framework_amd as grus
from grus_framework_amd import capi

ALPHA, ITERATIONS = 0.85, 20


def listed():
    return [
        # the smallest call: a query on a graph that fits a cache; the levels
        # come back in a new array, as from the Python call
        dict(name="bfs_small", app="bfs", graph="rmat", scale=10, ef=16, wmax=0, sources=1,
             resident=1.0),
        # the benchmark's headline graph: traversals in a row, results digested
        # on the device, the last one read out
        dict(name="bfs_large", app="bfs", graph="rmat", scale=24, ef=16, wmax=0, sources=6,
             resident=1.0),
        # road-like input: thousands of thin levels
        dict(name="bfs_grid", app="bfs", graph="grid", rows=1300, cols=1700, wmax=0, sources=1,
             resident=1.0),
        # a graph larger than its share of HBM: most edges in host memory
        dict(name="bfs_capped", app="bfs", graph="rmat", scale=21, ef=16, wmax=0, sources=1,
             resident=0.25),
        # shortest paths on a small-world graph
        dict(name="sssp_rmat", app="sssp", graph="rmat", scale=20, ef=16, wmax=255, sources=1,
             resident=1.0),
        # shortest paths on road-like input
        dict(name="sssp_grid", app="sssp", graph="grid", rows=1500, cols=1100, wmax=1000,
             sources=1, resident=1.0),
        # ranks of a directed graph of some ten thousand pages
        dict(name="pagerank_directed", app="pagerank", graph="directed", V=20011, E=300000,
             wmax=0, sources=0, resident=1.0),
        # the benchmark's PageRank
        dict(name="pagerank_large", app="pagerank", graph="rmat", scale=24, ef=16, wmax=0,
             sources=0, resident=1.0),
        # components of a large graph
        dict(name="cc_rmat", app="cc", graph="rmat", scale=22, ef=16, wmax=0, sources=0,
             method="hook", resident=1.0),
        # one full batch of each kind (level and distance tables of landmarks)
        dict(name="bfs_batch", app="bfs_multi", graph="rmat", scale=18, ef=16, wmax=0, sources=64,
             resident=1.0),
        dict(name="sssp_batch", app="sssp_multi", graph="rmat", scale=18, ef=16, wmax=255,
             sources=128, resident=1.0),
        # the query server under a burst of mixed queries
        dict(name="serve_mixed", app="serve", graph="rmat", scale=16, ef=16, wmax=255,
             sources=256, resident=1.0),
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], spread evenly over its logarithm."""
    return min(hi, max(lo, int(round(float(np.exp(rng.uniform(np.log(lo), np.log(hi))))))))


def draw(rng):
    app = rng.choice(["bfs", "bfs", "bfs_grid", "bfs_capped", "sssp", "sssp", "sssp_grid", "pagerank",
                      "pagerank", "cc", "bfs_multi", "sssp_multi", "serve"])
    case = dict(graph="rmat", wmax=0, sources=1, resident=1.0)
    if app in ("bfs_grid", "sssp_grid"):
        case.update(app=app[:-5], graph="grid", rows=_log(rng, 16, 1500), cols=_log(rng, 16, 1500))
        if app == "sssp_grid":
            case.update(wmax=rng.choice([10, 255, 1000, 20000]))
        return case
    if app in ("bfs", "sssp", "pagerank") and rng.random() < 0.4:
        V = _log(rng, 500, 700000)
        case.update(app=app, graph="directed", V=V, E=V * rng.randint(3, 24))
    elif app == "bfs_capped":
        case.update(app="bfs", scale=rng.randint(16, 21), ef=rng.randint(8, 20),
                    resident=round(rng.uniform(0.1, 0.7), 3))
    else:
        lo, hi = {"bfs": (8, 23), "sssp": (8, 22), "pagerank": (8, 23), "cc": (9, 23),
                  "bfs_multi": (9, 18), "sssp_multi": (9, 18), "serve": (10, 16)}[app]
        case.update(app=app, scale=rng.randint(lo, hi), ef=rng.randint(4, 22))
    if app in ("sssp", "sssp_multi", "serve"):
        case.update(wmax=rng.choice([10, 255, 1000, 20000]))
    if app == "pagerank":
        case.update(sources=0)
    elif app == "cc":
        case.update(sources=0, method=rng.choice(["hook", "hook", "lp"]))
    elif app == "bfs_multi":
        case.update(sources=rng.randint(2, 64))
    elif app == "sssp_multi":
        case.update(sources=rng.randint(2, 128))
    elif app == "serve":
        case.update(sources=rng.randint(24, 256))
    elif app in ("bfs", "sssp"):
        case.update(sources=rng.choice([1, 1, 4]))
    return case


# ------------------------------------------------------------------ inputs
_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        torch.cuda.init()
        _ctx = grus.Context(0)
    return _ctx


def _directed(case, seed):
    """CSR of a directed graph with skewed in- and out-degrees, rows sorted."""
    V, n = case["V"], case["E"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    u = torch.rand((2, n), generator=gen, device="cuda", dtype=torch.float64)
    where = torch.randperm(V, generator=gen, device="cuda")
    src = where[(u[0] ** 2 * V).long().clamp_(max=V - 1)]
    dst = where[(u[1] ** 3 * V).long().clamp_(max=V - 1)]
    key = torch.unique((src * V + dst)[src != dst])
    deg = torch.bincount(key // V, minlength=V)
    off = np.zeros(V + 1, np.uint64)
    off[1:] = torch.cumsum(deg, 0).cpu().numpy()
    col = (key % V).to(torch.int32).cpu().numpy().view(np.uint32)
    w = None
    if case["wmax"]:
        w = torch.randint(1, case["wmax"] + 1, (len(col),), generator=gen, device="cuda",
                          dtype=torch.int32).cpu().numpy().view(np.uint32)
    return off, col, w


def _graph(case, seed):
    ctx = _context()
    weights = (1, case["wmax"]) if case["wmax"] else None
    if case["graph"] == "directed":
        return grus.Graph.from_csr(ctx, *_directed(case, seed))
    if case["graph"] == "grid":
        return grus.Graph.grid(ctx, case["rows"], case["cols"], weights=weights, wseed=seed + 1)
    place = None
    if case["resident"] < 1.0:
        V, E = _size(case)
        place = grus.place("capped", hbm_cap_bytes=int(12 * V + 64 + 4 * E * case["resident"]))
    return grus.Graph.rmat(ctx, case["scale"], case["ef"], seed=seed + 1, weights=weights,
                           wseed=seed + 2, placement=place)


def _sources(g, n, seed):
    """n distinct vertices with edges (with repeats where there are too few)."""
    off = np.empty(g.V + 1, np.uint64)
    capi.check(capi.lib().grus_graph_copy_csr(g.h, off.ctypes.data_as(C.c_void_p), None, None))
    live = np.nonzero(np.diff(off))[0]
    rng = np.random.default_rng(seed)
    return rng.choice(live, n, replace=len(live) < n).astype(np.uint32)


class _State:
    """A graph, what a program keeps beside it, and the call's sources."""

    def __init__(self, case, seed):
        self.case = case
        self.server = None
        self.g = _graph(case, seed)
        n = case["sources"]
        self.srcs = _sources(self.g, n, seed) if n else None
        app = case["app"]
        rows = n if app in ("bfs_multi", "sssp_multi", "serve") else 1
        self.pinned = torch.zeros((rows, self.g.V), pin_memory=True,
                                  dtype=torch.float32 if app == "pagerank" else torch.int32)
        self.out = self.pinned.numpy()
        if app != "pagerank":
            self.out = self.out.view(np.uint32)
        if app == "serve":
            self.server = grus.Server(self.g, copy_results=True)

    def __del__(self):
        if getattr(self, "server", None):
            self.server.close()
        if getattr(self, "g", None):
            self.g.close()


def prepare(case, seed):
    return _State(case, seed)


# ------------------------------------------------------------------ one pass
def _traverse(s):
    g, app = s.g, s.case["app"]
    call = grus.bfs if app == "bfs" else grus.sssp
    if len(s.srcs) == 1 and g.V < (1 << 20):
        values, st = call(g, int(s.srcs[0]))  # a new array
        return dict(values=values, reached=st.vertices_reached, edges=st.edges_reached)
    reached, edges, digests = [], [], []
    for src in s.srcs:
        _, st = call(g, int(src), copy=False)
        reached.append(st.vertices_reached)
        edges.append(st.edges_reached)
        digests.append(g.digest()[1])
    capi.check(capi.lib().grus_result_copy(g.h, s.out.ctypes.data_as(C.c_void_p)))
    return dict(values=s.out[0], reached=np.array(reached), edges=np.array(edges),
                digests=np.array(digests, np.uint64).view(np.int64))


def run(s):
    g, app = s.g, s.case["app"]
    if app in ("bfs", "sssp"):
        return _traverse(s)
    lib, st = capi.lib(), capi.Stats()
    out = s.out.ctypes.data_as(C.c_void_p)
    if app == "pagerank":
        capi.check(lib.grus_pagerank(g.h, ALPHA, ITERATIONS, out, C.byref(st)))
        return s.out[0]
    if app == "cc":
        method = {"hook": 0, "lp": 1}[s.case["method"]]
        capi.check(lib.grus_cc(g.h, method, out, C.byref(st)))
        return s.out[0]
    if app in ("bfs_multi", "sssp_multi"):
        call = lib.grus_bfs_multi if app == "bfs_multi" else lib.grus_sssp_multi
        capi.check(call(g.h, s.srcs.ctypes.data_as(C.c_void_p), len(s.srcs), out, C.byref(st)))
        return dict(values=s.out, reached=st.vertices_reached)
    # serve: every query offered at once, half of each kind, then collected
    first = None
    for i, src in enumerate(s.srcs):
        qid = s.server.submit(grus.capi.Q_BFS if i % 2 == 0 else grus.capi.Q_SSSP, int(src),
                              s.out[i])
        first = qid if first is None else first
    reached = np.zeros(len(s.srcs), np.int64)
    digests = np.zeros(len(s.srcs), np.uint64)
    for _ in s.srcs:
        r = s.server.poll()
        capi.check(r.status)
        reached[r.id - first] = r.reached
        digests[r.id - first] = r.checksum
    return dict(values=s.out, reached=reached, digests=digests.view(np.int64))


# ------------------------------------------------------------------ work
def _size(case):
    """Vertices and (about) directed edges of the case's graph."""
    if case["graph"] == "grid":
        r, c = case["rows"], case["cols"]
        return r * c, 2 * (r * (c - 1) + c * (r - 1))
    if case["graph"] == "directed":
        return case["V"], case["E"]
    V = 1 << case["scale"]
    return V, int(2 * case["ef"] * V * (1 - 0.35 * 2.0 ** (-(case["scale"] - 10) / 4)))


def work(case):
    """Offsets, edges and (where the app reads them) weights once, results
    once; PageRank: once an iteration."""
    V, E = _size(case)
    per_edge = 8 if case["wmax"] and case["app"] in ("sssp", "sssp_multi", "serve") else 4
    graph = 8 * (V + 1) + per_edge * E
    n = max(1, case["sources"])
    if case["app"] == "pagerank":
        return dict(bytes=ITERATIONS * (graph + 12 * V) + 4 * V, flops=ITERATIONS * (E + 3 * V))
    if case["app"] in ("bfs", "sssp"):
        return dict(bytes=n * (graph + 4 * V), flops=n * E)
    if case["app"] == "cc":
        return dict(bytes=graph + 4 * V, flops=E)
    return dict(bytes=graph + 4 * V * n, flops=n * E)  # one sweep shared by the batch


# ------------------------------------------------------------------ exact
def exact(case, seed):
    """PageRank in 64 bits; everything else is whole numbers."""
    if case["app"] != "pagerank":
        return None
    if case["graph"] == "directed":
        off, col, _ = _directed(case, seed)
    else:
        g = _graph(case, seed)
        off, col, _ = g.csr()
        g.close()
    V = len(off) - 1
    alpha = float(np.float32(ALPHA))
    deg = torch.from_numpy(np.diff(off).astype(np.int64)).cuda()
    dst = torch.from_numpy(col.view(np.int32)).cuda().long()
    rank = torch.full((V,), (1 - alpha) / V, dtype=torch.float64, device="cuda")
    per = torch.where(deg > 0, 1.0 / deg.clamp(min=1).double(), torch.zeros_like(rank))
    for _ in range(ITERATIONS):
        sums = torch.zeros_like(rank)
        sums.index_add_(0, dst, torch.repeat_interleave(rank * per, deg))
        rank = (1 - alpha) / V + alpha * sums
    return rank
