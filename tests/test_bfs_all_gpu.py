"""A whole traversal in one launch (graphs of at most 2^18 vertices): one
workgroup and a grid, bitmap words that end inside a word, rows that a wave, a
workgroup and the whole grid expand or scan, and traversals that switch
direction both ways.  Levels and counts against the oracle."""
import numpy as np
import pytest

import grus_framework_amd as grus

pytestmark = pytest.mark.gpu

INF = grus.INFINIT


def csr(V, u, v, both=True):
    u, v = np.asarray(u, np.int64), np.asarray(v, np.int64)
    key = u * V + v
    if both:
        key = np.concatenate([key, v * V + u])
    key = np.unique(key)
    key = key[key // V != key % V]
    off = np.zeros(V + 1, np.uint64)
    np.add.at(off, key // V + 1, 1)
    return np.cumsum(off).astype(np.uint64), (key % V).astype(np.uint32)


def random_graph(V, edges, hubs, both=True):
    """Random edges, and hubs with rows of the given lengths spread over V."""
    rng = np.random.default_rng(V + edges)
    u, v = rng.integers(0, V, edges), rng.integers(0, V, edges)
    for n in hubs:
        n = min(n, V - 1)
        u = np.concatenate([u, np.full(n, rng.integers(0, V))])
        v = np.concatenate([v, rng.choice(V, n, replace=False)])
    return csr(V, u, v, both)


def build(kind):
    if kind == "star":  # one row past the whole-grid size, and a tail behind a leaf
        n = 20000
        u = [0] * (n - 1) + list(range(n - 1, n + 300))
        v = list(range(1, n)) + list(range(n, n + 301))
        return csr(n + 302, u, v)
    if kind == "stars":  # rows of 511 to 9000 edges, centre last, along a chain
        u, v, at, last = [], [], 0, None
        for n in [30, 511, 512, 513, 3000, 8191, 8192, 8193, 9000]:
            u += [at + n] * n
            v += list(range(at, at + n))
            if last is not None:
                u.append(last)
                v.append(at)
            last, at = at + n - 1, at + n + 1
        return csr(at, u, v)
    if kind == "directed":
        return random_graph(30000, 90000, [40, 700, 9000], both=False)
    V, deg = (int(x) for x in kind.split("x"))
    return random_graph(V, V * deg, [20, 600] if V > 700 else [20])


CASES = ["40x2", "63x1", "1023x3", "1024x3", "1025x3", "5000x1", "60001x8", "262144x2", "262145x2",
         "star", "stars", "directed"]


@pytest.mark.parametrize("kind", CASES)
def test_whole_traversal_vs_oracle(ctx, oracle, kind):
    off, col = build(kind)
    h = oracle.CSR(off, col, None)
    deg = np.diff(off).astype(np.int64)
    V = len(deg)
    assert deg.max() > 16  # not the padded low-degree path
    srcs = {0, V - 1, V // 2, int(np.argmax(deg))} | set(np.nonzero(deg == 0)[0][:1].tolist())
    with grus.Graph.from_csr(ctx, off, col, symmetric=kind != "directed") as g:
        for src in sorted(srcs):
            want = oracle.bfs(h, src)
            hit = want != INF
            for _ in range(2):  # the second finds the first one's bitmaps and flags
                got, st = grus.bfs(g, src)
                assert (got == want).all(), src
                assert st.iterations == int(want[hit].max()) + 1
                assert st.vertices_reached == hit.sum()
                assert st.edges_reached == deg[hit].sum()


@pytest.mark.parametrize("alpha,beta,cut", [(1e-9, 64, 32), (1e9, 64, 1), (1e9, 1e9, 3), (14, 1, 200),
                                            (3, 2, 32)])
def test_whole_traversal_direction_rules(oracle, alpha, beta, cut):
    c = grus.Context(0)
    try:
        t = c.tuning
        t.bfs_alpha, t.bfs_beta, t.bu_thread_edges = alpha, beta, cut
        c.tuning = t
        with grus.Graph.rmat(c, 14) as g:
            off, col, _ = g.csr()
            h = oracle.CSR(off, col, None)
            for src in (g.info.max_degree_vertex, 77):
                got, st = grus.bfs(g, src)
                assert (got == oracle.bfs(h, src)).all()
                assert alpha < 1 or st.pull_iterations > 0 or st.iterations < 3
    finally:
        c.close()


@pytest.mark.parametrize("scale", [9, 13])
def test_whole_traversal_under_a_cu_mask(oracle, scale):
    # one workgroup still runs it; a grid does not, and levels are launched
    c = grus.Context(0)
    try:
        c.set_cu_limit(16)
        with grus.Graph.rmat(c, scale) as g:
            off, col, _ = g.csr()
            want = oracle.bfs(oracle.CSR(off, col, None), g.info.max_degree_vertex)
            got, _ = grus.bfs(g, g.info.max_degree_vertex)
            assert (got == want).all()
    finally:
        c.close()
