"""SSSP rounds that one workgroup runs back to back: near queues and far
queues around the limits at which it takes over and hands back (1024 vertices,
16384 out-edges, 8192 far vertices), bucket widths with mostly empty buckets,
and the one-pass far split.  Distances against Dijkstra."""
import numpy as np
import pytest

import grus_framework_amd as grus

pytestmark = pytest.mark.gpu

INF = grus.INFINIT


def csr(V, u, v, w):
    u, v, w = (np.asarray(x, np.int64) for x in (u, v, w))
    key, at = np.unique(u * V + v, return_index=True)
    off = np.zeros(V + 1, np.uint64)
    np.add.at(off, key // V + 1, 1)
    return (np.cumsum(off).astype(np.uint64), (key % V).astype(np.uint32),
            w[at].astype(np.uint32))


def fan(leaves, per, wmax):
    """source -> leaves -> per targets each: a near queue of `leaves` vertices
    and leaves * per edges; the last target has edges back (a long row)."""
    rng = np.random.default_rng(leaves + per)
    first, n = 1, leaves * per // 2 + 50
    V = 1 + leaves + n
    u = [0] * leaves + list(np.repeat(np.arange(first, first + leaves), per))
    v = list(range(first, first + leaves))
    for _ in range(leaves):
        v += list(first + leaves + rng.choice(n, per, replace=False))
    u += [V - 1] * 60
    v += list(rng.choice(V - 1, 60, replace=False))
    return csr(V, u, v, rng.integers(1, wmax + 1, len(u)))


def build(kind):
    rng = np.random.default_rng(2)
    if kind.startswith("fan"):
        leaves, per = (int(x) for x in kind.split("_")[1:])
        return fan(leaves, per, 9)
    if kind.startswith("far"):  # a hub offers `n` far distances at once
        n = int(kind.split("_")[1])
        u = [0] * n + list(range(1, n + 1))
        v = list(range(1, n + 1)) + list(rng.permutation(n) + 1)
        keep = np.array(u) != np.array(v)
        return csr(n + 2, np.array(u)[keep], np.array(v)[keep],
                   rng.integers(1, 1 << 15, keep.sum()))  # (sums stay below 2^32)
    V = 3000
    u, v = rng.integers(0, V, 9 * V), rng.integers(0, V, 9 * V)
    u = np.concatenate([u, np.full(200, 17)])  # one row past the low-degree path
    v = np.concatenate([v, rng.choice(V, 200, replace=False)])
    keep = u != v
    wmax = {"random_unit": 1, "random_wide": 1 << 26}.get(kind, 5000)
    return csr(V, u[keep], v[keep], rng.integers(1, wmax + 1, keep.sum()))


@pytest.mark.parametrize("delta", [0, 1, 700, 1 << 24])
@pytest.mark.parametrize("kind", ["fan_1023_16", "fan_1024_16", "fan_1025_15", "fan_1024_17",
                                  "fan_300_55", "far_8191", "far_8193", "far_12000", "random",
                                  "random_unit", "random_wide"])
def test_small_rounds_vs_dijkstra(ctx, oracle, kind, delta):
    off, col, w = build(kind)
    h = oracle.CSR(off, col, w)
    deg = np.diff(off).astype(np.int64)
    assert deg.max() > 32  # not the persistent low-degree path
    t0 = ctx.tuning
    with grus.Graph.from_csr(ctx, off, col, w) as g:
        try:
            t = ctx.tuning
            t.sssp_delta = delta
            ctx.tuning = t
            for src in (0, 17, len(deg) - 1):
                want = oracle.sssp(h, src)
                got, st = grus.sssp(g, src)
                assert (got == want).all(), (kind, delta, src)
                assert st.vertices_reached == (want != INF).sum()
                assert st.edges_reached == deg[want != INF].sum()
        finally:
            ctx.tuning = t0
