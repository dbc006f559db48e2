"""SSSP batch steps over the in-edges: rows around the wave's 64 edges and the
workgroup's 256, rows that several workgroups share, both entry widths, and
the graphs for which steps keep pushing."""
import numpy as np
import pytest

import grus_framework_amd as grus

pytestmark = pytest.mark.gpu


def symmetric(V, pairs, wmax, seed, mirror=True):
    """CSR of the undirected pairs; mirror: both directions weigh the same."""
    a, b = pairs.min(1).astype(np.int64), pairs.max(1).astype(np.int64)
    key = np.unique((a * V + b)[a != b])
    a, b = key // V, key % V
    rng = np.random.default_rng(seed)
    w = rng.integers(1, wmax + 1, len(key))
    w2 = w if mirror else rng.integers(1, wmax + 1, len(key))
    s, d, w = np.r_[a, b], np.r_[b, a], np.r_[w, w2]
    order = np.lexsort((d, s))
    off = np.zeros(V + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(s, minlength=V))
    return off, d[order].astype(np.uint32), w[order].astype(np.uint32)


def shape(name, seed):
    rng = np.random.default_rng(seed)
    if name == "sparse":  # degrees 0..12, runs of empty rows
        V = 4001
        return V, rng.integers(0, V // 2, (3 * V, 2)) * 2
    if name == "hubs":  # rows of 60..70, 250..260 and 3000 edges beside leaves
        V = 3500
        hub = [np.c_[np.full(n, 7 * i), rng.choice(V, n, replace=False)]
               for i, n in enumerate((62, 64, 65, 127, 255, 257, 512, 3000))]
        return V, np.concatenate(hub + [rng.integers(0, V, (V, 2))])
    if name == "complete":  # more edges than 64 a vertex
        V = 210
        return V, np.argwhere(np.ones((V, V)))
    V = 130  # "tiny": fewer edges than one workgroup takes
    return V, np.c_[np.arange(100), np.arange(1, 101)]


def check(g, oracle, csr, srcs):
    h = oracle.CSR(*csr)
    want = np.array([oracle.sssp(h, int(s)) for s in srcs])
    for _ in range(2):
        got, _ = grus.sssp_multi(g, srcs)
        assert (got == want).all()


@pytest.mark.parametrize("wmax", [5, 30000, 1 << 20])  # 16 bits; some and all slots widened
@pytest.mark.parametrize("name", ["sparse", "hubs", "complete", "tiny"])
@pytest.mark.parametrize("k", [15, 128])
def test_sssp_batch(ctx, oracle, name, k, wmax):
    V, pairs = shape(name, k)
    csr = symmetric(V, pairs, wmax, k)
    srcs = np.random.default_rng(k).integers(0, V, k)
    with grus.Graph.from_csr(ctx, *csr, symmetric=True) as g:
        check(g, oracle, csr, srcs)


@pytest.mark.parametrize("name", ["hubs", "complete"])
def test_weights_differ_by_direction(ctx, oracle, name):
    # declared symmetric, and only the edges are: the out-edges' weights hold
    V, pairs = shape(name, 3)
    csr = symmetric(V, pairs, 200, 3, mirror=False)
    with grus.Graph.from_csr(ctx, *csr, symmetric=True) as g:
        check(g, oracle, csr, np.arange(64))


@pytest.mark.parametrize("in_edges", [False, True])
def test_directed(ctx, oracle, in_edges):
    rng = np.random.default_rng(8)
    V = 1500
    key = np.unique((rng.random(40000) ** 2 * V).astype(np.int64) * V + rng.integers(0, V, 40000))
    off = np.zeros(V + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(key // V, minlength=V))
    csr = off, (key % V).astype(np.uint32), rng.integers(1, 90, len(key)).astype(np.uint32)
    with grus.Graph.from_csr(ctx, *csr) as g:
        if in_edges:  # built for another traversal
            grus.bfs_multi(g, [0, 1])
        check(g, oracle, csr, rng.integers(0, V, 100))


def test_unweighted(ctx, oracle):
    V, pairs = shape("hubs", 5)
    off, col, _ = symmetric(V, pairs, 1, 5)
    with grus.Graph.from_csr(ctx, off, col, symmetric=True) as g:
        check(g, oracle, (off, col, None), np.arange(20, 60))
