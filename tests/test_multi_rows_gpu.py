"""Rows of a batch copied out together: widths around the transposing tile
(32 slots x 64 vertices), 16- and 32-bit entries, more rows than the staging
buffer holds, and one row at a time under a device budget."""
import numpy as np
import pytest

import grus_framework_amd as grus

pytestmark = pytest.mark.gpu

INF = grus.INFINIT


def directed(V, M, wmax, seed):
    rng = np.random.default_rng(seed)
    key = np.unique(rng.integers(0, V, M) * V + rng.integers(0, V, M))
    off = np.zeros(V + 1, np.uint64)
    np.add.at(off, key // V + 1, 1)
    w = rng.integers(1, wmax + 1, len(key)).astype(np.uint32)
    return np.cumsum(off).astype(np.uint64), (key % V).astype(np.uint32), w


@pytest.mark.parametrize("wmax", [9, 1 << 20])  # 16-bit rows, and rows widened on the way
@pytest.mark.parametrize("V", [63, 64, 1029])
@pytest.mark.parametrize("k", [1, 31, 33, 127, 128])
def test_sssp_rows(ctx, oracle, V, k, wmax):
    off, col, w = directed(V, 6 * V, wmax, V + k)
    h = oracle.CSR(off, col, w)
    srcs = np.random.default_rng(k).integers(0, V, k)
    want = np.array([oracle.sssp(h, int(s)) for s in srcs])
    with grus.Graph.from_csr(ctx, off, col, w) as g:
        for _ in range(2):  # the second batch finds the first one's entries
            got, st = grus.sssp_multi(g, srcs)
            assert (got == want).all()
            assert st.vertices_reached == (want != INF).sum()
        few, st = grus.sssp_multi(g, srcs[:1])  # the other slots still hold finite entries
        assert (few == want[:1]).all()
        assert st.vertices_reached == (want[:1] != INF).sum()


@pytest.mark.parametrize("V,k", [(63, 64), (1029, 33), (1029, 1)])
def test_bfs_rows(ctx, oracle, V, k):
    off, col, _ = directed(V, 2 * V, 1, V + k)
    h = oracle.CSR(off, col, None)
    srcs = np.random.default_rng(k).integers(0, V, k)
    want = np.array([oracle.bfs(h, int(s)) for s in srcs])
    with grus.Graph.from_csr(ctx, off, col) as g:
        for n in (k, 1):
            got, st = grus.bfs_multi(g, srcs[:n])
            assert (got == want[:n]).all()
            assert st.vertices_reached == (want[:n] != INF).sum()


def test_sssp_rows_past_the_staging_buffer(ctx):
    # 128 rows of 2^18 vertices are twice what is staged at a time
    with grus.Graph.rmat(ctx, 18, 4, weights=(1, 255), wseed=2) as g:
        rng = np.random.default_rng(1)
        srcs = rng.choice(g.V, 128, replace=False)
        got, _ = grus.sssp_multi(g, srcs)
        for i in (0, 31, 32, 63, 64, 65, 127):
            want, _ = grus.sssp(g, int(srcs[i]))
            assert (got[i] == want).all(), i


def test_sssp_rows_under_a_device_budget(oracle):
    c = grus.Context(0)
    try:
        off, col, w = directed(1029, 6000, 9, 4)
        h = oracle.CSR(off, col, w)
        srcs = np.arange(40)
        with grus.Graph.from_csr(c, off, col, w) as g:
            c.set_device_budget(c.device_memory()[0] + (64 << 20))
            got, st = grus.sssp_multi(g, srcs)
        want = np.array([oracle.sssp(h, int(s)) for s in srcs])
        assert (got == want).all()
        assert st.vertices_reached == (want != INF).sum()
    finally:
        c.set_device_budget(0)
        c.close()
