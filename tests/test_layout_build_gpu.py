"""Layouts built over the edges, 64 a wave at a time: rows that span several
waves, runs of empty rows longer than the 64 row ends a wave reads, edge counts
around a wave's, and more edges than one sweep of the launch takes."""
import numpy as np
import pytest

import grus_framework_amd as grus

pytestmark = pytest.mark.gpu

PR_TOL = 1e-6


def shape(name):
    rng = np.random.default_rng(len(name))
    if name == "gaps":  # one row in 131 has edges, some more than 64
        V = 20000
        src = np.repeat(np.arange(7, V, 131), rng.integers(1, 150, len(range(7, V, 131))))
    elif name == "hub":  # rows 0 and V - 1 hold most edges
        V = 9000
        src = np.r_[np.zeros(3000, int), rng.integers(1, V - 1, 4000), np.full(5000, V - 1)]
    elif name == "ones":  # a row per edge, more rows than a chunk's sources
        V = 9001
        src = np.arange(V)
    else:  # that many edges
        V = 300
        src = rng.integers(40, V, int(name))
    key = np.unique(src * V + rng.integers(0, V, len(src)))
    off = np.zeros(V + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(key // V, minlength=V))
    return off, (key % V).astype(np.uint32), rng.integers(1, 300, len(key)).astype(np.uint32)


@pytest.mark.parametrize("name", ["gaps", "hub", "ones", "1", "64", "70", "1100"])
def test_directed_layouts(oracle, name):
    off, col, w = shape(name)
    h = oracle.CSR(off, col, w)
    want = oracle.pagerank(h, csc=oracle.transpose(h))
    src = int(np.argmax(np.diff(off.astype(np.int64))))
    c = grus.Context(0)
    try:
        t = c.tuning
        t.sssp_pull_div = 1 << 20
        for layout, bits in ((2, 0), (3, 9), (4, 11), (4, 13)):
            t.pr_layout, t.pr_bin_bits = layout, bits
            c.tuning = t
            with grus.Graph.from_csr(c, off, col, w) as g:  # its in-edges: sorted by head
                ranks, _ = grus.pagerank(g)
                assert np.abs(ranks - want).sum() <= PR_TOL, (layout, bits)
                d, _ = grus.sssp(g, src)
                assert (d == oracle.sssp(h, src)).all(), (layout, bits)
    finally:
        c.close()


def test_more_edges_than_a_sweep():
    # a symmetric graph's in-edges are its own rows; declared directed, the
    # same rows come out of the transposition
    c = grus.Context(0)
    try:
        t = c.tuning
        with grus.Graph.rmat(c, 20, 16) as g:
            off, col, _ = g.csr()
            assert g.E > 1 << 24
            for layout in (1, 2, 3, 4):
                t.pr_layout = layout
                c.tuning = t
                a, _ = grus.pagerank(g)
                with grus.Graph.from_csr(c, off, col) as d:
                    b, _ = grus.pagerank(d)
                assert np.abs(a.astype(np.float64) - b).sum() <= PR_TOL, layout
                if layout == 2:
                    assert (a.view(np.uint32) == b.view(np.uint32)).all()
    finally:
        c.close()
