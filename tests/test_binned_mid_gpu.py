"""The binned layout at each accumulator size (bins of 2^12, 2^13 and 2^14
vertices and the automatic width), with tasks that split bins and tasks that
do not: SSSP pull rounds against Dijkstra, PageRank ranks equal bit for bit
and within the FP64 oracle's tolerance."""
import numpy as np
import pytest

import grus_framework_amd as grus

pytestmark = pytest.mark.gpu

PR_TOL = 1e-6


@pytest.mark.parametrize("wmax", [200, 60000, 1 << 20])  # 1-, 2- and 4-byte weight streams
@pytest.mark.parametrize("bits,task", [(0, 0), (11, 0), (12, 700), (13, 0), (13, 900), (14, 700)])
def test_binned_sizes(oracle, bits, task, wmax):
    c = grus.Context(0)
    try:
        t = c.tuning
        t.pr_layout, t.pr_bin_bits, t.pr_task_edges, t.sssp_pull_div = 4, bits, task, 1 << 20
        c.tuning = t
        with grus.Graph.rmat(c, 15, 6, weights=(1, wmax), wseed=5) as g:
            off, col, w = g.csr()
            h = oracle.CSR(off, col, w)
            src = g.info.max_degree_vertex
            ranks, _ = grus.pagerank(g)
            d, st = grus.sssp(g, src)
            again, _ = grus.pagerank(g)  # after SSSP cut its own tasks
            assert st.pull_iterations >= 1
            assert (d == oracle.sssp(h, src)).all()
            assert (ranks == again).all()
            assert np.abs(ranks - oracle.pagerank(h)).sum() <= PR_TOL
            t.pr_bin_bits, t.pr_task_edges = 14, 1 << 18
            c.tuning = t
            wide, _ = grus.pagerank(g)
            assert (ranks.view(np.uint32) == wide.view(np.uint32)).all()
    finally:
        c.close()
