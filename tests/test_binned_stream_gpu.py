"""The binned layout's phase 2 over long streams: more slabs per wave than the
64 whose first groups it holds at a time, the last ones partly filled, for
each width of the weight stream and of the accumulators."""
import numpy as np
import pytest

import grus_framework_amd as grus

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wmax", [255, 65535, 1 << 20])  # 1-, 2- and 4-byte weight streams
@pytest.mark.parametrize("bits", [12, 13, 14])
def test_long_tasks(bits, wmax):
    c = grus.Context(0)
    try:
        t = c.tuning
        t.pr_layout, t.pr_bin_bits, t.sssp_pull_div = 4, bits, 1 << 20
        with grus.Graph.rmat(c, 18, 17, weights=(1, wmax), wseed=3) as g:
            src = g.info.max_degree_vertex
            t.pr_task_edges = 20000  # a slab or three per wave
            c.tuning = t
            want, _ = grus.pagerank(g)
            t.sssp_pull_layout = 1
            c.tuning = t
            dist, _ = grus.sssp(g, src)
            t.sssp_pull_layout, t.pr_task_edges = 0, 1 << 23  # bins whole: millions of edges
            c.tuning = t
            ranks, _ = grus.pagerank(g)
            assert (ranks.view(np.uint32) == want.view(np.uint32)).all()
            got, st = grus.sssp(g, src)
            assert st.pull_iterations >= 1
            assert (got == dist).all()
            t.pr_layout = 2
            c.tuning = t
            plain, _ = grus.pagerank(g)
            assert np.abs(ranks.astype(np.float64) - plain).sum() <= 1e-6
    finally:
        c.close()
