"""The task size of SSSP's pull rounds follows the tuning from one run to the
next, as PageRank's does."""
import numpy as np
import pytest

import grus_framework_amd as grus

pytestmark = pytest.mark.gpu


def test_task_size_between_runs(oracle):
    with grus.Context(0) as c:
        t = c.tuning
        t.sssp_pull_div, t.pr_layout = 1 << 20, 4
        c.tuning = t
        with grus.Graph.rmat(c, 14, 8, weights=(1, 200), wseed=5) as g:
            off, col, w = g.csr()
            src = g.info.max_degree_vertex
            want = oracle.sssp(oracle.CSR(off, col, w), src)
            held = {}
            for size in (0, 300, 0, 100000):
                t.pr_task_edges = size
                c.tuning = t
                got, st = grus.sssp(g, src)
                assert st.pull_iterations >= 1 and (got == want).all()
                held[size] = c.device_memory()[0]  # with the table of tasks, 16 bytes each
                ranks = grus.pagerank(g)[0].view(np.uint32)
                assert size == 0 or (ranks == first).all()
                first = ranks
            tasks = g.E // 300
            assert held[300] - held[100000] > 16 * tasks // 2
