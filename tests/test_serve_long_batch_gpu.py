"""A batch that keeps admitting arrivals runs for as long as they come; what the
server learns of a batch's time from it must not make every queue look short
enough to be served one query at a time."""
import time

import numpy as np
import pytest

import grus_framework_amd as grus

pytestmark = pytest.mark.gpu


def closed_loop_ms(g, live, kind, outstanding, n, **options):
    rng = np.random.default_rng(5)
    ms = []
    with grus.Server(g, **options) as server:
        for _ in range(5):
            srcs = [int(s) for s in rng.choice(live, n)]
            t0 = time.perf_counter()
            for s in srcs[:outstanding]:
                server.submit(kind, s)
            for k in range(n):
                assert server.poll(timeout_ms=30000).status == 0
                if k + outstanding < n:
                    server.submit(kind, srcs[k + outstanding])
            ms.append((time.perf_counter() - t0) * 1e3)
    return np.mean(ms[2:])


@pytest.mark.parametrize("kind,scale", [(grus.Q_BFS, 18), (grus.Q_SSSP, 21)])
def test_a_wide_queue_stays_in_batches(ctx, kind, scale):
    with grus.Graph.rmat(ctx, scale, weights=(1, 255), wseed=3) as g:
        off = np.empty(g.V + 1, np.uint64)
        grus.capi.check(grus.capi.lib().grus_graph_copy_csr(g.h, grus._p(off), None, None))
        live = np.nonzero(np.diff(off))[0]
        alone = closed_loop_ms(g, live, kind, 128, 600, solo_max=1000)
        assert closed_loop_ms(g, live, kind, 128, 600, admit_window=1000) < 0.8 * alone
