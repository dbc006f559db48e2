"""Bursts of one kind of query that a large graph's kernels serve faster alone
than in a batch: after the server has seen a batch it has to take no longer than
a server that runs no batches, whose single queries it measured beside one."""
import time

import numpy as np
import pytest

import grus_framework_amd as grus

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def graph(ctx):
    with grus.Graph.rmat(ctx, 24, weights=(1, 255), wseed=3) as g:
        off = np.empty(g.V + 1, np.uint64)
        grus.capi.check(grus.capi.lib().grus_graph_copy_csr(g.h, grus._p(off), None, None))
        yield g, np.nonzero(np.diff(off))[0]


def burst_ms(server, kind, srcs):
    t0 = time.perf_counter()
    for s in srcs:
        server.submit(kind, int(s))
    for _ in srcs:
        assert server.poll(timeout_ms=30000).status == 0
    return (time.perf_counter() - t0) * 1e3


def mean_burst(g, live, kind, n, **options):
    rng = np.random.default_rng(n)
    with grus.Server(g, **options) as server:
        burst_ms(server, kind, rng.choice(live, 4))
        burst_ms(server, kind, rng.choice(live, 64))  # a batch runs
        return np.mean([burst_ms(server, kind, rng.choice(live, n)) for _ in range(10)])


@pytest.mark.parametrize("kind,n", [(grus.Q_BFS, 32), (grus.Q_SSSP, 24)])
def test_no_slower_than_alone(graph, kind, n):
    g, live = graph
    alone = mean_burst(g, live, kind, n, solo_max=1000)
    assert mean_burst(g, live, kind, n) < 1.3 * alone
