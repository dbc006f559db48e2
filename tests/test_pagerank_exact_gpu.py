"""The exact pull of small graphs: bit for bit the binned layout's ranks (both
add the same 64-bit fixed-point terms), within the FP64 oracle's tolerance,
on rows that meet its 1024-edge windows in every way."""
import numpy as np
import pytest

import grus_framework_amd as grus

pytestmark = pytest.mark.gpu

PR_TOL = 1e-6  # L1 over normalised ranks vs the FP64 oracle
WIN = 1024


def from_in_degrees(indeg, seed):
    """Directed CSR whose vertex v has indeg[v] distinct in-neighbours."""
    rng = np.random.default_rng(seed)
    V = len(indeg)
    src = np.concatenate([rng.choice(V, d, replace=False) for d in indeg] + [np.zeros(0, int)])
    dst = np.repeat(np.arange(V), indeg)
    order = np.lexsort((dst, src))
    off = np.zeros(V + 1, np.uint64)
    np.add.at(off, src + 1, 1)
    return np.cumsum(off).astype(np.uint64), dst[order].astype(np.uint32)


def in_degrees(kind):
    rng = np.random.default_rng(11)
    if kind == "hub_spans_windows":
        return [3] * 500 + [5000] + [0] * 300 + [2] * 5200
    if kind == "row_is_a_window":  # rows that begin and end on window boundaries
        return [WIN, WIN, WIN - 1, 1, 2 * WIN, 0, 0, WIN + 1, WIN - 1] + [0] * 3000
    if kind == "one_edge_past":
        return [1] * (WIN - 1) + [2] + [0] * 70 + [1] * WIN
    if kind == "edges_end_on_window":
        return [4] * (WIN // 2) + [0] * 40
    if kind == "one_edge":
        return [0, 1, 0]
    if kind == "no_edges":
        return [0] * 300
    return list(rng.choice([0, 1, 3, 7, 40, 900, 1100, 2500], 900,
                           p=[.3, .3, .2, .1, .06, .02, .01, .01])) + [0] * 1700


@pytest.mark.parametrize("iters", [0, 1, 2, 20])
@pytest.mark.parametrize("kind", ["hub_spans_windows", "row_is_a_window", "one_edge_past",
                                  "edges_end_on_window", "one_edge", "no_edges", "mixed"])
def test_exact_pull_equals_binned(ctx, oracle, kind, iters):
    off, col = from_in_degrees(in_degrees(kind), 5)
    h = oracle.CSR(off, col, None)
    want = oracle.pagerank(h, iters=iters, csc=oracle.transpose(h))
    t0 = ctx.tuning
    with grus.Graph.from_csr(ctx, off, col) as g:
        try:
            got, _ = grus.pagerank(g, iters=iters)
            again, _ = grus.pagerank(g, iters=iters)  # sums and counts were left at zero
            t = ctx.tuning
            t.pr_layout = 4
            ctx.tuning = t
            binned, _ = grus.pagerank(g, iters=iters)
        finally:
            ctx.tuning = t0
    assert (got == again).all()
    if len(col):  # (a graph without edges has no binned layout)
        assert (got.view(np.uint32) == binned.view(np.uint32)).all()
    assert np.abs(got - want).sum() <= PR_TOL


def test_exact_pull_symmetric_hubs(ctx, oracle):
    with grus.Graph.rmat(ctx, 15) as g:
        off, col, _ = g.csr()
        want = oracle.pagerank(oracle.CSR(off, col, None))
        got, st = grus.pagerank(g)
        assert st.kernel_launches == 1 + 20
        assert np.abs(got - want).sum() <= PR_TOL
