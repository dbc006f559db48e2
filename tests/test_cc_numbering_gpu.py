"""Connected components where a vertex's first neighbour is not its smallest or
says little: numberings without order, rows in any order, and many components.
Labels against the union-find oracle, and the time against the same graph with
its rows ascending."""
import numpy as np
import pytest

import grus_framework_amd as grus

pytestmark = pytest.mark.gpu


def csr(V, u, v, row_order=None):
    """Symmetric CSR of the pairs; rows ascend, or follow a random order."""
    key = np.unique(np.concatenate([u * V + v, v * V + u]))
    key = key[key // V != key % V]
    a, b = key // V, key % V
    if row_order is not None:
        p = np.random.default_rng(row_order).permutation(len(a))
        p = p[np.argsort(a[p], kind="stable")]
        a, b = a[p], b[p]
    off = np.zeros(V + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(a, minlength=V))
    return off, b.astype(np.uint32)


def uniform(V, n, seed=1):
    rng = np.random.default_rng(seed)
    return V, rng.integers(0, V, n), rng.integers(0, V, n)


def blocks(V, size, per):
    """Components of at most `size` vertices, their ids shuffled."""
    rng = np.random.default_rng(4)
    u = rng.integers(0, V, per * V)
    v = np.minimum(u // size * size + rng.integers(0, size, per * V), V - 1)
    p = rng.permutation(V)
    return V, p[u], p[v]


def two_sided(V, few, n):
    rng = np.random.default_rng(5)
    return V, rng.integers(few, V, n), rng.integers(0, few, n)


GRAPHS = {
    "two_vertices": (2, np.array([0]), np.array([1])),
    "uniform_300": uniform(300, 200),
    "uniform_5000": uniform(5000, 20000),
    "uniform_70001": uniform(70001, 500000),
    "sparse_70001": uniform(70001, 40000),  # a giant component beside thousands of others
    "blocks_30000": blocks(30000, 100, 6),
    "pairs_20000": blocks(20000, 2, 1),
    "two_sided_40000": two_sided(40000, 300, 200000),
}


@pytest.mark.parametrize("row_order", [None, 3])
@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_labels(ctx, oracle, name, row_order):
    off, col = csr(*GRAPHS[name], row_order)
    want = oracle.cc(oracle.CSR(off, col, None))
    with grus.Graph.from_csr(ctx, off, col, symmetric=True) as g:
        for _ in range(2):
            got, _ = grus.cc(g)
            assert (got == want).all()


def device_ms(ctx, off, col):
    with grus.Graph.from_csr(ctx, off, col, symmetric=True) as g:
        grus.cc(g, copy=False)
        return min(grus.cc(g, copy=False)[1].device_ms for _ in range(5))


def test_row_order_costs_little(ctx):
    with grus.Graph.rmat(ctx, 18) as g:
        off, col, _ = g.csr()
    V = len(off) - 1
    u = np.repeat(np.arange(V), np.diff(off).astype(np.int64))
    any_order = csr(V, u, col.astype(np.int64), 7)
    # one list of edges in two orders: what is read is the same, the links that
    # rows in ascending order save are those of a few neighbours a vertex
    assert device_ms(ctx, *any_order) < 5 * device_ms(ctx, off, col)
