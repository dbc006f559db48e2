"""Connected components by first-neighbour hooks: the graphs where the hooks,
the sampled mode or the mapping of the left-over rows can go wrong, bit-exact
against the union-find oracle."""
import numpy as np
import pytest

import grus_framework_amd as grus

pytestmark = pytest.mark.gpu


def symmetric(V, u, v):
    u, v = np.asarray(u, np.int64), np.asarray(v, np.int64)
    key = np.unique(np.concatenate([u * V + v, v * V + u]))
    off = np.zeros(V + 1, np.uint64)
    np.add.at(off, key // V + 1, 1)
    return np.cumsum(off).astype(np.uint64), (key % V).astype(np.uint32)


def build(kind):
    rng = np.random.default_rng(7)
    if kind == "chain":  # hooks form one chain through every vertex
        n = 70001
        return symmetric(n, np.arange(n - 1), np.arange(1, n))
    if kind == "chain_shuffled":  # about a third of the vertices are local minima
        p = rng.permutation(50000)
        return symmetric(50000, p[:-1], p[1:])
    if kind == "stars":  # centre above its leaves; rows of 15, 16, 17, 63..65, 200 edges, no giant
        sizes = [15, 16, 17, 63, 64, 65, 200] * 30
        u, v, at = [], [], 0
        for s in sizes:
            u += [at + s] * s
            v += list(range(at, at + s))
            at += s + 1
        return symmetric(at, u, v)
    if kind == "giant_and_rows":  # a giant by sampling, and rows around a wave outside it
        n = 20000
        u, v = list(rng.integers(0, n, 60000)), list(rng.integers(0, n, 60000))
        at = n
        for s in [16, 17, 64, 65, 1000]:
            ids = at + rng.permutation(s + 1)
            u += [ids[0]] * s
            v += list(ids[1:])
            at += s + 1
        keep = np.array(u) != np.array(v)
        return symmetric(at, np.array(u)[keep], np.array(v)[keep])
    if kind == "no_edges":
        return np.zeros(1001, np.uint64), np.zeros(0, np.uint32)
    if kind == "one":
        return np.zeros(2, np.uint64), np.zeros(0, np.uint32)
    off, col = build("giant_and_rows")  # rows in descending order
    for i in range(len(off) - 1):
        col[int(off[i]):int(off[i + 1])] = col[int(off[i]):int(off[i + 1])][::-1]
    return off, col


@pytest.mark.parametrize("kind", ["chain", "chain_shuffled", "stars", "giant_and_rows", "no_edges",
                                  "one", "descending_rows"])
def test_cc_hooks_vs_oracle(ctx, oracle, kind):
    off, col = build(kind)
    want = oracle.cc(oracle.CSR(off, col, None))
    with grus.Graph.from_csr(ctx, off, col, symmetric=True) as g:
        for _ in range(2):
            got, _ = grus.cc(g)
            assert (got == want).all(), kind
