"""Thin levels of low-degree graphs run on the device: frontiers that stay
within one workgroup, that outgrow it, that outgrow the cooperative grid, and
that shrink again; padded rows of 4, 8 and 16 columns.  Levels and counts
against the oracle."""
import numpy as np
import pytest

import grus_framework_amd as grus

pytestmark = pytest.mark.gpu

INF = grus.INFINIT


def csr(V, u, v, both=True):
    u, v = np.asarray(u, np.int64), np.asarray(v, np.int64)
    key = u * V + v
    if both:
        key = np.concatenate([key, v * V + u])
    key = np.unique(key)
    key = key[key // V != key % V]
    off = np.zeros(V + 1, np.uint64)
    np.add.at(off, key // V + 1, 1)
    return np.cumsum(off).astype(np.uint64), (key % V).astype(np.uint32)


def grid(R, C, diagonals=False):
    i = np.arange(R * C).reshape(R, C)
    pairs = [(i[:, :-1], i[:, 1:]), (i[:-1], i[1:])]
    if diagonals:
        pairs += [(i[:-1, :-1], i[1:, 1:]), (i[:-1, 1:], i[1:, :-1])]
    return csr(R * C, np.concatenate([a.ravel() for a, _ in pairs]),
               np.concatenate([b.ravel() for _, b in pairs]))


def build(kind):
    rng = np.random.default_rng(3)
    if kind == "path":
        return grid(1, 9000)
    if kind == "grid_small":
        return grid(37, 53)
    if kind == "grid_wide":  # frontiers past one workgroup and back
        return grid(900, 1100)
    if kind == "grid_eight":  # 8 columns a row; square rings, up to 4 x 700 vertices
        return grid(700, 750, diagonals=True)
    if kind == "tree":  # doubles past every limit: 1, 2, 4, ... 65536
        n = (1 << 17) - 1
        k = np.arange(1, n)
        return csr(n, (k - 1) // 2, k)
    if kind == "tree16":  # one 16-column level fills the LDS list of a workgroup
        n = 70000
        k = np.arange(1, n)
        return csr(n, (k - 1) // 15, k)
    if kind == "lollipops":  # trees hung along a path: thin, wide, thin again
        n = 40 * 5000
        u, v = [], []
        for s in range(40):
            k = np.arange(1, 4000) + s * 5000
            u += list((k - s * 5000 - 1) // 3 + s * 5000)
            v += list(k)
            p = np.arange(4000, 5000) + s * 5000
            u += list(p - 1)
            v += list(p)
            if s:
                u.append(s * 5000 - 1)
                v.append(s * 5000)
        return csr(n, u, v)
    # directed, out-degree at most 3, long cycles and unreached parts
    n = 60000
    k = np.arange(n)
    return csr(n, np.concatenate([k, k, rng.integers(0, n, 500)]),
               np.concatenate([(k + 1) % n, np.minimum(k + 40, n - 1), rng.integers(0, n, 500)]),
               both=False)


@pytest.mark.parametrize("kind", ["path", "grid_small", "grid_wide", "grid_eight", "tree", "tree16",
                                  "lollipops", "directed"])
def test_thin_levels_vs_oracle(ctx, oracle, kind):
    off, col = build(kind)
    h = oracle.CSR(off, col, None)
    deg = np.diff(off).astype(np.int64)
    assert deg.max() <= 16
    V = len(deg)
    with grus.Graph.from_csr(ctx, off, col, symmetric=kind != "directed") as g:
        for src in (0, V // 2 + 7, V - 1):
            want = oracle.bfs(h, src)
            hit = want != INF
            for direction in ("auto", "push"):
                print(kind, src, direction, flush=True)
                got, st = grus.bfs(g, src, direction=direction)
                assert (got == want).all()
                assert st.iterations == int(want[hit].max()) + 1
                assert st.vertices_reached == hit.sum()
                assert st.edges_reached == deg[hit].sum()


def test_thin_levels_without_cooperative_grid(ctx, oracle):
    # under a CU mask only the single workgroup runs; wider levels are launched
    off, col = build("grid_wide")
    h = oracle.CSR(off, col, None)
    want = oracle.bfs(h, 450 * 1100 + 500)
    c = grus.Context(0)
    try:
        c.set_cu_limit(64)
        with grus.Graph.from_csr(c, off, col, symmetric=True) as g:
            got, st = grus.bfs(g, 450 * 1100 + 500)
            assert (got == want).all()
            assert st.iterations == int(want.max()) + 1
    finally:
        c.close()
