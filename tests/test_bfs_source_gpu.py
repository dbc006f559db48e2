"""The first launch counts the source's edges: sources with none, with as many
as one workgroup expands, with one more, and with most of the graph's; the
digest of a result, against its definition, at sizes around a thread's share."""
import numpy as np
import pytest

import grus_framework_amd as grus

pytestmark = pytest.mark.gpu

INF = grus.INFINIT


def stars(V, degs, more):
    """Hub i (vertex i) with degs[i] leaves of its own, the leaves in a chain
    and joined by `more` edges: symmetric."""
    leaf = len(degs)
    pairs = []
    for i, d in enumerate(degs):
        pairs.append(np.c_[np.full(d, i), leaf + np.arange(d)])
        leaf += d
    assert leaf <= V
    p = np.concatenate(pairs)
    p = np.concatenate([p, np.c_[len(degs) + np.arange(leaf - len(degs) - 1),
                                 len(degs) + 1 + np.arange(leaf - len(degs) - 1)]])
    p = np.concatenate([p, np.random.default_rng(1).integers(len(degs), leaf, (more, 2))])
    s, d = np.r_[p[:, 0], p[:, 1]], np.r_[p[:, 1], p[:, 0]]
    order = np.lexsort((d, s))
    off = np.zeros(V + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(s, minlength=V))
    return off, d[order].astype(np.uint32)


@pytest.mark.parametrize("V", [40000, (1 << 18) + 70])  # one launch / level by level
@pytest.mark.parametrize("more", [0, 100000])  # the largest star is a fifth / a thirtieth of it
@pytest.mark.parametrize("direction", ["auto", "push", "pull"])
def test_source_degrees(ctx, oracle, V, direction, more):
    off, col = stars(V, [1, 4095, 4096, 4097, 9000], more)
    h = oracle.CSR(off, col, None)
    with grus.Graph.from_csr(ctx, off, col, symmetric=True) as g:
        for src in (0, 1, 2, 3, 4, 5, 700, V - 1):  # the last one is isolated
            want = oracle.bfs(h, src)
            got, st = grus.bfs(g, src, direction=direction)
            assert (got == want).all(), src
            assert st.vertices_reached == (want != INF).sum()
            assert st.edges_reached == np.diff(off.astype(np.int64))[want != INF].sum()


def mix64(z):
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 85), (16, 16), (1, 257), (512, 512),
                                       (1024, 2047), (1024, 2048), (1449, 1448)])
def test_digest(ctx, rows, cols):
    with grus.Graph.grid(ctx, rows, cols) as g:
        for _ in range(2):
            lv, _ = grus.bfs(g, 0)
            v = np.arange(rows * cols, dtype=np.uint64)
            with np.errstate(over="ignore"):
                want = mix64((v << np.uint64(32)) | lv).sum(dtype=np.uint64)
            assert g.digest() == ((lv != INF).sum(), want)
