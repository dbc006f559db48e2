"""Whole traversals of deep graphs: thin levels are handed from the one-launch
kernel to the small-levels kernel and wide frontiers back, with a chain's worth
of levels on either side of the hand-over, rows of every mapping at the return,
one workgroup and a grid.  Levels and counts against the oracle; and the
automatic direction takes no longer than the levels pushed by themselves."""
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
    off = np.zeros(V + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(key // V, minlength=V))
    return off, (key % V).astype(np.uint32)


def beads(links, leaves):
    """Stars of the given leaves along a chain: links[i] vertices, then star i."""
    u, v, at, last = [], [], 0, None
    for n, k in zip(links, leaves):
        for x in range(at, at + n):
            if last is not None:
                u.append(last)
                v.append(x)
            last = x
        at += n
        u += [last] * k
        v += list(range(at, at + k))
        # the chain goes on behind the star's last leaf
        last, at = at + k - 1, at + k
    return csr(at, u, v)


def grid(r, c, leaves):
    i = np.arange(r * c).reshape(r, c)
    u = np.concatenate([i[:, :-1].ravel(), i[:-1].ravel(), np.full(leaves, r * c // 2)])
    v = np.concatenate([i[:, 1:].ravel(), i[1:].ravel(), np.arange(r * c, r * c + leaves)])
    return csr(r * c + leaves, u, v)


def ring(n, reach):
    i = np.arange(n)
    return csr(n, np.tile(i, reach), np.concatenate([(i + k) % n for k in range(1, reach + 1)]))


def tails(n, edges, count, length):
    """A directed core and chains hanging off it."""
    rng = np.random.default_rng(1)
    u, v = [rng.integers(0, n, edges)], [rng.integers(0, n, edges)]
    for k in range(count):
        t = np.arange(n + k * length, n + (k + 1) * length)
        u.append(np.r_[rng.integers(0, n), t[:-1]])
        v.append(t)
    return csr(n + count * length, np.concatenate(u), np.concatenate(v), both=False)


GRAPHS = {
    # around the levels that are waited for, and more than one launch of small levels
    "links": lambda: beads([7, 8, 9, 10, 11, 63, 64, 65, 140, 3], [1500] * 10),
    # returns at a row of a wave, a workgroup and the whole grid, and at the ends
    # of what the small levels take (4096 edges)
    "rows": lambda: beads([20] * 9, [30, 513, 4094, 4095, 4096, 8191, 8192, 8193, 20000]),
    "one_workgroup": lambda: beads([300, 12, 9, 30], [40, 300, 17, 60]),
    "small": lambda: beads([9, 10, 40], [17, 17, 17]),
    "grid": lambda: grid(40, 700, 50),
    "ring": lambda: ring(9000, 9),
    "tails": lambda: tails(4000, 40000, 30, 200),
}


@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_levels(ctx, oracle, name):
    off, col = GRAPHS[name]()
    h = oracle.CSR(off, col, None)
    deg = np.diff(off).astype(np.int64)
    V = len(deg)
    assert deg.max() > 16  # not the padded low-degree path
    with grus.Graph.from_csr(ctx, off, col, symmetric=name != "tails") as g:
        for src in (0, V - 1, V // 3, int(np.argmax(deg))):
            want = oracle.bfs(h, src)
            hit = want != INF
            for _ in range(2):  # the second finds the first one's bitmaps and flags
                got, st = grus.bfs(g, src)
                assert (got == want).all(), src
                assert st.iterations == int(want[hit].max()) + 1
                assert st.vertices_reached == hit.sum()
                assert st.edges_reached == deg[hit].sum()
            if name == "grid":  # most levels thin: a few launches, and not one a level
                assert 1 < st.kernel_launches < st.iterations // 5


@pytest.mark.parametrize("name,graph", [("chain", lambda: beads([8000, 8000], [20, 20])),
                                        ("grid", lambda: grid(300, 300, 40)),
                                        ("ring", lambda: ring(20000, 10))])
def test_no_slower_than_pushing(ctx, name, graph):
    with grus.Graph.from_csr(ctx, *graph(), symmetric=True) as g:
        ms = {}
        for d in ("auto", "push"):
            grus.bfs(g, 0, direction=d, copy=False)
            ms[d] = min(grus.bfs(g, 0, direction=d, copy=False)[1].device_ms for _ in range(3))
        # a few launches more, and the last levels pull
        assert ms["auto"] < 1.35 * ms["push"]
