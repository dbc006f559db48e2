"""That the paths the other tests compare with the oracle are the ones that ran:
whole traversals in one launch, thin levels in a few, batch steps over the
in-edges; and that those do not depend on what was called first."""
import numpy as np
import pytest

import grus_framework_amd as grus

pytestmark = pytest.mark.gpu


def csr(V, u, v, weights=None, mirror=True, both=True):
    u, v = np.asarray(u, np.int64), np.asarray(v, np.int64)
    if both:
        u, v = np.minimum(u, v), np.maximum(u, v)
    key = np.unique(u * V + v)
    key = key[key // V != key % V]
    u, v = key // V, key % V
    rng = np.random.default_rng(9)
    w = rng.integers(1, weights + 1, len(key)) if weights else np.ones(len(key), np.int64)
    if both:
        w2 = w if mirror else rng.integers(1, weights + 1, len(key))
        u, v, w = np.r_[u, v], np.r_[v, u], np.r_[w, w2]
    order = np.lexsort((v, u))
    off = np.zeros(V + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(u, minlength=V))
    return off, v[order].astype(np.uint32), w[order].astype(np.uint32) if weights else None


def random_pairs(V, n, seed=1):
    rng = np.random.default_rng(seed)
    return (rng.random(n) ** 2 * V).astype(np.int64), rng.integers(0, V, n)


@pytest.mark.parametrize("V", [40, 1023, 1025, 60001, 262144, 262145])
def test_whole_traversal_launches(ctx, V):
    u, v = random_pairs(V, 6 * V)
    with grus.Graph.from_csr(ctx, *csr(V, u, v), symmetric=True) as g:
        assert g.info.max_degree > 16
        st = grus.bfs(g, int(g.info.max_degree_vertex))[1]
        assert (st.kernel_launches == 1) == (V <= 262144)
        assert grus.bfs(g, int(g.info.max_degree_vertex), direction="push")[1].kernel_launches > 1


@pytest.mark.parametrize("rows,cols", [(300, 300), (1500, 1700)])  # one workgroup, a grid of them
def test_thin_level_launches(ctx, rows, cols):
    with grus.Graph.grid(ctx, rows, cols) as g:
        st = grus.bfs(g, rows // 2 * cols + cols // 2)[1]
        # launched one by one, a level takes two launches and more
        assert st.kernel_launches < st.iterations // 10


@pytest.mark.parametrize("mirror", [True, False])
def test_batch_steps_over_in_edges(ctx, mirror):
    u, v = random_pairs(3000, 30000)
    with grus.Graph.from_csr(ctx, *csr(3000, u, v, 90, mirror), symmetric=True) as g:
        st = grus.sssp_multi(g, np.arange(64))[1]
        assert (st.pull_iterations > 0) == mirror
        assert st.pull_iterations < st.iterations
        assert grus.sssp_multi(g, [1, 2, 3])[1].pull_iterations == 0  # two lanes: pushed
        assert grus.bfs_multi(g, np.arange(64))[1].pull_iterations > 0


def test_batches_do_not_depend_on_what_was_called_first(ctx, oracle):
    u, v = random_pairs(2500, 40000)
    data = csr(2500, u, v, 60, both=False)
    srcs = np.arange(100)
    want = np.array([oracle.sssp(oracle.CSR(*data), int(s)) for s in srcs])
    with grus.Graph.from_csr(ctx, *data) as g:
        got, st = grus.sssp_multi(g, srcs)  # no in-edges are built for it
        assert st.pull_iterations == 0 and (got == want).all()
        grus.bfs(g, 0)  # builds them
        got, st = grus.sssp_multi(g, srcs)
        assert st.pull_iterations > 0 and (got == want).all()
