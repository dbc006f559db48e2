"""Batch steps commit their bits in spans of vertices: sizes around a
workgroup's span, at both workgroup sizes and past one item a thread."""
import numpy as np
import pytest

import grus_framework_amd as grus

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [255, 256, 257, 1 << 15, (1 << 15) + 1, (1 << 19) + 1023,
                               (1 << 20) + 1])
def test_spans(ctx, oracle, V):
    rng = np.random.default_rng(V)
    key = np.unique(np.r_[rng.integers(0, V, 2 * V) * V + rng.integers(0, V, 2 * V),
                          (np.arange(min(V, 70)) + 1) * V - 1])  # edges to the last vertex
    off = np.zeros(V + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(key // V, minlength=V))
    col, w = (key % V).astype(np.uint32), rng.integers(1, 20, len(key)).astype(np.uint32)
    h = oracle.CSR(off, col, w)
    srcs = np.r_[0, V - 1, rng.integers(0, V, 6)]
    with grus.Graph.from_csr(ctx, off, col, w) as g:
        lv, st = grus.bfs_multi(g, srcs)
        d, _ = grus.sssp_multi(g, srcs)
        for i, s in enumerate(srcs):
            assert (lv[i] == oracle.bfs(h, int(s))).all()
            assert (d[i] == oracle.sssp(h, int(s))).all()
