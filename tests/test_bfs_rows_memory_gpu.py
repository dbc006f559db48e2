"""The padded rows of low-degree graphs are optional: traversals run without
them where the device lacks the memory, and a server's workers share one copy."""
import ctypes as C

import numpy as np
import pytest

import grus_framework_amd as grus

pytestmark = pytest.mark.gpu

GB = 1 << 30


class Ballast:
    """Device memory taken until about `leave` bytes are free."""

    def __init__(self, leave):
        self.hip, self.held = C.CDLL("libamdhip64.so"), []
        for size in (64 * GB, 16 * GB, 4 * GB, GB, GB // 4, GB // 16):
            while self.free() > leave + size:
                p = C.c_void_p()
                if self.hip.hipMalloc(C.byref(p), C.c_size_t(size)) != 0:
                    self.hip.hipGetLastError()
                    break
                self.held.append(p)

    def free(self):
        free, total = C.c_size_t(), C.c_size_t()
        assert self.hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    def release(self):
        for p in self.held:
            self.hip.hipFree(p)
        self.held = []


def stars(n, leaves):
    """n stars of the given number of leaves, centre first."""
    V = n * (leaves + 1)
    centre = np.arange(n, dtype=np.uint32) * np.uint32(leaves + 1)
    deg = np.ones(V, np.uint64)
    deg[centre] = leaves
    off = np.zeros(V + 1, np.uint64)
    off[1:] = np.cumsum(deg)
    col = np.empty((n, 2 * leaves), np.uint32)
    col[:, :leaves] = centre[:, None] + np.arange(1, leaves + 1, dtype=np.uint32)
    col[:, leaves:] = centre[:, None]
    return off, col.ravel()


def test_traversal_without_room_for_the_rows(ctx):
    off, col = stars(1 << 20, 15)  # 2^24 vertices: rows padded to 16 columns take 1 GB
    with grus.Graph.from_csr(ctx, off, col, symmetric=True) as g:
        grus.bfs(g, 0, direction="pull", copy=False)  # the workspace, without the rows
        ballast = Ballast(GB * 7 // 8)  # (room for everything else)
        try:
            assert ballast.free() < GB
            for src in (0, 16 * 70001 + 3):
                got, st = grus.bfs(g, src)
                assert st.vertices_reached == 16 and st.iterations == (2 if src == 0 else 3)
                first = src // 16 * 16
                want = np.full(16, 1 if src == 0 else 2, np.uint32)
                want[0] = 0 if src == 0 else 1
                want[src - first] = 0
                assert (got[first:first + 16] == want).all()
                assert (got != grus.INFINIT).sum() == 16
        finally:
            ballast.release()


def test_workers_share_the_rows():
    c = grus.Context(0)
    try:
        with grus.Graph.grid(c, 1500, 1500) as g:
            before = c.device_memory()[0]
            grus.bfs(g, 0, direction="pull", copy=False)
            workspace = c.device_memory()[0] - before  # of one traversal, without the rows
            with grus.Server(g, solo_max=1000) as server:
                held = c.device_memory()[0]
                for s in range(64):
                    server.submit(grus.Q_BFS, s)
                for _ in range(64):
                    assert server.poll(timeout_ms=30000).status == 0
                grown = c.device_memory()[0] - held
            rows = 16 * g.V
            assert grown <= 4 * workspace + rows // 2  # four workers
    finally:
        c.close()
