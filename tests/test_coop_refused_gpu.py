"""Traversals of a process that is refused cooperative launches, because another
one holds the device's cooperative queue: levels and distances against the
oracle, by the paths that launch level by level and round by round."""
import os
import subprocess
import sys

import numpy as np
import pytest

import grus_framework_amd as grus

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = r"""
import sys
import numpy as np
import grus_framework_amd as grus
with grus.Context(0) as c:
    with grus.Graph.rmat(c, 14) as g, grus.Graph.grid(c, 90, 70, weights=(1, 50), wseed=4) as grid, \
            grus.Graph.grid(c, 700, 700) as wide:
        out = {}
        for i in range(2):  # refused, and remembered
            out["bfs%d" % i], st = grus.bfs(g, 5)
            out["launches%d" % i] = np.array(st.kernel_launches)
            out["thin%d" % i] = grus.bfs(wide, 350 * 700 + 350)[0]  # thin levels past one workgroup's
            out["sssp%d" % i] = grus.sssp(grid, 11)[0]
np.savez(sys.argv[1], **out)
"""


def test_second_process(oracle, tmp_path):
    with grus.Context(0) as c:
        with grus.Graph.rmat(c, 14) as g, grus.Graph.grid(c, 90, 70, weights=(1, 50), wseed=4) as grid, \
                grus.Graph.grid(c, 700, 700) as wide:
            assert grus.bfs(g, 5)[1].kernel_launches == 1  # this process holds the queue
            want = {"bfs": oracle.bfs(oracle.CSR(*g.csr()[:2], None), 5),
                    "thin": oracle.bfs(oracle.CSR(*wide.csr()[:2], None), 350 * 700 + 350),
                    "sssp": oracle.sssp(oracle.CSR(*grid.csr()), 11)}
            path = str(tmp_path / "out.npz")
            r = subprocess.run([sys.executable, "-c", CHILD, path], cwd=ROOT, timeout=100,
                               capture_output=True, text=True, env=dict(os.environ, GRUS_TRACE="1"))
            assert r.returncode == 0, r.stderr[-2000:]
    got = np.load(path)
    for name, levels in want.items():
        for i in range(2):
            assert (got["%s%d" % (name, i)] == levels).all(), name
    if "cooperative launch refused" in r.stderr:  # (the runtime may serve two processes)
        assert got["launches0"] > 1 and got["launches1"] > 1
        assert r.stderr.count("cooperative launch refused") == 1
    print("refusals:", r.stderr.count("cooperative launch refused"))
