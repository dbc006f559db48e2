"""What the query server learns of a single query's time, compiled for the host:
a worker's slow first query and queries beside a batch stand in at most until a
query has run by itself, and never for more than the least of them."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "serve_time.hpp"

int main() {
  using namespace mgg;
  {  // first queries side by side: one waited for another's allocations
    SoloTime t;
    const double ms[] = {296, 1.5, 297, 1.8};
    for (double x : ms) t.add(x, true);
    t.add(14, true);  // beside a batch
    if (t.mean.n != 1 || t.mean.ms != 1.5 || t.quiet) return 1;
    for (int i = 0; i < 8; i++) t.add(2, false);
    t.add(300, true);
    t.add(0.5, true);
    if (!t.quiet || t.mean.ms != 2) return 2;
    t.add(10, false);
    if (t.mean.n != 8 || t.mean.ms != 3) return 3;
  }
  {  // a first query in its stead is dropped by the first quiet one
    SoloTime t;
    t.add(0.1, true);
    t.add(4, false);
    if (t.mean.n != 1 || t.mean.ms != 4) return 4;
  }
  {
    Slow s;
    uint64_t m = s.mark();
    if (!s.quiet_since(m)) return 5;
    s.begin();
    if (s.quiet_since(m)) return 6;
    uint64_t during = s.mark();
    s.end();
    if (s.quiet_since(during) || s.quiet_since(m)) return 7;  // it ran beside both
    if (!s.quiet_since(s.mark())) return 8;
    s.begin();
    s.begin();
    s.end();
    if (s.quiet_since(s.mark())) return 9;  // one is still running
    s.end();
    if (!s.quiet_since(s.mark())) return 10;
  }
  return 0;
}
"""


def test_learned_times(tmp_path):
    src, exe = tmp_path / "times.cpp", tmp_path / "times"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-O1",
                           "-I" + os.path.join(ROOT, "grus_framework_amd", "csrc"),
                           str(src), "-o", str(exe)])
    assert subprocess.run([str(exe)]).returncode == 0
