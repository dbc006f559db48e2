"""The wave's 64-way search, its steps run on the host over offsets that are a
formula: tables of up to 2^32 entries, the offsets of the largest graphs."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "device.hpp"
#include <cstdio>

// entry i of a table of n: i / 3 rows of one length (empty rows between)
static uint64_t entry(uint64_t i) { return i / 3 * 2; }

static uint64_t search(uint64_t n, uint64_t key, int *steps) {
  mgg::WaveSearch w{0, n};
  for (;; ++*steps) {
    uint32_t c = 0;
    for (uint32_t l = 0; l < mgg::WAVE; l++) c += w.probe(l) < w.hi && entry(w.probe(l)) <= key;
    if (w.advance(c)) return w.lo;
    if (w.lo > w.hi || *steps > 10) return ~0ull;
  }
}

static uint64_t want(uint64_t n, uint64_t key) {
  const uint64_t i = (key / 2 + 1) * 3;  // the first entry above key
  return i < n ? i : n;
}

int main() {
  const uint64_t sizes[] = {1, 2, 3, 63, 64, 65, 127, 4095, 4096, 4097, 262145, 1ull << 24,
                            (1ull << 31) + 5, (1ull << 32) - 65, (1ull << 32) - 64,
                            (1ull << 32) - 63, (1ull << 32) - 1, 1ull << 32};
  for (uint64_t n : sizes) {
    const uint64_t last = entry(n - 1);
    const uint64_t keys[] = {0, 1, 2, 3, last / 3, last / 2, last - (last > 0), last, last + 9};
    for (uint64_t key : keys) {
      int steps = 0;
      if (search(n, key, &steps) != want(n, key) || steps > 6) {
        printf("n %llu key %llu\n", (unsigned long long)n, (unsigned long long)key);
        return 1;
      }
    }
  }
  return 0;
}
"""


def test_search_over_offsets(tmp_path):
    src, exe = tmp_path / "search.hip", tmp_path / "search"
    src.write_text(PROGRAM)
    subprocess.check_call(["/opt/rocm/bin/hipcc", "-O1", "-std=c++17", "--cuda-host-only",
                           "-I" + os.path.join(ROOT, "grus_framework_amd", "csrc"),
                           str(src), "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
