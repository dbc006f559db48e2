// serve_time.hpp -- what the query server learns of how long queries take.
#pragma once

#include <algorithm>
#include <cstdint>

namespace mgg {

// Running mean: plain up to 8 values, then weight 1/8 to the newest (with 1/8
// from the second value on, the first stood for the others for dozens).
struct Mean {
  double ms = 0;
  int n = 0;  // 0: none yet
  void add(double x) {
    n = std::min(n + 1, 8);
    ms += (x - ms) / n;
  }
};

// What runs that makes single queries beside it slower than they are.
struct Slow {
  int running = 0;
  uint64_t begun = 0;
  void begin() { running++, begun++; }
  void end() { running--; }
  uint64_t mark() const { return running ? ~0ull : begun; }
  // nothing ran at the mark, or has begun since
  bool quiet_since(uint64_t mark) const { return mark == begun; }
};

// Time of a single query of a kind.  A query beside a batch takes as long as
// the batch: means of such times made batches of 6 queries look worth starting,
// several side by side (32 SSSP queries at RMAT s24: 264 ms instead of 134 in
// one).  Such times are upper bounds of the query's own, and only the least of
// them stands in until a query has run with nothing slow beside it.  Too low, it
// has the next queries served alone, which tells; too high, it would have a
// batch beside every further query (one worker's first allocations, 300 ms,
// averaged in: bursts of 32 BFS queries at s24 24 ms for good, 15.5 without).
struct SoloTime {
  Mean mean;
  bool quiet = false;  // mean is of queries with nothing slow beside them
  void add(double x, bool beside) {
    if (beside) {
      if (quiet) return;
      mean.ms = mean.n ? std::min(mean.ms, x) : x;
      mean.n = 1;
      return;
    }
    if (!quiet) mean = Mean();
    quiet = true;
    mean.add(x);
  }
};

}  // namespace mgg
