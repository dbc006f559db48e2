// device.hpp -- wave64 intrinsics and bitmap frontier primitives for gfx950.
//
// atomicAggInc (reference include/intrinsics.cuh:96-103) aggregates one
// atomicAdd per 32-lane coalesced group through cooperative_groups; here the
// same slot allocation is a 64-lane ballot + popcount + mbcnt, one atomic
// per wave, with the leader's base broadcast by a lane shuffle.
#pragma once

#include "common.hpp"

namespace mgg {

__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }

// XCD-aware workgroup order.  Workgroups are dispatched round-robin over
// the XCDs, so block b runs on XCD b % NXCD.  Giving XCD x the contiguous
// item range [x*per, (x+1)*per) keeps the working set of neighbouring items
// in that XCD's own L2 instead of spreading it over all eight.  gridDim.x
// must be a multiple of NXCD; the map is a bijection on [0, gridDim.x).
__device__ __forceinline__ uint64_t xcd_block() {
  const uint64_t per = gridDim.x / NXCD;
  return (uint64_t)(blockIdx.x % NXCD) * per + blockIdx.x / NXCD;
}

// number of set bits of m in lanes below this one
__device__ __forceinline__ uint32_t lane_rank(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Wave-aggregated append: every active lane of the wave must call it.
// Returns the slot for lanes with pred set, UINT32_MAX otherwise.
__device__ __forceinline__ uint32_t wave_append(uint32_t *count, bool pred) {
  uint64_t m = __ballot(pred);
  if (m == 0) return 0xFFFFFFFFu;
  int leader = __ffsll((unsigned long long)m) - 1;
  uint32_t base = 0;
  if ((int)lane_id() == leader) base = atomicAdd(count, (uint32_t)__popcll(m));
  base = __shfl(base, leader);
  return pred ? base + lane_rank(m) : 0xFFFFFFFFu;
}

// Workgroup-aggregated append: every thread of the workgroup must call it
// (block-uniform control flow).  One atomic per workgroup; lanes get their
// slot in wave order, lane order within a wave.  `lds` holds >= waves + 1
// u32 of shared scratch.  Returns UINT32_MAX for threads with pred unset.
__device__ __forceinline__ uint32_t block_append(uint32_t *count, bool pred, uint32_t *lds) {
  const uint32_t nwaves = blockDim.x / WAVE;
  const uint32_t wid = threadIdx.x / WAVE;
  uint64_t m = __ballot(pred);
  if (lane_id() == 0) lds[wid] = (uint32_t)__popcll(m);
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t s = 0;
    for (uint32_t i = 0; i < nwaves; i++) {
      uint32_t c = lds[i];
      lds[i] = s;
      s += c;
    }
    lds[nwaves] = s ? atomicAdd(count, s) : 0u;
  }
  __syncthreads();
  uint32_t slot = lds[nwaves] + lds[wid] + lane_rank(m);
  __syncthreads();  // lds reusable by the next call
  return pred ? slot : 0xFFFFFFFFu;
}

// Reserves n slots per thread at *count with one atomic per workgroup and
// returns the thread's first slot (a workgroup's slots are contiguous, in
// thread order).  Every thread of the workgroup must call it; lds holds
// blockDim.x / WAVE + 1 entries.
__device__ __forceinline__ uint32_t block_reserve(uint32_t *count, uint32_t n, uint32_t *lds) {
  const uint32_t nwaves = blockDim.x / WAVE;
  const uint32_t wid = threadIdx.x / WAVE;
  uint32_t x = n;  // inclusive wave scan
#pragma unroll
  for (int o = 1; o < WAVE; o <<= 1) {
    const uint32_t y = __shfl_up(x, o);
    if ((int)lane_id() >= o) x += y;
  }
  if (lane_id() == WAVE - 1) lds[wid] = x;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t s = 0;
    for (uint32_t i = 0; i < nwaves; i++) {
      const uint32_t c = lds[i];
      lds[i] = s;
      s += c;
    }
    lds[nwaves] = s ? atomicAdd(count, s) : 0u;
  }
  __syncthreads();
  const uint32_t slot = lds[nwaves] + lds[wid] + (x - n);
  __syncthreads();  // lds reusable by the next call
  return slot;
}

template <class T>
__device__ __forceinline__ T wave_sum(T x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
  return x;
}

// Adds every thread's two numbers up, with one atomic pair per workgroup
// (skipped where zero).  Every thread of the workgroup must call it, at the
// end of the kernel; blockDim.x <= 1024.  The sums go into the context's
// control block, to 32 slots of 64 bytes by turns (16 cache lines), and
// publish_ctl puts them together: atomics on one line run one after the other,
// 12 ns each, and the workgroups of a launch end together (RMAT scale 20,
// digest of 1 M entries: 2048 workgroups 52 us, 256 of them 9).  `field` is
// the first of two words of a slot: CTL_STEP for StepCounters' next_count and
// next_edges, CTL_REACHED for words 40 and 41, CTL_DIGEST for words 48 and 49.
constexpr uint32_t CTL_SPREAD = 128;  // first word; 8 words a slot
constexpr uint32_t CTL_LINES = 32;
constexpr uint32_t CTL_STEP = 0, CTL_REACHED = 2, CTL_DIGEST = 4;
__device__ __forceinline__ void block_add_spread(unsigned long long a, unsigned long long b,
                                                 void *ctl, uint32_t field) {
  __shared__ unsigned long long s_a[1024 / WAVE], s_b[1024 / WAVE];
  a = wave_sum(a);
  b = wave_sum(b);
  const uint32_t wid = threadIdx.x / WAVE, nwaves = blockDim.x / WAVE;
  if (lane_id() == 0) {
    s_a[wid] = a;
    s_b[wid] = b;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t w = 1; w < nwaves; w++) {
      a += s_a[w];
      b += s_b[w];
    }
    auto *line = reinterpret_cast<unsigned long long *>(ctl) + CTL_SPREAD +
                 8 * (blockIdx.x % CTL_LINES) + field;
    if (a) atomicAdd(&line[0], a);
    if (b) atomicAdd(&line[1], b);
  }
}

// One 64-bit sum, to one address (skipped when zero).
__device__ __forceinline__ void block_add_u64(unsigned long long sum, unsigned long long *out) {
  __shared__ unsigned long long s_s[1024 / WAVE];
  sum = wave_sum(sum);
  const uint32_t wid = threadIdx.x / WAVE, nwaves = blockDim.x / WAVE;
  if (lane_id() == 0) s_s[wid] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t w = 1; w < nwaves; w++) sum += s_s[w];
    if (sum) atomicAdd(out, sum);
  }
}

__device__ __forceinline__ bool bm_test(const uint64_t *bm, uint32_t v) {
  return (bm[v >> 6] >> (v & 63)) & 1ull;
}

// Sets bit v; true when this call flipped it from 0 to 1.
__device__ __forceinline__ bool bm_claim(uint64_t *bm, uint32_t v) {
  unsigned long long bit = 1ull << (v & 63);
  unsigned long long old = atomicOr((unsigned long long *)&bm[v >> 6], bit);
  return (old & bit) == 0;
}

__device__ __forceinline__ uint32_t atomic_min_u32(uint32_t *p, uint32_t v) {
  return atomicMin(p, v);
}

// 64-bit splitmix64 output function (Steele, Lea, Flood 2014).
__host__ __device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

__device__ __forceinline__ uint64_t readlane_u64(uint64_t x, uint32_t i) {
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)x, i);
  const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(x >> 32), i);
  return ((uint64_t)hi << 32) | lo;
}

// One search step of a wave over the indexes [lo, hi): WAVE probes at equal
// distances.  In 64 bits: a graph may have 2^32 - 1 vertices, and one offset
// more.
struct WaveSearch {
  uint64_t lo, hi;
  __host__ __device__ uint64_t step() const { return (hi - lo + WAVE - 1) / WAVE; }
  __host__ __device__ uint64_t probe(uint32_t lane) const { return lo + lane * step(); }
  // c: the probes below hi that hold at most the key, which are the first ones;
  // true when lo is the result
  __host__ __device__ bool advance(uint32_t c) {
    const uint64_t s = step();
    if (s <= 1 || c == 0) {
      lo += c;
      return true;
    }
    const uint64_t end = lo + c * s;
    lo += (c - 1) * s + 1;
    if (end < hi) hi = end;
    return false;
  }
};

// First index in [lo, hi) whose entry is above key, or hi, by a whole wave
// (every lane calls it with the same arguments; a is non-decreasing): a queue
// of 4096 takes two dependent loads and one of 2^24 four, where one thread's
// binary search took 12 and 24.
__device__ __forceinline__ uint64_t wave_upper_bound_u64(const uint64_t *a, uint64_t lo,
                                                         uint64_t hi, uint64_t key) {
  WaveSearch w{lo, hi};
  for (;;) {
    const uint64_t i = w.probe(lane_id());
    if (w.advance((uint32_t)__popcll(__ballot(i < w.hi && a[i] <= key)))) return w.lo;
  }
}

// f(e, u, first) for the edges [e0, e1) of a wave (e0 and e1 the same in every
// lane), a lane per edge, 64 consecutive edges at a time: u is e's row, first
// whether e begins it.  Rows are walked 64 row ends a read, in scalar
// registers, so a row costs about ten instructions and short rows share the
// wave; a wave per row left most lanes idle (RMAT scale 24, 16.7 M rows of 31
// edges on average, half of them empty: a pass that writes 4 bytes an edge
// took 68 ms, with this 2.2).
template <class F>
__device__ __forceinline__ void wave_edge_rows(const uint64_t *off, uint64_t V, uint64_t e0,
                                               uint64_t e1, F &&f) {
  if (e0 >= e1) return;
  const uint32_t lane = lane_id();
  uint64_t r = wave_upper_bound_u64(off, 0, V + 1, e0) - 1, rb = r;
  uint64_t ends = off[rb + 1 + lane < V ? rb + 1 + lane : V];  // of rows rb .. rb + 63
  uint64_t row_beg = off[r];
  for (uint64_t base = e0; base < e1; base += WAVE) {
    const uint32_t n = (uint32_t)(e1 - base < WAVE ? e1 - base : WAVE);
    uint32_t my_r = 0, pos = 0;
    bool first = false;
    while (pos < n) {
      const uint64_t row_end = readlane_u64(ends, (uint32_t)(r - rb));
      if (lane >= pos) {
        my_r = (uint32_t)r;
        first = base + lane == row_beg;
      }
      pos = row_end - base < n ? (uint32_t)(row_end - base) : n;
      if (base + pos != row_end || row_end >= e1) break;
      row_beg = row_end;
      uint64_t later;  // the rows read that end past row_end
      while ((later = __ballot(ends > row_end)) == 0) {  // (there is one: e1 <= off[V])
        rb += WAVE;
        ends = off[rb + 1 + lane < V ? rb + 1 + lane : V];
      }
      r = rb + (uint32_t)__ffsll((unsigned long long)later) - 1;
    }
    if (lane < n) f(base + lane, my_r, first);
  }
}

// The same over all E edges by a whole launch, 1024 edges a wave at a time:
// a share of the edges in one piece left the waves that hold the short rows
// last (RMAT scale 24, 16384 waves: 15 ms).
template <class F>
__device__ __forceinline__ void grid_edge_rows(const uint64_t *off, uint64_t V, uint64_t E, F &&f) {
  const uint32_t per_wg = blockDim.x / WAVE;
  const uint64_t wave =
      blockIdx.x * (uint64_t)per_wg + __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const uint64_t nw = (uint64_t)gridDim.x * per_wg;
  const uint64_t per = E / nw < 1024 ? (E / nw + WAVE) / WAVE * WAVE : 1024;
  for (uint64_t e0 = wave * per; e0 < E; e0 += nw * per)
    wave_edge_rows(off, V, e0, e0 + per < E ? e0 + per : E, f);
}

}  // namespace mgg
