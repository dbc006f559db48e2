// bfs_thin.hpp -- top-down levels of low-degree graphs run on the device.
//
// Grids, meshes and road networks have thousands of levels of a few hundred
// to a few thousand vertices.  Launched level by level from the host such a
// level costs ~18 us of kernel and ~27 us of launches and read-back, whatever
// it holds.  Here one launch runs level after level while the frontier stays
// thin; what bounds a level is the latency of one dependent chain: the row
// load, the claim, the barrier.
//
// Rows come padded (D = 4, 8 or 16 columns per vertex, GRUS_NO_VERTEX in
// unused slots; graphs of maximum degree <= 16), so a vertex's row is one or
// a few 16-byte loads with no offset lookup before them, and the row of the
// vertex a thread expands next is requested before the barrier (grid 1300 x
// 1700: 3.9 -> 3.1 us a level, with the barrier polled by a wave of its own).
// Per call, launched level by level / thin: grid 64 x 64 1.1 / 0.2 ms, 300 x
// 300 3.2 / 1.1 ms, 1300 x 1700 51 / 7.5 ms, 4096 x 4096 268 / 28 ms.  A workgroup keeps
// the vertices it discovers in LDS and expands them itself in the next level;
// what exceeds its share goes to the global queue, which the next level deals
// round-robin over all workgroups.
//
//   k_thin<T, true>   one workgroup, barriers within the workgroup only
//   k_thin<T, false>  a cooperative grid.  Barrier and level sums are one
//                     64-bit flag per workgroup (level tag, new vertices,
//                     queued vertices), stored once and polled by one wave of
//                     every workgroup, a lane per flag: no atomic is shared
//
// What crosses workgroups inside a launch (the visited bits, the queue, the
// flags) is read and written with device-scope atomics; levels are
// plain stores that nobody reads before the kernel ends.  Plain reads of the
// visited bits may be stale-clear, which costs a claim that fails.  Every
// wait is bounded by a wall-clock limit that raises the abort flag.
#pragma once

#include "persist.hpp"

namespace mgg {
namespace bfs {

struct ThinCtl {
  uint32_t queued[4];  // global queue reservations of step s, in slot s & 3
  uint32_t abort, status;
  uint32_t levels, nf, cur, prev_nf;
  unsigned long long mf, v_add, e_add;
};

struct ThinParams {
  const uint4 *pad;  // pad_q uint4 per vertex
  uint32_t pad_q;
  const uint64_t *off;
  uint32_t *q0, *q1;  // queues; the frontier is in q[cur]
  uint32_t cur, nf;
  uint64_t mf;  // out-edges of that frontier
  uint32_t lo, hi;  // leave when a frontier has fewer (but some) or more vertices
  uint32_t max_levels;
  uint32_t level;
  uint32_t tag;               // of the launch's first level; never used before
  unsigned long long *flags;  // [2][THIN_MAX_G], by level parity
  uint32_t *label;
  uint64_t *visited;
  ThinCtl *ctl;
  uint64_t timeout;
};

// columns of every row, padded to D
__global__ __launch_bounds__(BLOCK) void k_pad_cols(CsrView g, uint32_t D, uint32_t *pad) {
  const uint64_t stride = (uint64_t)gridDim.x * BLOCK;
  for (uint64_t i = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; i < g.V * D; i += stride) {
    const uint64_t v = i / D, e = g.off[v] + i % D;
    pad[i] = e < g.off[v + 1] ? edge_col(g, e) : GRUS_NO_VERTEX;
  }
}

// a workgroup's flag: tag | new vertices | those of them queued.  A workgroup
// expands at most GRID_HI frontier vertices of 16 columns, and the sums of 64
// workgroups stay below the same 20 bits (GRID_HI * 16 = 2^18).
constexpr int THIN_TAG = 40, THIN_NF = 20;
constexpr uint32_t THIN_MAX_G = WAVE;

// threads of a launch: T that expand, and in a grid one more wave that only
// waits at the barrier (its polls do not queue behind the rows requested ahead)
constexpr int thin_threads(int T, bool solo) { return solo ? T : T + WAVE; }

template <int T, bool kSolo>
__global__ __launch_bounds__((thin_threads(T, kSolo))) void k_thin(ThinParams p) {
  constexpr uint32_t TT = thin_threads(T, kSolo);
  // a workgroup's next vertices: the first KEEP stay, the rest is queued
  constexpr uint32_t CAP = kSolo ? 4096 : 2048, KEEP = kSolo ? 4096 : T;
  __shared__ uint32_t s_v[2][CAP];
  __shared__ uint32_t s_n[2], s_base, s_abort;
  __shared__ unsigned long long s_word;
  ThinCtl *c = p.ctl;
  const uint32_t t = threadIdx.x, G = gridDim.x;
  uint32_t *q[2] = {p.q0, p.q1};
  uint32_t cur = p.cur, nf = p.nf, prev = 0, lv = 0, n_loc = 0, n_glob = p.nf, b = 0;
  uint64_t v_add = 0, edges = 0;  // edges: out-edges of the vertices this thread expanded
  bool ok = true;
  // The first four columns of the vertex this thread expands first in the
  // next level, and the visited words of those: requested before the barrier,
  // so that their latency passes beside the barrier's.
  uint4 px = make_uint4(0, 0, 0, 0);
  uint64_t pw[4] = {0, 0, 0, 0};
  auto words = [&](const uint4 &x, uint64_t *w) {
    const uint32_t d[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
    for (int j = 0; j < 4; j++) w[j] = d[j] != GRUS_NO_VERTEX ? p.visited[d[j] >> 6] : 0ull;
  };
  auto ahead = [&](const uint32_t *next) {
    if (t < n_loc) {
      px = p.pad[(uint64_t)next[t] * p.pad_q];
      words(px, pw);
    }
  };
  if (t < 2) s_n[t] = 0;
  __syncthreads();
  while (nf >= p.lo && nf <= p.hi && lv < p.max_levels) {
    uint32_t *next = s_v[b ^ 1], *count = &s_n[b ^ 1];
    uint32_t *gcount = &c->queued[lv & 3], *gq = q[cur ^ 1];
    // claims of four columns in flight together, then their outcomes
    auto claim = [&](const uint4 &x, const uint64_t *w) {
      const uint32_t d[4] = {x.x, x.y, x.z, x.w};
      unsigned long long old[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const unsigned long long bit = 1ull << (d[j] & 63);
        const bool in = d[j] != GRUS_NO_VERTEX;
        edges += in;
        old[j] = (!in || (w[j] & bit))
                     ? bit
                     : atomicOr((unsigned long long *)&p.visited[d[j] >> 6], bit);
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        if (old[j] & (1ull << (d[j] & 63))) continue;
        p.label[d[j]] = p.level + lv + 1;
        const uint32_t s = atomicAdd(count, 1u);
        if (s < CAP) next[s] = d[j];
        else st_agent(&gq[atomicAdd(gcount, 1u)], d[j]);  // LDS full: straight to the queue
      }
    };
    const uint32_t mine = n_loc + (n_glob > blockIdx.x ? (n_glob - blockIdx.x - 1) / G + 1 : 0);
    for (uint32_t i = t; t < T && i < mine; i += T) {
      const bool ready = i < T;  // (i == t) its first columns were requested before the barrier
      const uint32_t v = i < n_loc ? s_v[b][i] : ld_agent(&q[cur][(i - n_loc) * G + blockIdx.x]);
      for (uint32_t g = 0; g < p.pad_q; g++) {
        if (g == 0 && ready && i < n_loc) {
          claim(px, pw);
        } else {
          const uint4 x = p.pad[(uint64_t)v * p.pad_q + g];
          uint64_t w[4];
          words(x, w);
          claim(x, w);
        }
      }
    }
    __syncthreads();
    const uint32_t n = *count;
    n_loc = n < KEEP ? n : KEEP;
    const uint32_t extra = (n < CAP ? n : CAP) - n_loc;
    prev = nf;
    if (kSolo) {
      if (n > CAP) __builtin_amdgcn_s_waitcnt(0);
      n_glob = n > CAP ? n - CAP : 0;
      nf = n;
      if (t == 0) s_n[b] = 0;
      ahead(next);
    } else {
      if (extra) {
        if (t == 0) s_base = atomicAdd(gcount, extra);
        __syncthreads();
        for (uint32_t i = t; i < extra; i += TT) st_agent(&gq[s_base + i], next[KEEP + i]);
      }
      if (n > KEEP) {  // the queued entries are in place before this workgroup arrives
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
      }
      if (t < T) {
        ahead(next);
      } else {
        const uint32_t l = t - T;
        // arrive: this workgroup's flag; then wait until every workgroup's
        // flag carries the level's tag (lane l polls workgroup l)
        unsigned long long *flags = p.flags + (lv & 1) * THIN_MAX_G;
        const uint64_t tag = (uint64_t)(p.tag + lv) << THIN_TAG;
        if (l == 0) {
          s_n[b] = 0;
          // every workgroup has left step lv - 2, the last to add to this
          // slot, and the polls below wait for this store, so it is done
          // before any workgroup enters step lv + 2
          if (blockIdx.x == 0) st_agent(&c->queued[(lv + 2) & 3], 0);
          __hip_atomic_store(&flags[blockIdx.x], tag | ((uint64_t)n << THIN_NF) | (n - n_loc),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        const uint64_t t0 = wall_clock64();
        uint32_t a = 0;
        uint64_t x = tag;
        for (uint32_t poll = 1;; poll++) {
          if (l < G) x = __hip_atomic_load(&flags[l], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          if (!__ballot((x >> THIN_TAG) != (tag >> THIN_TAG))) break;
          if (poll % 64 == 0) {  // (uniform in the wave)
            a = ld_agent(&c->abort);
            if (!a && wall_clock64() - t0 > p.timeout) {
              if (l == 0) st_agent(&c->abort, 1);
              a = 1;
            }
            if (__ballot(a)) {
              a = 1;
              break;
            }
          }
          __builtin_amdgcn_s_sleep(1);
        }
        const unsigned long long sum = wave_sum((unsigned long long)(x & ((1ull << THIN_TAG) - 1)));
        if (l == 0) {
          s_word = sum;
          s_abort = a;
        }
      }
      __syncthreads();
      if (s_abort) {
        ok = false;
        break;
      }
      nf = (uint32_t)(s_word >> THIN_NF);
      n_glob = (uint32_t)(s_word & ((1ull << THIN_NF) - 1));
    }
    __syncthreads();  // s_word, s_n read before the next level changes them
    v_add += nf;
    b ^= 1;
    cur ^= 1;
    lv++;
  }
  // hand the frontier back in q[cur], behind what is queued there already,
  // with its out-degree sum
  uint64_t mf = 0;
  if (ok && nf && lv) {
    uint32_t *gcount = &c->queued[(lv - 1) & 3];
    for (uint64_t i = (uint64_t)blockIdx.x * TT + t; i < n_glob; i += (uint64_t)G * TT) {
      const uint32_t v = ld_agent(&q[cur][i]);
      mf += p.off[v + 1] - p.off[v];
    }
    if (n_loc) {
      if (t == 0) s_base = kSolo ? n_glob : atomicAdd(gcount, n_loc);
      __syncthreads();
      for (uint32_t i = t; i < n_loc; i += TT) {
        const uint32_t v = s_v[b][i];
        q[cur][s_base + i] = v;
        mf += p.off[v + 1] - p.off[v];
      }
    }
  }
  block_add_u64(mf, &c->mf);
  __syncthreads();  // block_add_u64's scratch is used twice
  block_add_u64(edges, &c->e_add);
  if (blockIdx.x == 0 && t == 0) {
    c->levels = lv;
    c->nf = nf;
    c->cur = cur;
    c->prev_nf = prev;
    c->v_add = v_add;
    c->status = ok ? 0u : 1u;
  }
}

}  // namespace bfs
}  // namespace mgg
