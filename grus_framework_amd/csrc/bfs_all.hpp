// bfs_all.hpp -- a whole direction-optimizing traversal in one launch, for
// graphs whose frontier bitmap fits LDS.
//
// On a graph of up to 2^18 vertices a level is a few microseconds of work and
// ~20 us of launches and read-back when the host runs the level loop.  Here
// one grid runs it, in 4-10 us a level; up to 1024 vertices one workgroup does,
// with no grid barrier.  Per call with the levels copied out, host loop / here:
// RMAT s8 134 / 53 us, s10 145 / 61, s12 166 / 95, s14 214 / 118, s16 198 /
// 126, s18 282 / 218; directed 50 K vertices 253 / 137.  Four words per
// workgroup: 1, 2 and 8 measured within 5% (s14, s16), 16 9% slower (s12).
// Above 2^18 vertices a level's work outweighs its launch.  Workgroup b owns the bitmap words w with w % G == b (64
// vertices each; interleaved, because RMAT's hubs have low ids): it alone
// keeps their visited bits (in LDS), writes their levels and, bottom-up,
// finds their parents.
//   bottom-up: every workgroup copies the whole frontier bitmap to LDS and
//     scans the in-edges of its unvisited vertices against it, so a test
//     costs an LDS read;
//   top-down:  the frontier's vertices are dealt to the workgroups in id order;
//     a wave per vertex (the workgroup for a long row, the whole grid for a
//     huge one, which whoever discovers it lists) claims its neighbours in
//     the shared visited bitmap and sets their bits in the next frontier,
//     which their owner picks up in the next level.
// Three frontier bitmaps rotate: level L reads L % 3, writes (L + 1) % 3, and
// clears (L + 2) % 3, which nobody has read since the barrier before.  The
// direction rule is the host loop's.  Levels end in a grid barrier of one
// flag per workgroup that carries its counts (see bfs_thin.hpp); what crosses
// workgroups moves in device-scope atomics, completed before the flag is
// stored (s_waitcnt).  Every wait is bounded.
#pragma once

#include "persist.hpp"

namespace mgg {
namespace bfs {

constexpr int ALL_T = 1024;
constexpr uint32_t ALL_MAX_G = 256;       // 4 flags per polling lane
constexpr uint64_t ALL_MAX_V = 1ull << 18;  // 32 KB of frontier bitmap
constexpr uint32_t ALL_OWN = 16;          // words per workgroup at most
// rows of 512 edges and more by the workgroup, past 8192 by the grid: by a wave
// each they took s18 600 us (a 25 K-edge row alone), by the workgroup 350
constexpr uint64_t ALL_BIG = 512;         // edges of a row that a whole workgroup scans or expands
constexpr uint64_t ALL_HUGE = 8192;       // out-edges of a row that the whole grid expands
constexpr int ALL_TAG = 40;               // flags: tag | huge rows | vertices, tag | out-edges
constexpr int ALL_NF = 20;
static_assert(ALL_MAX_V < (1ull << ALL_NF), "a frontier's size fits its field");

// A launch ends early after ALL_THIN thin levels in a row, pushes of at most
// thin_nf vertices and thin_mf out-edges: k_small_levels runs those at 2.7 us
// each, and here every one costs the whole grid a bitmap's reads and a barrier
// (4.5 us in one workgroup, 5.7 to 9 in a grid).  What k_small_levels leaves
// comes back here.  Chains, grids and rings with a hub, ms without / with the
// hand-over: 20000 levels 114 / 55, 599 levels 4.9 / 2.8, 10001 levels 96 / 40.
// RMAT never has so many thin levels in a row.
constexpr uint32_t ALL_THIN = 8;

struct AllCtl {
  uint32_t status, levels, pulls, abort;  // levels: of this launch; status 1: aborted
  unsigned long long v_reached, e_reached;
  uint32_t huge[4];  // huge rows listed for the frontier of level L, in slot L % 3
  // left at a thin frontier: its vertices (in the queue, `queued` of them
  // counted there), their out-edges, the unexplored edges, the level before
  uint32_t nf, queued;
  unsigned long long mf, mu;
  uint32_t prev_nf, pad;
};

struct AllParams {
  CsrView out, in;
  const uint32_t *first_in;
  const uint64_t *unreachable;
  uint64_t *visited, *front[3];
  uint32_t *huge[2];  // huge rows of the frontier of level L, in list L % 2
  uint32_t *label;
  uint32_t src, K, W, own;  // own = words per workgroup at most
  // a traversal that goes on: level > 0, its frontier in front[level % 3],
  // visited and levels in place, and the counts as AllCtl has them
  uint32_t level, nf, prev_nf;
  uint64_t mf, mu;
  uint32_t thin_nf;
  uint64_t thin_mf;
  uint32_t *queue;  // of the frontier left (may be huge[0]: a thin frontier lists none)
  double alpha, beta;
  unsigned long long *flags;  // [2 parities][2 counts][ALL_MAX_G]
  uint32_t tag;               // of the first barrier; never used before
  AllCtl *ctl;
  uint64_t timeout;
};

__device__ __forceinline__ uint64_t ld_agent64(const uint64_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent64(uint64_t *p, uint64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ __launch_bounds__(ALL_T) void k_bfs_all(AllParams p) {
  extern __shared__ uint64_t s_mem[];
  uint64_t *s_front = s_mem;           // W words: the frontier, bottom-up
  uint64_t *s_vis = s_front + p.W;     // own words: visited
  uint64_t *s_cur = s_vis + p.own;     // own words: this level's frontier
  __shared__ unsigned long long s_n, s_e, s_tot[2];
  __shared__ uint32_t s_abort, s_nbig, s_nlist, s_wave[ALL_T / WAVE];
  // a workgroup's frontier vertices, top-down (every G-th of at most ALL_OWN *
  // 64 * G), and its long rows, either way
  __shared__ uint32_t s_list[ALL_OWN * 64], s_big[ALL_OWN * 64];
  const uint32_t t = threadIdx.x, lane = lane_id(), wid = t / WAVE, b = blockIdx.x, G = gridDim.x;
  constexpr uint32_t NW = ALL_T / WAVE;
  const uint64_t V = p.out.V;
  const uint32_t mine = p.W > b ? (p.W - b - 1) / G + 1 : 0;  // own words
  // grid barrier number `bar`, adding every thread's counts; false: aborted
  uint32_t bar = 0;
  auto barrier = [&](uint64_t n, uint64_t e, uint64_t *nf, uint64_t *mf) {
    const unsigned long long wn = wave_sum((unsigned long long)n), we = wave_sum((unsigned long long)e);
    if (lane == 0 && wn) {
      atomicAdd(&s_n, wn);
      atomicAdd(&s_e, we);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (G == 1) {
      *nf = s_n;
      *mf = s_e;
      bar++;
      __syncthreads();
      if (t == 0) s_n = s_e = 0;
      __syncthreads();
      return true;
    }
    if (wid == 0) {
      unsigned long long *f0 = p.flags + (bar & 1) * 2 * ALL_MAX_G, *f1 = f0 + ALL_MAX_G;
      const uint64_t tag = p.tag + bar;
      if (lane == 0) {
        __hip_atomic_store(&f0[b], (tag << ALL_TAG) | s_n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&f1[b], (tag << ALL_TAG) | s_e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_n = s_e = 0;
      }
      const uint64_t t0 = wall_clock64();
      uint32_t a = 0;
      uint64_t x[4], y[4];
      for (uint32_t poll = 1;; poll++) {
        bool late = false;
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) {
          const uint32_t i = lane + k * WAVE;
          x[k] = y[k] = tag << ALL_TAG;
          if (i < G) {
            x[k] = ld_agent64((const uint64_t *)&f0[i]);
            y[k] = ld_agent64((const uint64_t *)&f1[i]);
          }
        }
#pragma unroll
        for (uint32_t k = 0; k < 4; k++)
          late = late || (x[k] >> ALL_TAG) != tag || (y[k] >> ALL_TAG) != tag;
        if (!__ballot(late)) break;
        if (poll % 64 == 0) {
          a = ld_agent(&p.ctl->abort);
          if (!a && wall_clock64() - t0 > p.timeout) {
            if (lane == 0) st_agent(&p.ctl->abort, 1);
            a = 1;
          }
          if (__ballot(a)) {
            a = 1;
            break;
          }
        }
        __builtin_amdgcn_s_sleep(1);
      }
      constexpr uint64_t M = (1ull << ALL_TAG) - 1;
      const unsigned long long sn =
          wave_sum((unsigned long long)((x[0] & M) + (x[1] & M) + (x[2] & M) + (x[3] & M)));
      const unsigned long long se =
          wave_sum((unsigned long long)((y[0] & M) + (y[1] & M) + (y[2] & M) + (y[3] & M)));
      if (lane == 0) {
        s_tot[0] = sn;
        s_tot[1] = se;
        s_abort = a;
      }
    }
    __syncthreads();
    *nf = s_tot[0];
    *mf = s_tot[1];
    const bool ok = !s_abort;
    bar++;
    __syncthreads();  // read before the next barrier rewrites them
    return ok;
  };

  // own words: visited = unreachable | source, levels, the first frontier
  if (t == 0) {
    s_n = s_e = 0;
    s_abort = 0;
  }
  uint32_t level = p.level, pulls = 0, streak = 0;
  const bool fresh = level == 0;
  uint64_t found = 0;  // huge rows of a frontier that goes on
  for (uint32_t k = wid; k < mine; k += NW) {
    const uint32_t w = k * G + b;
    const uint64_t v = (uint64_t)w * 64 + lane;
    uint64_t at = w == (p.src >> 6) ? 1ull << (p.src & 63) : 0ull, vis;
    if (fresh) {
      vis = p.unreachable[w] | at;
      if (v < V) p.label[v] = v == p.src ? 0u : INFINIT;
    } else {
      vis = p.visited[w];
      at = p.front[level % 3][w];
      if (((at >> lane) & 1ull) && p.out.off[v + 1] - p.out.off[v] > ALL_HUGE) {
        found += 1ull << ALL_NF;
        st_agent(&p.huge[level & 1][atomicAdd(&p.ctl->huge[level % 3], 1u)], (uint32_t)v);
      }
    }
    if (lane == 0) {
      s_vis[k] = vis;
      s_cur[k] = at;
      if (fresh) {
        st_agent64(&p.visited[w], vis);
        st_agent64(&p.front[0][w], at);
      }
      st_agent64(&p.front[(level + 1) % 3][w], 0);
    }
  }
  uint64_t nf = p.nf, mf = p.mf, mu = p.mu, prev_nf = p.prev_nf, x, y;
  if (fresh) {
    nf = 1;
    mf = p.out.off[p.src + 1] - p.out.off[p.src];
    mu = p.out.E >= mf ? p.out.E - mf : 0;
    if (mf > ALL_HUGE && b == 0 && t == 0) {
      found = 1ull << ALL_NF;
      st_agent(&p.huge[0][0], p.src);
    }
  }
  uint64_t v_reached = fresh ? 1 : 0, e_reached = fresh ? mf : 0;
  bool pull = false, pushed = false;  // pushed: own frontier words await their owner
  __syncthreads();
  bool ok = barrier(found, 0, &x, &y);
  uint32_t nhuge = (uint32_t)(x >> ALL_NF);
  while (ok && nf) {
    if (!pull && (double)mf > (double)mu / p.alpha) pull = true;
    else if (pull && (double)nf < (double)V / p.beta && nf < prev_nf) pull = false;
    streak = !pull && nf <= p.thin_nf && mf <= p.thin_mf ? streak + 1 : 0;
    if (streak > ALL_THIN) break;
    const uint64_t *cur = p.front[level % 3];
    uint64_t *next = p.front[(level + 1) % 3], *clear = p.front[(level + 2) % 3];
    uint64_t n = 0;  // new vertices, and huge rows among them from bit ALL_NF on
    uint64_t e = 0;
    auto count = [&](uint64_t v) {  // v joins the next frontier
      const uint64_t deg = p.out.off[v + 1] - p.out.off[v];
      n++;
      e += deg;
      if (deg > ALL_HUGE) {
        n += 1ull << ALL_NF;
        st_agent(&p.huge[(level + 1) & 1][atomicAdd(&p.ctl->huge[(level + 1) % 3], 1u)], (uint32_t)v);
      }
    };
    if (pushed) {  // what others found among this workgroup's vertices
      for (uint32_t k = wid; k < mine; k += NW) {
        const uint64_t m = ld_agent64(&cur[k * G + b]);
        if ((m >> lane) & 1ull) p.label[(uint64_t)(k * G + b) * 64 + lane] = level;
        if (lane == 0) {
          s_cur[k] = m;
          s_vis[k] |= m;
        }
      }
    }
    if (pull) {
      for (uint32_t i = t; i < p.W; i += ALL_T) s_front[i] = ld_agent64(&cur[i]);
      if (t == 0) s_nbig = 0;
      __syncthreads();
      for (uint32_t k = wid; k < mine; k += NW) {
        const uint32_t w = k * G + b;
        const uint64_t vis = s_vis[k];
        uint64_t m = 0;
        if (vis != ~0ull) {  // (wave-uniform; bits past V are set)
          const uint64_t v = (uint64_t)w * 64 + lane;
          const bool active = !((vis >> lane) & 1ull);
          uint64_t beg = 0, end = 0;
          bool found = false;
          if (active) {
            const uint32_t f = p.first_in[v];
            beg = p.in.off[v];
            end = p.in.off[v + 1];
            found = f != GRUS_NO_VERTEX && bm_test(s_front, f);
          }
          const uint64_t lim = end - beg > p.K ? beg + p.K : end;
          if (active && !found) {
            for (uint64_t i = beg + 1; i < lim && !found; i += 4) {
              uint32_t c[4];
#pragma unroll
              for (int q = 0; q < 4; q++) c[q] = i + q < lim ? p.in.col[i + q] : GRUS_NO_VERTEX;
#pragma unroll
              for (int q = 0; q < 4; q++)
                found = found || (c[q] != GRUS_NO_VERTEX && bm_test(s_front, c[q]));
            }
          }
          // what is left of a row: the wave shares it, or the workgroup, below
          const bool rest = active && !found && lim < end, big = rest && end - lim > ALL_BIG;
          if (big) s_big[atomicAdd(&s_nbig, 1u)] = (k << 6) | lane;
          for (uint64_t r = __ballot(rest && !big); r; r &= r - 1) {
            const int l = __ffsll((unsigned long long)r) - 1;
            const uint64_t rb = __shfl(lim, l), re = __shfl(end, l);
            bool hit = false;
            for (uint64_t i = rb; i < re && !hit; i += 4 * WAVE) {
              uint32_t c[4];
#pragma unroll
              for (int q = 0; q < 4; q++) {
                const uint64_t at = i + (uint64_t)q * WAVE + lane;
                c[q] = at < re ? p.in.col[at] : GRUS_NO_VERTEX;
              }
              bool mine_hit = false;
#pragma unroll
              for (int q = 0; q < 4; q++)
                mine_hit = mine_hit || (c[q] != GRUS_NO_VERTEX && bm_test(s_front, c[q]));
              hit = __ballot(mine_hit) != 0;
            }
            if ((int)lane == l) found = hit;
          }
          m = __ballot(found);
          if (found) {
            p.label[v] = level + 1;
            count(v);
          }
        }
        if (lane == 0) {
          s_cur[k] = m;
          st_agent64(&next[w], m);
          if (m) {
            s_vis[k] = vis | m;
            st_agent64(&p.visited[w], vis | m);
          }
        }
      }
      __syncthreads();
      const uint32_t nbig = s_nbig;
      for (uint32_t i = 0; i < nbig; i++) {
        const uint32_t k = s_big[i] >> 6, bit = s_big[i] & 63, w = k * G + b;
        const uint64_t v = (uint64_t)w * 64 + bit, end = p.in.off[v + 1];
        bool hit = false;
        for (uint64_t at = p.in.off[v] + p.K + t; !hit; at += 4 * ALL_T) {
          uint32_t c[4];
#pragma unroll
          for (int q = 0; q < 4; q++)
            c[q] = at + (uint64_t)q * ALL_T < end ? p.in.col[at + (uint64_t)q * ALL_T] : GRUS_NO_VERTEX;
          int mine_hit = 0;
#pragma unroll
          for (int q = 0; q < 4; q++)
            mine_hit |= c[q] != GRUS_NO_VERTEX && bm_test(s_front, c[q]);
          hit = __syncthreads_or(mine_hit);
          if (at - t + 4 * ALL_T >= end) break;  // (uniform) the row is done
        }
        if (hit && t == 0) {
          const uint64_t m = s_cur[k] | (1ull << bit), vis = s_vis[k] | (1ull << bit);
          p.label[v] = level + 1;
          s_cur[k] = m;
          s_vis[k] = vis;
          st_agent64(&next[w], m);
          st_agent64(&p.visited[w], vis);
          count(v);
        }
      }
      pushed = false;
      pulls++;
    } else {
      // claims the columns [at, end) of a row, `stride` threads side by side
      auto expand = [&](uint64_t at, uint64_t end, uint64_t stride) {
        for (; at < end; at += 4 * stride) {
          uint32_t d[4];
          unsigned long long old[4];
#pragma unroll
          for (int q = 0; q < 4; q++)
            d[q] = at + q * stride < end ? p.out.col[at + q * stride] : GRUS_NO_VERTEX;
#pragma unroll
          for (int q = 0; q < 4; q++)
            old[q] = d[q] == GRUS_NO_VERTEX ? ~0ull : ld_agent64(&p.visited[d[q] >> 6]);
          // the claims in flight together, and only of clear bits: most edges
          // of a wide level lead to a few words of hubs, where atomics queue
          // up one behind the other
#pragma unroll
          for (int q = 0; q < 4; q++)
            if (!((old[q] >> (d[q] & 63)) & 1ull))
              old[q] = atomicOr((unsigned long long *)&p.visited[d[q] >> 6], 1ull << (d[q] & 63));
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const unsigned long long bit = 1ull << (d[q] & 63);
            if (old[q] & bit) continue;
            atomicOr((unsigned long long *)&next[d[q] >> 6], bit);
            count(d[q]);
          }
        }
      };
      // this workgroup's share of the frontier: every G-th of its vertices in
      // id order, so that neighbouring hubs go to different workgroups
      const uint32_t per = (p.W + ALL_T - 1) / ALL_T, w0 = t * per;
      uint32_t ones = 0;
      for (uint32_t j = 0; j < per && w0 + j < p.W; j++) {
        const uint64_t m = ld_agent64(&cur[w0 + j]);
        s_front[w0 + j] = m;
        ones += (uint32_t)__popcll(m);
      }
      uint32_t r = ones;  // inclusive scan
#pragma unroll
      for (int o = 1; o < WAVE; o <<= 1) {
        const uint32_t z = __shfl_up(r, o);
        if ((int)lane >= o) r += z;
      }
      if (lane == WAVE - 1) s_wave[wid] = r;
      if (t == 0) s_nbig = s_nlist = 0;
      __syncthreads();
      for (uint32_t j = 0; j < wid; j++) r += s_wave[j];
      r -= ones;
      for (uint32_t j = 0; j < per && w0 + j < p.W; j++)
        for (uint64_t m = s_front[w0 + j]; m; m &= m - 1, r++)
          if (r % G == b)
            s_list[atomicAdd(&s_nlist, 1u)] = (w0 + j) * 64 + (uint32_t)__ffsll((unsigned long long)m) - 1;
      __syncthreads();
      const uint32_t nlist = s_nlist;
      for (uint32_t i = wid; i < nlist; i += NW) {
        const uint32_t u = s_list[i];
        const uint64_t at = p.out.off[u], end = p.out.off[u + 1];
        if (end - at > ALL_HUGE) continue;  // for the whole grid, below
        if (end - at > ALL_BIG) {           // for the whole workgroup, below
          if (lane == 0) s_big[atomicAdd(&s_nbig, 1u)] = u;
        } else {
          expand(at + lane, end, WAVE);
        }
      }
      __syncthreads();
      for (uint32_t i = 0; i < s_nbig; i++)
        expand(p.out.off[s_big[i]] + t, p.out.off[s_big[i] + 1], ALL_T);
      for (uint32_t i = 0; i < nhuge; i++) {
        const uint32_t u = ld_agent(&p.huge[level & 1][i]);
        expand(p.out.off[u] + (uint64_t)b * ALL_T + t, p.out.off[u + 1], (uint64_t)G * ALL_T);
      }
      pushed = true;
    }
    for (uint32_t k = t; k < mine; k += ALL_T) st_agent64(&clear[k * G + b], 0);
    if (b == 0 && t == 0) st_agent(&p.ctl->huge[(level + 2) % 3], 0);
    prev_nf = nf;
    ok = barrier(n, e, &nf, &mf);
    nhuge = (uint32_t)(nf >> ALL_NF);
    nf &= (1ull << ALL_NF) - 1;
    mu = mu >= mf ? mu - mf : 0;
    v_reached += nf;
    e_reached += mf;
    level++;
  }
  if (ok && nf) {  // left at a thin frontier: its levels, if they await their owner, and the queue
    for (uint32_t k = wid; k < mine; k += NW) {
      const uint64_t m = ld_agent64(&p.front[level % 3][k * G + b]);
      const uint32_t v = (k * G + b) * 64 + lane;
      uint32_t at = 0;
      if (lane == 0 && m) at = atomicAdd(&p.ctl->queued, (uint32_t)__popcll(m));
      at = __shfl(at, 0);
      if ((m >> lane) & 1ull) {
        p.label[v] = level;
        p.queue[at + lane_rank(m)] = v;
      }
    }
  }
  if (b == 0 && t == 0) {
    p.ctl->nf = ok ? (uint32_t)nf : 0u;
    p.ctl->mf = mf;
    p.ctl->mu = mu;
    p.ctl->prev_nf = (uint32_t)prev_nf;
    p.ctl->status = ok ? 0u : 1u;
    p.ctl->levels = level - p.level;
    p.ctl->pulls = pulls;
    p.ctl->v_reached = v_reached;
    p.ctl->e_reached = e_reached;
  }
}

}  // namespace bfs
}  // namespace mgg
