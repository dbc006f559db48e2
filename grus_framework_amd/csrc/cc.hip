// cc.hip -- connected components, label = minimum vertex id of the component.
//
// Reference: samples/cc/cc.cu (CCInit :35-40 label = id, updater :69-79
// atomicMin(label[dst], label[src]), push driver :155-190 from a full
// frontier).  Its fixed point on a symmetric graph is the minimum vertex id
// of each component; both methods below reach exactly that labelling.
//
// method 0 (default) -- hooking + pointer jumping (after Sutton et al.,
//   IPDPS'18 "Afforest"): hook every vertex under its first neighbour where
//   that is smaller (one store, no atomic), compress, find the most frequent
//   root by sampling, then link every edge of the vertices outside that
//   component.  A link hooks the larger root under the smaller one with a
//   CAS, so parent[x] <= x holds throughout and every root is the minimum of
//   its tree.  Rows of generated graphs ascend, so the first neighbour is the
//   lowest: on RMAT s20 the hooks alone put 93% of the vertices with edges
//   into the giant component, and the rest hold 0.3% of the edges.  Where the
//   sample finds too many edges outside, every vertex's first two neighbours
//   are linked before the rest.
// method 1 -- the reference's min-label propagation through the push
//   operator (advance.hpp), frontier deduplicated by round stamps.
#include <algorithm>
#include <cstring>
#include <string>

#include "advance.hpp"
#include "apps.hpp"
#include "device.hpp"
#include "prims.hpp"

namespace mgg {

struct CcWork {
  Buf q[2], stamp, giant;
  PushWork push;
  uint64_t cap_v = 0;
  uint32_t stamp_id = 0;
};

namespace cc {

__global__ void k_init(uint32_t *label, uint64_t V) {
  uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
  uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (; i < V; i += stride) label[i] = (uint32_t)i;  // CCInit cc.cu:38
}

__device__ __forceinline__ uint32_t ld(const uint32_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// hook the larger root under the smaller (CAS); parent[x] <= x is invariant
__device__ __forceinline__ void link(uint32_t u, uint32_t v, uint32_t *parent) {
  uint32_t p1 = ld(&parent[u]), p2 = ld(&parent[v]);
  while (p1 != p2) {
    uint32_t hi = p1 > p2 ? p1 : p2, lo = p1 > p2 ? p2 : p1;
    uint32_t ph = ld(&parent[hi]);
    if (ph == lo) return;
    if (ph == hi && atomicCAS(&parent[hi], hi, lo) == hi) return;
    p1 = ld(&parent[ld(&parent[hi])]);
    p2 = ld(&parent[lo]);
  }
}

// parent[u] = u's first neighbour where that is smaller, else u.  Bound by
// the gather of one cache line per row.
__global__ __launch_bounds__(BLOCK) void k_hook_first(CsrView g, uint32_t *parent) {
  uint64_t u = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
  uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (; u < g.V; u += stride) {
    const uint64_t e = g.off[u];
    uint32_t p = (uint32_t)u;
    if (e < g.off[u + 1]) p = min(p, edge_col(g, e));
    parent[u] = p;
  }
}

// v's root, or `stop` if it lies on the way, climbing at most `hops` steps
// past v's parent.  v takes every ancestor it reaches as its parent, so that
// the vertices below it skip what it has climbed: on a grid, whose hooks form
// chains as long as its side, storing only the root made each vertex climb
// its whole chain.  (A vertex that is not a root never becomes one, and only
// its own thread stores its parent, so the stores race with no CAS.)
__device__ __forceinline__ uint32_t climb(uint32_t v, uint32_t *parent, uint32_t stop,
                                          uint32_t hops) {
  uint32_t p = parent[v];  // cached: a stale parent is an older ancestor
  uint32_t pp = p == stop ? p : ld(&parent[p]);
  for (uint32_t i = 0; p != pp && i < hops; i++) {
    __hip_atomic_store(&parent[v], pp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    p = pp;
    pp = p == stop ? p : ld(&parent[p]);
  }
  return p;
}

// What the sampled edges tell, in the scratch.
struct Giant {
  uint32_t root;  // the most frequent root
  uint32_t more;  // too many edges lie outside it
};

// A full climb by every vertex at once is slow on long chains (each starts
// before those above it have shortened theirs), so the first pass stops
// after FIRST_HOPS and k_link_rest climbs the rest: 4096 x 4096 grid 1.19 ->
// 0.44 ms in all; RMAT s22, where FIRST_HOPS reach every root, 0.13 either way.
constexpr uint32_t FIRST_HOPS = 8;
__global__ __launch_bounds__(BLOCK) void k_compress(uint32_t *parent, uint64_t V, uint32_t hops,
                                                    const Giant *if_more) {
  if (if_more && !if_more->more) return;
  uint64_t v = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
  uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (; v < V; v += stride) climb((uint32_t)v, parent, GRUS_NO_VERTEX, hops);
}

// The most frequent root among the heads of kSample pseudo-random edges
// (ties: the smaller root) to *out, in one workgroup with an edge per thread:
// each thread counts the samples equal to its own, so the mode needs no sort
// and no trip to the host (256 of them 5 us, 1024 in 16 waves 22).  Edges and
// not vertices, because what is left to do is the edges outside: more of them
// than half the vertices, and the links of k_link_two cost less than theirs.
// `again`: only if `more` was found before.
constexpr uint32_t kSample = 256;
__global__ __launch_bounds__(kSample) void k_sample_mode(CsrView g, uint32_t *parent,
                                                         uint64_t seed, bool again, Giant *out) {
  __shared__ uint4 s_root[kSample / 4];
  __shared__ unsigned long long s_best[kSample / WAVE];
  if (again && !out->more) return;
  const uint32_t t = threadIdx.x;
  uint32_t mine = GRUS_NO_VERTEX;
  if (g.E)
    mine = climb(edge_col(g, mix64(seed + t) % g.E), parent, GRUS_NO_VERTEX, 0xFFFFFFFFu);
  reinterpret_cast<uint32_t *>(s_root)[t] = mine;
  __syncthreads();
  uint32_t n = 0;
  for (uint32_t i = 0; i < kSample / 4; i++) {
    const uint4 x = s_root[i];
    n += (x.x == mine) + (x.y == mine) + (x.z == mine) + (x.w == mine);
  }
  unsigned long long best = ((unsigned long long)n << 32) | (0xFFFFFFFFu - mine);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long y = __shfl_xor(best, o);
    best = y > best ? y : best;
  }
  if (lane_id() == 0) s_best[t / WAVE] = best;
  __syncthreads();
  if (t == 0) {
    for (uint32_t w = 1; w < kSample / WAVE; w++) best = s_best[w] > best ? s_best[w] : best;
    const uint32_t outside = kSample - (uint32_t)(best >> 32);
    *out = {0xFFFFFFFFu - (uint32_t)best, (double)outside * g.E > (double)kSample / 2 * g.V};
  }
}

// The hooks alone join few vertices where first neighbours are not often the
// smallest of a neighbourhood (numberings without order, rows in any order):
// half of the edges and more are then outside the giant component, and to link
// them all takes longer than everything else.  There the edges to every
// vertex's first two neighbours are linked too, as Afforest does.  ms per call
// without / with them: uniform edges, V = 2^16, 8 a vertex 0.134 / 0.080; V =
// 2^20, 16 a vertex 1.76 / 0.25; RMAT s20 with its rows in random order 19.3 /
// 0.19.  Where the hooks do (RMAT s22) the three idle launches take 13 us.
__global__ __launch_bounds__(BLOCK) void k_link_two(CsrView g, const Giant *giant,
                                                    uint32_t *parent) {
  if (!giant->more) return;
  uint64_t u = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (; u < g.V; u += stride) {
    const uint64_t beg = g.off[u], end = g.off[u + 1];
    for (uint64_t e = beg; e < end && e < beg + 2; e++)
      link((uint32_t)u, edge_col(g, e), parent);
  }
}

// Every edge of the vertices outside the giant component.  A lane tests one
// vertex and links its row itself up to REST_LANE edges; the wave shares
// longer rows.  Nearly every vertex fails the test, so this costs one
// coalesced read of the parents: RMAT s22 spent 325 of 503 us here with a
// wave per vertex; the whole call now takes 126 us on the device.
constexpr uint64_t REST_LANE = 16;
__global__ __launch_bounds__(BLOCK) void k_link_rest(CsrView g, const Giant *giant_p,
                                                     uint32_t *parent) {
  const uint32_t giant = giant_p->root;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const uint64_t first = blockIdx.x * (uint64_t)blockDim.x + (threadIdx.x & ~(uint32_t)(WAVE - 1));
  for (uint64_t base = first; base < g.V; base += stride) {  // wave-uniform
    const uint64_t u = base + lane_id();
    uint64_t beg = 0, end = 0;
    if (u < g.V && climb((uint32_t)u, parent, giant, 0xFFFFFFFFu) != giant) {
      beg = g.off[u];
      end = g.off[u + 1];
    }
    const bool shared_row = end - beg > REST_LANE;
    if (!shared_row)
      for (uint64_t e = beg; e < end; e++) link((uint32_t)u, edge_col(g, e), parent);
    for (uint64_t m = __ballot(shared_row); m; m &= m - 1) {
      const int l = __ffsll((unsigned long long)m) - 1;
      const uint64_t b = __shfl(beg, l), x = __shfl(end, l);
      for (uint64_t e = b + lane_id(); e < x; e += WAVE)
        link((uint32_t)(base + l), edge_col(g, e), parent);
    }
  }
}

__global__ void k_iota(uint32_t *q, uint64_t n) {
  uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
  uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) q[i] = (uint32_t)i;
}

// job_t of samples/cc/cc.cu:42-67 for min-label propagation
struct job_t {
  static constexpr bool kFar = false;
  uint32_t *label;
  uint32_t *stamp;
  const uint64_t *out_off;
  uint32_t stamp_id;
  // updater cc.cu:69-79
  __device__ __forceinline__ bool update(vtx_t src, vtx_t dst, eid_t, weight_t, uint32_t *) const {
    uint32_t ls = ld(&label[src]);
    if (ld(&label[dst]) <= ls) return false;
    return atomicMin(&label[dst], ls) > ls;
  }
  // generator cc.cu:86-91 (the byte CAS flag becomes a round stamp)
  __device__ __forceinline__ int generate(bool updated, vtx_t dst, uint32_t) const {
    // stamps are unique per round: a plain read showing this round's is exact
    if (!updated || stamp[dst] == stamp_id) return 0;
    return atomicExch(&stamp[dst], stamp_id) != stamp_id ? 1 : 0;
  }
  __device__ __forceinline__ uint64_t out_degree(vtx_t v) const {
    return out_off[v + 1] - out_off[v];
  }
};

}  // namespace cc

// The device buffers of one CC run beyond the graph and the labels.
struct CcSpace {
  cc::Giant *giant = nullptr;           // method 0: what the sampled edges tell
  uint32_t *q[2] = {nullptr, nullptr};  // method 1: frontier queues, V + 1 each
  uint32_t *stamp = nullptr;            // method 1: round stamps, V + 1
  uint32_t *stamp_id = nullptr;         // method 1: last stamp handed out (host)
  PushWork *push = nullptr;             // method 1: the push operator's scans
};

namespace {
constexpr uint64_t kGiantBytes = 256;

void cc_core(Graph &g, int method, uint32_t *label, CcSpace &sp, grus_stats *st) {
  Context &ctx = *g.ctx;
  const uint64_t V = g.V;
  const CsrView gr = g.csr();
  uint64_t launches = 0;
  uint32_t iterations = 0;
  GRUS_HIP(hipEventRecord(ctx.ev0, ctx.stream));
  if (method == 0) {
    const unsigned grid = grid_cap(ctx, V, BLOCK);
    if (V) {
      cc::k_hook_first<<<grid, BLOCK, 0, ctx.stream>>>(gr, label);
      GRUS_LAUNCH_CHECK();
      cc::k_compress<<<grid, BLOCK, 0, ctx.stream>>>(label, V, cc::FIRST_HOPS, nullptr);
      GRUS_LAUNCH_CHECK();
      cc::k_sample_mode<<<1, cc::kSample, 0, ctx.stream>>>(gr, label, 0x5EEDull, false, sp.giant);
      GRUS_LAUNCH_CHECK();
      cc::k_link_two<<<grid, BLOCK, 0, ctx.stream>>>(gr, sp.giant, label);
      GRUS_LAUNCH_CHECK();
      cc::k_compress<<<grid, BLOCK, 0, ctx.stream>>>(label, V, cc::FIRST_HOPS, sp.giant);
      GRUS_LAUNCH_CHECK();
      cc::k_sample_mode<<<1, cc::kSample, 0, ctx.stream>>>(gr, label, 0x5EEDull, true, sp.giant);
      GRUS_LAUNCH_CHECK();
      cc::k_link_rest<<<grid, BLOCK, 0, ctx.stream>>>(gr, sp.giant, label);
      GRUS_LAUNCH_CHECK();
      cc::k_compress<<<grid, BLOCK, 0, ctx.stream>>>(label, V, 0xFFFFFFFFu, nullptr);
      GRUS_LAUNCH_CHECK();
      launches += 8;
    }
    iterations = 2;  // the hooks, then the rest
  } else {
    auto *cnt = reinterpret_cast<StepCounters *>(ctx.d_ctl.p);
    const StepCounters *hc = reinterpret_cast<const StepCounters *>(ctx.h_ctl);
    uint32_t &stamp_id = *sp.stamp_id;
    cc::k_init<<<grid_cap(ctx, V, BLOCK), BLOCK, 0, ctx.stream>>>(label, V);
    GRUS_LAUNCH_CHECK();
    launches++;
    cc::k_iota<<<grid_cap(ctx, V, BLOCK), BLOCK, 0, ctx.stream>>>(sp.q[0], V);
    GRUS_LAUNCH_CHECK();
    uint64_t nf = V, mf = g.E;
    int cur = 0;
    while (nf) {
      if (iterations > V + 1) raise(GRUS_E_HIP, "label propagation did not converge");
      if (stamp_id >= 0xFFFFFF00u) {
        fill_u32(ctx, sp.stamp, V + 1, 0);
        stamp_id = 0;
      }
      fill_u64(ctx, reinterpret_cast<uint64_t *>(cnt), sizeof(StepCounters) / 8, 0);
      push_scan_degrees(ctx, *sp.push, gr.off, sp.q[cur], (uint32_t)nf);
      cc::job_t job{label, sp.stamp, gr.off, ++stamp_id};
      push_advance(ctx, *sp.push, gr, sp.q[cur], (uint32_t)nf, mf, job, sp.q[cur ^ 1], cnt);
      launches += 4;
      ctx.read_ctl(2);
      nf = hc->next_count;
      mf = hc->next_edges;
      cur ^= 1;
      iterations++;
    }
  }
  GRUS_HIP(hipEventRecord(ctx.ev1, ctx.stream));
  GRUS_HIP(hipEventSynchronize(ctx.ev1));
  float ms = 0;
  GRUS_HIP(hipEventElapsedTime(&ms, ctx.ev0, ctx.ev1));
  if (st) {
    *st = grus_stats{};
    st->device_ms = ms;
    st->iterations = iterations;
    st->vertices_reached = V;
    st->edges_reached = g.E;
    st->kernel_launches = launches;
  }
}

void cc_check(Graph &g, int method) {
  g.ctx->activate();
  if (method != 0 && method != 1) raise(GRUS_E_INVALID, "cc method");
  if (!g.symmetric)
    raise(GRUS_E_UNSUPPORTED, "connected components need a symmetric graph (weak CC)");
}
}  // namespace

void run_cc(Graph &g, int method, grus_stats *st) {
  cc_check(g, method);
  g.make_room(Graph::App::CC);
  if (!g.cc) g.cc = std::make_shared<CcWork>();
  CcWork &w = *g.cc;
  Context &ctx = *g.ctx;
  const uint64_t V = g.V;
  g.result.ensure(V * 4);
  CcSpace sp;
  if (method == 0) {
    w.giant.ensure(kGiantBytes);
    sp.giant = w.giant.as<cc::Giant>();
  } else {
    if (w.cap_v < V) {
      w.q[0].alloc((V + 1) * 4);
      w.q[1].alloc((V + 1) * 4);
      w.stamp.alloc((V + 1) * 4);
      fill_u32(ctx, w.stamp.as<uint32_t>(), V + 1, 0);
      w.push.ensure(V);
      w.cap_v = V;
      w.stamp_id = 0;
    }
    sp.q[0] = w.q[0].as<uint32_t>();
    sp.q[1] = w.q[1].as<uint32_t>();
    sp.stamp = w.stamp.as<uint32_t>();
    sp.stamp_id = &w.stamp_id;
    sp.push = &w.push;
  }
  cc_core(g, method, g.result.as<uint32_t>(), sp, st);
}

uint64_t cc_scratch_bytes(Context &ctx, uint64_t V, int method) {
  if (method == 0) return kGiantBytes;
  // queues and stamps (3 x (V + 1) u32), degree and scan (2 x (V + 2) u64),
  // the scan's temporaries, each start aligned to 256 bytes
  auto up = [](uint64_t x) { return (x + 255) & ~255ull; };
  return 3 * up((V + 1) * 4) + 2 * up((V + 2) * 8) + up(scan_excl_u64_bytes(ctx, V + 1));
}

void run_cc_in(Graph &g, int method, uint32_t *label, void *scratch, uint64_t scratch_bytes,
               grus_stats *st) {
  cc_check(g, method);
  Context &ctx = *g.ctx;
  const uint64_t V = g.V;
  const uint64_t need = cc_scratch_bytes(ctx, V, method);
  if (need > scratch_bytes)
    raise(GRUS_E_BUDGET, "connected components (method " + std::to_string(method) + ") on " +
                             std::to_string(V) + " vertices need " + std::to_string(need) +
                             " bytes of scratch; " + std::to_string(scratch_bytes) +
                             " are available");
  auto *base = static_cast<unsigned char *>(scratch);
  auto up = [](uint64_t x) { return (x + 255) & ~255ull; };
  CcSpace sp;
  PushWork push;  // borrowed buffers only: its own Bufs stay empty
  uint32_t stamp_id = 0;
  if (method == 0) {
    sp.giant = reinterpret_cast<cc::Giant *>(base);
  } else {
    uint64_t at = 0;
    auto take = [&](uint64_t bytes) {
      unsigned char *p = base + at;
      at += up(bytes);
      return p;
    };
    sp.q[0] = reinterpret_cast<uint32_t *>(take((V + 1) * 4));
    sp.q[1] = reinterpret_cast<uint32_t *>(take((V + 1) * 4));
    sp.stamp = reinterpret_cast<uint32_t *>(take((V + 1) * 4));
    push.deg_ext = reinterpret_cast<uint64_t *>(take((V + 2) * 8));
    push.scan_ext = reinterpret_cast<uint64_t *>(take((V + 2) * 8));
    push.tmp_bytes = up(scan_excl_u64_bytes(ctx, V + 1));
    push.tmp = take(push.tmp_bytes);
    // the scratch keeps the last call's contents: stamps start from zero
    fill_u32(ctx, sp.stamp, V + 1, 0);
    sp.stamp_id = &stamp_id;
    sp.push = &push;
  }
  cc_core(g, method, label, sp, st);
}

}  // namespace mgg
