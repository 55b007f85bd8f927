// sssp.hip -- weighted min-plus SSSP on the device (the reference's traversal
// Ingress loop, sum_sync_traversal_worker.h:1146-1159 with the weighted
// SSSPIngress::Compute of sssp/sssp_ingress.h:131-175; replaces the unit-weight
// tjnsssp kernels, cudaCode/my_ssspworker.cu:374-495).
//
// State: dp[v] = dist << 32 | parent (u64).  One 64-bit atomicMin both lowers
// the distance and, on equal distance, picks the smaller parent id, so the fixed
// point is unique: dist = shortest distance, parent = smallest-id predecessor on
// a shortest path (the reference's DependencyData CAS keeps whichever proposal
// lands first, dependency_data.h:21-34; distances are identical, parents are a
// deterministic choice among the reference's valid ones).
//
// Frontier: double-buffered vertex lists + bitmaps.  A vertex whose distance
// drops is appended to the next list once (atomicOr on its bitmap word, then a
// wave64-aggregated append).  Per round: k_sssp_push (light tiles, heavy
// vertices deferred to 2048-edge chunks), k_sssp_heavy, k_sssp_end.  The lists,
// bitmaps and the count of pending seeds belong to the SSSP state: batches append
// seeds, and each query takes them at its start (k_sssp_begin).
//
// A run from scratch has a few rounds in which most of the graph is relaxed; a push pays
// an atomic minimum per edge that may win and an append per vertex reached there (about
// 6 and 8 G edges a second at 2^20 and 2^22 vertices).  Once the frontier holds more than
// 1 / kPullFrontier of the vertices, such a run pulls instead: k_sssp_pull streams the
// CSC in tiles of kPullTile edges, tests each source's frontier bit and keeps the minimum
// of every row in LDS, so a row costs one store; rows that no frontier vertex can improve
// (their word is at most the frontier's smallest) are passed over without reading their
// edges; k_sssp_collect makes the next list from the bitmap.  The fixed point is the same
// unique one (SSWP: the same widths).  MI355X, from
// scratch: SSSP on 1,000,003 vertices, 12M edges, weights to 64, 9 rounds, 3.86 -> 0.63 ms
// (4 of them pulls, 0.1 ms each); BFS on 2^22 vertices, 50M edges, 7 rounds, 6.55 -> 0.92 ms
// (3 pulls, 0.2 ms each, where the columns alone are 0.04 ms: bound by the gathers of
// frontier bits and words).
#include <algorithm>

#include "ctx.hpp"
#include "device.hpp"
#include "pr.hpp"
#include "readback.hpp"

namespace suminc {

struct SsspArgs {
  const uint32_t* off;
  const uint32_t* col;
  const uint32_t* w;  // null: unit weights
  unsigned long long* dp;
  uint32_t* wl[2];
  uint32_t* bits[2];
  uint2* heavy;
  Counters* cnt;
  int app;  // SUMINC_APP_*
};

__device__ __forceinline__ void sssp_relax(const SsspArgs& a, int nxt, uint32_t u, uint32_t du, uint32_t e) {
  uint32_t v = a.col[e];
  uint32_t w = a.w ? a.w[e] : 1u;
  unsigned long long nd = trav_extend(a.app, du, w);  // < 2^32 - 1 unless the path saturates
  bool add = false;
  if (nd < INF32) {
    unsigned long long cand = (nd << 32) | u;
    // words only decrease while the rounds run: a candidate no smaller than a
    // plain (possibly stale) read cannot win, so it skips the atomic.  SSWP takes
    // strictly better values only (trav_commit)
    const unsigned long long seen = a.dp[v];
    if (a.app == SUMINC_APP_SSWP ? nd < (seen >> 32) : cand < seen) {
      unsigned long long old = trav_commit(a.app, &a.dp[v], cand, seen);
      add = (old >> 32) > nd;
    }
  }
  if (add) {
    uint32_t bit = 1u << (v & 31);
    uint32_t prev = atomicOr(&a.bits[nxt][v >> 5], bit);
    add = !(prev & bit);
  }
  // every lane reaches the ballot, active or not
  unsigned long long slot = wave_append(add, &a.cnt->wl_count[nxt]);
  if (add) a.wl[nxt][slot] = v;
}

// Push kernels: done and mode != 0 (a pull round of sssp_run) return at entry.
__global__ void __launch_bounds__(kBlock) k_sssp_push(SsspArgs a) {
  __shared__ uint32_t s_scan[kBlock + 1];
  __shared__ uint32_t s_start[kBlock];
  __shared__ uint32_t s_warp[kBlock / 64 + 1];
  __shared__ uint32_t s_u[kBlock];
  __shared__ uint32_t s_du[kBlock];
  __shared__ unsigned long long s_edges;
  if (a.cnt->done || a.cnt->mode != 0) return;
  const int cur = (int)(a.cnt->aux[1] & 1), nxt = cur ^ 1;
  const unsigned long long nl = a.cnt->wl_count[cur];
  const uint32_t vt = frontier_tile<kBlock>(nl);
  const unsigned long long tiles = (nl + vt - 1) / vt;
  if (threadIdx.x == 0) s_edges = 0;
  __syncthreads();
  for (unsigned long long t = blockIdx.x; t < tiles; t += gridDim.x) {
    unsigned long long i = t * vt + threadIdx.x;
    uint32_t start = 0, len = 0;
    if (threadIdx.x < vt && i < nl) {
      uint32_t u = a.wl[cur][i];
      atomicAnd(&a.bits[cur][u >> 5], ~(1u << (u & 31)));
      uint32_t du = (uint32_t)(a.dp[u] >> 32);
      uint32_t b = a.off[u], e = a.off[u + 1];
      if (du != INF32 && e > b) {
        if (e - b <= kHeavyDeg) {
          start = b;
          len = e - b;
        } else {
          uint32_t nch = (e - b + kChunk - 1) / kChunk;
          unsigned long long slot = atomicAdd(&a.cnt->heavy_count, (unsigned long long)nch);
          for (uint32_t k = 0; k < nch; ++k) a.heavy[slot + k] = make_uint2(u, k);
        }
        atomicAdd(&s_edges, (unsigned long long)(e - b));
      }
      s_u[threadIdx.x] = u;
      s_du[threadIdx.x] = du;
    }
    block_adjacency<kBlock>(start, len, s_scan, s_start, s_warp,
                            [&](int slot, uint32_t, uint32_t e) { sssp_relax(a, nxt, s_u[slot], s_du[slot], e); });
  }
  __syncthreads();
  if (threadIdx.x == 0 && s_edges) atomicAdd(&a.cnt->edges, s_edges);
}

__global__ void __launch_bounds__(kBlock) k_sssp_heavy(SsspArgs a) {
  if (a.cnt->done || a.cnt->mode != 0) return;
  const int cur = (int)(a.cnt->aux[1] & 1), nxt = cur ^ 1;
  const unsigned long long nh = a.cnt->heavy_count;
  for (unsigned long long h = blockIdx.x; h < nh; h += gridDim.x) {
    uint2 hv = a.heavy[h];
    uint32_t u = hv.x;
    uint32_t du = (uint32_t)(a.dp[u] >> 32);
    uint32_t b = a.off[u] + hv.y * kChunk;
    uint32_t e = min(a.off[u + 1], b + kChunk);
    // all lanes iterate the same trip count so wave_append sees full waves
    for (uint32_t k0 = b; k0 < e; k0 += kBlock) {
      uint32_t k = k0 + threadIdx.x;
      if (k < e) sssp_relax(a, nxt, u, du, k);
    }
  }
}

// ---- pull rounds --------------------------------------------------------------------
constexpr uint32_t kPullTile = 1024;     // CSC edges per workgroup
constexpr uint32_t kPullFrontier = 64;   // a pull from n / 64 frontier vertices on
// Rounds are enqueued without the pull's launches after a group of rounds that had no pull
// and left a frontier below n / 256, and from the start where the last run from scratch
// had none.  Long paths and road graphs are such runs: two of their five launches a round
// return at once (BFS of 4999 rounds on a 2500 x 2500 grid: 193 ms with them, 154 without;
// of 20,000 rounds on a path of a graph of 340,000 edges: 249 and 198).  A frontier that
// grows past n / 64 all the same stops the group (k_sssp_end).
constexpr uint32_t kPushFrontier = 256;
constexpr uint64_t kPullMinEdges = 1u << 18;  // below, a push round costs less than the further launches

struct SsspPull {
  const uint32_t* ioff;
  const uint32_t* icol;
  const uint32_t* iw;        // null: unit weights
  const uint32_t* tile_row;  // row of the first edge of every tile, then the last row
  uint32_t* edges;           // per tile: edges out of frontier vertices
  uint32_t n;
  uint64_t m;
};

__global__ void k_sssp_tiles(const uint32_t* __restrict__ off, uint32_t n, uint32_t tiles,
                             uint32_t* __restrict__ tile_row) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t > tiles) return;
  if (t == tiles) {
    tile_row[t] = n - 1;
    return;
  }
  const uint32_t e = t * kPullTile;
  uint32_t lo = 0, hi = n - 1;  // the last row that starts at or before e is the row of e
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo + 1) / 2;
    if (off[mid] <= e) lo = mid; else hi = mid - 1;
  }
  tile_row[t] = lo;
}

// Whether the word cand may replace old (its value's word: old_hi).
__device__ __forceinline__ bool sssp_better(int app, unsigned long long cand, unsigned long long old, uint32_t old_hi) {
  return cand < old && (app != SUMINC_APP_SSWP || (uint32_t)(cand >> 32) < old_hi);
}

__device__ __forceinline__ void sssp_mark(uint32_t* bits, uint32_t v) { atomicOr(&bits[v >> 5], 1u << (v & 31)); }

// A tile's rows are named by the slot of their first edge in the tile (slot 0: the row
// that the tile begins in).
__global__ void __launch_bounds__(kBlock) k_sssp_pull(SsspArgs a, SsspPull p) {
  constexpr int kPer = kPullTile / kBlock;
  __shared__ unsigned long long s_min[kPullTile];
  __shared__ uint32_t s_old[kPullTile];  // the value's word before the round
  __shared__ uint32_t s_id[kPullTile];
  __shared__ uint16_t s_slot[kPullTile];
  __shared__ uint32_t s_w[kBlock / 64], s_ed[kBlock / 64];
  if (a.cnt->done || a.cnt->mode == 0) return;
  const int cur = (int)(a.cnt->aux[1] & 1), nxt = cur ^ 1;
  const uint32_t least = (uint32_t)a.cnt->rc[cur];
  const uint32_t* front = a.bits[cur];
  const uint32_t t = blockIdx.x;
  const uint64_t e0 = (uint64_t)t * kPullTile;
  const uint32_t ne = (uint32_t)(p.m - e0 < kPullTile ? p.m - e0 : kPullTile);
  const uint32_t r0 = p.tile_row[t], r1 = p.tile_row[t + 1];
  uint32_t ed = 0;
  if (r1 - r0 > 32 * kPullTile) {  // mostly empty rows: a search per edge passes over fewer of them
    for (uint32_t i = threadIdx.x; i < ne; i += kBlock) {
      const uint32_t e = (uint32_t)e0 + i, u = p.icol[e];
      if (!(front[u >> 5] >> (u & 31) & 1)) continue;
      ++ed;
      uint32_t lo = r0, hi = r1;
      while (lo < hi) {
        const uint32_t mid = lo + (hi - lo + 1) / 2;
        if (p.ioff[mid] <= e) lo = mid; else hi = mid - 1;
      }
      const unsigned long long nd = trav_extend(a.app, (uint32_t)(a.dp[u] >> 32), p.iw ? p.iw[e] : 1u);
      if (nd >= INF32) continue;
      const unsigned long long cand = nd << 32 | u, was = a.dp[lo];
      if (!sssp_better(a.app, cand, was, (uint32_t)(was >> 32))) continue;
      if ((trav_commit(a.app, &a.dp[lo], cand, was) >> 32) > nd) sssp_mark(a.bits[nxt], lo);
    }
  } else {
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const uint32_t i = j * kBlock + threadIdx.x;
      s_slot[i] = 0;
      s_id[i] = i == 0 ? r0 : INF32;
    }
    __syncthreads();
    for (uint32_t r = r0 + 1 + threadIdx.x; r <= r1; r += kBlock) {
      const uint32_t b = p.ioff[r], e = p.ioff[r + 1];
      if (e > b && b - e0 < ne) {
        s_slot[b - (uint32_t)e0] = (uint16_t)(b - (uint32_t)e0);
        s_id[b - (uint32_t)e0] = r;
      }
    }
    __syncthreads();
    // the rows' words (0: passed over), and a running maximum gives each edge its slot
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const uint32_t i = j * kBlock + threadIdx.x;
      if (s_id[i] != INF32) {
        const unsigned long long x = a.dp[s_id[i]];
        s_old[i] = (uint32_t)(x >> 32);
        s_min[i] = (uint32_t)(x >> 32) <= least ? 0ull : x;
      }
    }
    uint32_t x[kPer], run = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      run = max(run, (uint32_t)s_slot[threadIdx.x * kPer + j]);
      x[j] = run;
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(run, o);
      if (lane_id() >= o) run = max(run, y);
    }
    if (lane_id() == 63) s_w[threadIdx.x >> 6] = run;
    uint32_t before = __shfl_up(run, 1);
    if (lane_id() == 0) before = 0;
    __syncthreads();
    for (uint32_t w = 0; w < threadIdx.x >> 6; ++w) before = max(before, s_w[w]);
#pragma unroll
    for (int j = 0; j < kPer; ++j) s_slot[threadIdx.x * kPer + j] = (uint16_t)max(before, x[j]);
    __syncthreads();
    // the sources of the rows that can still improve, then their frontier bits, then
    // the words and weights of the sources in the frontier: each step's loads together
    uint32_t u[kPer], sl[kPer], bw[kPer];
    bool on[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const uint32_t i = j * kBlock + threadIdx.x;
      sl[j] = i < ne ? s_slot[i] : 0u;
      on[j] = i < ne && s_min[sl[j]] != 0ull;
      u[j] = on[j] ? p.icol[e0 + i] : 0u;
    }
#pragma unroll
    for (int j = 0; j < kPer; ++j) bw[j] = on[j] ? front[u[j] >> 5] : 0u;
    unsigned long long du[kPer];
    uint32_t w[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      on[j] = bw[j] >> (u[j] & 31) & 1;
      ed += on[j];
      du[j] = on[j] ? a.dp[u[j]] : ~0ull;
      w[j] = on[j] && p.iw ? p.iw[e0 + j * kBlock + threadIdx.x] : 1u;
    }
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      if (!on[j]) continue;
      const unsigned long long nd = trav_extend(a.app, (uint32_t)(du[j] >> 32), w[j]);
      if (nd >= INF32) continue;
      const unsigned long long cand = nd << 32 | u[j];
      if (sssp_better(a.app, cand, s_min[sl[j]], s_old[sl[j]])) atomicMin(&s_min[sl[j]], cand);
    }
    __syncthreads();
    // rows inside the tile have no other writer; the first and the last may reach over
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const uint32_t i = j * kBlock + threadIdx.x, v = s_id[i];
      if (v == INF32) continue;
      const unsigned long long best = s_min[i];
      if (best == 0ull) continue;
      const unsigned long long seen = a.dp[v];
      if (best >= seen) continue;
      if (p.ioff[v] >= e0 && p.ioff[v + 1] <= e0 + ne) {
        a.dp[v] = best;
        if ((uint32_t)(best >> 32) < s_old[i]) sssp_mark(a.bits[nxt], v);
      } else if ((trav_commit(a.app, &a.dp[v], best, seen) >> 32) > (best >> 32)) {
        sssp_mark(a.bits[nxt], v);
      }
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) ed += __shfl_xor(ed, o);
  if (lane_id() == 0) s_ed[threadIdx.x >> 6] = ed;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t total = 0;
    for (int w = 0; w < kBlock / 64; ++w) total += s_ed[w];
    p.edges[t] = total;
  }
}

// After a pull: the frontier that was is cleared and the next one's list made from its
// bitmap (a word a thread); before a pull also the smallest word of the next frontier
// (cnt->rc).
__global__ void __launch_bounds__(kBlock) k_sssp_collect(SsspArgs a, uint32_t n) {
  __shared__ uint32_t s_warp[kBlock / 64 + 1], s_least[kBlock / 64];
  __shared__ unsigned long long s_base;
  if (a.cnt->done) return;
  const int cur = (int)(a.cnt->aux[1] & 1), nxt = cur ^ 1;
  const bool pull = a.cnt->mode != 0;
  if (!pull && a.cnt->wl_count[nxt] * kPullFrontier <= n) return;
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x, words = (n + 31) / 32;
  uint32_t b = i < words ? a.bits[nxt][i] : 0u;
  uint32_t at = 0;
  if (pull) {
    if (i < words) a.bits[cur][i] = 0;
    uint32_t total;
    at = block_exclusive_scan<kBlock>(__popc(b), s_warp, &total);
    if (threadIdx.x == 0) s_base = total ? atomicAdd(&a.cnt->wl_count[nxt], (unsigned long long)total) : 0ull;
    __syncthreads();
  }
  uint32_t least = INF32;
  for (; b; b &= b - 1) {
    const uint32_t v = i * 32 + __ffs(b) - 1;
    if (pull) a.wl[nxt][s_base + at++] = v;
    least = min(least, (uint32_t)(a.dp[v] >> 32));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) least = min(least, (uint32_t)__shfl_xor((int)least, o));
  if (lane_id() == 0) s_least[threadIdx.x >> 6] = least;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kBlock / 64; ++w) least = min(least, s_least[w]);
    if (least != INF32) atomicMin(&a.cnt->rc[nxt], (unsigned long long)least);
  }
}

// Closes a round of a run that may pull, and chooses the next one's direction.
__global__ void __launch_bounds__(1024) k_sssp_turn(Counters* cnt, uint32_t n, const uint32_t* __restrict__ edges,
                                                    uint32_t tiles, int max_rounds) {
  __shared__ unsigned long long s[1024 / 64];
  if (cnt->done) return;
  unsigned long long ed = 0;
  if (cnt->mode) {
    for (uint32_t i = threadIdx.x; i < tiles; i += 1024) ed += edges[i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ed += __shfl_xor(ed, o);
  }
  if (lane_id() == 0) s[threadIdx.x >> 6] = ed;
  __syncthreads();
  if (threadIdx.x) return;
  for (int w = 1; w < 1024 / 64; ++w) ed += s[w];
  const int cur = (int)(cnt->aux[1] & 1), nxt = cur ^ 1;
  cnt->edges += ed;
  cnt->aux[6] += cnt->wl_count[cur];
  cnt->pull_rounds += cnt->mode;
  cnt->wl_count[cur] = 0;
  cnt->heavy_count = 0;
  cnt->rc[cur] = INF32;
  cnt->rounds += 1;
  cnt->aux[1] ^= 1ull;
  cnt->mode = cnt->wl_count[nxt] * kPullFrontier > n;
  if (cnt->wl_count[nxt] == 0 || (long long)cnt->rounds >= (long long)max_rounds) cnt->done = 1;
}

// Closes a push round.  n_pull (0: no pulls): the vertices of a run that may pull but whose
// rounds are enqueued without it; a frontier to pull from stops the group, and the first
// round of the next one is a pull that passes over no row for its word (cnt->rc).
__global__ void k_sssp_end(Counters* cnt, int max_rounds, uint32_t n_pull) {
  if (threadIdx.x != 0 || cnt->done) return;
  const int cur = (int)(cnt->aux[1] & 1), nxt = cur ^ 1;
  cnt->aux[6] += cnt->wl_count[cur];  // frontier vertices processed
  cnt->wl_count[cur] = 0;
  cnt->heavy_count = 0;
  cnt->rounds += 1;
  cnt->aux[1] ^= 1ull;
  if (cnt->wl_count[nxt] == 0 || (long long)cnt->rounds >= (long long)max_rounds) {
    cnt->done = 1;
  } else if (n_pull && cnt->wl_count[nxt] * kPullFrontier > n_pull) {
    cnt->mode = 1;
    cnt->rc[nxt] = 0;
    cnt->done = 1;
  }
}

__global__ void k_sssp_resume(Counters* cnt) {
  if (threadIdx.x == 0) cnt->done = 0;
}

__global__ void k_sssp_init(uint32_t n, unsigned long long* dp, uint32_t src) {
  uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n) return;
  dp[v] = (v == src) ? (unsigned long long)src : ((unsigned long long)INF32 << 32) | v;
}

__global__ void k_sssp_seed(unsigned long long* seeds, uint32_t* wl0, uint32_t* bits0, uint32_t src) {
  if (threadIdx.x) return;
  *seeds = 1;
  wl0[0] = src;
  bits0[src >> 5] = 1u << (src & 31);
}

// Start of a query: list 0 holds the pending seeds; the round state starts clear.
__global__ void k_sssp_begin(Counters* cnt, unsigned long long* seeds) {
  if (threadIdx.x) return;
  cnt->wl_count[0] = *seeds;
  *seeds = 0;
  cnt->wl_count[1] = 0;
  cnt->heavy_count = 0;
  cnt->aux[1] = 0;
  cnt->aux[6] = 0;
  cnt->done = 0;
  cnt->rounds = 0;
  cnt->edges = 0;
  cnt->mode = 0;
  cnt->pull_rounds = 0;
  cnt->rc[0] = cnt->rc[1] = INF32;
}

// one half of the words of n vertices: the parents, or the values of the app
__global__ void __launch_bounds__(kBlock) k_sssp_unpack(uint32_t n, const unsigned long long* __restrict__ dp, int app,
                                                        int parent, uint32_t* __restrict__ out) {
  const uint32_t v = blockIdx.x * kBlock + threadIdx.x;
  if (v >= n) return;
  const unsigned long long x = dp[v];
  const uint32_t hi = (uint32_t)(x >> 32);
  out[v] = parent ? (uint32_t)x : app == SUMINC_APP_SSWP ? ~hi : hi;
}

SsspArgs sssp_args(suminc_ctx* c) {
  SsspArgs a;
  a.off = c->out_off.as<uint32_t>();
  a.col = c->out_col.as<uint32_t>();
  a.w = c->wkind == SUMINC_W_U32 && c->sssp_app != SUMINC_APP_BFS ? c->out_w.as<uint32_t>() : nullptr;
  a.dp = c->sssp_dp.as<unsigned long long>();
  a.app = c->sssp_app;
  a.wl[0] = c->sssp_wl0.as<uint32_t>();
  a.wl[1] = c->sssp_wl1.as<uint32_t>();
  a.bits[0] = c->sssp_flag0.as<uint32_t>();
  a.bits[1] = c->sssp_flag1.as<uint32_t>();
  a.heavy = c->heavy.as<uint2>();
  a.cnt = dev_counters(c);
  return a;
}

void sssp_alloc(suminc_ctx* c) {
  const size_t n = c->n;
  c->sssp_dp.ensure(n * 8);
  const size_t words = (n + 31) / 32 + 1;
  c->sssp_flag0.ensure(words * 4);
  c->sssp_flag1.ensure(words * 4);
  c->sssp_wl0.ensure(n * 4 + 4);
  c->sssp_wl1.ensure(n * 4 + 4);
  c->sssp_seeds.ensure(8);
  c->heavy.ensure_slack((c->m / kChunk + c->m / kHeavyDeg + 2) * sizeof(uint4));
}

void sssp_clear_flags(suminc_ctx* c) {
  const size_t words = ((size_t)c->n + 31) / 32 + 1;
  SUMINC_HIP(hipMemsetAsync(c->sssp_flag0.p, 0, words * 4, c->stream));
  SUMINC_HIP(hipMemsetAsync(c->sssp_flag1.p, 0, words * 4, c->stream));
}

void traversal_init(suminc_ctx* c, int app, uint32_t source) {
  SUMINC_REQUIRE(app == SUMINC_APP_SSSP || app == SUMINC_APP_BFS || app == SUMINC_APP_SSWP, SUMINC_E_INVALID,
                 "unknown traversal app");
  c->sssp_app = app;
  sssp_init(c, source);
}

void sssp_init(suminc_ctx* c, uint32_t source) {
  SUMINC_REQUIRE(c->has_graph, SUMINC_E_STATE, "no graph");
  SUMINC_REQUIRE(source < c->n, SUMINC_E_INVALID, "source out of range");
  sssp_alloc(c);
  c->sssp_src = source;
  k_sssp_init<<<grid_for(c->n), kBlock, 0, c->stream>>>(c->n, c->sssp_dp.as<unsigned long long>(), source);
  sssp_clear_flags(c);
  k_sssp_seed<<<1, 64, 0, c->stream>>>(c->sssp_seeds.as<unsigned long long>(), c->sssp_wl0.as<uint32_t>(),
                                       c->sssp_flag0.as<uint32_t>(), source);
  SUMINC_HIP(hipGetLastError());
  c->sssp_ready = true;
  c->sssp_pending = true;
}

// Runs rounds from the frontier currently held in list 0 (set by sssp_init or
// by the batch repair) until it empties.
void sssp_run(suminc_ctx* c, suminc_stats* st) {
  SUMINC_REQUIRE(c->sssp_ready, SUMINC_E_STATE, "SSSP state not initialised");
  const int max_rounds = c->prm.max_rounds > 0 ? c->prm.max_rounds : 1000000;
  SsspArgs a = sssp_args(c);
  // pulls only where they can pay: a run from scratch (a batch's seeds are few) on more
  // than a small graph
  const bool pulls = c->sssp_pending && c->m >= kPullMinEdges;
  const uint32_t tiles = (uint32_t)((c->m + kPullTile - 1) / kPullTile);
  SsspPull p{};
  if (pulls) {
    c->sssp_tile.ensure_slack(((size_t)tiles * 2 + 1) * 4);
    p.ioff = c->in_off.as<uint32_t>();
    p.icol = c->in_col.as<uint32_t>();
    p.iw = a.w ? c->in_w.as<uint32_t>() : nullptr;
    p.tile_row = c->sssp_tile.as<uint32_t>();
    p.edges = c->sssp_tile.as<uint32_t>() + tiles + 1;
    p.n = c->n;
    p.m = c->m;
  }
  c->sssp_pending = false;
  SUMINC_HIP(hipEventRecord(c->ev_start, c->stream));
  if (pulls)
    k_sssp_tiles<<<grid_for((uint64_t)tiles + 1), kBlock, 0, c->stream>>>(p.ioff, c->n, tiles,
                                                                         c->sssp_tile.as<uint32_t>());
  k_sssp_begin<<<1, 64, 0, c->stream>>>(a.cnt, c->sssp_seeds.as<unsigned long long>());
  int group = c->hint_sssp;  // rounds of the previous query + 1 first
  bool pulling = pulls && !c->hint_sssp_push;  // this group's rounds may pull
  unsigned long long pulled = 0;
  size_t slot = 0;
  while (true) {
    for (int i = 0; i < group; ++i, ++slot) {
      if (c->prof_on) SUMINC_HIP(hipEventRecord(prof_event(c, 2 * slot), c->stream));
      k_sssp_push<<<push_grid(), kBlock, 0, c->stream>>>(a);
      k_sssp_heavy<<<push_grid(), kBlock, 0, c->stream>>>(a);
      if (pulling) k_sssp_pull<<<tiles, kBlock, 0, c->stream>>>(a, p);
      if (c->prof_on) SUMINC_HIP(hipEventRecord(prof_event(c, 2 * slot + 1), c->stream));
      if (pulling) {
        k_sssp_collect<<<grid_for((c->n + 31) / 32), kBlock, 0, c->stream>>>(a, c->n);
        k_sssp_turn<<<1, 1024, 0, c->stream>>>(a.cnt, c->n, p.edges, tiles, max_rounds);
      } else {
        k_sssp_end<<<1, 64, 0, c->stream>>>(a.cnt, max_rounds, pulls ? c->n : 0u);
      }
    }
    SUMINC_HIP(hipGetLastError());
    read_counters(c);
    const Counters* h = c->host_counters;
    const unsigned long long front = h->wl_count[h->aux[1] & 1];
    if (h->done) {
      if (pulling || !pulls || front == 0 || h->rounds >= (unsigned long long)max_rounds) break;
      // stopped for its frontier: the group's other rounds did nothing
      k_sssp_resume<<<1, 64, 0, c->stream>>>(a.cnt);
      slot = (size_t)h->rounds;
      group = 8;
      pulling = true;
      continue;
    }
    if (group < 64) group *= 2;
    pulling = pulls && (h->mode != 0 || h->pull_rounds != pulled || front * kPushFrontier > c->n);
    pulled = h->pull_rounds;
  }
  SUMINC_HIP(hipEventRecord(c->ev_stop, c->stream));
  SUMINC_HIP(hipEventSynchronize(c->ev_stop));
  float ms = 0;
  SUMINC_HIP(hipEventElapsedTime(&ms, c->ev_start, c->ev_stop));
  Counters* h = c->host_counters;
  c->hint_sssp = std::max(2, std::min(64, (int)h->rounds + 1));
  if (pulls) c->hint_sssp_push = h->pull_rounds == 0;
  if (c->prof_on) {
    prof_collect(c, SUMINC_KERNEL_SSSP_PUSH, (size_t)h->rounds, 0, 2);
    suminc_kernel_profile& p = c->prof[SUMINC_KERNEL_SSSP_PUSH];
    // algorithmic bytes of the min-plus push: column + weight (8 B) and a 32-bit
    // distance read-modify-write (8 B) per edge, 16 B per frontier vertex (list
    // entry, row pointers, distance); the packed 64-bit {dist, parent} word moves
    // 8 B more per edge than this count
    p.edges += (double)h->edges;
    p.vertices += (double)h->aux[6];
    p.alg_bytes += 16.0 * (double)h->edges + 16.0 * (double)h->aux[6];
  }
  c->stats = suminc_stats{};
  c->stats.rounds = (double)h->rounds;
  c->stats.edges_traversed = (double)h->edges;
  c->stats.kernel_ms = ms;
  c->stats.pull_rounds = (double)h->pull_rounds;
  c->stats.push_rounds = (double)(h->rounds - h->pull_rounds);
  if (st) *st = c->stats;
  // leave list 0 as the (empty) current list for the next repair
  const int cur = (int)(h->aux[1] & 1);
  SUMINC_REQUIRE(h->wl_count[cur] == 0 || h->rounds < (unsigned long long)max_rounds, SUMINC_E_NOT_CONVERGED,
                 "round cap reached with a non-empty frontier");
  if (cur != 0) {
    // swap buffers so that list/bitmap 0 is current
    c->sssp_wl0.swap(c->sssp_wl1);
    c->sssp_flag0.swap(c->sssp_flag1);
  }
}

// the next frontier (list 1 after a round) becomes the pending seeds of list 0
__global__ void k_sssp_carry(const Counters* cnt, unsigned long long* seeds) {
  if (threadIdx.x == 0) *seeds = cnt->wl_count[1];
}

// One min-plus round from the pending frontier (the seeds of init or a batch, or
// the previous step's output): tjnsssp::g_function + setCurSize/getAllSize
// (sum_sync_traversal_worker.h:1090, 1136-1142).  The frontier the round produced
// becomes the pending one; *frontier_out gets its size (0: fixed point).
void sssp_step(suminc_ctx* c, uint32_t* frontier_out) {
  SUMINC_REQUIRE(c->sssp_ready, SUMINC_E_STATE, "SSSP state not initialised");
  SsspArgs a = sssp_args(c);
  c->sssp_pending = false;
  k_sssp_begin<<<1, 64, 0, c->stream>>>(a.cnt, c->sssp_seeds.as<unsigned long long>());
  k_sssp_push<<<push_grid(), kBlock, 0, c->stream>>>(a);
  k_sssp_heavy<<<push_grid(), kBlock, 0, c->stream>>>(a);
  k_sssp_end<<<1, 64, 0, c->stream>>>(a.cnt, 1 << 30, 0);
  k_sssp_carry<<<1, 64, 0, c->stream>>>(a.cnt, c->sssp_seeds.as<unsigned long long>());
  SUMINC_HIP(hipGetLastError());
  read_counters(c);
  const Counters* h = c->host_counters;
  c->stats = suminc_stats{};
  c->stats.rounds = 1;
  c->stats.edges_traversed = (double)h->edges;
  c->stats.push_rounds = 1;
  // list 1 holds the next frontier with its bitmap: make it list 0
  c->sssp_wl0.swap(c->sssp_wl1);
  c->sssp_flag0.swap(c->sssp_flag1);
  if (frontier_out) *frontier_out = (uint32_t)h->wl_count[1];
}

void sssp_download(suminc_ctx* c, uint32_t* dist, uint32_t* parent) {
  SUMINC_REQUIRE(c->sssp_ready, SUMINC_E_STATE, "SSSP state not initialised");
  auto unpack = [c](int part, uint64_t first, uint64_t count, void* out) {
    k_sssp_unpack<<<grid_for(count), kBlock, 0, c->stream>>>(
        (uint32_t)count, c->sssp_dp.as<unsigned long long>() + first, c->sssp_app, part, reinterpret_cast<uint32_t*>(out));
  };
  uint32_t* to[2] = {dist, parent};
  if (readback(c, {{dist, c->n, 4}, {parent, c->n, 4}}, unpack)) return;
  DevBuf tmp;
  tmp.ensure((size_t)c->n * 4);
  for (int k = 0; k < 2; ++k) {
    if (!to[k]) continue;
    unpack(k, 0, c->n, tmp.p);
    SUMINC_HIP(hipGetLastError());
    SUMINC_HIP(hipMemcpyAsync(to[k], tmp.p, (size_t)c->n * 4, hipMemcpyDeviceToHost, c->stream));
  }
  SUMINC_HIP(hipStreamSynchronize(c->stream));
}

}  // namespace suminc
