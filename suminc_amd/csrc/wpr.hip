// wpr.hip -- weighted personalized PageRank and its adjoint on the device.
//
// No reference counterpart: the reference's nearest app is the weighted
// personalized PHP Ingress (php/php_ingress.h:15-120), and nothing in it has
// gradients.  The forward keeps the delta-accumulative form of the plain path:
//   r = (1-d) p + d W^T r,  W[u,v] = w_uv / s_u,  s_u = sum_k w_uk (rows of
//   dangling vertices are zero, their mass leaks like the plain path's),
// computed as r = sum_t delta_t with delta_0 = (1-d) p, delta_{t+1} = d W^T delta_t:
// a pull over the in-CSR (CSC) with per-edge coefficient a_e = d w_e / s_src.
// The adjoint of L = sum_i c_i r_i is the same delta iteration on the transpose
// graph (the out-CSR): lambda = sum_t mu_t, mu_0 = c, mu_{t+1} = d W mu_t, and
//   dL/dp_v    = (1-d) lambda_v
//   dL/dw_uv   = (d r_u / s_u) (lambda_v - sum_k W[u,k] lambda_k).
//
// Rows are classified once per graph version and direction (short rows: one
// thread; medium: one wave; long: 2048-edge chunks with one atomic each), so a
// round has no per-edge atomics.  State: FP32 deltas with Kahan-compensated FP32
// sums, or FP64; the stop rule and every residual are FP64 block partials.
#include <cstring>
#include <mutex>
#include <rocprim/rocprim.hpp>

#include "ctx.hpp"
#include "device.hpp"
#include "extrap.hpp"
#include "pr.hpp"
#include "readback.hpp"

namespace suminc {

// ---- row classes of one direction -----------------------------------------------
__global__ void k_wpr_lists(uint32_t n, const uint32_t* off, uint32_t* short_list, uint32_t* wave_list, uint2* heavy,
                            unsigned long long* counts) {
  uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t deg = v < n ? off[v + 1] - off[v] : 0;
  const bool is_short = deg >= 1 && deg <= kPullThread;
  const bool is_wave = deg > kPullThread && deg <= kHeavyDeg;
  unsigned long long s1 = wave_append(is_short, &counts[0]);
  if (is_short) short_list[s1] = v;
  unsigned long long s2 = wave_append(is_wave, &counts[1]);
  if (is_wave) wave_list[s2] = v;
  if (deg > kHeavyDeg) {
    uint32_t nch = (deg + kChunk - 1) / kChunk;
    unsigned long long slot = atomicAdd(&counts[2], (unsigned long long)nch);
    for (uint32_t k = 0; k < nch; ++k) heavy[slot + k] = make_uint2(v, k);
  }
}

struct RowLists {
  const uint32_t* off;
  const uint32_t* col;
  const uint32_t* shrt;
  const uint32_t* wave;
  const uint2* heavy;
  uint32_t n_short, n_wave;
  uint64_t n_heavy;
};

// Sum of a[k] * x[col[k]] over k = k0 + r * stride (r < U, k < e).  The U column
// and coefficient loads are issued before the U gathers, so a thread keeps U
// independent gathers in flight.
template <class T, int U>
__device__ __forceinline__ T spmv_sum(const uint32_t* __restrict__ col, const T* __restrict__ a,
                                      const T* __restrict__ x, uint32_t k0, uint32_t stride, uint32_t e) {
  uint32_t u[U];
  T w[U];
#pragma unroll
  for (int r = 0; r < U; ++r) {
    const uint32_t k = k0 + r * stride;
    const bool in = k < e;
    u[r] = in ? col[k] : 0u;
    w[r] = in ? a[k] : T(0);
  }
  T acc = T(0);
#pragma unroll
  for (int r = 0; r < U; ++r)
    if (w[r] != T(0)) acc += w[r] * x[u[r]];
  return acc;
}

// y[v] = sum_{e in row v} a[e] x[col[e]]; y must be zero before (heavy rows add).
// One launch for the three row classes: workgroups [0, gh) take the heavy
// chunks (one workgroup per chunk, one atomic), [gh, gh + gw) the wave rows (one
// wave per row), the rest the short rows (one thread per row).
template <class T>
__global__ void __launch_bounds__(kBlock) k_spmv(RowLists L, const T* __restrict__ a, const T* __restrict__ x,
                                                 T* __restrict__ y, const Counters* cnt, uint32_t gh, uint32_t gw) {
  __shared__ T s_red[kBlock / 64];
  if (cnt && cnt->done) return;
  const uint32_t bid = blockIdx.x;
  if (bid < gh) {
    for (uint64_t h = bid; h < L.n_heavy; h += gh) {
      const uint2 ch = L.heavy[h];
      const uint32_t b = L.off[ch.x] + ch.y * kChunk;
      const uint32_t e = min(L.off[ch.x + 1], b + kChunk);
      T acc = spmv_sum<T, kChunk / kBlock>(L.col, a, x, b + threadIdx.x, kBlock, e);
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
      if (lane_id() == 0) s_red[threadIdx.x >> 6] = acc;
      __syncthreads();
      if (threadIdx.x == 0) {
        T s = T(0);
        for (int w = 0; w < kBlock / 64; ++w) s += s_red[w];
        if (s != T(0)) atomicAdd(&y[ch.x], s);
      }
      __syncthreads();
    }
  } else if (bid < gh + gw) {
    const uint32_t waves = gw * (kBlock / 64);
    for (uint32_t i = (bid - gh) * (kBlock / 64) + (threadIdx.x >> 6); i < L.n_wave; i += waves) {
      const uint32_t v = L.wave[i];
      const uint32_t b = L.off[v], e = L.off[v + 1];
      T acc = T(0);
      for (uint32_t k = b + lane_id(); k < e; k += 4 * 64) acc += spmv_sum<T, 4>(L.col, a, x, k, 64, e);
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
      if (lane_id() == 0) y[v] = acc;
    }
  } else {
    const uint32_t nb = gridDim.x - gh - gw;
    for (uint32_t i = (bid - gh - gw) * kBlock + threadIdx.x; i < L.n_short; i += nb * kBlock) {
      const uint32_t v = L.shrt[i];
      const uint32_t b = L.off[v], e = L.off[v + 1];
      T acc = T(0);
      for (uint32_t k = b; k < e; k += 4) acc += spmv_sum<T, 4>(L.col, a, x, k, 1, e);
      y[v] = acc;
    }
  }
}

template <class T>
__device__ __forceinline__ void kahan(T* sum, float* comp, uint32_t v, T x) {
  if constexpr (sizeof(T) == 4) {
    float r = sum[v], cc = comp[v];
    float yv = (float)x - cc;
    float t = r + yv;
    comp[v] = (t - r) - yv;
    sum[v] = t;
  } else {
    sum[v] += x;
  }
}

// A series' rounds: product, count, decision, step.  The decision comes before the
// step, so that a step can be an extrapolation (extrap.hpp) at no further array: x and y
// are its two points.  Up to kBlock partials (2^18 vertices) every workgroup of the step
// decides by itself (k_wpr_turn), which spares a launch of the four: the adjoint on a random
// bipartite graph of 16,384 vertices, which never lines up, takes 59 rounds in 1.15 ms
// (1.59 with a launch for the decision and groups that doubled; 1.52 for as many plain
// rounds of three launches).
// The vertex passes of a round take kStepPer vertices a thread (vertex base +
// j * kBlock + t, coalesced), their loads issued first.  k_wpr_count: FP64 block
// partials of sum |y|, and with a candidate extrapolation (cnt->ex.cand > 0) of the
// extrapolated sum in the second gridDim.x partials.  k_wpr_step, after the decision:
// sum += x (compensated) and x <- y, or with a chosen extrapolation beta (extrap.hpp)
// sum += (1 + beta) x and x <- y + beta (y - x); y <- 0.
constexpr int kStepPer = 4;

template <class T>
__global__ void __launch_bounds__(kBlock) k_wpr_count(uint32_t n, const T* __restrict__ x, const T* __restrict__ y,
                                                      double* __restrict__ partial, const Counters* cnt,
                                                      const Extrap* __restrict__ ex) {
  __shared__ double s_p[2][kBlock / 64];
  if (cnt->done) return;
  const double cand = ex->cand;
  const uint32_t base = blockIdx.x * (kBlock * kStepPer);
  T xo[kStepPer], xn[kStepPer];
#pragma unroll
  for (int j = 0; j < kStepPer; ++j) {
    const uint32_t v = base + j * kBlock + threadIdx.x;
    xn[j] = v < n ? y[v] : T(0);
    xo[j] = cand > 0.0 && v < n ? x[v] : T(0);
  }
  double a = 0, e = 0;
#pragma unroll
  for (int j = 0; j < kStepPer; ++j) {
    a += fabs((double)xn[j]);
    if (cand > 0.0) e += fabs((double)extrap_value<T>(xn[j], xo[j], cand));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    a += __shfl_xor(a, o);
    e += __shfl_xor(e, o);
  }
  if (lane_id() == 0) {
    s_p[0][threadIdx.x >> 6] = a;
    s_p[1][threadIdx.x >> 6] = e;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    double t = 0;
    for (int w = 0; w < kBlock / 64; ++w) t += s_p[threadIdx.x][w];
    partial[(size_t)threadIdx.x * gridDim.x + blockIdx.x] = t;
  }
}

template <class T>
__device__ __forceinline__ void wpr_step_load(uint32_t n, const T* __restrict__ x, const T* __restrict__ y,
                                              T (&xo)[kStepPer], T (&xn)[kStepPer]) {
  const uint32_t base = blockIdx.x * (kBlock * kStepPer);
#pragma unroll
  for (int j = 0; j < kStepPer; ++j) {
    const uint32_t v = base + j * kBlock + threadIdx.x;
    xo[j] = v < n ? x[v] : T(0);
    xn[j] = v < n ? y[v] : T(0);
  }
}

template <class T>
__device__ __forceinline__ void wpr_step(uint32_t n, T* __restrict__ x, T* __restrict__ y, T* __restrict__ sum,
                                         float* __restrict__ comp, double beta, const uint32_t* __restrict__ pos,
                                         T* __restrict__ xc, const T (&xo)[kStepPer], T (&xn)[kStepPer]) {
  const uint32_t base = blockIdx.x * (kBlock * kStepPer);
#pragma unroll
  for (int j = 0; j < kStepPer; ++j) {
    const uint32_t v = base + j * kBlock + threadIdx.x;
    if (v < n) {
      if (beta > 0.0) {
        if (xo[j] != T(0)) rank_add_wide<T>(sum, comp, v, (1.0 + beta) * (double)xo[j]);
        xn[j] = extrap_value<T>(xn[j], xo[j], beta);
      } else if (xo[j] != T(0)) {
        kahan(sum, comp, v, xo[j]);
      }
      x[v] = xn[j];
      y[v] = T(0);
      if (pos && pos[v] != INF32) xc[pos[v]] = xn[j];  // the next round gathers the compact copy
    }
  }
}

template <class T>
__global__ void __launch_bounds__(kBlock) k_wpr_step(uint32_t n, T* __restrict__ x, T* __restrict__ y,
                                                     T* __restrict__ sum, float* __restrict__ comp,
                                                     const Counters* cnt, const uint32_t* __restrict__ pos,
                                                     T* __restrict__ xc) {
  if (cnt->done) return;
  T xo[kStepPer], xn[kStepPer];
  wpr_step_load<T>(n, x, y, xo, xn);
  wpr_step<T>(n, x, y, sum, comp, cnt->ex.beta, pos, xc, xo, xn);
}

// l1: sum |seed|; the series stops at tol (relative: times l1).
__global__ void __launch_bounds__(1024) k_wpr_decide(const double* __restrict__ partial, uint32_t nparts,
                                                     Counters* cnt, const double* __restrict__ l1, double tol_abs,
                                                     int relative, int max_rounds,
                                                     unsigned long long edges_per_round) {
  __shared__ double s[1024 / 64][2];
  if (cnt->done) return;
  sum_parts<2, 0u>(partial, nparts, s);
  if (threadIdx.x) return;
  const double tol = relative ? tol_abs * *l1 : tol_abs;
  const double s1 = s[0][0];
  const double r = extrap_decide(cnt->ex, s1, s[0][1], tol);
  cnt->dpad[0] = tol;
  cnt->residual = r;
  cnt->rounds += 1;
  cnt->edges += edges_per_round;
  if (s1 != s1 || s1 > 1e300) cnt->aux[0] = 1;
  if (!(r >= tol) || (long long)cnt->rounds >= (long long)max_rounds || cnt->aux[0]) cnt->done = 1;
}

// Decision and step of a round (its number from 0), gridDim.x <= kBlock: the same sums in
// every workgroup, so the same decision.  The state it comes from is left alone
// (ex2[round & 1]); the first workgroup writes the next one's and the counters.  One that
// begins after the first has stopped the series finds `done` and would have stopped too.
template <class T>
__global__ void __launch_bounds__(kBlock) k_wpr_turn(uint32_t n, T* __restrict__ x, T* __restrict__ y,
                                                     T* __restrict__ sum, float* __restrict__ comp, Counters* cnt,
                                                     const uint32_t* __restrict__ pos, T* __restrict__ xc,
                                                     const double* __restrict__ partial,
                                                     const double* __restrict__ l1, double tol_abs, int relative,
                                                     int round, int max_rounds, unsigned long long edges_per_round) {
  __shared__ double s[kBlock / 64][2];
  __shared__ double s_beta;
  __shared__ int s_done, s_stop;
  // everything that the decision and the step read, before either waits for it
  T xo[kStepPer], xn[kStepPer];
  wpr_step_load<T>(n, x, y, xo, xn);
  Extrap ex = cnt->ex2[round & 1];
  if (threadIdx.x == 0)  // one read for the workgroup: `done` may change meanwhile
    s_done = __hip_atomic_load(&cnt->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
  sum_parts<2, 0u, kBlock>(partial, gridDim.x, s);  // waits for the workgroup
  if (s_done) return;
  if (threadIdx.x == 0) {
    const double tol = relative ? tol_abs * *l1 : tol_abs;
    const double s1 = s[0][0];
    const double r = extrap_decide(ex, s1, s[0][1], tol);
    const bool failed = s1 != s1 || s1 > 1e300;
    s_beta = ex.beta;
    s_stop = !(r >= tol) || round + 1 >= max_rounds || failed;
    if (blockIdx.x == 0) {
      cnt->ex2[~round & 1] = ex;
      cnt->ex = ex;
      cnt->dpad[0] = tol;
      cnt->residual = r;
      cnt->rounds = round + 1;
      cnt->edges += edges_per_round;
      if (failed) cnt->aux[0] = 1;
      if (s_stop) __hip_atomic_store(&cnt->done, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  __syncthreads();
  if (!s_stop) wpr_step<T>(n, x, y, sum, comp, s_beta, pos, xc, xo, xn);
}

// x = scale * seed, y = sum = 0; block partials of sum |x|
template <class T>
__global__ void __launch_bounds__(kBlock) k_wpr_seed(uint32_t n, const float* __restrict__ src, T scale,
                                                     T* __restrict__ x, T* __restrict__ y, T* __restrict__ sum,
                                                     float* __restrict__ comp, double* __restrict__ partial,
                                                     const uint32_t* __restrict__ pos, T* __restrict__ xc) {
  __shared__ double s_p[kBlock / 64];
  const uint32_t v = blockIdx.x * kBlock + threadIdx.x;
  double a = 0;
  if (v < n) {
    const T s = scale * (T)src[v];
    x[v] = s;
    if (pos && pos[v] != INF32) xc[pos[v]] = s;
    y[v] = T(0);
    sum[v] = T(0);
    comp[v] = 0.f;
    a = fabs((double)s);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o);
  if (lane_id() == 0) s_p[threadIdx.x >> 6] = a;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0;
    for (int w = 0; w < kBlock / 64; ++w) t += s_p[w];
    partial[blockIdx.x] = t;
  }
}

// zeroes the counters block (a kernel, not a memset: callers may capture the series)
__global__ void k_wpr_clear(Counters* cnt) {
  if (threadIdx.x == 0) {
    Counters z{};
    *cnt = z;
  }
}

// sum |seed| of the block partials, the first residual of the series' ratios
__global__ void __launch_bounds__(1024) k_wpr_start(const double* __restrict__ partial, uint32_t nparts, double* l1,
                                                    Counters* cnt) {
  __shared__ double s[1024 / 64][1];
  sum_parts<1, 0u>(partial, nparts, s);
  if (threadIdx.x == 0) {
    *l1 = s[0][0];
    cnt->ex.last = cnt->ex2[0].last = s[0][0];
  }
}

// the step of the round that stopped, and the last delta (it belongs to the series)
template <class T>
__global__ void k_wpr_finish(uint32_t n, const T* __restrict__ x, const T* __restrict__ y, T* __restrict__ sum,
                             float* __restrict__ comp, const Counters* cnt, float* __restrict__ out32,
                             double* __restrict__ out64) {
  const uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n) return;
  const double beta = cnt->ex.beta;
  const T xo = x[v];
  T xn = y[v];
  if (beta > 0.0) {
    if (xo != T(0)) rank_add_wide<T>(sum, comp, v, (1.0 + beta) * (double)xo);
    xn = extrap_value<T>(xn, xo, beta);
  } else if (xo != T(0)) {
    kahan(sum, comp, v, xo);
  }
  if (xn != T(0)) kahan(sum, comp, v, xn);
  double val = (double)sum[v];
  if constexpr (sizeof(T) == 4) val -= (double)comp[v];
  if (out32) out32[v] = (float)val;
  if (out64) out64[v] = val;
}

// Wave-per-row kernels stride over the rows with at most this many workgroups (a
// grid of one wave per row would pass 2^32 threads at 2^26 rows).
constexpr unsigned kWaveGrid = 65536;

// ---- per-edge passes over the out-CSR --------------------------------------------
// Half of R-MAT's rows are empty and most of the others short, so a wave a row left
// most lanes idle (2^22 vertices, 50M edges: row sums 1.55 ms, coefficients 1.81 ms,
// gradients 4.04 ms, each against about 0.1 ms for the bytes).  Sums over rows take the
// row classes with 8 lanes a short row (k_row_sum: 0.17 ms); passes that only need to
// know an edge's row take tiles of consecutive edges whatever the rows
// (for_tile_edges: coefficients 0.19 ms, gradients 0.41 ms, bound by the gather of
// lambda).

// Per-edge terms of the row sums.
struct TermWeight {  // w_uv
  const float* w;
  __device__ double operator()(uint32_t e) const { return (double)w[e]; }
};
struct TermPhp {  // w_uv, edges into the source left out; integer, float or unit weights
  const uint32_t* col;
  const uint32_t* wu;
  const float* wf;
  uint32_t src;
  __device__ double operator()(uint32_t e) const {
    return col[e] == src ? 0.0 : wu ? (double)wu[e] : wf ? (double)wf[e] : 1.0;
  }
};
struct TermDot {  // w_uv x_v
  const float* w;
  const uint32_t* col;
  const double* x;
  __device__ double operator()(uint32_t e) const { return (double)w[e] * x[col[e]]; }
};

// out[v] = FP64 sum of f over the edges of row v, the rows with edges (a row of more
// than kHeavyDeg: its chunks' sums in part, k_row_sum_heavy adds them), in a fixed order.
// Workgroups as k_spmv's.
template <class F>
__global__ void __launch_bounds__(kBlock) k_row_sum(RowLists L, F f, double* __restrict__ out,
                                                    double* __restrict__ part, uint32_t gh, uint32_t gw) {
  __shared__ double s_red[kBlock / 64];
  const uint32_t bid = blockIdx.x;
  if (bid < gh) {
    for (uint64_t h = bid; h < L.n_heavy; h += gh) {
      const uint2 ch = L.heavy[h];
      const uint32_t b = L.off[ch.x] + ch.y * kChunk;
      const uint32_t e = min(L.off[ch.x + 1], b + kChunk);
      double acc = 0;
      for (uint32_t k = b + threadIdx.x; k < e; k += kBlock) acc += f(k);
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
      if (lane_id() == 0) s_red[threadIdx.x >> 6] = acc;
      __syncthreads();
      if (threadIdx.x == 0) {
        double t = 0;
        for (int w = 0; w < kBlock / 64; ++w) t += s_red[w];
        part[h] = t;
      }
      __syncthreads();
    }
    return;
  }
  const bool wave = bid < gh + gw;
  const uint32_t lanes = wave ? 64u : 8u;
  const uint32_t groups = (wave ? gw : gridDim.x - gh - gw) * (kBlock / lanes);
  const uint32_t first = (bid - gh - (wave ? 0u : gw)) * (kBlock / lanes) + threadIdx.x / lanes;
  const uint32_t count = wave ? L.n_wave : L.n_short;
  const uint32_t* list = wave ? L.wave : L.shrt;
  const uint32_t lane = threadIdx.x & (lanes - 1);
  // whole waves: the shuffles below need every lane of a group
  for (uint32_t i = first; i - threadIdx.x / lanes % (64 / lanes) < count; i += groups) {
    double acc = 0;
    const uint32_t v = i < count ? list[i] : 0u;
    if (i < count) {
      const uint32_t e = L.off[v + 1];
      for (uint32_t k = L.off[v] + lane; k < e; k += lanes) acc += f(k);
    }
    for (uint32_t o = lanes >> 1; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
    if (lane == 0 && i < count) out[v] = acc;
  }
}

// One wave per row of more than kHeavyDeg edges (the entries of chunk 0; a row's
// chunks follow each other): its chunk sums added up.
__global__ void __launch_bounds__(kBlock) k_row_sum_heavy(RowLists L, const double* __restrict__ part,
                                                          double* __restrict__ out) {
  const uint64_t h = (uint64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  if (h >= L.n_heavy) return;
  const uint2 ch = L.heavy[h];
  if (ch.y != 0) return;
  const uint32_t nch = (L.off[ch.x + 1] - L.off[ch.x] + kChunk - 1) / kChunk;
  double acc = 0;
  for (uint32_t k = lane_id(); k < nch; k += 64) acc += part[h + k];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
  if (lane_id() == 0) out[ch.x] = acc;
}

// A tile of kTileE consecutive edges of a CSR per workgroup; tile_row[t] is the row of
// edge t * kTileE (tile_row[tiles]: the last row), made once per graph.
constexpr uint32_t kTileE = 2048;

__global__ void k_tile_rows(const uint32_t* __restrict__ off, uint32_t n, uint64_t m, uint32_t tiles,
                            uint32_t* __restrict__ tile_row) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t > tiles) return;
  if (t == tiles) {
    tile_row[t] = n - 1;
    return;
  }
  const uint32_t e = t * kTileE;
  uint32_t lo = 0, hi = n - 1;  // the last row that starts at or before e is the row of e
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo + 1) / 2;
    if (off[mid] <= e) lo = mid; else hi = mid - 1;
  }
  tile_row[t] = lo;
}

// fn(edge, row) for the edges of the workgroup's tile, consecutive threads taking
// consecutive edges.  Every row that starts inside the tile marks its first edge; a
// running maximum over the tile gives each edge its row.
template <class Fn>
__device__ __forceinline__ void for_tile_edges(const uint32_t* __restrict__ off, uint64_t m,
                                               const uint32_t* __restrict__ tile_row, Fn&& fn) {
  constexpr int kPer = kTileE / kBlock;
  __shared__ uint32_t s_row[kTileE];
  __shared__ uint32_t s_w[kBlock / 64];
  const uint32_t t = blockIdx.x;
  const uint64_t e0 = (uint64_t)t * kTileE;
  const uint32_t ne = (uint32_t)(m - e0 < kTileE ? m - e0 : kTileE);
  const uint32_t r0 = tile_row[t], r1 = tile_row[t + 1];
  if (r1 - r0 > 32 * kTileE) {  // mostly empty rows: a search per edge passes over fewer of them
    for (uint32_t i = threadIdx.x; i < ne; i += kBlock) {
      const uint32_t e = (uint32_t)e0 + i;
      uint32_t lo = r0, hi = r1;
      while (lo < hi) {
        const uint32_t mid = lo + (hi - lo + 1) / 2;
        if (off[mid] <= e) lo = mid; else hi = mid - 1;
      }
      fn(e, lo);
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < kPer; ++j) s_row[j * kBlock + threadIdx.x] = 0;
  __syncthreads();
  for (uint32_t r = r0 + 1 + threadIdx.x; r <= r1; r += kBlock) {
    const uint32_t b = off[r], e = off[r + 1];
    if (e > b && b - e0 < ne) s_row[b - (uint32_t)e0] = r - r0;
  }
  __syncthreads();
  uint32_t x[kPer], run = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    run = max(run, s_row[threadIdx.x * kPer + j]);
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
  for (int j = 0; j < kPer; ++j) s_row[threadIdx.x * kPer + j] = max(before, x[j]);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const uint32_t i = j * kBlock + threadIdx.x;
    if (i < ne) fn((uint32_t)e0 + i, r0 + s_row[i]);
  }
}

// a_e = d f(e) / s_row
template <class T, class F>
__global__ void __launch_bounds__(kBlock) k_wpr_coef(const uint32_t* __restrict__ off, uint64_t m,
                                                     const uint32_t* __restrict__ tile_row, F f,
                                                     const double* __restrict__ s, double d, T* __restrict__ a) {
  for_tile_edges(off, m, tile_row, [&](uint32_t e, uint32_t v) {
    const double sv = s[v];
    const double inv = sv > 0 ? d / sv : 0.0;
    a[e] = (T)(f(e) * inv);
  });
}

// dst[i] = src[eid[i]]: the coefficients in CSC or layout order.  kGatherPer values a
// thread, their loads in flight together.
constexpr int kGatherPer = 4;
template <class T>
__global__ void __launch_bounds__(kBlock) k_wpr_gather(uint64_t m, const uint32_t* __restrict__ eid,
                                                       const T* __restrict__ src, T* __restrict__ dst) {
  const uint64_t base = (uint64_t)blockIdx.x * (kBlock * kGatherPer) + threadIdx.x;
  uint32_t e[kGatherPer];
#pragma unroll
  for (int j = 0; j < kGatherPer; ++j) e[j] = base + j * kBlock < m ? __builtin_nontemporal_load(eid + base + j * kBlock) : 0u;
  T x[kGatherPer];
#pragma unroll
  for (int j = 0; j < kGatherPer; ++j) x[j] = src[e[j]];
#pragma unroll
  for (int j = 0; j < kGatherPer; ++j)
    if (base + j * kBlock < m) __builtin_nontemporal_store(x[j], dst + base + j * kBlock);
}

// CSR edge id of every CSC position: sort (dst, src) keys with the edge index
__global__ void k_wpr_edge_keys(const uint32_t* __restrict__ off, uint32_t n, uint64_t m,
                                const uint32_t* __restrict__ col, unsigned long long* keys, uint32_t* idx) {
  const uint32_t waves = gridDim.x * (kBlock / 64);
  for (uint32_t v = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6); v < n; v += waves) {
    for (uint32_t e = off[v] + lane_id(); e < off[v + 1]; e += 64) {
      keys[e] = ((unsigned long long)col[e] << 32) | v;
      idx[e] = e;
    }
  }
  (void)m;
}

// ---- gradients -------------------------------------------------------------------
// grad_w[e] for CSR edge e = (u -> v): (d r_u / s_u) lambda_v - (r_u / s_u) y_u with
// y_u = sum_k a_uk lambda_k = (d / s_u) sum_k w_uk lambda_k.  rows: per vertex
// (d r_u / s_u, r_u y_u / s_u).
__global__ void __launch_bounds__(kBlock) k_wpr_grad_rows(uint32_t n, const double* __restrict__ s,
                                                          const double* __restrict__ r,
                                                          const double* __restrict__ dot, double d,
                                                          double2* __restrict__ rows) {
  const uint32_t u = blockIdx.x * kBlock + threadIdx.x;
  if (u >= n) return;
  const double su = s[u];
  const double ru = su > 0 ? r[u] / su : 0.0;  // a row without weight mass has no gradient
  rows[u] = make_double2(d * ru, su > 0 ? ru * (d * dot[u] / su) : 0.0);
}

__global__ void __launch_bounds__(kBlock) k_wpr_grad_w(const uint32_t* __restrict__ off,
                                                       const uint32_t* __restrict__ col, uint64_t m,
                                                       const uint32_t* __restrict__ tile_row,
                                                       const double2* __restrict__ rows,
                                                       const double* __restrict__ lam, float* __restrict__ g) {
  for_tile_edges(off, m, tile_row, [&](uint32_t e, uint32_t u) {
    const double2 x = rows[u];
    g[e] = (float)(x.x * lam[col[e]] - x.y);
  });
}

__global__ void k_wpr_grad_p(uint32_t n, const double* __restrict__ lam, double d, float* __restrict__ g) {
  const uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v < n) g[v] = (float)((1.0 - d) * lam[v]);
}

// the layout's edges as indices of the CSR: eid[i] <- csr_of[eid[i]]
__global__ void k_wpr_compose(uint64_t m, const uint32_t* __restrict__ csr_of, uint32_t* __restrict__ eid) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < m) eid[i] = csr_of[eid[i]];
}

// ---------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------
// Row lists of one direction and, on large graphs, compact positions of the
// columns (by decreasing number of appearances) with the columns renamed to them,
// so a round gathers from an array of the vertices that can be gathered at all.
struct WprDir {
  DevBuf shrt, wave, heavy, counts;
  uint64_t n_short = 0, n_wave = 0, n_heavy = 0;
  bool compact = false;
  DevBuf pos, scratch, colc;
};

static void build_lists(suminc_ctx* c, WprDir& L, const DevBuf& off) {
  const uint32_t n = c->n;
  L.shrt.ensure((size_t)n * 4 + 4);
  L.wave.ensure((size_t)n * 4 + 4);
  L.heavy.ensure((c->m / kChunk + c->m / kHeavyDeg + 2) * sizeof(uint2));
  L.counts.ensure(32);
  SUMINC_HIP(hipMemsetAsync(L.counts.p, 0, 32, c->stream));
  k_wpr_lists<<<grid_for(n), kBlock, 0, c->stream>>>(n, off.as<uint32_t>(), L.shrt.as<uint32_t>(),
                                                     L.wave.as<uint32_t>(), L.heavy.as<uint2>(),
                                                     L.counts.as<unsigned long long>());
  unsigned long long h[3];
  SUMINC_HIP(hipMemcpyAsync(h, L.counts.p, 24, hipMemcpyDeviceToHost, c->stream));
  SUMINC_HIP(hipStreamSynchronize(c->stream));
  L.n_short = h[0];
  L.n_wave = h[1];
  L.n_heavy = h[2];
}

struct WprState {
  uint64_t graph_version = ~0ull;    // version the lists / edge ids were built for
  uint64_t coef_version = ~0ull;     // weights version the coefficients belong to
  int coef_prec = -1;
  uint64_t weights_version = 0;
  bool fwd_ready = false;
  uint64_t fwd_coef_version = ~0ull;
  int hint_fwd = 12, hint_bwd = 12, hint_php = 12;  // rounds of the last run + 1: a series' first group
  WprDir out, in;
  DevBuf eid;                        // CSR edge id per CSC position
  DevBuf tile_row;                   // the row of the first edge of every edge tile of the CSR
  DevBuf row_part;                   // chunk sums of the long rows
  DevBuf s;                          // row sums (f64)
  DevBuf in_f, out_f, grad_w;        // FP32 vectors in and out of host or foreign memory
  DevBuf dot, grad_rows;             // sum_k w_uk lambda_k; the gradient's two terms per row
  DevBuf a_out, a_in;                // coefficients d w / s (T) in CSR / CSC order
  DevBuf x, y, sum, comp;            // round state (T)
  DevBuf xc;                         // x at the compact positions (large graphs)
  DevBuf r64, lam64;                 // FP64 results of the last forward / backward
  DevBuf l1;                         // sum |seed|
  DevBuf php_a_out, php_a_in, php64;  // PHP: coefficients (T) in CSR / CSC order, FP64 result
  DevBuf php_s;                      // PHP: row sums (f64)
  // binned series rounds (large graphs, the PageRank pull's rule): the forward over
  // the CSC, the adjoint over the CSR, their coefficients in layout order; built for
  // elements of bin_es bytes
  BinLayout bin_in, bin_out;
  uint64_t bin_es = 0;
};

static WprState& wstate(suminc_ctx* c) {
  if (!c->wpr) c->wpr = new WprState();
  return *reinterpret_cast<WprState*>(c->wpr);
}

void wpr_release(suminc_ctx* c) {
  delete reinterpret_cast<WprState*>(c->wpr);
  c->wpr = nullptr;
}

static void wpr_prepare_graph(suminc_ctx* c, WprState& S) {
  const uint64_t es = c->prm.pr_precision == SUMINC_PR_FP64 ? 8 : 4;
  if (S.graph_version == c->graph_version && S.bin_es == es) return;
  const uint32_t n = c->n;
  const uint64_t m = c->m;
  build_lists(c, S.out, c->out_off);
  build_lists(c, S.in, c->in_off);
  // the forward gathers over the CSC (columns: sources, counted by out-degree), the
  // adjoint over the CSR (columns: destinations, counted by in-degree)
  const bool compact = compact_pull(c, c->prm.pr_precision == SUMINC_PR_FP64 ? 8 : 4);
  S.in.compact = S.out.compact = compact && m > 0;
  if (S.in.compact) {
    build_positions_by_degree(c, c->out_off.as<uint32_t>(), c->in_off.as<uint32_t>(), c->in_col.as<uint32_t>(), m,
                              S.in.pos, S.in.scratch, S.in.colc);
    build_positions_by_degree(c, c->in_off.as<uint32_t>(), c->out_off.as<uint32_t>(), c->out_col.as<uint32_t>(),
                              m, S.out.pos, S.out.scratch, S.out.colc);
  }
  S.eid.ensure(m * 4 + 4);
  if (m) {
    DevBuf ka, kb, ia;
    ka.ensure(m * 8); kb.ensure(m * 8); ia.ensure(m * 4);
    k_wpr_edge_keys<<<grid_for(n, kBlock / 64, kWaveGrid), kBlock, 0, c->stream>>>(c->out_off.as<uint32_t>(), n, m,
                                                                       c->out_col.as<uint32_t>(),
                                                                       ka.as<unsigned long long>(), ia.as<uint32_t>());
    // keys (dst << 32 | src): the bits above 32 + log2(n) are zero
    int hi_bits = 1;
    while (hi_bits < 32 && (1ull << hi_bits) < n) ++hi_bits;
    const unsigned end_bit = 32 + hi_bits;
    size_t bytes = 0;
    SUMINC_HIP(rocprim::radix_sort_pairs(nullptr, bytes, ka.as<uint64_t>(), kb.as<uint64_t>(), ia.as<uint32_t>(),
                                         S.eid.as<uint32_t>(), (size_t)m, 0, end_bit, c->stream));
    c->tmp.ensure(bytes);
    SUMINC_HIP(rocprim::radix_sort_pairs(c->tmp.p, bytes, ka.as<uint64_t>(), kb.as<uint64_t>(), ia.as<uint32_t>(),
                                         S.eid.as<uint32_t>(), (size_t)m, 0, end_bit, c->stream));
    SUMINC_HIP(hipStreamSynchronize(c->stream));
  }
  // binned series rounds, by the PageRank pull's rule (on above 8 MiB of elements
  // or when a window is given): the gather pass multiplies by the coefficient
  S.bin_in.n_parts = S.bin_out.n_parts = 0;
  const int kib = c->prm.pull_bin_kib;
  if (m && kib >= 0 && (kib > 0 || (uint64_t)n * es > (8ull << 20))) {
    const uint64_t win = (uint64_t)(kib ? kib : 2048) * 1024;
    const unsigned long long src_in =
        S.in.compact ? nonempty_rows(c, c->out_off.as<uint32_t>(), S.bin_in.hist) : n;
    bin_layout_build(c, S.bin_in, n, c->in_off.as<uint32_t>(),
                     S.in.compact ? S.in.colc.as<uint32_t>() : c->in_col.as<uint32_t>(), src_in, es, win,
                     c->prm.pull_bin_direct, m, true);
    const unsigned long long src_out =
        S.out.compact ? nonempty_rows(c, c->in_off.as<uint32_t>(), S.bin_out.hist) : n;
    bin_layout_build(c, S.bin_out, n, c->out_off.as<uint32_t>(),
                     S.out.compact ? S.out.colc.as<uint32_t>() : c->out_col.as<uint32_t>(), src_out, es, win,
                     c->prm.pull_bin_direct, m, true);
  }
  if (S.bin_in.n_parts)  // its coefficients come from the CSR order directly
    k_wpr_compose<<<grid_for(m), kBlock, 0, c->stream>>>(m, S.eid.as<uint32_t>(), S.bin_in.eid.as<uint32_t>());
  const uint32_t tiles = (uint32_t)((m + kTileE - 1) / kTileE);
  S.tile_row.ensure((size_t)tiles * 4 + 4);
  k_tile_rows<<<grid_for((uint64_t)tiles + 1), kBlock, 0, c->stream>>>(c->out_off.as<uint32_t>(), n, m, tiles,
                                                                      S.tile_row.as<uint32_t>());
  SUMINC_HIP(hipGetLastError());
  S.row_part.ensure(S.out.n_heavy * 8 + 8);
  S.bin_es = es;
  S.graph_version = c->graph_version;
  S.coef_version = ~0ull;
  S.fwd_ready = false;
}

// compact: the renamed columns when the direction has them (then the gathered
// vector must be at the compact positions)
static RowLists lists_of(const WprDir& L, const DevBuf& off, const DevBuf& col, bool compact) {
  RowLists R;
  R.off = off.as<uint32_t>();
  R.col = compact && L.compact ? L.colc.as<uint32_t>() : col.as<uint32_t>();
  R.shrt = L.shrt.as<uint32_t>();
  R.wave = L.wave.as<uint32_t>();
  R.heavy = L.heavy.as<uint2>();
  R.n_short = (uint32_t)L.n_short;
  R.n_wave = (uint32_t)L.n_wave;
  R.n_heavy = L.n_heavy;
  return R;
}

template <class T>
static void spmv(suminc_ctx* c, const RowLists& R, const T* a, const T* x, T* y, const Counters* cnt) {
  const uint32_t gh = R.n_heavy ? push_grid() : 0u;
  const uint32_t gw = R.n_wave ? grid_for(R.n_wave, kBlock / 64, 8192) : 0u;
  const uint32_t gs = R.n_short ? grid_for(R.n_short, kBlock, 8192) : 0u;
  if (gh + gw + gs) k_spmv<T><<<gh + gw + gs, kBlock, 0, c->stream>>>(R, a, x, y, cnt, gh, gw);
}

// out = per row FP64 sums of f over the out-edges (0 for empty rows).
template <class F>
static void row_sum(suminc_ctx* c, WprState& S, F f, double* out) {
  const RowLists R = lists_of(S.out, c->out_off, c->out_col, false);
  SUMINC_HIP(hipMemsetAsync(out, 0, (size_t)c->n * 8, c->stream));
  const uint32_t gh = (uint32_t)std::min<uint64_t>(R.n_heavy, 8192);
  const uint32_t gw = R.n_wave ? grid_for(R.n_wave, kBlock / 64, 8192) : 0u;
  const uint32_t gs = R.n_short ? grid_for(R.n_short, kBlock / 8, 16384) : 0u;
  if (gh + gw + gs)
    k_row_sum<F><<<gh + gw + gs, kBlock, 0, c->stream>>>(R, f, out, S.row_part.as<double>(), gh, gw);
  if (R.n_heavy)
    k_row_sum_heavy<<<grid_for(R.n_heavy, kBlock / 64), kBlock, 0, c->stream>>>(R, S.row_part.as<double>(), out);
  SUMINC_HIP(hipGetLastError());
}

// a = d f / s in CSR order, and in CSC order for the row classes (the binned rounds
// take theirs from the CSR order).
template <class T, class F>
static void edge_coefs(suminc_ctx* c, WprState& S, F f, const double* s, double d, T* a_out, DevBuf& a_in) {
  const uint64_t m = c->m;
  if (!m) return;
  k_wpr_coef<T, F><<<(unsigned)((m + kTileE - 1) / kTileE), kBlock, 0, c->stream>>>(
      c->out_off.as<uint32_t>(), m, S.tile_row.as<uint32_t>(), f, s, d, a_out);
  if (!S.bin_in.n_parts) {
    a_in.ensure(m * sizeof(T) + 8);
    k_wpr_gather<T><<<grid_for(m, kBlock * kGatherPer), kBlock, 0, c->stream>>>(m, S.eid.as<uint32_t>(), a_out,
                                                                              a_in.as<T>());
  }
  SUMINC_HIP(hipGetLastError());
}

template <class T>
static void wpr_prepare_coef(suminc_ctx* c, WprState& S) {
  const int prec = sizeof(T) == 8 ? SUMINC_PR_FP64 : SUMINC_PR_FP32_KAHAN;
  if (S.coef_version == S.weights_version && S.coef_prec == prec) return;
  S.s.ensure((size_t)c->n * 8 + 8);
  S.a_out.ensure(c->m * sizeof(T) + 8);
  const TermWeight w{c->out_w.as<float>()};
  row_sum(c, S, w, S.s.as<double>());
  edge_coefs<T>(c, S, w, S.s.as<double>(), c->prm.damping, S.a_out.as<T>(), S.a_in);
  S.coef_version = S.weights_version;
  S.coef_prec = prec;
}

// Device buffers of one series run: the round state (x, y, the compensated sum),
// the compact copy of x (large graphs), the FP64 block partials and sum |seed|.
template <class T>
struct SeriesBufs {
  T *x, *y, *sum, *xc;
  float* comp;
  double *partial, *l1;
};

// Bytes of the series buffers for n vertices (partials: the seed pass leaves one value per
// vertex block, the count two per workgroup of kStepPer vertices a thread: room for three
// per vertex block, which also fixes the largest n that the scratch array takes).
template <class T>
static size_t series_bytes(uint32_t n, bool compact) {
  auto al = [](size_t b) { return (b + 255) & ~size_t(255); };
  const size_t g = grid_for(n);
  return 3 * al((size_t)n * sizeof(T) + 8) + (compact ? al((size_t)n * sizeof(T) + 8) : 0) + al((size_t)n * 4 + 4) +
         al((g + 1) * 8 * 3) + al(8);
}

// Carves the series buffers out of `base` (series_bytes<T>(n, compact) bytes).
template <class T>
static SeriesBufs<T> series_carve(unsigned char* base, uint32_t n, bool compact) {
  auto al = [](size_t b) { return (b + 255) & ~size_t(255); };
  const size_t g = grid_for(n);
  SeriesBufs<T> B;
  size_t o = 0;
  auto take = [&](size_t bytes) { unsigned char* p = base + o; o += al(bytes); return p; };
  B.x = reinterpret_cast<T*>(take((size_t)n * sizeof(T) + 8));
  B.y = reinterpret_cast<T*>(take((size_t)n * sizeof(T) + 8));
  B.sum = reinterpret_cast<T*>(take((size_t)n * sizeof(T) + 8));
  B.xc = compact ? reinterpret_cast<T*>(take((size_t)n * sizeof(T) + 8)) : nullptr;
  B.comp = reinterpret_cast<float*>(take((size_t)n * 4 + 4));
  B.partial = reinterpret_cast<double*>(take((g + 1) * 8 * 3));
  B.l1 = reinterpret_cast<double*>(take(8));
  return B;
}

// The series buffers in the context's weighted-PageRank state (grown on demand).
template <class T>
static SeriesBufs<T> series_state(suminc_ctx* c, WprState& S, bool compact) {
  const uint32_t n = c->n;
  S.x.ensure((size_t)n * sizeof(T) + 8);
  if (compact) S.xc.ensure((size_t)n * sizeof(T) + 8);
  S.y.ensure((size_t)n * sizeof(T) + 8);
  S.sum.ensure((size_t)n * sizeof(T) + 8);
  S.comp.ensure((size_t)n * 4 + 4);
  S.l1.ensure(8);
  c->partial.ensure((size_t)(grid_for(n) + 1) * 8 * 3);
  SeriesBufs<T> B;
  B.x = S.x.as<T>();
  B.y = S.y.as<T>();
  B.sum = S.sum.as<T>();
  B.xc = compact ? S.xc.as<T>() : nullptr;
  B.comp = S.comp.as<float>();
  B.partial = c->partial.as<double>();
  B.l1 = S.l1.as<double>();
  return B;
}

// Runs sum = sum_t x_t with x_{t+1} = A x_t from x_0 = scale * seed until
// sum|x| < tol.  A's coefficients: a in the order of R's rows, a_csr in the CSR's (the
// binned rounds).  Result (FP64) in out64, optionally FP32 in out32 (either may be
// null); a series that fails leaves out32 alone unless out32_always.  hint: the rounds to
// enqueue first, then what the next run of this series is to.  pos != nullptr: R's columns are compact positions, and the rounds
// gather the compact copy of x (B.xc).  Allocates nothing itself.
template <class T>
static void wpr_series(suminc_ctx* c, int& hint, const SeriesBufs<T>& B, const RowLists& R, const BinLayout* L,
                       const uint32_t* pos, const T* a, const T* a_csr, const float* seed_dev, T scale, double tol_abs, bool relative,
                       float* out32, double* out64, suminc_stats* st, bool out32_always = false) {
  const uint32_t n = c->n;
  // the binned layout of R's direction when it exists: its coefficients taken in layout
  // order, the rounds through the gather and summing passes
  const bool binned = L && L->n_parts;
  if (binned && L->m)
    k_wpr_gather<T><<<grid_for(L->m, kBlock * kGatherPer), kBlock, 0, c->stream>>>(L->m, L->eid.as<uint32_t>(), a_csr,
                                                                                  L->coef.as<T>());
  T* xc = pos ? B.xc : nullptr;
  const unsigned g = grid_for(n);
  const unsigned gs = grid_for(n, kBlock * kStepPer);  // the round's vertex pass and its partials
  Counters* cnt = dev_counters(c);
  k_wpr_clear<<<1, 64, 0, c->stream>>>(cnt);
  k_wpr_seed<T><<<g, kBlock, 0, c->stream>>>(n, seed_dev, scale, B.x, B.y, B.sum, B.comp, B.partial, pos, xc);
  k_wpr_start<<<1, 1024, 0, c->stream>>>(B.partial, g, B.l1, cnt);
  const int max_rounds = c->prm.max_rounds > 0 ? c->prm.max_rounds : 100000;
  SUMINC_HIP(hipEventRecord(c->ev_start, c->stream));
  // extrapolated series take 9-20 rounds, others up to hundreds, loose tolerances one or
  // two; a look at the counters costs about as much as three empty rounds
  int group = hint, enqueued = 0;
  const bool turn = gs <= (unsigned)kBlock;
  while (true) {
    for (int i = 0; i < group; ++i, ++enqueued) {
      if (binned) bin_layout_spmv<T, true>(c, *L, pos ? xc : B.x, B.y, cnt, 2);
      else spmv<T>(c, R, a, pos ? xc : B.x, B.y, cnt);
      k_wpr_count<T><<<gs, kBlock, 0, c->stream>>>(n, B.x, B.y, B.partial, cnt,
                                                  turn ? &cnt->ex2[enqueued & 1] : &cnt->ex);
      if (turn) {
        k_wpr_turn<T><<<gs, kBlock, 0, c->stream>>>(n, B.x, B.y, B.sum, B.comp, cnt, pos, xc, B.partial, B.l1, tol_abs,
                                                   relative, enqueued, max_rounds, c->m);
        continue;
      }
      k_wpr_decide<<<1, 1024, 0, c->stream>>>(B.partial, gs, cnt, B.l1, tol_abs, relative, max_rounds, c->m);
      k_wpr_step<T><<<gs, kBlock, 0, c->stream>>>(n, B.x, B.y, B.sum, B.comp, cnt, pos, xc);
    }
    SUMINC_HIP(hipGetLastError());
    read_counters(c);
    if (c->host_counters->done) break;
    group = enqueued < 12 ? 12 - enqueued : enqueued < 24 ? 4 : std::min(64, enqueued / 2);
  }
  const Counters* h = c->host_counters;
  hint = std::max(4, std::min(64, (int)h->rounds + 1));
  const bool capped = h->residual >= h->dpad[0];
  if ((h->aux[0] || capped) && !out32_always) out32 = nullptr;
  k_wpr_finish<T><<<g, kBlock, 0, c->stream>>>(n, B.x, B.y, B.sum, B.comp, cnt, out32, out64);
  SUMINC_HIP(hipGetLastError());
  SUMINC_HIP(hipEventRecord(c->ev_stop, c->stream));
  SUMINC_HIP(hipEventSynchronize(c->ev_stop));
  float ms = 0;
  SUMINC_HIP(hipEventElapsedTime(&ms, c->ev_start, c->ev_stop));
  SUMINC_REQUIRE(!h->aux[0], SUMINC_E_NUMERIC, "NaN/Inf in the weighted PageRank state");
  SUMINC_REQUIRE(!capped, SUMINC_E_NOT_CONVERGED, "round cap reached before sum|delta| < tolerance");
  suminc_stats out{};
  out.rounds = (double)h->rounds;
  out.edges_traversed = (double)h->edges;
  out.residual = h->residual;
  out.kernel_ms = ms;
  out.pull_rounds = (double)h->rounds;
  c->stats = out;
  if (st) *st = out;
}

static void check_weighted(suminc_ctx* c) {
  SUMINC_REQUIRE(c->has_graph, SUMINC_E_STATE, "no graph");
  SUMINC_REQUIRE(c->wkind == SUMINC_W_F32, SUMINC_E_STATE, "weighted PageRank needs SUMINC_W_F32 edge weights");
}

void wpr_set_weights(suminc_ctx* c, const float* w) {
  check_weighted(c);
  SUMINC_REQUIRE(w || c->m == 0, SUMINC_E_INVALID, "null weights");
  WprState& S = wstate(c);
  if (c->m) {
    SUMINC_HIP(hipMemcpyAsync(c->out_w.p, w, c->m * 4, hipMemcpyDefault, c->stream));
    wpr_prepare_graph(c, S);
    k_wpr_gather<float><<<grid_for(c->m, kBlock * kGatherPer), kBlock, 0, c->stream>>>(
        c->m, S.eid.as<uint32_t>(), c->out_w.as<float>(), c->in_w.as<float>());
    SUMINC_HIP(hipGetLastError());
    SUMINC_HIP(hipStreamSynchronize(c->stream));
  }
  S.weights_version++;
  S.fwd_ready = false;
}

// Device memory of the context's GPU, which a kernel can be handed as it is.
static bool own_device(const suminc_ctx* c, const void* p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type == hipMemoryTypeDevice && a.device == c->device;
}

// A caller's vector as kernels read it: itself, or its copy in buf.
static const float* vector_in(suminc_ctx* c, const float* p, uint64_t count, DevBuf& buf) {
  if (own_device(c, p)) return p;
  buf.ensure(count * 4 + 4);
  SUMINC_HIP(hipMemcpyAsync(buf.p, p, count * 4, hipMemcpyDefault, c->stream));
  return buf.as<float>();
}

// Where kernels write a result of the caller's (null: nowhere to bring it), and its way
// there afterwards.
static float* vector_out(suminc_ctx* c, float* p, uint64_t count, DevBuf& buf) {
  if (p && own_device(c, p)) return p;
  buf.ensure(count * 4 + 4);
  return buf.as<float>();
}
__global__ void __launch_bounds__(kBlock) k_copy_f32(uint32_t n, const float* __restrict__ src,
                                                     float* __restrict__ dst) {
  const uint32_t v = blockIdx.x * kBlock + threadIdx.x;
  if (v < n) dst[v] = src[v];
}
static void vector_home(suminc_ctx* c, float* p, const float* dev, uint64_t count) {
  if (!p || p == dev || !count) return;
  if (readback(c, {{p, count, 4}}, [c, dev](int, uint64_t first, uint64_t k, void* out) {
        k_copy_f32<<<grid_for(k), kBlock, 0, c->stream>>>((uint32_t)k, dev + first, reinterpret_cast<float*>(out));
      }))
    return;
  SUMINC_HIP(hipMemcpyAsync(p, dev, count * 4, hipMemcpyDefault, c->stream));
}

template <class T>
static void wpr_forward_t(suminc_ctx* c, const float* p, float* r, suminc_stats* st) {
  WprState& S = wstate(c);
  wpr_prepare_graph(c, S);
  wpr_prepare_coef<T>(c, S);
  const uint32_t n = c->n;
  const float* pd = vector_in(c, p, n, S.in_f);
  S.r64.ensure((size_t)n * 8 + 8);
  float* rd = r ? vector_out(c, r, n, S.out_f) : nullptr;
  const RowLists R = lists_of(S.in, c->in_off, c->in_col, true);
  const uint32_t* pos = S.in.compact ? S.in.pos.as<uint32_t>() : nullptr;
  wpr_series<T>(c, S.hint_fwd, series_state<T>(c, S, pos != nullptr), R, &S.bin_in, pos, S.a_in.as<T>(), S.a_out.as<T>(), pd,
                (T)(1.0 - c->prm.damping), c->prm.termcheck_threshold, false, rd, S.r64.as<double>(), st);
  vector_home(c, r, rd, n);
  SUMINC_HIP(hipStreamSynchronize(c->stream));
  S.fwd_ready = true;
  S.fwd_coef_version = S.weights_version;
}

template <class T>
static void wpr_backward_t(suminc_ctx* c, const float* cvec, float* grad_p, float* grad_w, suminc_stats* st) {
  WprState& S = wstate(c);
  SUMINC_REQUIRE(S.fwd_ready && S.fwd_coef_version == S.weights_version && S.graph_version == c->graph_version,
                 SUMINC_E_STATE, "backward needs a forward on the current graph and weights");
  wpr_prepare_coef<T>(c, S);
  const uint32_t n = c->n;
  const uint64_t m = c->m;
  const double d = c->prm.damping;
  const float* cd = vector_in(c, cvec, n, S.in_f);
  S.lam64.ensure((size_t)n * 8 + 8);
  const RowLists R = lists_of(S.out, c->out_off, c->out_col, true);
  const uint32_t* pos = S.out.compact ? S.out.pos.as<uint32_t>() : nullptr;
  wpr_series<T>(c, S.hint_bwd, series_state<T>(c, S, pos != nullptr), R, &S.bin_out, pos, S.a_out.as<T>(), S.a_out.as<T>(), cd,
                (T)1, c->prm.termcheck_threshold, true, nullptr, S.lam64.as<double>(), st);
  const double* lam = S.lam64.as<double>();
  if (grad_p) {
    float* gp = vector_out(c, grad_p, n, S.out_f);
    k_wpr_grad_p<<<grid_for(n), kBlock, 0, c->stream>>>(n, lam, d, gp);
    SUMINC_HIP(hipGetLastError());
    vector_home(c, grad_p, gp, n);
  }
  if (grad_w && m) {
    // one more product, in FP64 from the weights themselves
    S.dot.ensure((size_t)n * 8 + 8);
    S.grad_rows.ensure((size_t)n * 16 + 16);
    row_sum(c, S, TermDot{c->out_w.as<float>(), c->out_col.as<uint32_t>(), lam}, S.dot.as<double>());
    k_wpr_grad_rows<<<grid_for(n), kBlock, 0, c->stream>>>(n, S.s.as<double>(), S.r64.as<double>(), S.dot.as<double>(),
                                                          d, S.grad_rows.as<double2>());
    float* gw = vector_out(c, grad_w, m, S.grad_w);
    k_wpr_grad_w<<<(unsigned)((m + kTileE - 1) / kTileE), kBlock, 0, c->stream>>>(
        c->out_off.as<uint32_t>(), c->out_col.as<uint32_t>(), m, S.tile_row.as<uint32_t>(), S.grad_rows.as<double2>(),
        lam, gw);
    SUMINC_HIP(hipGetLastError());
    vector_home(c, grad_w, gw, m);
  }
  SUMINC_HIP(hipStreamSynchronize(c->stream));
}

void wpr_forward(suminc_ctx* c, const float* p, float* r, suminc_stats* st) {
  check_weighted(c);
  SUMINC_REQUIRE(p, SUMINC_E_INVALID, "null personalization");
  if (c->prm.pr_precision == SUMINC_PR_FP64) wpr_forward_t<double>(c, p, r, st);
  else wpr_forward_t<float>(c, p, r, st);
}

void wpr_backward(suminc_ctx* c, const float* cvec, float* grad_p, float* grad_w, suminc_stats* st) {
  check_weighted(c);
  SUMINC_REQUIRE(cvec, SUMINC_E_INVALID, "null loss weights");
  if (c->prm.pr_precision == SUMINC_PR_FP64) wpr_backward_t<double>(c, cvec, grad_p, grad_w, st);
  else wpr_backward_t<float>(c, cvec, grad_p, grad_w, st);
}

// ---- PHP: penalized hitting probability on the series kernels --------------------
// PHPIngress (php/php_ingress.h:15-120): value = sum of the deltas a vertex takes,
// delta_0 = 1 at the source and 0 elsewhere, and a vertex u sends
// d * w_uv / s_u of its delta along every out-edge u -> v with v != source, where
// s_u = the sum of u's out-edge weights to vertices other than the source
// (frag.weight_sum, :30-45); nothing enters the source again.  That is the weighted
// series x_{t+1} = A x_t with a_uv = d w_uv / s_u (0 into the source), x_0 = e_src,
// value = sum_t x_t: the weighted-PageRank rounds over the same CSC row classes.
__global__ void __launch_bounds__(kBlock) k_copy_f64(uint32_t n, const double* __restrict__ src,
                                                     double* __restrict__ dst) {
  const uint32_t v = blockIdx.x * kBlock + threadIdx.x;
  if (v < n) dst[v] = src[v];
}

__global__ void k_php_seed(uint32_t n, uint32_t src, float* __restrict__ p) {
  const uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v < n) p[v] = v == src ? 1.f : 0.f;
}

template <class T>
static void php_run_t(suminc_ctx* c, uint32_t src, double d, double* values, suminc_stats* st) {
  WprState& S = wstate(c);
  wpr_prepare_graph(c, S);
  const uint32_t n = c->n;
  const uint64_t m = c->m;
  S.php_a_out.ensure(m * sizeof(T) + 8);
  S.php64.ensure((size_t)n * 8 + 8);
  S.php_s.ensure((size_t)n * 8 + 8);
  const TermPhp w{c->out_col.as<uint32_t>(), c->wkind == SUMINC_W_U32 ? c->out_w.as<uint32_t>() : nullptr,
                  c->wkind == SUMINC_W_F32 ? c->out_w.as<float>() : nullptr, src};
  row_sum(c, S, w, S.php_s.as<double>());
  edge_coefs<T>(c, S, w, S.php_s.as<double>(), d, S.php_a_out.as<T>(), S.php_a_in);
  S.in_f.ensure((size_t)n * 4 + 4);
  k_php_seed<<<grid_for(n), kBlock, 0, c->stream>>>(n, src, S.in_f.as<float>());
  SUMINC_HIP(hipGetLastError());
  const RowLists R = lists_of(S.in, c->in_off, c->in_col, true);
  const uint32_t* pos = S.in.compact ? S.in.pos.as<uint32_t>() : nullptr;
  wpr_series<T>(c, S.hint_php, series_state<T>(c, S, pos != nullptr), R, &S.bin_in, pos, S.php_a_in.as<T>(),
                S.php_a_out.as<T>(), S.in_f.as<float>(), (T)1, c->prm.termcheck_threshold, false, nullptr, S.php64.as<double>(), st);
  if (readback(c, {{values, n, 8}}, [c, &S](int, uint64_t first, uint64_t count, void* out) {
        k_copy_f64<<<grid_for(count), kBlock, 0, c->stream>>>((uint32_t)count, S.php64.as<double>() + first,
                                                             reinterpret_cast<double*>(out));
      }))
    return;
  if (values) SUMINC_HIP(hipMemcpyAsync(values, S.php64.p, (size_t)n * 8, hipMemcpyDefault, c->stream));
  SUMINC_HIP(hipStreamSynchronize(c->stream));
}

void php_run(suminc_ctx* c, uint32_t source, double damping, double* values, suminc_stats* st) {
  SUMINC_REQUIRE(c->has_graph, SUMINC_E_STATE, "no graph");
  SUMINC_REQUIRE(source < c->n, SUMINC_E_INVALID, "source out of range");
  SUMINC_REQUIRE(damping > 0.0 && damping < 1.0, SUMINC_E_INVALID, "damping must be in (0, 1)");
  if (c->prm.pr_precision == SUMINC_PR_FP64) php_run_t<double>(c, source, damping, values, st);
  else php_run_t<float>(c, source, damping, values, st);
}

// ---- the allocation-free forward -------------------------------------------------
// Its round state lives in `scratch`, one fixed array per GPU that the library
// holds until the process ends.  Host code never passes the array's name to a
// kernel: wpr_scratch_setup() takes the array's device address once per device
// (with that device current) and every launch uses that address.
constexpr size_t kScratchBytes = size_t(64) << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];
constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static unsigned char* g_scratch_dev[kMaxDevices] = {};

void wpr_scratch_setup(int device) {
  SUMINC_REQUIRE(device >= 0 && device < kMaxDevices, SUMINC_E_INVALID, "device index beyond the scratch table");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_dev[device]) return;
  void* p = nullptr;
  SUMINC_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  SUMINC_REQUIRE(p, SUMINC_E_HIP, "no device address for the scratch array");
  g_scratch_dev[device] = reinterpret_cast<unsigned char*>(p);
}

static unsigned char* scratch_of(int device) {
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  return device >= 0 && device < kMaxDevices ? g_scratch_dev[device] : nullptr;
}

static bool on_device(const void* p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type == hipMemoryTypeDevice || a.type == hipMemoryTypeManaged;
}

template <class T>
static void wpr_forward_noalloc_t(suminc_ctx* c, const float* p, float* r, suminc_stats* st) {
  SUMINC_REQUIRE(c->wpr, SUMINC_E_STATE, "no weighted PageRank state: call suminc_wpr_set_weights and one "
                                        "suminc_wpr_forward first");
  WprState& S = *reinterpret_cast<WprState*>(c->wpr);
  const int prec = sizeof(T) == 8 ? SUMINC_PR_FP64 : SUMINC_PR_FP32_KAHAN;
  SUMINC_REQUIRE(S.graph_version == c->graph_version && S.coef_version == S.weights_version && S.coef_prec == prec,
                 SUMINC_E_STATE, "the coefficients of the current graph, weights and precision are not prepared: "
                                 "run one suminc_wpr_forward first");
  const uint32_t n = c->n;
  const bool compact = S.in.compact;
  const size_t need = series_bytes<T>(n, compact);
  if (need > kScratchBytes)
    throw Error(SUMINC_E_TOO_LARGE, "suminc_wpr_forward_noalloc: " + std::to_string(n) + " vertices need " +
                                        std::to_string(need) + " bytes of scratch, the fixed array holds " +
                                        std::to_string(kScratchBytes));
  unsigned char* base = scratch_of(c->device);
  SUMINC_REQUIRE(base, SUMINC_E_STATE, "scratch array not set up on this device");
  const SeriesBufs<T> B = series_carve<T>(base, n, compact);
  const RowLists R = lists_of(S.in, c->in_off, c->in_col, true);
  const uint32_t* pos = compact ? S.in.pos.as<uint32_t>() : nullptr;
  S.fwd_ready = false;  // the rank of this forward is not kept for a backward
  wpr_series<T>(c, S.hint_fwd, B, R, &S.bin_in, pos, S.a_in.as<T>(), S.a_out.as<T>(), p, (T)(1.0 - c->prm.damping),
                c->prm.termcheck_threshold, false, r, nullptr, st, true);
  SUMINC_HIP(hipStreamSynchronize(c->stream));
}

void wpr_forward_noalloc(suminc_ctx* c, const float* p, float* r, suminc_stats* st) {
  check_weighted(c);
  SUMINC_REQUIRE(p && r, SUMINC_E_INVALID, "null personalization or rank");
  SUMINC_REQUIRE(on_device(p) && on_device(r), SUMINC_E_INVALID,
                 "suminc_wpr_forward_noalloc needs device memory for the personalization and the rank");
  if (c->prm.pr_precision == SUMINC_PR_FP64) wpr_forward_noalloc_t<double>(c, p, r, st);
  else wpr_forward_noalloc_t<float>(c, p, r, st);
}

void wpr_download(suminc_ctx* c, double* r, double* lam) {
  WprState& S = wstate(c);
  SUMINC_REQUIRE(S.fwd_ready, SUMINC_E_STATE, "no weighted PageRank forward yet");
  if (r) SUMINC_HIP(hipMemcpy(r, S.r64.p, (size_t)c->n * 8, hipMemcpyDeviceToHost));
  if (lam) {
    SUMINC_REQUIRE(S.lam64.p, SUMINC_E_STATE, "no backward yet");
    SUMINC_HIP(hipMemcpy(lam, S.lam64.p, (size_t)c->n * 8, hipMemcpyDeviceToHost));
  }
}

}  // namespace suminc
