// extrap.hpp -- the choice of extrapolation steps in a delta series.
//
// Every iteration here is the series r += delta, delta <- M delta (M = d P^T of
// PageRank, its weighted and transposed forms, a round of the supernode sketch), and
// delta is the exact residual of r: for any y, r += y with delta <- delta - (I - M) y
// keeps that.  A plain round takes y = delta.  Once delta has lined up with M's
// dominant eigenvector (eigenvalue rho), taking y = delta / (1 - rho) removes that
// component at once: with p the delta before a round and g the one after it, the state
//   r + beta p,   g + beta (g - p),   beta = rho / (1 - rho)
// is the one that y = (1 + beta) p leads to (power extrapolation: Kamvar, Haveliwala,
// Manning and Golub, "Extrapolation methods for accelerating PageRank computations",
// WWW 2003).  R-MAT graphs have rho = 0.84 and a next eigenvalue near 0.16, so the
// 80 plain rounds from 0.15 to 1e-7 become 10.
//
// The stop rule stays sum |delta| < T on the state that is kept.  The vertex pass that
// counts S1 = sum |g| also counts S2 = sum |g + beta (g - p)| for the candidate of the
// rounds before (rho = the last round's ratio of sums), and a step is taken only when
// S2 is known to be the smaller: when it ends the run (S2 < T), or when S2 < S1 / 2 and
// waiting another round no longer pays (S2 / S1 fell by less than kExtrapStall: as
// the steps' polynomials commute, an extrapolation is worth the more the better rho is
// known).  A series that never lines up (an isolated cycle, a path, signed mass on a
// regular grid) runs its plain rounds.
//
// What bounds the rounds: where M contracts the 1-norm by d (all forms but the adjoint's),
// sum |delta| after t rounds is at most d^t of the first, steps or not, so a run ends by
// the round at which that bound passes T.  A plain run may beat the bound by more than one
// with steps does, from a single seed or where mass leaks through layers.  The adjoint's
// transposed M contracts the maximum norm instead; its steps still halve the 1-norm each,
// but there is no such bound.  Over some thousands of small random graphs (bipartite,
// layered, cliques, stars, skewed, rings) the most was three rounds more than plain (45 ->
// 48), two in the adjoint (32 -> 34), and none did not end.
#pragma once
#include "ctx.hpp"
#include "device.hpp"

namespace suminc {

constexpr double kExtrapStall = 0.7;
constexpr double kExtrapMaxRho = 0.98;

// One thread, after the sums are known: the round's residual (of the state as the next
// vertex pass leaves it), ex.beta for that pass and ex.cand for the next count.
__device__ __forceinline__ double extrap_decide(Extrap& ex, double s1, double s2, double T) {
  bool take = false;
  double q = 0.0;
  if (ex.cand > 0.0 && s1 >= T) {
    q = s2 / s1;
    take = s2 < T || (q < 0.5 && ex.ratio > 0.0 && q > kExtrapStall * ex.ratio);
  }
  const double res = take ? s2 : s1;
  const double rho = !take && ex.last > 0.0 ? fmin(s1 / ex.last, kExtrapMaxRho) : 0.0;
  ex.beta = take ? ex.cand : 0.0;
  ex.ratio = take ? 0.0 : q;
  ex.cand = rho / (1.0 - rho);
  ex.last = res;
  return res;
}

// A value of the extrapolated delta.
template <class T>
__device__ __forceinline__ T extrap_value(T g, T p, double beta) {
  return (T)((double)g + beta * ((double)g - (double)p));
}

// rank[v] += x for an FP64 x: in FP32 mode the sum rank - comp is formed in FP64 and
// split again, so a step several times the delta loses no more than a plain one.
template <class T>
__device__ __forceinline__ void rank_add_wide(T* rank, float* comp, uint32_t v, double x) {
  if constexpr (sizeof(T) == 4) {
    const double t = (double)rank[v] - (double)comp[v] + x;
    const float r = (float)t;
    rank[v] = r;
    comp[v] = (float)((double)r - t);
  } else {
    rank[v] += x;
  }
}

// Sums of a block's values of each of the K arrays of nparts (double or u64 bits per
// kU bit k) into out[K], in a fixed order; all threads of a block of kThreads.  Up to
// kThreads parts the sums are the same for every kThreads.
template <int K, unsigned kU, int kThreads = 1024>
__device__ __forceinline__ void sum_parts(const double* __restrict__ partial, uint32_t nparts, double (*s)[K]) {
  double acc[K];
#pragma unroll
  for (int k = 0; k < K; ++k) acc[k] = 0.0;  // the bits of u64 zero too
  for (uint32_t i = threadIdx.x; i < nparts; i += kThreads) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const double x = partial[(size_t)k * nparts + i];
      if (kU >> k & 1)
        acc[k] = __longlong_as_double(__double_as_longlong(acc[k]) + __double_as_longlong(x));
      else
        acc[k] += x;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (kU >> k & 1)
        acc[k] = __longlong_as_double(__double_as_longlong(acc[k]) +
                                      __shfl_xor((long long)__double_as_longlong(acc[k]), o));
      else
        acc[k] += __shfl_xor(acc[k], o);
    }
  }
  if (lane_id() == 0) {
#pragma unroll
    for (int k = 0; k < K; ++k) s[threadIdx.x >> 6][k] = acc[k];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kThreads / 64; ++w) {
#pragma unroll
      for (int k = 0; k < K; ++k) {
        if (kU >> k & 1)
          s[0][k] = __longlong_as_double(__double_as_longlong(s[0][k]) + __double_as_longlong(s[w][k]));
        else
          s[0][k] += s[w][k];
      }
    }
  }
}

}  // namespace suminc
