// One CG iteration of a column by one workgroup, for the single and the batched
// solver.
#pragma once

#include "common.hpp"

namespace mplak {

// A column of up to kCgStepMax elements stays in the registers of one workgroup
// of 16 waves, so the two dot products are block reductions and the iteration's
// vector work is one launch instead of three (dz, update, direct), each of which
// is mostly launch latency and a reduction of partial sums at these sizes.  Per
// iteration in a graph, three launches and this one: one column of n = 1000, 8.0
// and 4.5 us; n = 4000, 8.9 and 6.5; n = 6000, 8.9 and 8.1; 64 columns of n =
// 4000 (with the group's state), 12.2 and 9.3.  Beyond, one CU's share of the
// cache bandwidth is the bound (n = 8192: 9.0 and 9.8; n = 10000: 8.9 and 16.4)
// and the grids of the three kernels win.
constexpr int kCgStepThreads = 1024;
constexpr int64_t kCgStepMax = 6 * kCgStepThreads;

__device__ __forceinline__ double cg_stop_value(int rule, double rr, double bnorm2, double n_global) {
  return rule == MPLAK_STOP_RMS ? sqrt(rr / n_global) : sqrt(rr) / sqrt(bnorm2);
}

// alpha = rr / <d,z>, x += alpha d, r -= alpha z, stopping test on <r,r>, d = r +
// beta d unless it converged (the reference breaks before the direction update
// only then; on its last iteration it still updates d).  n <= 1024 E.
template <int E>
__device__ __forceinline__ void cg_step(int64_t n, double* __restrict__ x, double* __restrict__ r,
                                        double* __restrict__ d, const double* __restrict__ z,
                                        const mplak_cg_state* __restrict__ in, mplak_cg_state* __restrict__ out,
                                        double* scratch) {
  const mplak_cg_state s_in = *in;
  if (s_in.done != MPLAK_RUNNING) {
    if (threadIdx.x == 0) *out = s_in;
    return;
  }
  double dv[E], zv[E], rv[E];
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int64_t i = threadIdx.x + (int64_t)u * kCgStepThreads;
    const bool in_range = i < n;
    dv[u] = in_range ? d[i] : 0.0;
    zv[u] = in_range ? z[i] : 0.0;
    rv[u] = in_range ? r[i] : 0.0;
  }
  double s = 0.0;
#pragma unroll
  for (int u = 0; u < E; ++u) s = fma(dv[u], zv[u], s);
  const double dz = block_sum<kCgStepThreads>(s, scratch);
  const double alpha = s_in.rr / dz;
  double rr = 0.0;
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int64_t i = threadIdx.x + (int64_t)u * kCgStepThreads;
    rv[u] = fma(-alpha, zv[u], rv[u]);
    if (i < n) {
      rr = fma(rv[u], rv[u], rr);
      r[i] = rv[u];
      x[i] = fma(alpha, dv[u], x[i]);
    }
  }
  const double rr_new = block_sum<kCgStepThreads>(rr, scratch);
  const double beta = rr_new / s_in.rr;
  const int k = s_in.k + 1;
  const double rel = cg_stop_value(s_in.rule, rr_new, s_in.bnorm2, s_in.n_global);
  const bool conv = rel < s_in.eps;
  const bool limit = k >= s_in.iter_max - 1;
  if (!conv) {
#pragma unroll
    for (int u = 0; u < E; ++u) {
      const int64_t i = threadIdx.x + (int64_t)u * kCgStepThreads;
      if (i < n) d[i] = fma(beta, dv[u], rv[u]);
    }
  }
  if (threadIdx.x == 0) {
    mplak_cg_state o = s_in;
    o.rr = rr_new;
    o.rel = rel;
    o.alpha = alpha;
    o.beta = beta;
    o.k = k;
    o.done = conv ? MPLAK_CONVERGED : (limit ? MPLAK_ITER_LIMIT : MPLAK_RUNNING);
    *out = o;
  }
}

}  // namespace mplak
