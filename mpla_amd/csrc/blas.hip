// Dense FP64 level-1/2 kernels and synthetic-input fills for gfx950.
//
//   dgemv  : y = A x, A column-major, HBM-streaming row panels with split-K
//   ddot   : deterministic two-pass reduction
//   daxpy / waxpby / fill / copy : grid-stride elementwise kernels
//   fill_uniform : counter-based SplitMix64 inputs (bitwise equal to the host)

#include <algorithm>

#include "common.hpp"
#include "rng.hpp"

namespace mplak {
namespace {

// ---------------------------------------------------------------------------
// Elementwise kernels
// ---------------------------------------------------------------------------

inline int elementwise_grid(int64_t n) {
  int64_t blocks = (n + kBlock * 4 - 1) / (kBlock * 4);
  if (blocks < 1) blocks = 1;
  if (blocks > 8192) blocks = 8192;
  return static_cast<int>(blocks);
}

__global__ __launch_bounds__(kBlock) void fill_kernel(double* __restrict__ out, int64_t n,
                                                      double v) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) out[i] = v;
}

__global__ __launch_bounds__(kBlock) void copy_kernel(double* __restrict__ dst,
                                                      const double* __restrict__ src, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    dst[i] = src[i];
}

__global__ __launch_bounds__(kBlock) void axpy_kernel(int64_t n, double alpha,
                                                      const double* __restrict__ x,
                                                      double* __restrict__ y) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    y[i] = fma(alpha, x[i], y[i]);
}

// w may alias x or y, so no __restrict__ here.
__global__ __launch_bounds__(kBlock) void waxpby_kernel(int64_t n, double a, const double* x,
                                                        double b, const double* y, double* w) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    w[i] = a * x[i] + b * y[i];
}

__global__ __launch_bounds__(kBlock) void uniform_kernel(double* __restrict__ out, int64_t n,
                                                         uint64_t key, uint64_t first, double lo,
                                                         double span) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    out[i] = rng_uniform_ab(key, first + (uint64_t)i, lo, span);
}

// ---------------------------------------------------------------------------
// Deterministic dot product
// ---------------------------------------------------------------------------

constexpr int kDotMaxBlocks = 1024;

inline int dot_blocks(int64_t n) {
  int64_t b = (n + kBlock * 8 - 1) / (kBlock * 8);
  if (b < 1) b = 1;
  if (b > kDotMaxBlocks) b = kDotMaxBlocks;
  return static_cast<int>(b);
}

__global__ __launch_bounds__(kBlock) void dot_partial_kernel(int64_t n,
                                                             const double* __restrict__ x,
                                                             const double* __restrict__ y,
                                                             double* __restrict__ part) {
  __shared__ double scratch[kBlock / kWave];
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  double s = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    s = fma(x[i], y[i], s);
  s = block_sum<kBlock>(s, scratch);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ __launch_bounds__(kBlock) void dot_final_kernel(const double* __restrict__ part,
                                                           int count, double* __restrict__ out) {
  __shared__ double scratch[kBlock / kWave];
  double s = reduce_partials<kBlock>(part, count, scratch);
  if (threadIdx.x == 0) *out = s;
}

// ---------------------------------------------------------------------------
// dgemv: y = A x, column-major A.
//
// A workgroup of NW waves owns a panel of 2 RL rows and one slab of columns.
// RL lanes of a wave hold two rows each (one 16-byte load per column), its
// 64 / RL lane groups take column pairs side by side, and the waves take
// contiguous shares of the slab.  Lane groups are added by xor-shuffles, waves
// in wave order through LDS, and a second kernel adds the slabs in slab order;
// every split depends only on (m, n).
//
// Column strides are whatever lda is: a 16-byte load needs 4-byte alignment
// only, so matrices of odd lda (or a base that is 8-byte aligned) take the
// same loads as even ones.  Two 8-byte loads per lane and column, as such
// matrices had before, ran a 30001 x 20003 product at 2.9 TB/s; 16-byte loads
// run it at 6.4 TB/s (1663 -> 751 us).
//
// Geometries:
// * streamed (RL = 64, 4 waves): each load instruction reads 1 KiB of one
//   column; bound by HBM or the Infinity Cache.  A product keeps the memory
//   system busy from about 152 workgroups, and above 256 (one per CU) a last
//   round that is nearly empty costs up to a third (n = 16385: 465 us at 258
//   workgroups, 363 us at 2064), so the slab count is the smallest with 152
//   to 256 workgroups, or else with at least 90 % of the last round filled; one
//   from 4 rounds of panels (200000 x 256: 63 us, in two slabs 67 us).
// * panels of 16 rows (RL = 8, 16 waves): a matrix of up to 40 MB and 4096
//   rows has too few 128-row panels to fill the chip and is bound by latency;
//   16-row panels put 16 waves on each of m / 16 CUs with every load of a wave
//   in flight at once and mostly need no second kernel (1000 x 1000: 4.9 us
//   against 9.9 us streamed, 1500 x 1500: 7.0 us against 7.4 us, 226 x 208: 3.6
//   us against 6.0 us).  Matrices of up to 64 rows take it at any size: most
//   lanes of a 128-row panel would hold no row (64 x 30000: 7.5 us in 32 slabs).
// * the panels between (RL = 16 or 32 with 16 waves, RL = 64 with 8), the
//   lowest that give at most one panel per CU, for matrices that fit the
//   Infinity Cache: all columns in one workgroup save the slab sum and its
//   launch (streamed / so: 4096 x 4000 24.4 / 21.5 us, 4200 x 1000 12.7 / 8.4
//   us, 10000 x 2500 32.5 / 29.8 us, 16384 x 4000 83 / 75 us, 20000 x 1000
//   23.9 / 23.4 us; 120 MB as 3000 x 5000, on 94 panels, 23.6 / 25.2 us).
//   Fewer than 128 columns leave too little for their waves and are streamed in
//   one slab (12000 x 64: 3.5 us, panels 3.9 us, two slabs 6.5 us), and so are
//   small matrices whose 32-row panels are more than the CUs (8200 x 256: 4.0
//   us, 64-row panels 4.3 us; 12000 x 256, 25 MB: 5.8 and 5.0 us).
//
// A matrix larger than the 256 MiB Infinity Cache is read with nontemporal
// loads (STREAM): every element is used once, and the hint keeps the stream
// from churning L2 and the Infinity Cache.  At N = 65536 that raises the read
// rate from 6.26 to about 6.85 TB/s; a smaller matrix that stays cached
// between calls reads faster with ordinary loads (N = 4096: 29 us against
// 32 us).
// ---------------------------------------------------------------------------

constexpr int kGvUnroll = 8;                                // columns of a lane in flight
constexpr int kGvSumRounds = 256 / kGvUnroll;               // rounds of them in one running sum
constexpr int kGvStreamLanes = 64, kGvPanelLanes = 8;       // 128-row and 16-row panels
constexpr double kGvPanelBytes = 40e6;                      // largest matrix of the 16-row panels
constexpr int64_t kGvPanelRows = 64;                        // or most rows at any size
constexpr int64_t kGvPanelCols = 128;                       // fewest columns of the panels between,
constexpr int64_t kGvWholeTiles = 120;                      // fewest of those panels
constexpr double kGvSmallBytes = 22e6;                      // and smallest matrix of more than 8192 rows
constexpr int64_t kGvCus = 256;
constexpr int64_t kGvBusy = 152;                            // workgroups that saturate the memory system
constexpr int64_t kGvStreamBytes = int64_t(256) << 20;      // Infinity Cache capacity

typedef double gv_f64x2 __attribute__((ext_vector_type(2), aligned(8)));

template <bool STREAM>
__device__ __forceinline__ gv_f64x2 gv_load2(const double* p) {
  const gv_f64x2* q = reinterpret_cast<const gv_f64x2*>(p);
  if constexpr (STREAM) return __builtin_nontemporal_load(q);
  else return *q;
}

struct GemvPlan {
  int lanes, waves;  // RL, NW
  int64_t row_tiles, slabs, slab_cols;
};

inline GemvPlan gemv_plan(int64_t m, int64_t n) {
  GemvPlan p;
  const double bytes = (double)m * (double)n * sizeof(double);
  auto tiles = [&](int lanes) { return (m + 2 * lanes - 1) / (2 * lanes); };
  p.lanes = kGvStreamLanes;
  p.waves = 4;
  bool whole = false;  // one slab
  if (m <= kGvPanelRows || (m <= kGvCus * 2 * kGvPanelLanes && bytes <= kGvPanelBytes)) {
    p.lanes = kGvPanelLanes;
  } else if (n < kGvPanelCols || (tiles(2 * kGvPanelLanes) > kGvCus && bytes <= kGvSmallBytes)) {
    whole = true;
  } else if (bytes <= kGvStreamBytes) {
    int lanes = 2 * kGvPanelLanes;
    while (lanes < kGvStreamLanes && tiles(lanes) > kGvCus) lanes *= 2;
    whole = tiles(lanes) >= kGvWholeTiles;
    if (whole) p.lanes = lanes;
    if (whole && tiles(lanes) <= kGvCus) p.waves = 8;
  }
  if (p.lanes < kGvStreamLanes) p.waves = 16;
  p.row_tiles = tiles(p.lanes);
  int64_t ks = 1;
  if (p.lanes == kGvPanelLanes) {
    // a lane walks n / 128 columns: wide matrices of few rows are split further
    if (n >= 4096) ks = std::min((kGvCus + p.row_tiles - 1) / p.row_tiles, n / 1024);
  } else if (!whole && p.row_tiles < 4 * kGvCus) {
    const int64_t most = std::min<int64_t>(std::max<int64_t>(n / (8 * kGvUnroll), 1), 4096);
    double best = 0.0;
    for (int64_t k = 1; k <= most; ++k) {
      const int64_t w = p.row_tiles * k;
      const double full = (double)w / (double)(kGvCus * ((w + kGvCus - 1) / kGvCus));
      if (full > best) best = full, ks = k;
      if ((w >= kGvBusy && w <= kGvCus) || (w > kGvCus && full >= 0.9)) {
        ks = k;
        break;
      }
    }
  }
  if (ks < 1) ks = 1;
  p.slab_cols = (n + ks - 1) / ks;
  p.slabs = (n + p.slab_cols - 1) / p.slab_cols;
  return p;
}

// ROWS = 2: the lane holds rows b and b + 1; the last lane of an odd m holds
// m - 2 and m - 1, so no load leaves the matrix.  ROWS = 1 (m == 1): one row.
template <int RL, int NW, int ROWS, bool STREAM>
__global__ __launch_bounds__(NW* kWave) void dgemv_partial_kernel(int64_t m, int64_t n, const double* __restrict__ A,
                                                                  int64_t lda, const double* __restrict__ x,
                                                                  int64_t slab_cols, double* __restrict__ out,
                                                                  const int32_t* __restrict__ skip) {
  if (skip != nullptr && *skip != 0) return;
  constexpr int CG = kWave / RL;  // lane groups: column pairs side by side
  constexpr int U = kGvUnroll;
  constexpr int R = 2 * RL;
  __shared__ double red[NW][R];
  const int lane = threadIdx.x & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int rl = lane % RL;
  const int g = CG == 1 ? 0 : lane / RL;
  const int64_t panel = (int64_t)blockIdx.x * R;
  const int64_t row = panel + 2 * rl;
  const int64_t b = ROWS == 2 ? (row < m - 2 ? row : m - 2) : 0;
  const int64_t c0 = (int64_t)blockIdx.y * slab_cols;
  const int64_t c1 = c0 + slab_cols < n ? c0 + slab_cols : n;
  // the wave's columns: a whole number of pairs per lane group
  const int64_t share = ((slab_cols + NW - 1) / NW + 2 * CG - 1) / (2 * CG) * (2 * CG);
  const int64_t j0 = c0 + w * share < c1 ? c0 + w * share : c1;
  const int64_t j1 = j0 + share < c1 ? j0 + share : c1;
  auto load = [](const double* p) {
    if constexpr (ROWS == 2) {
      return gv_load2<STREAM>(p);
    } else {
      const gv_f64x2 v = {*p, 0.0};
      return v;
    }
  };
  // column offset of the lane's u-th load of a round
  auto col = [](int u) { return (u / 2) * 2 * CG + (u & 1); };

  // running sums of 256 columns, then their sum: a single one over the thousands
  // of columns of a wave would lose accuracy with the root of its length
  double sum0 = 0.0, sum1 = 0.0, acc0 = 0.0, acc1 = 0.0;
  int left = kGvSumRounds;
  int64_t j = j0 + 2 * g;
  const double* a = A + b + j * lda;
  int64_t jw = j0;
  for (; jw + U * CG <= j1; jw += U * CG) {
    gv_f64x2 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = load(a + col(u) * lda);
    double xv[U];
    if constexpr (CG == 1) {
#pragma unroll
      for (int u = 0; u < U; ++u) xv[u] = x[jw + u];  // wave-uniform: scalar loads
    } else {
#pragma unroll
      for (int u = 0; u < U; u += 2) {
        const gv_f64x2 q = *reinterpret_cast<const gv_f64x2*>(x + j + col(u));
        xv[u] = q.x;
        xv[u + 1] = q.y;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      acc0 = fma(v[u].x, xv[u], acc0);
      acc1 = fma(v[u].y, xv[u], acc1);
    }
    j += U * CG;
    a += (int64_t)(U * CG) * lda;
    if (--left == 0) {
      left = kGvSumRounds;
      sum0 += acc0;
      sum1 += acc1;
      acc0 = acc1 = 0.0;
    }
  }
  if (jw < j1) {
    // the last columns of the share, fewer than U CG: an absent column is
    // neither loaded nor multiplied
    gv_f64x2 v[U];
    double xv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const gv_f64x2 zero = {0.0, 0.0};
      v[u] = zero;
      xv[u] = 0.0;
      if (j + col(u) < j1) {
        v[u] = load(a + col(u) * lda);
        xv[u] = x[j + col(u)];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (j + col(u) < j1) {
        acc0 = fma(v[u].x, xv[u], acc0);
        acc1 = fma(v[u].y, xv[u], acc1);
      }
    }
  }
  acc0 += sum0;
  acc1 += sum1;
#pragma unroll
  for (int s = RL; s < kWave; s <<= 1) {
    acc0 += __shfl_xor(acc0, s, kWave);
    acc1 += __shfl_xor(acc1, s, kWave);
  }
  if (g == 0 && row < m) {
    // the last lane of an odd m repeats its neighbour's second row (the same
    // value) and may begin one row before the panel
    const int64_t k = b - panel;
    if (k >= 0) red[w][k] = acc0;
    if (ROWS == 2) red[w][k + 1] = acc1;
  }
  __syncthreads();
  if (threadIdx.x < R) {
    const int r = threadIdx.x;
    const int64_t gr = panel + r;
    if (gr < m) {
      double s = red[0][r];
#pragma unroll
      for (int q = 1; q < NW; ++q) s += red[q][r];
      out[(int64_t)blockIdx.y * m + gr] = s;
    }
  }
}

// y[i] = sum of the slab partials in slab order, eight loads in flight.
__global__ __launch_bounds__(kBlock) void slab_sum_kernel(int64_t m, int64_t slabs,
                                                          const double* __restrict__ part,
                                                          double* __restrict__ y,
                                                          const int32_t* __restrict__ skip) {
  if (skip != nullptr && *skip != 0) return;
  constexpr int kBatch = 8;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += stride) {
    double s = part[i];
    for (int64_t k = 1; k < slabs; k += kBatch) {
      double v[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) v[u] = k + u < slabs ? part[(k + u) * m + i] : 0.0;
#pragma unroll
      for (int u = 0; u < kBatch; ++u)
        if (k + u < slabs) s += v[u];
    }
    y[i] = s;
  }
}

template <int RL, int NW>
void launch_gemv(const GemvPlan& p, bool stream, int64_t m, int64_t n, const double* A, int64_t lda, const double* x,
                 double* out, const int32_t* skip, hipStream_t s) {
  const dim3 grid((unsigned)p.row_tiles, (unsigned)p.slabs);
  auto kern = m == 1 ? dgemv_partial_kernel<RL, NW, 1, false>
                     : (stream ? dgemv_partial_kernel<RL, NW, 2, true> : dgemv_partial_kernel<RL, NW, 2, false>);
  hipLaunchKernelGGL(kern, grid, dim3(NW * kWave), 0, s, m, n, A, lda, x, p.slab_cols, out, skip);
}

}  // namespace
}  // namespace mplak

using namespace mplak;

extern "C" {

const char* mplak_status_string(int status) {
  switch (status) {
    case MPLAK_OK: return "ok";
    case MPLAK_ERR_ARG: return "invalid argument";
    case MPLAK_ERR_HIP: return "HIP runtime error";
    case MPLAK_ERR_WORKSPACE: return "workspace too small";
    case MPLAK_ERR_UNSUPPORTED: return "unsupported request";
    case MPLAK_ERR_TOO_LARGE: return "problem needs more scratch than the no-allocation entry point holds";
    default: return "unknown status";
  }
}

int mplak_version(void) { return 100; }

int mplak_fill_uniform_f64(double* out, int64_t n, uint64_t seed, uint64_t stream,
                           uint64_t first_index, double lo, double hi, mplak_stream_t s) {
  if (n < 0 || (n > 0 && out == nullptr)) return MPLAK_ERR_ARG;
  if (n == 0) return MPLAK_OK;
  const uint64_t key = rng_key(seed, stream);
  hipLaunchKernelGGL(uniform_kernel, dim3(elementwise_grid(n)), dim3(kBlock), 0, as_stream(s), out,
                     n, key, first_index, lo, hi - lo);
  return launch_status();
}

int mplak_fill_f64(double* out, int64_t n, double value, mplak_stream_t s) {
  if (n < 0 || (n > 0 && out == nullptr)) return MPLAK_ERR_ARG;
  if (n == 0) return MPLAK_OK;
  hipLaunchKernelGGL(fill_kernel, dim3(elementwise_grid(n)), dim3(kBlock), 0, as_stream(s), out, n,
                     value);
  return launch_status();
}

int mplak_copy_f64(double* dst, const double* src, int64_t n, mplak_stream_t s) {
  if (n < 0 || (n > 0 && (dst == nullptr || src == nullptr))) return MPLAK_ERR_ARG;
  if (n == 0 || dst == src) return MPLAK_OK;
  hipLaunchKernelGGL(copy_kernel, dim3(elementwise_grid(n)), dim3(kBlock), 0, as_stream(s), dst,
                     src, n);
  return launch_status();
}

size_t mplak_dgemv_workspace_bytes(int64_t m, int64_t n) {
  if (m <= 0 || n <= 0) return 0;
  const GemvPlan p = gemv_plan(m, n);
  return p.slabs > 1 ? (size_t)p.slabs * (size_t)m * sizeof(double) : 0;
}

int mplak_dgemv_f64(int64_t m, int64_t n, const double* A, int64_t lda, const double* x, double* y,
                    void* work, size_t work_bytes, const int32_t* skip_if, mplak_stream_t s) {
  if (m < 0 || n < 0 || lda < (m > 1 ? m : 1)) return MPLAK_ERR_ARG;
  if (m == 0) return MPLAK_OK;
  if (y == nullptr) return MPLAK_ERR_ARG;
  if (n == 0) return mplak_fill_f64(y, m, 0.0, s);
  if (A == nullptr || x == nullptr) return MPLAK_ERR_ARG;
  const GemvPlan p = gemv_plan(m, n);
  const size_t need = mplak_dgemv_workspace_bytes(m, n);
  if (work_bytes < need || (need > 0 && work == nullptr)) return MPLAK_ERR_WORKSPACE;
  double* out = p.slabs > 1 ? static_cast<double*>(work) : y;
  const bool stream = (double)m * (double)n * sizeof(double) > (double)kGvStreamBytes;
  if (p.lanes == 8)
    launch_gemv<8, 16>(p, stream, m, n, A, lda, x, out, skip_if, as_stream(s));
  else if (p.lanes == 16)
    launch_gemv<16, 16>(p, stream, m, n, A, lda, x, out, skip_if, as_stream(s));
  else if (p.lanes == 32)
    launch_gemv<32, 16>(p, stream, m, n, A, lda, x, out, skip_if, as_stream(s));
  else if (p.waves == 8)
    launch_gemv<64, 8>(p, stream, m, n, A, lda, x, out, skip_if, as_stream(s));
  else
    launch_gemv<64, 4>(p, stream, m, n, A, lda, x, out, skip_if, as_stream(s));
  int st = launch_status();
  if (st != MPLAK_OK || p.slabs == 1) return st;
  hipLaunchKernelGGL(slab_sum_kernel, dim3(elementwise_grid(m)), dim3(kBlock), 0, as_stream(s), m,
                     p.slabs, out, y, skip_if);
  return launch_status();
}

size_t mplak_dot_workspace_bytes(int64_t n) {
  return (size_t)dot_blocks(n > 0 ? n : 1) * sizeof(double);
}

int mplak_ddot_f64(int64_t n, const double* x, const double* y, double* result, void* work,
                   size_t work_bytes, mplak_stream_t s) {
  if (n < 0 || result == nullptr || (n > 0 && (x == nullptr || y == nullptr))) return MPLAK_ERR_ARG;
  if (n == 0) return mplak_fill_f64(result, 1, 0.0, s);
  const int g = dot_blocks(n);
  if (work == nullptr || work_bytes < (size_t)g * sizeof(double)) return MPLAK_ERR_WORKSPACE;
  double* part = static_cast<double*>(work);
  hipLaunchKernelGGL(dot_partial_kernel, dim3(g), dim3(kBlock), 0, as_stream(s), n, x, y, part);
  int st = launch_status();
  if (st != MPLAK_OK) return st;
  hipLaunchKernelGGL(dot_final_kernel, dim3(1), dim3(kBlock), 0, as_stream(s), part, g, result);
  return launch_status();
}

int mplak_daxpy_f64(int64_t n, double alpha, const double* x, double* y, mplak_stream_t s) {
  if (n < 0 || (n > 0 && (x == nullptr || y == nullptr))) return MPLAK_ERR_ARG;
  if (n == 0) return MPLAK_OK;
  hipLaunchKernelGGL(axpy_kernel, dim3(elementwise_grid(n)), dim3(kBlock), 0, as_stream(s), n,
                     alpha, x, y);
  return launch_status();
}

int mplak_dwaxpby_f64(int64_t n, double a, const double* x, double b, const double* y, double* w,
                      mplak_stream_t s) {
  if (n < 0 || (n > 0 && (x == nullptr || y == nullptr || w == nullptr))) return MPLAK_ERR_ARG;
  if (n == 0) return MPLAK_OK;
  hipLaunchKernelGGL(waxpby_kernel, dim3(elementwise_grid(n)), dim3(kBlock), 0, as_stream(s), n, a,
                     x, b, y, w);
  return launch_status();
}

}  // extern "C"
