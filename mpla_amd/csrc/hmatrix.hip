// H-matrix operator kernels with closed-form kernel entries (C ABI of
// include/mplak.h): ACA compression of the admissible blocks, the far-field
// coefficient products and the near + far apply.  The block partition comes
// from the host (libmpla's H-matrix plugin, which replaces hmglib behind
// src/hmglib_adapter.cu:6-132).

#include <type_traits>

#include "common.hpp"
#include "entry.hpp"
#include "hmatrix_kernels.hpp"

namespace mplak {
namespace {

using hm::kHmThreads;

__global__ __launch_bounds__(kBlock) void gather_scaled_kernel(const double* const* __restrict__ points, int dim,
                                                               int64_t offset, const int64_t* __restrict__ perm,
                                                               int64_t n, double scale, double* __restrict__ out,
                                                               int64_t ld) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += stride) {
    const int64_t i = offset + perm[k];
    for (int d = 0; d < dim; ++d) out[d * ld + k] = scale * points[d][i];
  }
}

// One item: the item's columns against the block's rank terms.  Wave w takes
// the terms q = w, w + 4, ...: its lanes walk the item's columns two at a time
// for up to kFarTerms terms together (16-byte loads of V, x read once for all),
// then a butterfly sums the lanes.  No barriers; every sum has a fixed order.
// Bound by V's bandwidth: one term at a time left a wave two loads in flight
// and read 985 MB at 3.2 TB/s (n = 131072, 2-D, rank 20).
constexpr int kFarTerms = 5;
typedef double hm_f64x2 __attribute__((ext_vector_type(2), aligned(8)));

template <bool STREAM>
__device__ __forceinline__ hm_f64x2 factor_load2(const double* p) {
  const hm_f64x2* q = reinterpret_cast<const hm_f64x2*>(p);
  if constexpr (STREAM) return __builtin_nontemporal_load(q);
  else return *q;
}

template <bool STREAM>
__device__ __forceinline__ void far_item(const mplak_hm_block* __restrict__ blocks, const mplak_hm_item& it,
                                         const int32_t* __restrict__ rank, int kmax, const double* __restrict__ V,
                                         const double* __restrict__ xs, double* __restrict__ out) {
  constexpr int kWaves = kHmThreads / kWave;
  const mplak_hm_block B = blocks[it.block];
  const int rb = rank[it.block];
  const double* x = xs + B.c0;
  const int lane = threadIdx.x % kWave, w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int64_t j1 = it.j0 + it.count;
  for (int q0 = w; q0 < rb; q0 += kFarTerms * kWaves) {
    const double* v[kFarTerms];
    double s[kFarTerms];
#pragma unroll
    for (int u = 0; u < kFarTerms; ++u) {
      const int q = q0 + u * kWaves;
      v[u] = V + B.voff + (int64_t)(q < rb ? q : q0) * B.n;
      s[u] = 0.0;
    }
    const int terms = (rb - q0 + kWaves - 1) / kWaves;  // of this round, wave-uniform
    for (int64_t j = it.j0 + 2 * lane; j < j1; j += 2 * kWave) {
      if (j + 1 < j1) {
        hm_f64x2 a[kFarTerms];
#pragma unroll
        for (int u = 0; u < kFarTerms; ++u)
          if (u < terms) a[u] = factor_load2<STREAM>(v[u] + j);
        const hm_f64x2 xv = *reinterpret_cast<const hm_f64x2*>(x + j);
#pragma unroll
        for (int u = 0; u < kFarTerms; ++u)
          if (u < terms) s[u] = fma(a[u].y, xv.y, fma(a[u].x, xv.x, s[u]));
      } else {
#pragma unroll
        for (int u = 0; u < kFarTerms; ++u)
          if (u < terms) s[u] = fma(v[u][j], x[j], s[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < kFarTerms; ++u) {
      if (u >= terms) break;
      const double sum = wave_sum(s[u]);
      if (lane == 0) out[q0 + u * kWaves] = sum;
    }
  }
}

template <bool STREAM>
__global__ __launch_bounds__(kHmThreads) void far_partial_kernel(const mplak_hm_block* __restrict__ blocks,
                                                                 const mplak_hm_item* __restrict__ items,
                                                                 const int32_t* __restrict__ rank, int kmax,
                                                                 const double* __restrict__ V,
                                                                 const double* __restrict__ xs,
                                                                 double* __restrict__ part) {
  far_item<STREAM>(blocks, items[blockIdx.x], rank, kmax, V, xs, part + (int64_t)blockIdx.x * kmax);
}

// One thread per (block, term): the block's item partials in item order.
__global__ __launch_bounds__(kBlock) void far_sum_kernel(const int64_t* __restrict__ first_item, int64_t nblocks,
                                                         const int32_t* __restrict__ rank, int kmax,
                                                         const double* __restrict__ part, double* __restrict__ t) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= nblocks * kmax) return;
  const int64_t b = g / kmax;
  const int q = (int)(g % kmax);
  double s = 0.0;
  if (q < rank[b])
    for (int64_t i = first_item[b]; i < first_item[b + 1]; ++i) s += part[i * kmax + q];
  t[g] = s;
}

__global__ __launch_bounds__(kBlock) void scatter_nugget_kernel(const double* __restrict__ ys,
                                                                const int64_t* __restrict__ perm, int64_t n,
                                                                double nugget, const double* __restrict__ x,
                                                                int64_t shift, int64_t x_count,
                                                                double* __restrict__ y) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += stride) {
    const int64_t i = perm[k];
    const int64_t j = i + shift;
    double v = ys[k];
    if (nugget != 0.0 && j >= 0 && j < x_count) v = fma(nugget, x[j], v);
    y[i] = v;
  }
}

// ---- symmetric near field --------------------------------------------------
//
// One workgroup per pair (A, B) of near chunks (at most 512 sorted points
// each): 128-row blocks of A (two rows per lane) against the 64-point groups of
// B staged in LDS, block r against group g by wave (g + r) mod 4, so that the
// waves share whatever sizes the chunks have.  (A wave per 128-row block leaves
// the fourth wave idle at 312-point leaves, 40000 points in 3-D.)  Off the
// diagonal, lane l takes source (l + s) mod 64 at step s, so one evaluation of
// each entry feeds the row sums of its two A rows and a column sum for its B
// row that rotates one lane per step and ends in the lane of its source.  On
// the diagonal (A = B), block r meets the groups g >= 2 r only: its own two for
// the row sums, the later ones for both, their column sums being rows of A.
// Row sums are added over the waves, column sums over the row blocks, in order.
// Bound by the vector unit's FP64 entry evaluation.
constexpr int kPairRows = 2 * kBlock;
constexpr int kPairBlocks = kPairRows / (2 * kWave);

// LDS of a pair in doubles: the sources (x, y, z, value; afterwards the waves'
// row sums), the fourth coordinate, the blocks' column sums, the exp2 table.
constexpr int pair_lds(int dim) { return 4 * kPairRows + (dim > 3 ? kPairRows : 0) + kPairBlocks * kPairRows + kExp2Table; }

template <int KIND, int DIM>
__device__ __forceinline__ void near_pair(const double* __restrict__ pts, int64_t ld, const mplak_hm_pair& P,
                                          const double* __restrict__ xs, double* __restrict__ rows_a, double* lds) {
  double4* src = reinterpret_cast<double4*>(lds);
  double* crd4 = lds + 4 * kPairRows;
  double* col = crd4 + (DIM > 3 ? kPairRows : 0);
  double* tab = col + kPairBlocks * kPairRows;
  fill_exp2_table(tab);  // first read after the staging barrier
  const int tid = threadIdx.x, lane = tid & (kWave - 1), w = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int am = (int)P.am, bm = (int)P.bm;
  const bool diagonal = P.a0 == P.b0;
  // every global load of the staging is issued before the first use
  double sc[2][DIM], sv[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int k = u * kBlock + tid;
    const int64_t j = P.b0 + (k < bm ? k : bm - 1);
#pragma unroll
    for (int d = 0; d < DIM; ++d) sc[u][d] = pts[d * ld + j];
    sv[u] = k < bm ? xs[j] : 0.0;
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int k = u * kBlock + tid;
    double4 q;
    q.x = sc[u][0];
    q.y = DIM > 1 ? sc[u][DIM > 1 ? 1 : 0] : 0.0;
    q.z = DIM > 2 ? sc[u][DIM > 2 ? 2 : 0] : 0.0;
    q.w = sv[u];
    src[k] = q;
    if (DIM > 3) crd4[k] = sc[u][DIM - 1];
  }
  __syncthreads();
  const int groups = (bm + kWave - 1) / kWave;
  double rows[kPairBlocks][2];
#pragma unroll
  for (int r = 0; r < kPairBlocks; ++r) rows[r][0] = rows[r][1] = 0.0;
#pragma unroll 1
  for (int r = 0; r * 2 * kWave < am; ++r) {
    double pi[2][DIM], xi[2], acc[2] = {0.0, 0.0};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int k = r * 2 * kWave + h * kWave + lane;
      const int64_t i = P.a0 + (k < am ? k : am - 1);
#pragma unroll
      for (int d = 0; d < DIM; ++d) pi[h][d] = pts[d * ld + i];
      xi[h] = k < am ? xs[i] : 0.0;
    }
    // One group: entries of the lane's H rows, their row sums and, with COLS,
    // the group's column sums.
    auto group = [&](int g, auto rows_tag, auto cols_tag) {
      constexpr int H = decltype(rows_tag)::value;
      constexpr bool COLS = decltype(cols_tag)::value;
      double t = 0.0;
#pragma unroll 4
      for (int s = 0; s < kWave; ++s) {
        const int jj = g * kWave + (COLS ? (lane + s) & (kWave - 1) : s);
        const double4 q = src[jj];
#pragma unroll
        for (int h = 0; h < H; ++h) {
          const double dx = pi[h][0] - q.x;
          double s2 = dx * dx;
          if constexpr (DIM > 1) {
            const double dy = pi[h][1] - q.y;
            s2 = fma(dy, dy, s2);
          }
          if constexpr (DIM > 2) {
            const double dz = pi[h][2] - q.z;
            s2 = fma(dz, dz, s2);
          }
          if constexpr (DIM > 3) {
            const double dw = pi[h][DIM - 1] - crd4[jj];
            s2 = fma(dw, dw, s2);
          }
          const double e = kernel_entry<double, KIND>(s2, tab);
          acc[h] = fma(e, q.w, acc[h]);
          if constexpr (COLS) t = fma(e, xi[h], t);
        }
        if constexpr (COLS) t = wave_rotate(t);
      }
      col[r * kPairRows + g * kWave + lane] = t;
    };
    const bool two = am > r * 2 * kWave + kWave;  // the block's second 64 rows exist
    for (int g = (w - r) & 3; g < groups; g += kBlock / kWave) {
      const bool own = diagonal && g <= 2 * r + 1;
      if (diagonal && g < 2 * r) {
        col[r * kPairRows + g * kWave + lane] = 0.0;
      } else if (two) {
        if (own) group(g, std::integral_constant<int, 2>{}, std::false_type{});
        else group(g, std::integral_constant<int, 2>{}, std::true_type{});
      } else {
        if (own) group(g, std::integral_constant<int, 1>{}, std::false_type{});
        else group(g, std::integral_constant<int, 1>{}, std::true_type{});
      }
    }
#pragma unroll
    for (int q = 0; q < kPairBlocks; ++q)
      if (q == r) rows[q][0] = acc[0], rows[q][1] = acc[1];
  }
  __syncthreads();  // every wave is done with the sources
  double* sums = lds;
#pragma unroll
  for (int r = 0; r < kPairBlocks; ++r)
#pragma unroll
    for (int h = 0; h < 2; ++h) sums[w * kPairRows + r * 2 * kWave + h * kWave + lane] = rows[r][h];
  __syncthreads();
  const int blocks = (am + 2 * kWave - 1) / (2 * kWave);
  double* rows_b = rows_a + kPairRows;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int k = u * kBlock + tid;
    double ra = sums[k];
#pragma unroll
    for (int q = 1; q < kBlock / kWave; ++q) ra += sums[q * kPairRows + k];
    double cb = 0.0;
    if (k < groups * kWave)
      for (int r = 0; r < blocks; ++r) cb += col[r * kPairRows + k];
    rows_a[k] = diagonal ? ra + cb : ra;
    if (!diagonal) rows_b[k] = cb;
  }
}

// Far-field coefficients and near pairs in one launch: the coefficients are
// bound by V's bandwidth, the pairs by the vector unit.  Pairs first, so that
// they run beside the items from the start and none is left for the end.
template <int KIND, int DIM, bool STREAM>
__global__ __launch_bounds__(kBlock) void far_near_kernel(
    const mplak_hm_block* __restrict__ blocks, const mplak_hm_item* __restrict__ items, const int32_t* __restrict__ rank,
    int kmax, const double* __restrict__ V, const double* __restrict__ xs, double* __restrict__ fpart,
    const double* __restrict__ pts, int64_t ld, const mplak_hm_pair* __restrict__ pairs, int64_t npairs,
    double* __restrict__ part) {
  __shared__ __attribute__((aligned(16))) double lds[pair_lds(DIM)];
  const int64_t b = blockIdx.x;
  if (b < npairs)
    near_pair<KIND, DIM>(pts, ld, pairs[b], xs, part + b * 2 * kPairRows, lds);
  else
    far_item<STREAM>(blocks, items[b - npairs], rank, kmax, V, xs, fpart + (b - npairs) * kmax);
}

// Far-field rows and near pairs in one launch: U's bandwidth beside the vector
// unit.  A chunk's admissible blocks are split over the workgroup's four waves,
// whose sums are added in wave order.
template <int KIND, int DIM, bool STREAM>
__global__ __launch_bounds__(kBlock) void rows_near_kernel(
    const mplak_hm_chunk* __restrict__ chunks, const int64_t* __restrict__ far_ptr, const int32_t* __restrict__ far_blk,
    const mplak_hm_block* __restrict__ blocks, const int32_t* __restrict__ rank, int kmax, const double* __restrict__ U,
    const double* __restrict__ t, double* __restrict__ ys, const double* __restrict__ xs,
    const double* __restrict__ pts, int64_t ld, const mplak_hm_pair* __restrict__ pairs, int64_t npairs,
    double* __restrict__ part) {
  __shared__ __attribute__((aligned(16))) double lds[pair_lds(DIM)];
  const int64_t b = blockIdx.x;
  if (b < npairs) {
    near_pair<KIND, DIM>(pts, ld, pairs[b], xs, part + b * 2 * kPairRows, lds);
    return;
  }
  constexpr int kWaves = kBlock / kWave;
  const mplak_hm_chunk c = chunks[b - npairs];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  int64_t row[hm::kHmLaneRows];
  bool valid[hm::kHmLaneRows];
  hm::item_rows(c, row, valid);
  double acc[hm::kHmLaneRows] = {};
  hm::far_rows<STREAM>(row, valid, far_ptr, far_blk, c.leaf, blocks, rank, kmax, U, t, w, kWaves, acc);
#pragma unroll
  for (int h = 0; h < hm::kHmLaneRows; ++h) lds[w * hm::kHmRows + h * kWave + lane] = acc[h];
  __syncthreads();
  if ((int)threadIdx.x < c.count) {
    double v = lds[threadIdx.x];
#pragma unroll
    for (int q = 1; q < kWaves; ++q) v += lds[q * hm::kHmRows + threadIdx.x];
    ys[c.r0 + threadIdx.x] = v;
  }
}

// The near partials of a chunk's rows added to its far field, one row per
// thread, kEntBatch partials in flight: into ys (perm == nullptr), or with the
// nugget to the caller's row order.
constexpr int kEntBatch = 8;

__global__ __launch_bounds__(hm::kHmRows) void pairs_finish_kernel(
    const mplak_hm_chunk* __restrict__ chunks, const int64_t* __restrict__ chunk_near,
    const int64_t* __restrict__ near_start, const int64_t* __restrict__ ent_ptr, const int64_t* __restrict__ ent,
    const double* __restrict__ part, double* __restrict__ ys, const int64_t* __restrict__ perm, double nugget,
    const double* __restrict__ x, int64_t shift, int64_t x_count, double* __restrict__ y) {
  const mplak_hm_chunk c = chunks[blockIdx.x];
  if ((int)threadIdx.x >= c.count) return;
  const int64_t nc = chunk_near[blockIdx.x];
  const int64_t row = c.r0 + threadIdx.x;
  const double* p = part + (row - near_start[nc]);
  double s = 0.0;
  const int64_t k1 = ent_ptr[nc + 1];
  for (int64_t k = ent_ptr[nc]; k < k1; k += kEntBatch) {
    double v[kEntBatch];
#pragma unroll
    for (int u = 0; u < kEntBatch; ++u) v[u] = k + u < k1 ? p[ent[k + u] * kPairRows] : 0.0;
#pragma unroll
    for (int u = 0; u < kEntBatch; ++u)
      if (k + u < k1) s += v[u];
  }
  s += ys[row];
  if (perm == nullptr) {
    ys[row] = s;
    return;
  }
  const int64_t i = perm[row], j = i + shift;
  if (nugget != 0.0 && j >= 0 && j < x_count) s = fma(nugget, x[j], s);
  y[i] = s;
}

// Far field and near partials of one apply chunk in one launch: wave p of the
// workgroup's 8 adds the chunk's partial blocks p, p + 8, ... and its share of the
// admissible blocks; the eight sums of a row are added in wave order.
__global__ __launch_bounds__(hm::kHmApplyThreads) void apply_pairs_kernel(
    const mplak_hm_chunk* __restrict__ chunks, const int64_t* __restrict__ chunk_near,
    const int64_t* __restrict__ near_start, const int64_t* __restrict__ ent_ptr, const int64_t* __restrict__ ent,
    const double* __restrict__ part, const int64_t* __restrict__ far_ptr, const int32_t* __restrict__ far_blk,
    const mplak_hm_block* __restrict__ blocks, const int32_t* __restrict__ rank, int kmax,
    const double* __restrict__ U, const double* __restrict__ t, double* __restrict__ ys) {
  __shared__ double red[hm::kHmParts][hm::kHmRows];
  const mplak_hm_chunk c = chunks[blockIdx.x];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  int64_t row[hm::kHmLaneRows];
  bool valid[hm::kHmLaneRows];
  hm::item_rows(c, row, valid);
  const int64_t nc = chunk_near[blockIdx.x];
  const int64_t off = c.r0 - near_start[nc];
  double acc[hm::kHmLaneRows] = {};
  for (int64_t k = ent_ptr[nc] + w; k < ent_ptr[nc + 1]; k += hm::kHmParts) {
    const double* blk = part + ent[k] * kPairRows + off;
#pragma unroll
    for (int h = 0; h < hm::kHmLaneRows; ++h)
      if (valid[h]) acc[h] += blk[h * kWave + lane];
  }
  hm::far_rows<false>(row, valid, far_ptr, far_blk, c.leaf, blocks, rank, kmax, U, t, w, hm::kHmParts, acc);
  hm::finish_rows(acc, row, valid, ys, red);
}

// Kernel and dimension of `p` as compile-time values for `go`.
template <typename F>
void with_points(const mplak_hm_points* p, F&& go) {
  auto with_dim = [&](auto kind) {
    switch (p->dim) {
      case 1: go(kind, std::integral_constant<int, 1>{}); break;
      case 2: go(kind, std::integral_constant<int, 2>{}); break;
      case 3: go(kind, std::integral_constant<int, 3>{}); break;
      default: go(kind, std::integral_constant<int, 4>{}); break;
    }
  };
  if (p->kind == MPLAK_KERNEL_GAUSSIAN)
    with_dim(std::integral_constant<int, MPLAK_KERNEL_GAUSSIAN>{});
  else
    with_dim(std::integral_constant<int, MPLAK_KERNEL_MATERN32>{});
}

template <int KIND>
int launch_aca(const mplak_hm_points* p, const mplak_hm_block* blocks, int64_t nblocks, int kmax, double eps,
               double* U, double* V, int32_t* rank, hipStream_t s) {
  hm::KernelEntries<KIND> e{p->rows, p->cols, p->row_ld, p->col_ld, p->dim};
  hipLaunchKernelGGL(hm::aca_kernel<hm::KernelEntries<KIND>>, dim3((unsigned)nblocks), dim3(kHmThreads), 0, s, e,
                     blocks, kmax, eps, U, V, rank);
  return launch_status();
}

template <int KIND, int DIM>
void launch_apply(const hm::KernelEntries<KIND>& e, int64_t nchunks, hipStream_t s, const mplak_hm_chunk* chunks,
                  const int64_t* near_ptr, const int64_t* near_cols, const int64_t* far_ptr, const int32_t* far_blk,
                  const mplak_hm_block* blocks, const int32_t* rank, int kmax, const double* U, const double* t,
                  const double* xs, double* ys) {
  hipLaunchKernelGGL((hm::apply_kernel<KIND, DIM>), dim3((unsigned)nchunks), dim3(hm::kHmApplyThreads), 0, s, e, chunks,
                     near_ptr, near_cols, far_ptr, far_blk, blocks, rank, kmax, U, t, xs, ys);
}

template <int KIND>
int apply_kind(const mplak_hm_points* p, const mplak_hm_chunk* chunks, int64_t nchunks, const int64_t* near_ptr,
               const int64_t* near_cols, const int64_t* far_ptr, const int32_t* far_blk,
               const mplak_hm_block* blocks, const int32_t* rank, int kmax, const double* U, const double* t,
               const double* xs, double* ys, hipStream_t s) {
  hm::KernelEntries<KIND> e{p->rows, p->cols, p->row_ld, p->col_ld, p->dim};
  switch (p->dim) {
    case 1: launch_apply<KIND, 1>(e, nchunks, s, chunks, near_ptr, near_cols, far_ptr, far_blk, blocks, rank, kmax,
                                  U, t, xs, ys); break;
    case 2: launch_apply<KIND, 2>(e, nchunks, s, chunks, near_ptr, near_cols, far_ptr, far_blk, blocks, rank, kmax,
                                  U, t, xs, ys); break;
    case 3: launch_apply<KIND, 3>(e, nchunks, s, chunks, near_ptr, near_cols, far_ptr, far_blk, blocks, rank, kmax,
                                  U, t, xs, ys); break;
    default: launch_apply<KIND, 0>(e, nchunks, s, chunks, near_ptr, near_cols, far_ptr, far_blk, blocks, rank, kmax,
                                   U, t, xs, ys); break;
  }
  return launch_status();
}

int check_points(const mplak_hm_points* p) {
  if (p == nullptr || p->rows == nullptr || p->cols == nullptr || p->dim < 1 || p->dim > hm::kHmMaxDim ||
      p->row_ld < 0 || p->col_ld < 0)
    return MPLAK_ERR_ARG;
  if (p->kind != MPLAK_KERNEL_GAUSSIAN && p->kind != MPLAK_KERNEL_MATERN32) return MPLAK_ERR_ARG;
  return MPLAK_OK;
}

int64_t grid_for(int64_t n) {
  int64_t g = (n + kBlock - 1) / kBlock;
  return g < 1 ? 1 : (g > 4096 ? 4096 : g);
}

}  // namespace
}  // namespace mplak

using namespace mplak;

extern "C" {

int mplak_hm_gather_scaled(const double* const* points, int32_t dim, int64_t offset, const int64_t* perm, int64_t n,
                           int32_t kind, double length_scale, double* out, int64_t ld, mplak_stream_t stream) {
  if (points == nullptr || perm == nullptr || out == nullptr || dim < 1 || n < 0 || offset < 0 || ld < n ||
      !(length_scale > 0.0) || (kind != MPLAK_KERNEL_GAUSSIAN && kind != MPLAK_KERNEL_MATERN32))
    return MPLAK_ERR_ARG;
  if (n == 0) return MPLAK_OK;
  hipLaunchKernelGGL(gather_scaled_kernel, dim3((unsigned)grid_for(n)), dim3(kBlock), 0, as_stream(stream), points,
                     dim, offset, perm, n, coord_scale(kind, length_scale), out, ld);
  return launch_status();
}

int mplak_hm_aca(const mplak_hm_points* pts, const mplak_hm_block* blocks, int64_t nblocks, int32_t kmax, double eps,
                 double* U, double* V, int32_t* rank, mplak_stream_t stream) {
  int st = check_points(pts);
  if (st != MPLAK_OK) return st;
  if (nblocks < 0 || kmax < 1 || kmax > MPLAK_HM_MAX_RANK || !(eps >= 0.0) || nblocks > 0x7fffffff) return MPLAK_ERR_ARG;
  if (nblocks == 0) return MPLAK_OK;
  if (blocks == nullptr || U == nullptr || V == nullptr || rank == nullptr) return MPLAK_ERR_ARG;
  hipStream_t s = as_stream(stream);
  if (pts->kind == MPLAK_KERNEL_GAUSSIAN)
    return launch_aca<MPLAK_KERNEL_GAUSSIAN>(pts, blocks, nblocks, kmax, eps, U, V, rank, s);
  return launch_aca<MPLAK_KERNEL_MATERN32>(pts, blocks, nblocks, kmax, eps, U, V, rank, s);
}

int mplak_hm_far_partials(const mplak_hm_block* blocks, const mplak_hm_item* items, int64_t nitems,
                          const int32_t* rank, int32_t kmax, const double* V, const double* xs, double* part,
                          mplak_stream_t stream) {
  if (nitems < 0 || nitems > 0x7fffffff || kmax < 1 || kmax > MPLAK_HM_MAX_RANK) return MPLAK_ERR_ARG;
  if (nitems == 0) return MPLAK_OK;
  if (blocks == nullptr || items == nullptr || rank == nullptr || V == nullptr || xs == nullptr || part == nullptr)
    return MPLAK_ERR_ARG;
  hipLaunchKernelGGL(far_partial_kernel<false>, dim3((unsigned)nitems), dim3(kHmThreads), 0, as_stream(stream), blocks,
                     items, rank, kmax, V, xs, part);
  return launch_status();
}

int mplak_hm_far_sum(const int64_t* first_item, int64_t nblocks, const int32_t* rank, int32_t kmax,
                     const double* part, double* t, mplak_stream_t stream) {
  if (nblocks < 0 || kmax < 1 || kmax > MPLAK_HM_MAX_RANK) return MPLAK_ERR_ARG;
  if (nblocks == 0) return MPLAK_OK;
  if (first_item == nullptr || rank == nullptr || part == nullptr || t == nullptr) return MPLAK_ERR_ARG;
  const int64_t total = nblocks * kmax;
  const int64_t g = (total + kBlock - 1) / kBlock;
  if (g > 0x7fffffff) return MPLAK_ERR_ARG;
  hipLaunchKernelGGL(far_sum_kernel, dim3((unsigned)g), dim3(kBlock), 0, as_stream(stream), first_item, nblocks, rank,
                     kmax, part, t);
  return launch_status();
}

int mplak_hm_apply(const mplak_hm_points* pts, const mplak_hm_chunk* chunks, int64_t nchunks, const int64_t* near_ptr,
                   const int64_t* near_cols, const int64_t* far_ptr, const int32_t* far_blk,
                   const mplak_hm_block* blocks, const int32_t* rank, int32_t kmax, const double* U, const double* t,
                   const double* xs, double* ys, mplak_stream_t stream) {
  int st = check_points(pts);
  if (st != MPLAK_OK) return st;
  if (nchunks < 0 || nchunks > 0x7fffffff || kmax < 1 || kmax > MPLAK_HM_MAX_RANK) return MPLAK_ERR_ARG;
  if (nchunks == 0) return MPLAK_OK;
  if (chunks == nullptr || near_ptr == nullptr || far_ptr == nullptr || xs == nullptr || ys == nullptr)
    return MPLAK_ERR_ARG;
  hipStream_t s = as_stream(stream);
  if (pts->kind == MPLAK_KERNEL_GAUSSIAN)
    return apply_kind<MPLAK_KERNEL_GAUSSIAN>(pts, chunks, nchunks, near_ptr, near_cols, far_ptr, far_blk, blocks,
                                             rank, kmax, U, t, xs, ys, s);
  return apply_kind<MPLAK_KERNEL_MATERN32>(pts, chunks, nchunks, near_ptr, near_cols, far_ptr, far_blk, blocks, rank,
                                           kmax, U, t, xs, ys, s);
}

int mplak_hm_far_near(const mplak_hm_points* pts, const mplak_hm_block* blocks, const mplak_hm_item* items,
                      int64_t nitems, const int32_t* rank, int32_t kmax, const double* V, const double* xs,
                      double* fpart, const mplak_hm_pair* pairs, int64_t npairs, double* part, int32_t stream_factors,
                      mplak_stream_t stream) {
  int st = check_points(pts);
  if (st != MPLAK_OK) return st;
  if (nitems < 0 || npairs < 0 || nitems + npairs > 0x7fffffff || kmax < 1 || kmax > MPLAK_HM_MAX_RANK)
    return MPLAK_ERR_ARG;
  if (nitems + npairs == 0) return MPLAK_OK;
  if (nitems > 0 && (blocks == nullptr || items == nullptr || rank == nullptr || V == nullptr || fpart == nullptr))
    return MPLAK_ERR_ARG;
  if (xs == nullptr || (npairs > 0 && (pairs == nullptr || part == nullptr))) return MPLAK_ERR_ARG;
  with_points(pts, [&](auto kind, auto dim) {
    constexpr int K = decltype(kind)::value, D = decltype(dim)::value;
    hipLaunchKernelGGL((stream_factors ? far_near_kernel<K, D, true> : far_near_kernel<K, D, false>),
                       dim3((unsigned)(npairs + nitems)), dim3(kBlock), 0, as_stream(stream), blocks, items, rank, kmax,
                       V, xs, fpart, pts->rows, pts->row_ld, pairs, npairs, part);
  });
  return launch_status();
}

int mplak_hm_rows_near(const mplak_hm_points* pts, const mplak_hm_chunk* chunks, int64_t nchunks,
                       const int64_t* far_ptr, const int32_t* far_blk, const mplak_hm_block* blocks,
                       const int32_t* rank, int32_t kmax, const double* U, const double* t, double* ys,
                       const double* xs, const mplak_hm_pair* pairs, int64_t npairs, double* part,
                       int32_t stream_factors, mplak_stream_t stream) {
  int st = check_points(pts);
  if (st != MPLAK_OK) return st;
  if (nchunks < 0 || npairs < 0 || nchunks + npairs > 0x7fffffff || kmax < 1 || kmax > MPLAK_HM_MAX_RANK)
    return MPLAK_ERR_ARG;
  if (nchunks + npairs == 0) return MPLAK_OK;
  if (nchunks > 0 && (chunks == nullptr || far_ptr == nullptr || ys == nullptr)) return MPLAK_ERR_ARG;
  if (npairs > 0 && (pairs == nullptr || part == nullptr || xs == nullptr)) return MPLAK_ERR_ARG;
  with_points(pts, [&](auto kind, auto dim) {
    constexpr int K = decltype(kind)::value, D = decltype(dim)::value;
    hipLaunchKernelGGL((stream_factors ? rows_near_kernel<K, D, true> : rows_near_kernel<K, D, false>),
                       dim3((unsigned)(npairs + nchunks)), dim3(kBlock), 0, as_stream(stream), chunks, far_ptr, far_blk,
                       blocks, rank, kmax, U, t, ys, xs, pts->rows, pts->row_ld, pairs, npairs, part);
  });
  return launch_status();
}

int mplak_hm_pairs_finish(const mplak_hm_chunk* chunks, int64_t nchunks, const int64_t* chunk_near,
                          const int64_t* near_start, const int64_t* ent_ptr, const int64_t* ent, const double* part,
                          double* ys, const int64_t* perm, double nugget, const double* x, int64_t shift,
                          int64_t x_count, double* y, mplak_stream_t stream) {
  if (nchunks < 0 || nchunks > 0x7fffffff || x_count < 0) return MPLAK_ERR_ARG;
  if (nchunks == 0) return MPLAK_OK;
  if (chunks == nullptr || chunk_near == nullptr || near_start == nullptr || ent_ptr == nullptr || ys == nullptr ||
      (perm != nullptr && (y == nullptr || (nugget != 0.0 && x == nullptr))))
    return MPLAK_ERR_ARG;
  hipLaunchKernelGGL(pairs_finish_kernel, dim3((unsigned)nchunks), dim3(hm::kHmRows), 0, as_stream(stream), chunks,
                     chunk_near, near_start, ent_ptr, ent, part, ys, perm, nugget, x, shift, x_count, y);
  return launch_status();
}

int mplak_hm_near_pairs(const mplak_hm_points* pts, const mplak_hm_pair* pairs, int64_t npairs, const double* xs,
                        double* part, mplak_stream_t stream) {
  return mplak_hm_far_near(pts, nullptr, nullptr, 0, nullptr, 1, nullptr, xs, nullptr, pairs, npairs, part, 0, stream);
}

int mplak_hm_apply_pairs(const mplak_hm_chunk* chunks, int64_t nchunks, const int64_t* chunk_near,
                         const int64_t* near_start, const int64_t* ent_ptr, const int64_t* ent, const double* part,
                         const int64_t* far_ptr, const int32_t* far_blk, const mplak_hm_block* blocks,
                         const int32_t* rank, int32_t kmax, const double* U, const double* t, double* ys,
                         mplak_stream_t stream) {
  if (nchunks < 0 || nchunks > 0x7fffffff || kmax < 1 || kmax > MPLAK_HM_MAX_RANK) return MPLAK_ERR_ARG;
  if (nchunks == 0) return MPLAK_OK;
  if (chunks == nullptr || chunk_near == nullptr || near_start == nullptr || ent_ptr == nullptr || far_ptr == nullptr ||
      ys == nullptr)
    return MPLAK_ERR_ARG;
  hipLaunchKernelGGL(apply_pairs_kernel, dim3((unsigned)nchunks), dim3(hm::kHmApplyThreads), 0, as_stream(stream),
                     chunks, chunk_near, near_start, ent_ptr, ent, part, far_ptr, far_blk, blocks, rank, kmax, U, t,
                     ys);
  return launch_status();
}

int mplak_hm_apply_stored(const mplak_hm_chunk* chunks, int64_t nchunks, const int64_t* leaf_range,
                          const int64_t* near_ptr, const int64_t* near_cols, const int64_t* near_off,
                          const double* stored, const int64_t* far_ptr, const int32_t* far_blk,
                          const mplak_hm_block* blocks, const int32_t* rank, int32_t kmax, const double* U,
                          const double* t, const double* xs, double* ys, mplak_stream_t stream) {
  if (nchunks < 0 || nchunks > 0x7fffffff || kmax < 1 || kmax > MPLAK_HM_MAX_RANK) return MPLAK_ERR_ARG;
  if (nchunks == 0) return MPLAK_OK;
  if (chunks == nullptr || leaf_range == nullptr || near_ptr == nullptr || far_ptr == nullptr || xs == nullptr ||
      ys == nullptr)
    return MPLAK_ERR_ARG;
  hipLaunchKernelGGL(hm::apply_stored_kernel, dim3((unsigned)nchunks), dim3(hm::kHmApplyThreads), 0, as_stream(stream), chunks,
                     leaf_range, near_ptr, near_cols, near_off, stored, far_ptr, far_blk, blocks, rank, kmax, U, t, xs,
                     ys);
  return launch_status();
}

int mplak_hm_scatter_nugget(const double* ys, const int64_t* perm, int64_t n, double nugget, const double* x,
                            int64_t shift, int64_t x_count, double* y, mplak_stream_t stream) {
  if (n < 0 || x_count < 0) return MPLAK_ERR_ARG;
  if (n == 0) return MPLAK_OK;
  if (ys == nullptr || perm == nullptr || y == nullptr || (nugget != 0.0 && x == nullptr)) return MPLAK_ERR_ARG;
  hipLaunchKernelGGL(scatter_nugget_kernel, dim3((unsigned)grid_for(n)), dim3(kBlock), 0, as_stream(stream), ys, perm,
                     n, nugget, x, shift, x_count, y);
  return launch_status();
}

}  // extern "C"
