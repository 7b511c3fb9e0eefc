// Ragged batched kernels for serving many independent kernel-interpolation
// solves at once (no reference counterpart).
//
// A batch is a device array of systems (one per request: its own points, N,
// kernel, right-hand sides and buffers) plus a device table of work items.
// One launch covers every system in the batch: workgroup b processes item b,
// whose fields name the system and the tile of work.  Each system's tiles,
// slabs and vector blocks depend only on that system's own (n, nrhs,
// precision, bytes of its partials), never on what else is in the batch, so a
// system's arithmetic, and therefore its result, is bitwise the same alone and
// in any mix.
//
// Products, two work splits (mplak_ragged_plan picks one per system from its
// n alone, mplak_ragged_plan_within from the bytes of its partials too): SLABS,
// the VALU scheme of the multi-RHS product (one target per thread, RT columns per
// thread, sources through LDS, FP64 slab partials);
// PAIRS, the symmetric tile-pair form (each off-diagonal entry evaluated once
// for both of its rows).  The kernel function, dimension (<= 4) and scale
// come from the system record.
// CG: the batched recurrences of the multi-RHS solver with per-column
// scalars in a state pool, items (system, column, vector block).

#include <math.h>
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "entry.hpp"

namespace mplak {
namespace {

constexpr int kChunk = 256;
constexpr int kRagTargetBlocks = 2048;
constexpr int kMaxRaggedDim = 4;

inline int vec_blocks_r(int64_t n) {
  int64_t b = (n + kBlock * 8 - 1) / (kBlock * 8);
  if (b < 1) b = 1;
  if (b > 1024) b = 1024;
  return (int)b;
}

inline int rt_class(int64_t R) { return R <= 1 ? 1 : (R <= 2 ? 2 : (R <= 4 ? 4 : 8)); }

// LDS of the product of a slab item: sources, values, chunk boxes and the
// FP64 exponential's table.
template <typename T, int RT, int MD>
struct SlabLds {
  T lp[MD][kChunk];
  T lv[RT][kChunk];
  T cbox[kBlock / kWave][2 * MD];
  double exp_tab[Exp2Lds<T>::size];
};

// A mixed plan's FP32 slabs of one chunk leave FP32 partials, the values of the
// FP64 ones in half the bytes.
__host__ __device__ inline bool narrow_slabs(const mplak_ragged_system& S) { return S.reserved != 0; }

// DIM > 0: the system has that dimension; DIM == 0: any dimension <=
// kMaxRaggedDim (coordinates past it are zero).
template <typename T, int RT, int DIM>
__device__ __forceinline__ void slab_item(const mplak_ragged_item& it, const mplak_ragged_system& S, void* lds_raw) {
  constexpr int MD = DIM > 0 ? DIM : kMaxRaggedDim;
  auto& lds = *static_cast<SlabLds<T, RT, MD>*>(lds_raw);
  if (sizeof(T) == 8) fill_exp2_table(lds.exp_tab);  // first read after the chunk barrier below
  const int tid = threadIdx.x;
  const int64_t n = S.n;
  const int dim = S.dim;
  const int64_t R = S.nrhs;
  int64_t i = (int64_t)it.tile * kBlock + tid;
  const bool active = i < n;
  if (!active) i = n - 1;
  const int64_t r0 = (int64_t)it.ctile * RT;
  T pi[MD];
#pragma unroll
  for (int d = 0; d < MD; ++d) pi[d] = d < dim ? (T)(S.points[d * n + i] * S.scale) : T(0);
  const int64_t c0 = (int64_t)it.slab * S.slab_cols;
  const int64_t c1 = (c0 + S.slab_cols < n) ? c0 + S.slab_cols : n;
  // Screening (drop_s > 0): a wave skips a chunk when the bounding boxes of
  // its 64 targets and of the chunk's sources are further apart than drop_s,
  // i.e. every entry of the block is below the system's drop level, and
  // within a kept chunk each 64-source part whose box is that far.
  const bool screen = S.drop_s > 0.0;
  const int lane = tid & (kWave - 1), w = tid / kWave;
  T tbox[2 * MD];
  if (screen) {
#pragma unroll
    for (int d = 0; d < MD; ++d) {
      tbox[d] = wave_min(pi[d]);
      tbox[MD + d] = wave_max(pi[d]);
    }
  }
  double acc[RT];
#pragma unroll
  for (int q = 0; q < RT; ++q) acc[q] = 0.0;
  for (int64_t cb = c0; cb < c1; cb += kChunk) {
    __syncthreads();
    const int64_t j = cb + tid;
#pragma unroll
    for (int d = 0; d < MD; ++d) lds.lp[d][tid] = (j < c1 && d < dim) ? (T)(S.points[d * n + j] * S.scale) : T(0);
#pragma unroll
    for (int q = 0; q < RT; ++q) lds.lv[q][tid] = (j < c1 && r0 + q < R) ? (T)S.V[(r0 + q) * n + j] : T(0);
    if (screen) {  // this wave's part of the chunk box; sources past the slab do not count
#pragma unroll
      for (int d = 0; d < MD; ++d) {
        const T lo = wave_min(j < c1 ? lds.lp[d][tid] : (T)INFINITY);
        const T hi = wave_max(j < c1 ? lds.lp[d][tid] : (T)-INFINITY);
        if (lane == 0) {
          lds.cbox[w][d] = lo;
          lds.cbox[w][MD + d] = hi;
        }
      }
    }
    __syncthreads();
    if (screen) {
      T d2 = T(0);
#pragma unroll
      for (int d = 0; d < MD; ++d) {
        T lo = lds.cbox[0][d], hi = lds.cbox[0][MD + d];
#pragma unroll
        for (int q = 1; q < kBlock / kWave; ++q) {
          lo = fmin(lo, lds.cbox[q][d]);
          hi = fmax(hi, lds.cbox[q][MD + d]);
        }
        const T gap = fmax(T(0), fmax(lo - tbox[MD + d], tbox[d] - hi));
        d2 = fma(gap, gap, d2);
      }
      if (__builtin_amdgcn_readfirstlane((int)(d2 > (T)S.drop_s)) != 0) continue;
    }
    // then per 64-source part of the chunk (wave q staged part q and its box):
    // the wave skips the parts whose box is too far from its targets, and those
    // past the slab
    const int parts = (int)((std::min<int64_t>(c1 - cb, kChunk) + kWave - 1) / kWave);
    uint32_t far_parts = ~0u << parts;
    if (screen) {
#pragma unroll
      for (int q = 0; q < kBlock / kWave; ++q) {
        T d2 = T(0);
#pragma unroll
        for (int d = 0; d < MD; ++d) {
          const T gap = fmax(T(0), fmax(lds.cbox[q][d] - tbox[MD + d], tbox[d] - lds.cbox[q][MD + d]));
          d2 = fma(gap, gap, d2);
        }
        if (__builtin_amdgcn_readfirstlane((int)(d2 > (T)S.drop_s)) != 0) far_parts |= 1u << q;
      }
    }
    T cacc[RT];
#pragma unroll
    for (int q = 0; q < RT; ++q) cacc[q] = T(0);
    // specialised per kernel function (uniform over the workgroup)
    auto run = [&](auto kind_c) {
      constexpr int KIND = decltype(kind_c)::value;
#pragma unroll 1
      for (int part = 0; part < kBlock / kWave; ++part) {
        if ((far_parts >> part) & 1u) continue;
#pragma unroll 2
        for (int jj = part * kWave; jj < (part + 1) * kWave; ++jj) {
          T s = T(0);
#pragma unroll
          for (int d = 0; d < MD; ++d) {
            const T df = pi[d] - lds.lp[d][jj];
            s = fma(df, df, s);
          }
          const T k = kernel_entry<T, KIND>(s, lds.exp_tab);
#pragma unroll
          for (int q = 0; q < RT; ++q) cacc[q] = fma(k, lds.lv[q][jj], cacc[q]);
        }
      }
    };
    if (S.kind == MPLAK_KERNEL_GAUSSIAN)
      run(std::integral_constant<int, MPLAK_KERNEL_GAUSSIAN>{});
    else
      run(std::integral_constant<int, MPLAK_KERNEL_MATERN32>{});
#pragma unroll
    for (int q = 0; q < RT; ++q) acc[q] += (double)cacc[q];
  }
  if (active) {
    float* part32 = reinterpret_cast<float*>(S.part);
#pragma unroll
    for (int q = 0; q < RT; ++q) {
      if (r0 + q >= R) continue;
      const int64_t k = ((int64_t)it.slab * R + r0 + q) * n + i;
      if (narrow_slabs(S)) part32[k] = (float)acc[q];
      else S.part[k] = acc[q];
    }
  }
}

template <typename T, int RT, int DIM>
__global__ __launch_bounds__(kBlock) void ragged_product_kernel(const mplak_ragged_system* __restrict__ systems,
                                                                const mplak_ragged_item* __restrict__ items) {
  const mplak_ragged_item it = items[blockIdx.x];
  const mplak_ragged_system S = systems[it.sys];
  if (S.skip != nullptr && *S.skip != 0) return;
  __shared__ SlabLds<T, RT, (DIM > 0 ? DIM : kMaxRaggedDim)> lds;
  slab_item<T, RT, DIM>(it, S, &lds);
}

// ---- pair scheme ------------------------------------------------------------
//
// The system's points in tiles of 512; item (pair p = (I, J), I <= J, column
// tile).  Each wave holds 128 targets of tile I (two per lane) and walks the
// eight 64-source groups of tile J, all 512 sources staged in LDS with their
// RT values.  Off the diagonal, lane l takes source (l + s) mod 64 at step s:
// one evaluation of each entry feeds the row sums of its two targets and a
// column sum per right-hand side that rotates one lane per step, so after the
// group lane l holds the column sums of source l over the wave's targets.
// The four waves' column sums of a group are added in wave order (FP64) and
// stored; the diagonal pair evaluates its whole block for the row sums.
//
// A system planned for mixed launches may split its pairs: part u of `split`
// works on source groups u 8 / split .. of tile J (the item's slab field).
//
// Partials (entry precision T): rows of I at part_i[((p split + u) R + r) 512 +
// k], rows of J at part_j[(p R + r) 512 + k] (after part_i; each part writes its
// groups), one flag per pair and part after both: 0 when every 128 x 64 block of
// it is screened out (nothing else written), 1 otherwise.  The finish adds, for
// a row of tile X, the pairs (X, P) over P = 0 .. tiles - 1 in order and their
// parts in order.

constexpr int kPairTile = 2 * kBlock;
constexpr int kPairGroups = kPairTile / kWave;
constexpr int64_t kRagPairMinN = 8192;
// In mixed launches, where pairs are split and the chip is shared, evaluating
// an entry once for both of its rows pays from fewer points (alone, an FP32
// product of 2000 points takes 9.3 us either way, one of 4000 11.9 us in pairs
// and 12.1 us in slabs).
constexpr int64_t kMixedPairMinN = 2048;

__host__ __device__ inline int64_t pair_count(int64_t tiles) { return tiles * (tiles + 1) / 2; }

template <typename T>
__device__ __forceinline__ T* pair_rows(const mplak_ragged_system& S) {
  return reinterpret_cast<T*>(S.part);
}
__host__ __device__ inline int pair_split(const mplak_ragged_system& S) { return S.reserved > 1 ? S.reserved : 1; }
template <typename T>
__device__ __forceinline__ int32_t* pair_flags(const mplak_ragged_system& S) {
  const int64_t bytes =
      (pair_split(S) + 1) * pair_count(S.tiles) * (int64_t)S.nrhs * kPairTile * (int64_t)sizeof(T);
  return reinterpret_cast<int32_t*>(reinterpret_cast<char*>(S.part) + (bytes + 255) / 256 * 256);
}

// LDS of a pair item.  The values of a source are padded to an even count, so
// that the rotated reads stay 8-byte aligned.
template <typename T, int RT, int DIM>
struct PairLds {
  static constexpr int kVals = RT > 1 ? (RT + 1) / 2 * 2 : 1;
  typename Quad<T>::type src[kPairTile];              // scaled source coordinates
  __attribute__((aligned(16))) T sval[kPairTile][kVals];  // source values, column tile
  T gbox[kPairGroups][2 * DIM];
  T red[kBlock / kWave][RT][kWave];
  uint32_t wkeep[kBlock / kWave];
  double exp_tab[Exp2Lds<T>::size];
};

template <typename T, int RT, int DIM>
__device__ __forceinline__ void pair_item(const mplak_ragged_item& it, const mplak_ragged_system& S, void* lds_raw) {
  typedef typename Quad<T>::type Q;
  auto& lds = *static_cast<PairLds<T, RT, DIM>*>(lds_raw);
  auto& src = lds.src;
  auto& sval = lds.sval;
  auto& gbox = lds.gbox;
  auto& red = lds.red;
  auto& wkeep = lds.wkeep;
  auto& exp_tab = lds.exp_tab;
  if (sizeof(T) == 8) fill_exp2_table(exp_tab);  // first read after the staging barrier

  const int64_t n = S.n, R = S.nrhs;
  const int64_t p = it.tile;
  int64_t I, J;
  decode_pair(p, I, J);
  const int split = pair_split(S), part = it.slab;
  const int g0 = part * (kPairGroups / split), g1 = g0 + kPairGroups / split;
  const int64_t r0 = (int64_t)it.ctile * RT;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), w = tid / kWave;
  const double scale = S.scale;

  // every global load of the staging is issued before the first use
  double tc[2][DIM], tv[2][RT], sc[2][DIM], sv[2][RT];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int64_t i = I * kPairTile + w * 2 * kWave + h * kWave + lane;
    const int64_t ic = i < n ? i : n - 1;
#pragma unroll
    for (int d = 0; d < DIM; ++d) tc[h][d] = S.points[d * n + ic];
#pragma unroll
    for (int q = 0; q < RT; ++q) tv[h][q] = (i < n && r0 + q < R) ? S.V[(r0 + q) * n + i] : 0.0;
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int64_t j = J * kPairTile + u * kBlock + tid;
    const int64_t jc = j < n ? j : n - 1;
#pragma unroll
    for (int d = 0; d < DIM; ++d) sc[u][d] = S.points[d * n + jc];
#pragma unroll
    for (int q = 0; q < RT; ++q) sv[u][q] = (j < n && r0 + q < R) ? S.V[(r0 + q) * n + j] : 0.0;
  }
  T pi[2][DIM], xi[2][RT];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int d = 0; d < DIM; ++d) pi[h][d] = (T)(tc[h][d] * scale);
#pragma unroll
    for (int q = 0; q < RT; ++q) xi[h][q] = (T)tv[h][q];
  }
  const bool screen = S.drop_s > 0.0;
  T tbox[2 * DIM];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int k = u * kBlock + tid;  // group k / 64 = 4 u + w: one group per wave and pass
    T c[4] = {T(0), T(0), T(0), T(0)};
#pragma unroll
    for (int d = 0; d < DIM; ++d) c[d] = (T)(sc[u][d] * scale);
    Q q;
    q.x = c[0], q.y = c[1], q.z = c[2], q.w = c[3];
    src[k] = q;
#pragma unroll
    for (int r = 0; r < RT; ++r) sval[k][r] = (T)sv[u][r];
    if (screen) {  // padded sources repeat point n - 1 and do not widen the box
#pragma unroll
      for (int d = 0; d < DIM; ++d) {
        const T lo = wave_min(c[d]), hi = wave_max(c[d]);
        if (lane == 0) {
          gbox[k / kWave][d] = lo;
          gbox[k / kWave][DIM + d] = hi;
        }
      }
    }
  }
  if (screen) {
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      tbox[d] = wave_min(fmin(pi[0][d], pi[1][d]));
      tbox[DIM + d] = wave_max(fmax(pi[0][d], pi[1][d]));
    }
  }
  __syncthreads();
  // groups this wave keeps (bit g); a pair nobody keeps writes only its flag
  const uint32_t mine = (1u << g1) - (1u << g0);
  uint32_t keep = mine;
  if (screen) {
    keep = 0u;
#pragma unroll
    for (int g = 0; g < kPairGroups; ++g) {
      T d2 = T(0);
#pragma unroll
      for (int d = 0; d < DIM; ++d) {
        const T gap = fmax(T(0), fmax(gbox[g][d] - tbox[DIM + d], tbox[d] - gbox[g][DIM + d]));
        d2 = fma(gap, gap, d2);
      }
      if (__builtin_amdgcn_readfirstlane((int)(d2 > (T)S.drop_s)) == 0) keep |= 1u << g;
    }
    keep &= mine;
    if (lane == 0) wkeep[w] = keep;
    __syncthreads();
    const uint32_t any = wkeep[0] | wkeep[1] | wkeep[2] | wkeep[3];
    if (any == 0u) {
      if (tid == 0) pair_flags<T>(S)[p * split + part] = 0;
      return;
    }
  }
  if (tid == 0) pair_flags<T>(S)[p * split + part] = 1;

  T* part_i = pair_rows<T>(S);
  T* part_j = part_i + split * pair_count(S.tiles) * R * kPairTile;
  // the compute loop specialised per kernel function (the kind is uniform
  // over the workgroup: no per-entry branch)
  auto run = [&](auto kind_c) {
    constexpr int KIND = decltype(kind_c)::value;
    T acc[2][RT];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < RT; ++q) acc[h][q] = T(0);
    auto entries = [&](const Q& q, T (&e)[2]) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const T dx = pi[h][0] - q.x;
        T s = dx * dx;
        if constexpr (DIM > 1) {
          const T dy = pi[h][1] - q.y;
          s = fma(dy, dy, s);
        }
        if constexpr (DIM > 2) {
          const T dz = pi[h][2] - q.z;
          s = fma(dz, dz, s);
        }
        if constexpr (DIM > 3) {
          const T dw = pi[h][3] - q.w;
          s = fma(dw, dw, s);
        }
        e[h] = kernel_entry<T, KIND>(s, exp_tab);
      }
    };

    if (I == J) {
#pragma unroll 1
      for (int g = g0; g < g1; ++g) {
        if (((keep >> g) & 1u) == 0u) continue;
#pragma unroll 2
        for (int s = 0; s < kWave; ++s) {
          const int jj = g * kWave + s;
          T e[2];
          entries(src[jj], e);
#pragma unroll
          for (int q = 0; q < RT; ++q) {
            const T v = sval[jj][q];
            acc[0][q] = fma(e[0], v, acc[0][q]);
            acc[1][q] = fma(e[1], v, acc[1][q]);
          }
        }
      }
    } else {
#pragma unroll 1
      for (int g = g0; g < g1; ++g) {
        T t[RT];
#pragma unroll
        for (int q = 0; q < RT; ++q) t[q] = T(0);
        if ((keep >> g) & 1u) {
#pragma unroll 2
          for (int s = 0; s < kWave; ++s) {
            const int jj = g * kWave + ((lane + s) & (kWave - 1));
            T e[2];
            entries(src[jj], e);
#pragma unroll
            for (int q = 0; q < RT; ++q) {
              const T v = sval[jj][q];
              acc[0][q] = fma(e[0], v, acc[0][q]);
              acc[1][q] = fma(e[1], v, acc[1][q]);
              t[q] = fma(e[1], xi[1][q], fma(e[0], xi[0][q], t[q]));
              t[q] = wave_rotate(t[q]);
            }
          }
        }
#pragma unroll
        for (int q = 0; q < RT; ++q) red[w][q][lane] = t[q];
        __syncthreads();
        for (int v = tid; v < RT * kWave; v += kBlock) {
          const int q = v / kWave, l = v % kWave;
          double s = (double)red[0][q][l];
#pragma unroll
          for (int ww = 1; ww < kBlock / kWave; ++ww) s += (double)red[ww][q][l];
          if (r0 + q < R) part_j[(p * R + r0 + q) * kPairTile + g * kWave + l] = (T)s;
        }
        __syncthreads();
      }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < RT; ++q)
        if (r0 + q < R)
          part_i[((p * split + part) * R + r0 + q) * kPairTile + w * 2 * kWave + h * kWave + lane] = acc[h][q];
  };
  if (S.kind == MPLAK_KERNEL_GAUSSIAN)
    run(std::integral_constant<int, MPLAK_KERNEL_GAUSSIAN>{});
  else
    run(std::integral_constant<int, MPLAK_KERNEL_MATERN32>{});
}

template <typename T, int RT, int DIM>
__global__ __launch_bounds__(kBlock) void ragged_pair_kernel(const mplak_ragged_system* __restrict__ systems,
                                                             const mplak_ragged_item* __restrict__ items) {
  const mplak_ragged_item it = items[blockIdx.x];
  const mplak_ragged_system S = systems[it.sys];
  // a launch specialised for DIM reads DIM coordinates: other systems are not its items
  if ((S.skip != nullptr && *S.skip != 0) || S.dim != DIM) return;
  __shared__ PairLds<T, RT, DIM> lds;
  pair_item<T, RT, DIM>(it, S, &lds);
}

// Items of every scheme, dimension (<= 4) and column tile in one launch, for
// systems planned by mplak_ragged_plan_mixed: a column tile is min(nrhs, 8)
// wide, and work that a launch per class would queue behind the largest system
// runs beside it.  Bound by the vector unit (FP32 entries and, per right-hand
// side, four FMAs and a rotation for each pair of entries).
template <typename T>
__global__ __launch_bounds__(kBlock) void ragged_mixed_kernel(const mplak_ragged_system* __restrict__ systems,
                                                              const mplak_ragged_item* __restrict__ items) {
  const mplak_ragged_item it = items[blockIdx.x];
  const mplak_ragged_system S = systems[it.sys];
  if (S.skip != nullptr && *S.skip != 0) return;
  constexpr size_t kLds = std::max(sizeof(PairLds<T, 8, 4>), sizeof(SlabLds<T, 8, kMaxRaggedDim>));
  __shared__ __attribute__((aligned(16))) char lds[kLds];
  auto columns = [&](auto rt_c) {
    constexpr int RT = decltype(rt_c)::value;
    if (S.scheme == MPLAK_RAGGED_SLABS) {
      slab_item<T, RT, 0>(it, S, lds);
      return;
    }
    switch (S.dim) {
      case 1: pair_item<T, RT, 1>(it, S, lds); break;
      case 2: pair_item<T, RT, 2>(it, S, lds); break;
      case 3: pair_item<T, RT, 3>(it, S, lds); break;
      default: pair_item<T, RT, 4>(it, S, lds); break;
    }
  };
  switch (S.rt) {
    case 1: columns(std::integral_constant<int, 1>{}); break;
    case 2: columns(std::integral_constant<int, 2>{}); break;
    case 3: columns(std::integral_constant<int, 3>{}); break;
    case 4: columns(std::integral_constant<int, 4>{}); break;
    case 5: columns(std::integral_constant<int, 5>{}); break;
    case 6: columns(std::integral_constant<int, 6>{}); break;
    case 7: columns(std::integral_constant<int, 7>{}); break;
    default: columns(std::integral_constant<int, 8>{}); break;
  }
}

// The finish: 64 entries of Y per workgroup, each wave a slice of their terms
// (every fourth), the slices added in order.  Bound by the latency of the
// partials, which other dies' caches have just written: with one thread per
// entry walking all of its 40 or so terms a twelve-request batch took 27 us,
// with four slices and kFinishLoads terms of each in flight 11 us.
constexpr int kFinishLoads = 8;
constexpr int kFinishSlices = kBlock / kWave;

// Slice k of the partials of row i, right-hand side r: the pairs (X, P) of the
// row's tile X over P = 0 .. tiles - 1, from P = X on one term per part.  A
// partial counts only if its flag says that it was written (it is then never
// used, whatever the memory holds).  A batch past the end adds +0.0, which
// leaves a sum that started at +0.0 unchanged.
template <typename T>
__device__ __forceinline__ double pair_finish_row(const mplak_ragged_system& S, int64_t i, int64_t r, int k) {
  // pair indices and parts fit 32 bits (use_pairs, mixed_parts); the split is a
  // power of two, so there is no division in the loop
  const uint32_t X = (uint32_t)(i / kPairTile), t = (uint32_t)(i % kPairTile), tiles = (uint32_t)S.tiles;
  const uint32_t split = (uint32_t)pair_split(S), shift = (uint32_t)__builtin_ctz(split);
  const int64_t stride = S.nrhs * (int64_t)kPairTile;  // of a pair's rows
  const T* part_i = pair_rows<T>(S) + r * kPairTile + t;
  const T* part_j = part_i + split * pair_count(S.tiles) * stride;
  const int32_t* flags = pair_flags<T>(S);
  auto pair = [](uint32_t I, uint32_t J) { return J * (J + 1) / 2 + I; };
  const uint32_t own = (t / kWave) >> (3 - shift);  // the part of t's group, in pairs whose tile J is X
  const uint32_t terms = X + ((tiles - X) << shift);
  double s = 0.0;
  for (uint32_t m0 = k; m0 < terms; m0 += kFinishLoads * kFinishSlices) {
    double v[kFinishLoads];
#pragma unroll
    for (uint32_t u = 0; u < kFinishLoads; ++u) {
      const uint32_t m = m0 + u * kFinishSlices < terms ? m0 + u * kFinishSlices : m0;
      const uint32_t q = m - X;  // only used for m >= X
      const uint32_t p = m < X ? pair(m, X) : pair(X, X + (q >> shift));
      const uint32_t f = (p << shift) + (m < X ? own : (q & (split - 1)));
      const T w = *(m < X ? part_j + p * stride : part_i + f * stride);
      v[u] = m0 + u * kFinishSlices < terms && flags[f] != 0 ? (double)w : 0.0;
    }
#pragma unroll
    for (uint32_t u = 0; u < kFinishLoads; ++u) s += v[u];
  }
  return s;
}

// Slice k of the partials p[0], p[stride], ... of an entry's slabs.
template <typename T>
__device__ __forceinline__ double slab_finish_row(const T* __restrict__ p, int32_t slabs, int64_t stride, int k) {
  double s = 0.0;
  for (int64_t m0 = k; m0 < slabs; m0 += kFinishLoads * kFinishSlices) {
    double v[kFinishLoads];
#pragma unroll
    for (int u = 0; u < kFinishLoads; ++u) {
      const int64_t m = m0 + u * kFinishSlices;
      v[u] = m < slabs ? (double)p[m * stride] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < kFinishLoads; ++u) s += v[u];
  }
  return s;
}

// items: (system, block) over n * nrhs entries of Y, 256 per item in four
// workgroups
__global__ __launch_bounds__(kBlock) void ragged_finish_kernel(const mplak_ragged_system* __restrict__ systems,
                                                               const mplak_ragged_item* __restrict__ items) {
  __shared__ double red[kFinishSlices][kWave];
  const mplak_ragged_item it = items[blockIdx.x / (kBlock / kWave)];
  const mplak_ragged_system S = systems[it.sys];
  if (S.skip != nullptr && *S.skip != 0) return;
  const int lane = threadIdx.x % kWave, k = threadIdx.x / kWave;
  const int64_t g = (int64_t)it.tile * kBlock + (blockIdx.x % (kBlock / kWave)) * kWave + lane;
  const int64_t n = S.n, R = S.nrhs;
  const bool active = g < n * R;
  const bool narrow = n * R <= 0xffffffffll;
  const int64_t r = narrow ? (int64_t)((uint32_t)g / (uint32_t)n) : g / n, i = g - r * n;
  double s = 0.0;
  if (active) {
    if (S.scheme == MPLAK_RAGGED_PAIRS) {
      s = S.precision == MPLAK_PREC_F64 ? pair_finish_row<double>(S, i, r, k) : pair_finish_row<float>(S, i, r, k);
    } else {
      s = narrow_slabs(S) ? slab_finish_row(reinterpret_cast<const float*>(S.part) + r * n + i, S.slabs, R * n, k)
                          : slab_finish_row(S.part + r * n + i, S.slabs, R * n, k);
    }
  }
  red[k][lane] = s;
  __syncthreads();
  if (k != 0 || !active) return;
#pragma unroll
  for (int q = 1; q < kFinishSlices; ++q) s += red[q][lane];
  if (S.nugget != 0.0) s = fma(S.nugget, S.V[r * n + i], s);
  S.Y[r * n + i] = s;
}

// ---- ragged CG --------------------------------------------------------------

__device__ __forceinline__ mplak_cg_state* cg_in(const mplak_ragged_cg& S, int parity) {
  return S.states + (int64_t)parity * S.nrhs;
}

// items: (system, column, vector block)
__global__ __launch_bounds__(kBlock) void ragged_start_kernel(const mplak_ragged_cg* __restrict__ systems,
                                                              const mplak_ragged_item* __restrict__ items) {
  __shared__ double scratch[kBlock / kWave];
  const mplak_ragged_item it = items[blockIdx.x];
  const mplak_ragged_cg S = systems[it.sys];
  const int64_t n = S.n, off = (int64_t)it.slab * n;
  const int G = S.G;
  double rr = 0.0, bb = 0.0;
  for (int64_t i = (int64_t)it.tile * kBlock + threadIdx.x; i < n; i += (int64_t)G * kBlock) {
    const double bi = S.B[off + i];
    const double ri = bi - S.Z[off + i];
    S.R[off + i] = ri;
    S.D[off + i] = ri;
    rr = fma(ri, ri, rr);
    bb = fma(bi, bi, bb);
  }
  rr = block_sum<kBlock>(rr, scratch);
  bb = block_sum<kBlock>(bb, scratch);
  if (threadIdx.x == 0) {
    S.part[(2 * it.slab) * G + it.tile] = rr;
    S.part[(2 * it.slab + 1) * G + it.tile] = bb;
  }
}

// items: (system, column) in fields (sys, slab); writes states[column] of buffer 0
__global__ __launch_bounds__(kBlock) void ragged_start_final_kernel(const mplak_ragged_cg* __restrict__ systems,
                                                                    const mplak_ragged_item* __restrict__ items) {
  __shared__ double scratch[kBlock / kWave];
  const mplak_ragged_item it = items[blockIdx.x];
  const mplak_ragged_cg S = systems[it.sys];
  const int G = S.G, c = it.slab;
  double rr, bb;
  reduce_partials2<kBlock>(S.part + (2 * c) * G, S.part + (2 * c + 1) * G, G, scratch, rr, bb);
  if (threadIdx.x == 0) {
    mplak_cg_state s;
    s.rr = rr;
    s.bnorm2 = bb;
    s.eps = S.eps;
    s.n_global = (double)S.n;
    // a zero right-hand side with a zero residual is solved exactly (x = 0);
    // 0/0 would otherwise leave a NaN that never meets the tolerance
    s.rel = (bb == 0.0 && rr == 0.0) ? 0.0 : sqrt(rr) / sqrt(bb);
    s.alpha = s.beta = 0.0;
    s.k = 0;
    s.iter_max = 2;
    s.rule = MPLAK_STOP_RELATIVE;
    s.done = s.rel < S.eps ? MPLAK_CONVERGED : MPLAK_RUNNING;
    S.states[c] = s;
  }
}

// one workgroup per system (items: (system, -)); `parity` selects the buffer to read
__global__ __launch_bounds__(kBlock) void ragged_group_kernel(const mplak_ragged_cg* __restrict__ systems,
                                                              const mplak_ragged_item* __restrict__ items, int parity) {
  __shared__ int scratch[kBlock / kWave];
  const mplak_ragged_item it = items[blockIdx.x];
  const mplak_ragged_cg S = systems[it.sys];
  const mplak_cg_state* st = cg_in(S, parity);
  int running = 0;
  for (int c = threadIdx.x; c < S.nrhs; c += kBlock) running += st[c].done == MPLAK_RUNNING ? 1 : 0;
  running = block_sum<kBlock>(running, scratch);
  if (threadIdx.x == 0) {
    S.group->active = running;
    S.group->all_done = running == 0 ? 1 : 0;
  }
}

__global__ __launch_bounds__(kBlock) void ragged_dz_kernel(const mplak_ragged_cg* __restrict__ systems,
                                                           const mplak_ragged_item* __restrict__ items, int parity) {
  const mplak_ragged_item it = items[blockIdx.x];
  const mplak_ragged_cg S = systems[it.sys];
  const int c = it.slab;
  if (cg_in(S, parity)[c].done != MPLAK_RUNNING) return;
  __shared__ double scratch[kBlock / kWave];
  const int64_t n = S.n, off = (int64_t)c * n;
  const int G = S.G;
  double s = 0.0;
  for (int64_t i = (int64_t)it.tile * kBlock + threadIdx.x; i < n; i += (int64_t)G * kBlock)
    s = fma(S.D[off + i], S.Z[off + i], s);
  s = block_sum<kBlock>(s, scratch);
  if (threadIdx.x == 0) S.part[c * G + it.tile] = s;
}

__global__ __launch_bounds__(kBlock) void ragged_update_kernel(const mplak_ragged_cg* __restrict__ systems,
                                                               const mplak_ragged_item* __restrict__ items,
                                                               int parity) {
  const mplak_ragged_item it = items[blockIdx.x];
  const mplak_ragged_cg S = systems[it.sys];
  const int c = it.slab;
  const mplak_cg_state* in = cg_in(S, parity);
  if (in[c].done != MPLAK_RUNNING) return;
  __shared__ double scratch[kBlock / kWave];
  const int G = S.G;
  const double alpha = in[c].rr / reduce_partials<kBlock>(S.part + c * G, G, scratch);
  const int64_t n = S.n, off = (int64_t)c * n;
  double rr = 0.0;
  for (int64_t i = (int64_t)it.tile * kBlock + threadIdx.x; i < n; i += (int64_t)G * kBlock) {
    S.X[off + i] = fma(alpha, S.D[off + i], S.X[off + i]);
    const double ri = fma(-alpha, S.Z[off + i], S.R[off + i]);
    S.R[off + i] = ri;
    rr = fma(ri, ri, rr);
  }
  rr = block_sum<kBlock>(rr, scratch);
  if (threadIdx.x == 0) S.part[(S.nrhs + c) * G + it.tile] = rr;
}

__global__ __launch_bounds__(kBlock) void ragged_direct_kernel(const mplak_ragged_cg* __restrict__ systems,
                                                               const mplak_ragged_item* __restrict__ items,
                                                               int parity) {
  const mplak_ragged_item it = items[blockIdx.x];
  const mplak_ragged_cg S = systems[it.sys];
  const int c = it.slab;
  const mplak_cg_state s_in = cg_in(S, parity)[c];
  mplak_cg_state* out = cg_in(S, 1 - parity);
  if (s_in.done != MPLAK_RUNNING) {
    if (it.tile == 0 && threadIdx.x == 0) out[c] = s_in;
    return;
  }
  __shared__ double scratch[kBlock / kWave];
  const int G = S.G;
  double dz, rr_new;
  reduce_partials2<kBlock>(S.part + c * G, S.part + (S.nrhs + c) * G, G, scratch, dz, rr_new);
  const double beta = rr_new / s_in.rr;
  const int k = s_in.k + 1;
  const double rel = sqrt(rr_new) / sqrt(s_in.bnorm2);
  const bool conv = rel < s_in.eps;
  const bool limit = k >= s_in.iter_max - 1;
  if (!conv) {
    const int64_t n = S.n, off = (int64_t)c * n;
    for (int64_t i = (int64_t)it.tile * kBlock + threadIdx.x; i < n; i += (int64_t)G * kBlock)
      S.D[off + i] = fma(beta, S.D[off + i], S.R[off + i]);
  }
  if (it.tile == 0 && threadIdx.x == 0) {
    mplak_cg_state s = s_in;
    s.rr = rr_new;
    s.rel = rel;
    s.alpha = s_in.rr / dz;
    s.beta = beta;
    s.k = k;
    s.done = conv ? MPLAK_CONVERGED : (limit ? MPLAK_ITER_LIMIT : MPLAK_RUNNING);
    out[c] = s;
  }
}

// items: (system, column, vector block): X += E (E stored in Z's companion buffer `E`)
__global__ __launch_bounds__(kBlock) void ragged_axpy_kernel(const mplak_ragged_cg* __restrict__ systems,
                                                             const mplak_ragged_item* __restrict__ items) {
  const mplak_ragged_item it = items[blockIdx.x];
  const mplak_ragged_cg S = systems[it.sys];
  const int64_t n = S.n, off = (int64_t)it.slab * n;
  for (int64_t i = (int64_t)it.tile * kBlock + threadIdx.x; i < n; i += (int64_t)S.G * kBlock)
    S.Xout[off + i] += S.X[off + i];
}

__global__ __launch_bounds__(kBlock) void ragged_fill_kernel(const mplak_ragged_cg* __restrict__ systems,
                                                             const mplak_ragged_item* __restrict__ items,
                                                             double value) {
  const mplak_ragged_item it = items[blockIdx.x];
  const mplak_ragged_cg S = systems[it.sys];
  const int64_t n = S.n, off = (int64_t)it.slab * n;
  for (int64_t i = (int64_t)it.tile * kBlock + threadIdx.x; i < n; i += (int64_t)S.G * kBlock) S.X[off + i] = value;
}

template <typename T, int DIM>
void launch_product_dim(int rt, const mplak_ragged_system* sys, const mplak_ragged_item* items, int64_t count,
                        hipStream_t st) {
  const dim3 g((unsigned)count), b(kBlock);
  switch (rt) {
    case 1: hipLaunchKernelGGL((ragged_product_kernel<T, 1, DIM>), g, b, 0, st, sys, items); break;
    case 2: hipLaunchKernelGGL((ragged_product_kernel<T, 2, DIM>), g, b, 0, st, sys, items); break;
    case 4: hipLaunchKernelGGL((ragged_product_kernel<T, 4, DIM>), g, b, 0, st, sys, items); break;
    default: hipLaunchKernelGGL((ragged_product_kernel<T, 8, DIM>), g, b, 0, st, sys, items); break;
  }
}

template <typename T>
void launch_product(int rt, int dim, const mplak_ragged_system* sys, const mplak_ragged_item* items, int64_t count,
                    hipStream_t st) {
  switch (dim) {
    case 1: launch_product_dim<T, 1>(rt, sys, items, count, st); break;
    case 2: launch_product_dim<T, 2>(rt, sys, items, count, st); break;
    case 3: launch_product_dim<T, 3>(rt, sys, items, count, st); break;
    case 4: launch_product_dim<T, 4>(rt, sys, items, count, st); break;
    default: launch_product_dim<T, 0>(rt, sys, items, count, st); break;
  }
}

template <typename T, int DIM>
void launch_pairs_dim(int rt, const mplak_ragged_system* sys, const mplak_ragged_item* items, int64_t count,
                      hipStream_t st) {
  const dim3 g((unsigned)count), b(kBlock);
  switch (rt) {
    case 1: hipLaunchKernelGGL((ragged_pair_kernel<T, 1, DIM>), g, b, 0, st, sys, items); break;
    case 2: hipLaunchKernelGGL((ragged_pair_kernel<T, 2, DIM>), g, b, 0, st, sys, items); break;
    case 4: hipLaunchKernelGGL((ragged_pair_kernel<T, 4, DIM>), g, b, 0, st, sys, items); break;
    default: hipLaunchKernelGGL((ragged_pair_kernel<T, 8, DIM>), g, b, 0, st, sys, items); break;
  }
}

template <typename T>
void launch_pairs(int rt, int dim, const mplak_ragged_system* sys, const mplak_ragged_item* items, int64_t count,
                  hipStream_t st) {
  switch (dim) {
    case 1: launch_pairs_dim<T, 1>(rt, sys, items, count, st); break;
    case 2: launch_pairs_dim<T, 2>(rt, sys, items, count, st); break;
    case 3: launch_pairs_dim<T, 3>(rt, sys, items, count, st); break;
    default: launch_pairs_dim<T, 4>(rt, sys, items, count, st); break;
  }
}

// PAIRS for n >= least unless MPLAK_RAGGED_PAIRS says otherwise (0: never, 1:
// every n); the pair index must fit an item's 32-bit field.
bool use_pairs(int64_t n, int64_t least) {
  const char* v = getenv("MPLAK_RAGGED_PAIRS");
  bool on = n >= least;
  if (v != nullptr && *v != '\0') on = atoi(v) != 0;
  const int64_t tiles = (n + kPairTile - 1) / kPairTile;
  return on && pair_count(tiles) <= 0x7fffffff;
}

static_assert(kPairGroups == 8, "pair_finish_row: parts of 8 groups");

// Scale, tiles and, in slabs of whole `unit`s of sources, the split of a system
// whose column tiles are `rt` wide.
void plan_slabs(mplak_ragged_system* s, int rt, int64_t unit) {
  s->rt = rt;
  s->ctiles = (s->nrhs + s->rt - 1) / s->rt;
  s->tiles = (int32_t)((s->n + kBlock - 1) / kBlock);
  int64_t ks = (kRagTargetBlocks + (int64_t)s->tiles * s->ctiles - 1) / ((int64_t)s->tiles * s->ctiles);
  const int64_t units = (s->n + unit - 1) / unit;
  if (ks > units) ks = units;
  if (ks < 1) ks = 1;
  const int64_t per = (units + ks - 1) / ks;
  s->slab_cols = per * unit;
  s->slabs = (int32_t)((s->n + s->slab_cols - 1) / s->slab_cols);
  s->scale = coord_scale(s->kind, s->length_scale);
  s->drop_s = s->drop_log2 > 0.0 ? drop_distance2(s->kind, s->drop_log2) : 0.0;
  s->scheme = MPLAK_RAGGED_SLABS;
  s->reserved = 0;
}

size_t slab_part_bytes(const mplak_ragged_system* s) {
  return (size_t)s->slabs * (size_t)s->nrhs * (size_t)s->n * (narrow_slabs(*s) ? sizeof(float) : sizeof(double));
}

// Partials of a system in pairs shared by `parts` workgroups each.
size_t pair_part_bytes(const mplak_ragged_system* s, int parts) {
  const size_t es = s->precision == MPLAK_PREC_F64 ? sizeof(double) : sizeof(float);
  const size_t pairs = (size_t)pair_count((s->n + kPairTile - 1) / kPairTile);
  return align_up((size_t)(parts + 1) * pairs * (size_t)s->nrhs * kPairTile * es, 256) +
         align_up((size_t)parts * pairs * sizeof(int32_t), 256);
}

size_t plan_pairs(mplak_ragged_system* s, int parts) {
  s->scheme = MPLAK_RAGGED_PAIRS;
  s->tiles = (int32_t)((s->n + kPairTile - 1) / kPairTile);
  s->slabs = 0;
  s->slab_cols = 0;
  s->reserved = parts;
  return pair_part_bytes(s, parts);
}

bool plannable(const mplak_ragged_system* s) {
  return s != nullptr && s->n > 0 && s->nrhs > 0 && s->dim >= 1 && s->dim <= kMaxRaggedDim;
}

// Workgroups per tile pair in a mixed launch: the largest power of two up to 8
// that keeps pairs times workgroups below 1200 and the partials within `bytes`
// (0 if none does).  One workgroup a pair leaves a 13455-point system's 378 pairs
// on 256 CUs, two on some and one on the others; each further part is another
// row set for the finish to read (twelve requests of up to 24576 points: 60.1 ms
// at 1200, 61.8 ms at 600).
int mixed_parts(const mplak_ragged_system* s, size_t bytes) {
  const int64_t pairs = pair_count((s->n + kPairTile - 1) / kPairTile);
  int k = 1;
  while (k < kPairGroups && pairs * (2 * k) < 1200) k *= 2;
  while (k > 0 && pair_part_bytes(s, k) > bytes) k /= 2;
  return k;
}

}  // namespace
}  // namespace mplak

using namespace mplak;

extern "C" {

size_t mplak_ragged_plan(mplak_ragged_system* s) {
  if (!plannable(s)) return 0;
  plan_slabs(s, rt_class(s->nrhs), kChunk);
  return use_pairs(s->n, kRagPairMinN) ? plan_pairs(s, 1) : slab_part_bytes(s);
}

size_t mplak_ragged_plan_mixed(mplak_ragged_system* s) {
  if (!plannable(s)) return 0;
  mplak_ragged_system wide = *s;
  wide.precision = MPLAK_PREC_F64;
  return mplak_ragged_plan_within(s, mplak_ragged_plan(&wide));
}

size_t mplak_ragged_plan_within(mplak_ragged_system* s, size_t bytes) {
  // FP64 systems are launched by class
  if (!plannable(s) || s->precision == MPLAK_PREC_F64) return mplak_ragged_plan(s);
  const int rt = s->nrhs < 8 ? s->nrhs : 8;
  plan_slabs(s, rt, kWave);
  // whole pairs would sum 512 sources in FP32 where slabs sum 256
  const int parts = use_pairs(s->n, kMixedPairMinN) ? mixed_parts(s, bytes) : 0;
  if (parts > (use_pairs(s->n, kRagPairMinN) ? 0 : 1)) return plan_pairs(s, parts);
  for (int64_t unit = kWave;; unit *= 2) {
    plan_slabs(s, rt, unit);
    s->reserved = s->slab_cols <= kChunk;
    const size_t need = slab_part_bytes(s);
    if (need <= bytes || unit == kChunk) return need;
  }
}

int64_t mplak_ragged_product_items(const mplak_ragged_system* s, mplak_ragged_item* out, int32_t sys_index) {
  if (s == nullptr || s->tiles <= 0) return 0;
  if (s->scheme == MPLAK_RAGGED_PAIRS) {
    const int64_t pairs = pair_count(s->tiles);
    const int split = pair_split(*s);
    if (out) {
      int64_t k = 0;
      for (int32_t c = 0; c < s->ctiles; ++c)
        for (int64_t q = 0; q < pairs; ++q)
          for (int32_t u = 0; u < split; ++u) out[k++] = mplak_ragged_item{sys_index, (int32_t)q, u, c};
    }
    return pairs * split * s->ctiles;
  }
  const int64_t count = (int64_t)s->tiles * s->slabs * s->ctiles;
  if (out) {
    int64_t k = 0;
    for (int32_t c = 0; c < s->ctiles; ++c)
      for (int32_t sl = 0; sl < s->slabs; ++sl)
        for (int32_t t = 0; t < s->tiles; ++t) out[k++] = mplak_ragged_item{sys_index, t, sl, c};
  }
  return count;
}

int64_t mplak_ragged_finish_items(const mplak_ragged_system* s, mplak_ragged_item* out, int32_t sys_index) {
  if (s == nullptr || s->n <= 0) return 0;
  const int64_t count = (s->n * s->nrhs + kBlock - 1) / kBlock;
  if (out)
    for (int64_t b = 0; b < count; ++b) out[b] = mplak_ragged_item{sys_index, (int32_t)b, 0, 0};
  return count;
}

int mplak_ragged_product(const mplak_ragged_system* systems, const mplak_ragged_item* items, int64_t count, int rt,
                         int dim, int precision, int scheme, mplak_stream_t s) {
  if (count <= 0) return MPLAK_OK;
  if (!systems || !items || count > 0x7fffffff || dim < 0 || dim > kMaxRaggedDim) return MPLAK_ERR_ARG;
  if (scheme != MPLAK_RAGGED_SLABS && scheme != MPLAK_RAGGED_PAIRS) return MPLAK_ERR_ARG;
  if (scheme == MPLAK_RAGGED_PAIRS && dim == 0) return MPLAK_ERR_ARG;
  hipStream_t hs = as_stream(s);
  if (scheme == MPLAK_RAGGED_PAIRS) {
    if (precision == MPLAK_PREC_F64)
      launch_pairs<double>(rt, dim, systems, items, count, hs);
    else
      launch_pairs<float>(rt, dim, systems, items, count, hs);
  } else if (precision == MPLAK_PREC_F64) {
    launch_product<double>(rt, dim, systems, items, count, hs);
  } else {
    launch_product<float>(rt, dim, systems, items, count, hs);
  }
  return launch_status();
}

int mplak_ragged_product_mixed(const mplak_ragged_system* systems, const mplak_ragged_item* items, int64_t count,
                               mplak_stream_t s) {
  if (count <= 0) return MPLAK_OK;
  if (!systems || !items || count > 0x7fffffff) return MPLAK_ERR_ARG;
  hipLaunchKernelGGL(ragged_mixed_kernel<float>, dim3((unsigned)count), dim3(kBlock), 0, as_stream(s), systems, items);
  return launch_status();
}

int mplak_ragged_finish(const mplak_ragged_system* systems, const mplak_ragged_item* items, int64_t count,
                        mplak_stream_t s) {
  if (count <= 0) return MPLAK_OK;
  if (!systems || !items) return MPLAK_ERR_ARG;
  if (count > 0x7fffffff / (kBlock / kWave)) return MPLAK_ERR_ARG;
  hipLaunchKernelGGL(ragged_finish_kernel, dim3((unsigned)(count * (kBlock / kWave))), dim3(kBlock), 0, as_stream(s),
                     systems, items);
  return launch_status();
}

int32_t mplak_ragged_cg_blocks(int64_t n) { return vec_blocks_r(n); }

size_t mplak_ragged_cg_part_bytes(int64_t n, int32_t nrhs) {
  return (size_t)2 * vec_blocks_r(n) * (size_t)nrhs * sizeof(double);
}

int64_t mplak_ragged_cg_items(const mplak_ragged_cg* s, mplak_ragged_item* out, int32_t sys_index) {
  if (s == nullptr || s->n <= 0) return 0;
  const int64_t count = (int64_t)s->G * s->nrhs;
  if (out) {
    int64_t k = 0;
    for (int32_t c = 0; c < s->nrhs; ++c)
      for (int32_t b = 0; b < s->G; ++b) out[k++] = mplak_ragged_item{sys_index, b, c, 0};
  }
  return count;
}

int mplak_ragged_cg_op(int op, const mplak_ragged_cg* systems, const mplak_ragged_item* items, int64_t count,
                       int parity, double value, mplak_stream_t s) {
  if (count <= 0) return MPLAK_OK;
  if (!systems || !items) return MPLAK_ERR_ARG;
  hipStream_t hs = as_stream(s);
  const dim3 g((unsigned)count), b(kBlock);
  switch (op) {
    case MPLAK_RAGGED_START: hipLaunchKernelGGL(ragged_start_kernel, g, b, 0, hs, systems, items); break;
    case MPLAK_RAGGED_START_FINAL: hipLaunchKernelGGL(ragged_start_final_kernel, g, b, 0, hs, systems, items); break;
    case MPLAK_RAGGED_GROUP: hipLaunchKernelGGL(ragged_group_kernel, g, b, 0, hs, systems, items, parity); break;
    case MPLAK_RAGGED_DZ: hipLaunchKernelGGL(ragged_dz_kernel, g, b, 0, hs, systems, items, parity); break;
    case MPLAK_RAGGED_UPDATE: hipLaunchKernelGGL(ragged_update_kernel, g, b, 0, hs, systems, items, parity); break;
    case MPLAK_RAGGED_DIRECT: hipLaunchKernelGGL(ragged_direct_kernel, g, b, 0, hs, systems, items, parity); break;
    case MPLAK_RAGGED_AXPY: hipLaunchKernelGGL(ragged_axpy_kernel, g, b, 0, hs, systems, items); break;
    case MPLAK_RAGGED_FILL: hipLaunchKernelGGL(ragged_fill_kernel, g, b, 0, hs, systems, items, value); break;
    default: return MPLAK_ERR_ARG;
  }
  return launch_status();
}

}  // extern "C"
