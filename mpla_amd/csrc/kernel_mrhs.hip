// Multi-right-hand-side kernel-matrix products Y = K V (V is N x R) on gfx950.
//
// No counterpart in the reference (its only product is single-vector,
// src/kernel.cu:87-171).  Three kernels:
//
// * VALU kernel (FP64 and FP32 for narrow V): one target per thread, a tile
//   of RT columns of V accumulated per thread, sources streamed through LDS.
//   Each kernel entry is computed once per column tile.
//
// * MFMA kernel (BF16, split BF16 "bf16x3", FP32): a wave owns 64 targets
//   (two 32-row MFMA blocks) and all R columns.  For every step of 16 sources
//   each lane evaluates its 16 kernel entries in FP32 directly in the
//   A-operand layout of v_mfma_f32_32x32x16_bf16 (lane l: target l%32 of the
//   row block, sources 8*(l/32) .. +7 of the step), so entries never leave
//   registers.  V is packed once per call into an MFMA-native layout (one
//   16-byte B operand per lane per step and 32-column block, contiguous per
//   wave).  bf16x3 splits entries and V into hi + lo BF16 parts and adds the
//   three leading products (K_hi V_hi + K_hi V_lo + K_lo V_hi).  FP32 uses
//   v_mfma_f32_32x32x2_f32 with eight K=2 products per step.
//
// * FP64 MFMA kernel (FP64, wide V): below.
//
// All split the sources into slabs (accumulation within a slab in FP64 for
// FP64 entries, in FP32 on the matrix cores otherwise) and a finish kernel
// adds the slabs' partials in FP64, in slab order, with the nugget term:
// deterministic for a given shape.

#include <math.h>

#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "entry.hpp"

namespace mplak {
namespace {

constexpr int kChunk = 256;          // sources per LDS chunk
constexpr int kMaxDim = 16;
constexpr int kValuUnit = 32;  // sources a slab of the vector kernel is a multiple of

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

struct Slabs {
  int64_t tiles, slabs, slab_cols;
};

// Split of the sources for a kernel with `occ` workgroups resident
// per CU: the slab count (of whole chunks of sources) that minimises, in
// units of one workgroup's chunk on a full CU, the chunks of the busiest CU
// plus the slabs' partials, written and read back once each.  A CU with fewer
// than `occ` workgroups takes a chunk down to a quarter of that time.  Measured:
// partials 4 TB/s and 0.15 us of latency a slab (n = 3000, 16 columns: 47 slabs
// 27 us, 16 slabs 25 us), against 8 us for a 64-column BF16x3 chunk and 18 us for an
// FP64 one (n = 20001, 64 columns in FP64, at three waves a SIMD: 1.44 ms in 8
// slabs, five workgroups on the busiest CU; 1.66 ms in 4, three).  At most 16
// workgroups a CU, or four rounds of the resident ones.
// `drain`: share of a long workgroup's chunks (those past kDrainChunks) that the
// chip is partly idle at the end of a product.  Workgroups that start together
// end 10 % apart and more, so that one even round of long ones loses to several
// rounds of shorter ones (BF16, n = 131072, 64 columns: 6.41 ms in 2 slabs, 5.70
// ms in 8); short ones lose less than their slabs cost (n = 12000: 2 % per
// iteration with the share taken of every chunk).
// `longest`: most sources of a slab.
constexpr double kMfmaDrain = 0.12;
constexpr int64_t kDrainChunks = 64;
inline Slabs balanced_slabs(int64_t rows, int64_t cols, int tile_rows, int chunk, int occ, int64_t R,
                            int64_t col_tiles = 1, double slab_weight = 1.0, double drain = 0.0,
                            int64_t longest = INT64_MAX) {
  constexpr int64_t kCus = 256;
  Slabs p;
  p.tiles = (rows + tile_rows - 1) / tile_rows;
  const int64_t chunks = (cols + chunk - 1) / chunk;
  const int64_t least = longest < cols ? (chunks + longest / chunk - 1) / (longest / chunk) : 1;
  const int64_t most =
      std::min<int64_t>(chunks, std::max<int64_t>(kCus * std::max(4 * occ, 16) / (p.tiles * col_tiles), least));
  const double slab_cost = slab_weight * (0.02 + 2.4e-7 * (double)rows * (double)R);
  double best = 0.0;
  for (int64_t ks = least; ks <= most;) {
    const int64_t per = (chunks + ks - 1) / ks;
    const int64_t slabs = (chunks + per - 1) / per;
    const double m = (double)((p.tiles * col_tiles * slabs + kCus - 1) / kCus) / occ;  // of the busiest CU, in full CUs
    const double cost = (double)per * (m >= 1.0 ? m : 0.25 + 0.75 * m) +
                        drain * (double)std::max<int64_t>(per - kDrainChunks, 0) + slab_cost * (double)slabs;
    if (ks == least || cost < best) {
      best = cost;
      p.slabs = slabs;
      p.slab_cols = per * chunk;
    }
    if (per == 1) break;
    ks = (chunks + per - 2) / (per - 1);  // the next count has shorter slabs: few counts of many chunks do
  }
  return p;
}

// Most sources of a slab that the matrix cores add up in FP32.  The error of
// such a sum grows with the root of its length, so a slab is never longer than
// the share of one of 2048 workgroups of 256 targets: 256 sources up to 11520
// points, 512 to 16384, 1024 at 20001, 4608 at 50000, 32768 at 131072.  The
// balance alone would take 704 sources at 9000 points and 1344 at 16000 (relative
// error of FP32 products 5.0e-7 and 6.6e-7; so bounded 3.2e-7 and 4.3e-7).  The
// additional partials cost 64 columns, BF16x3, at 9000 points 82 -> 89 us, at 16000
// 179 -> 185 us, at 50000 nothing.
inline int64_t longest_fp32_slab(int64_t rows, int64_t cols) {
  constexpr int64_t kTile = 256, kWorkgroups = 2048;
  const int64_t tiles = (rows + kTile - 1) / kTile, chunks = (cols + kTile - 1) / kTile;
  const int64_t slabs = std::min((kWorkgroups + tiles - 1) / tiles, chunks);
  return (chunks + slabs - 1) / slabs * kTile;
}

// ---------------------------------------------------------------------------
// VALU kernel.  grid = (target tiles of 256, slabs, column tiles of RT).
// part layout: part[(slab * R + r) * rows + i].  Bound by the vector unit, and
// while slabs were whole 256-source chunks by a few waves of long serial loops;
// slabs are now multiples of 32 sources, as many as the balance below gives (2-D
// Matern in FP64, 5 columns: n = 1797 38 -> 15 us, n = 6000 86 -> 54 us, n =
// 12000 242 -> 181 us; 3-D Gaussian in FP32: 22 -> 13, 46 -> 31, 115 -> 100 us).

template <typename T, int KIND, int DIM, int RT>
__global__ __launch_bounds__(kBlock) void mrhs_valu_kernel(
    const double* const* __restrict__ points, int dim_rt, int64_t row_off, int64_t rows, int64_t col_off,
    int64_t cols, int64_t slab_cols, double scale, int64_t R, const double* __restrict__ V, int64_t ldv,
    double* __restrict__ part, const int32_t* __restrict__ skip) {
  if (skip != nullptr && *skip != 0) return;
  constexpr int MD = DIM > 0 ? DIM : kMaxDim;
  const int dim = DIM > 0 ? DIM : dim_rt;
  __shared__ T lp[MD][kChunk];
  __shared__ T lv[RT][kChunk];
  __shared__ double exp_tab[Exp2Lds<T>::size];
  if (sizeof(T) == 8) fill_exp2_table(exp_tab);  // first read after the chunk barrier below
  const int tid = threadIdx.x;
  int64_t i = (int64_t)blockIdx.x * kBlock + tid;
  const bool active = i < rows;
  if (!active) i = rows - 1;
  const int64_t r0 = (int64_t)blockIdx.z * RT;
  T pi[MD];
#pragma unroll
  for (int d = 0; d < MD; ++d) pi[d] = d < dim ? (T)(points[d][row_off + i] * scale) : T(0);
  const int64_t c0 = (int64_t)blockIdx.y * slab_cols;
  const int64_t c1 = (c0 + slab_cols < cols) ? c0 + slab_cols : cols;
  double acc[RT];
#pragma unroll
  for (int q = 0; q < RT; ++q) acc[q] = 0.0;
  for (int64_t cb = c0; cb < c1; cb += kChunk) {
    __syncthreads();
    const int64_t j = cb + tid;
#pragma unroll
    for (int d = 0; d < MD; ++d) lp[d][tid] = (j < c1 && d < dim) ? (T)(points[d][col_off + j] * scale) : T(0);
#pragma unroll
    for (int q = 0; q < RT; ++q) lv[q][tid] = (j < c1 && r0 + q < R) ? (T)V[(r0 + q) * ldv + j] : T(0);
    __syncthreads();
    T cacc[RT];
#pragma unroll
    for (int q = 0; q < RT; ++q) cacc[q] = T(0);
    const int jn = (int)(c1 - cb < kChunk ? c1 - cb : kChunk);
#pragma unroll 2
    for (int jj = 0; jj < jn; ++jj) {
      T s = T(0);
#pragma unroll
      for (int d = 0; d < MD; ++d)
        if (d < dim) {
          const T df = pi[d] - lp[d][jj];
          s = fma(df, df, s);
        }
      const T k = kernel_entry<T, KIND>(s, exp_tab);
#pragma unroll
      for (int q = 0; q < RT; ++q) cacc[q] = fma(k, lv[q][jj], cacc[q]);
    }
#pragma unroll
    for (int q = 0; q < RT; ++q) acc[q] += (double)cacc[q];
  }
  if (active) {
#pragma unroll
    for (int q = 0; q < RT; ++q)
      if (r0 + q < R) part[((int64_t)blockIdx.y * R + r0 + q) * rows + i] = acc[q];
  }
}

// ---------------------------------------------------------------------------
// MFMA kernel.
//
// Sources are packed once per call (pack_kernel) into blocks of 64, each the
// image of its LDS staging:
//   64 float4            scaled coordinates (padding: far away)
//   BF16 / BF16X3 : per 16-source step and 32-column block 64 lanes x 8 bf16,
//                   lane l holds V[16 s + 8 (l/32) + t][32 cb + l%32]; BF16X3
//                   stores the hi parts of the block, then its lo parts
//   FP32          : the same with 8 floats, V[16 s + 2 t + l/32][32 cb + l%32]
// (t = 0..7).  A workgroup copies two blocks at a time straight into LDS and
// its four waves read their operands from there: read from global memory by
// every wave, the operands (4 KiB per wave and step in BF16x3) took up to 45
// bytes a clock and CU through a 64-byte L1.

enum MfmaMode { kModeBf16 = 0, kModeBf16x3 = 1, kModeF32 = 2 };

constexpr int kWaveTargets = 64;                    // two 32-row MFMA blocks
constexpr int kMfmaTile = kWaveTargets * (kBlock / kWave);  // 256 targets per workgroup
constexpr int kMfmaSlab = 64;                       // sources per packed block
constexpr int kMfmaStage = 2;                       // blocks in LDS at a time
constexpr int kBlockSteps = kMfmaSlab / 16;
constexpr size_t kPackAlign = 16;                   // the copies into LDS move aligned 16-byte words
// resident waves per SIMD (and workgroups per CU) by 32-column blocks
constexpr int mfma_waves(int cblocks) { return cblocks == 1 ? 5 : 4; }
constexpr int64_t kMfmaGroup = 64;  // columns per MFMA launch (two 32-column blocks)

// Bytes of one step and column block, of one operand part and of a block.
constexpr int step_bytes(int mode) { return kWave * (mode == kModeF32 ? 32 : 16); }
constexpr int part_bytes(int mode, int cblocks) { return kBlockSteps * cblocks * step_bytes(mode); }
constexpr int block_bytes(int mode, int cblocks) {
  return kMfmaSlab * 16 + part_bytes(mode, cblocks) * (mode == kModeBf16x3 ? 2 : 1);
}

__global__ __launch_bounds__(kBlock) void pack_kernel(const double* const* __restrict__ points, int dim,
                                                      int64_t col_off, double scale, const double* __restrict__ V,
                                                      int64_t ldv, int64_t R, int64_t cols, int64_t blocks,
                                                      int cblocks, int mode, char* __restrict__ out) {
  // one workgroup per block; one thread per (step, cblock, lane)
  const int64_t bytes = kMfmaSlab * 16 + (int64_t)kBlockSteps * cblocks * step_bytes(mode) * (mode == kModeBf16x3 ? 2 : 1);
  for (int64_t b = blockIdx.x; b < blocks; b += gridDim.x) {
    char* image = out + b * bytes;
    char* ops = image + kMfmaSlab * 16;
    if (threadIdx.x < kMfmaSlab) {
      const int64_t j = b * kMfmaSlab + threadIdx.x;
      float4 q = make_float4(0.f, 0.f, 0.f, 0.f);
      if (j < cols) {
        q.x = (float)(points[0][col_off + j] * scale);
        if (dim > 1) q.y = (float)(points[1][col_off + j] * scale);
        if (dim > 2) q.z = (float)(points[2][col_off + j] * scale);
        if (dim > 3) q.w = (float)(points[3][col_off + j] * scale);
      } else {
        q.x = 1.0e4f;  // far away: entries of padded sources underflow to 0
      }
      reinterpret_cast<float4*>(image)[threadIdx.x] = q;
    }
    for (int g = threadIdx.x; g < kBlockSteps * cblocks * kWave; g += kBlock) {
      const int lane = g % kWave, cb = (g / kWave) % cblocks, st = g / (kWave * cblocks);
      const int64_t r = cb * 32 + (lane % 32), j0 = b * kMfmaSlab + 16 * st;
      if (mode == kModeF32) {
        float* o = reinterpret_cast<float*>(ops) + g * 8;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          const int64_t j = j0 + 2 * t + lane / 32;
          o[t] = (j < cols && r < R) ? (float)V[r * ldv + j] : 0.0f;
        }
      } else {
        bf16x8 hi, lo;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          const int64_t j = j0 + 8 * (lane / 32) + t;
          const float v = (j < cols && r < R) ? (float)V[r * ldv + j] : 0.0f;
          hi[t] = (__bf16)v;
          lo[t] = (__bf16)(v - (float)hi[t]);
        }
        reinterpret_cast<bf16x8*>(ops)[g] = hi;
        if (mode == kModeBf16x3) reinterpret_cast<bf16x8*>(ops)[kBlockSteps * cblocks * kWave + g] = lo;
      }
    }
  }
}

// DIM: the points' dimension (1..4); coordinates past it are not evaluated.
// Squared distance over the first DIM coordinates.
template <int DIM>
__device__ __forceinline__ float dist2(const float (&p)[4], const float4& q) {
  const float dx = p[0] - q.x;
  float s = dx * dx;
  if (DIM > 1) {
    const float dy = p[1] - q.y;
    s = fmaf(dy, dy, s);
  }
  if (DIM > 2) {
    const float dz = p[2] - q.z;
    s = fmaf(dz, dz, s);
  }
  if (DIM > 3) {
    const float dw = p[3] - q.w;
    s = fmaf(dw, dw, s);
  }
  return s;
}

// 16 bytes per lane from global memory straight into LDS (the wave's lanes at
// consecutive 16-byte slots from `lds`), counted by vmcnt.
__device__ __forceinline__ void load_to_lds(const char* global, char* lds) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)global,
                                   (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}

// Bound by the vector unit's entry evaluation (per entry 11 instructions, one
// square root and one exponential for Matern BF16x3) and, in BF16x3, by the
// matrix products, which overlap it only in part.
template <int KIND, int MODE, int CB, int DIM>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(mfma_waves(CB), mfma_waves(CB)))) void
mrhs_mfma_kernel(const double* const* __restrict__ points, int64_t row_off, int64_t rows, int64_t blocks,
                 int64_t slab_blocks, double scale, int64_t R, const char* __restrict__ packed,
                 float* __restrict__ part, const int32_t* __restrict__ skip) {
  if (skip != nullptr && *skip != 0) return;
  constexpr int kBytes = block_bytes(MODE, CB), kPart = part_bytes(MODE, CB);
  __shared__ __attribute__((aligned(16))) char image[kMfmaStage * kBytes];
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int64_t base = (int64_t)blockIdx.x * kMfmaTile + wave * kWaveTargets;

  // target coordinates for the two row blocks of this lane
  float pa[2][4];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    int64_t i = base + h * 32 + (lane % 32);
    if (i >= rows) i = rows - 1;
#pragma unroll
    for (int d = 0; d < 4; ++d) pa[h][d] = d < DIM ? (float)(points[d][row_off + i] * scale) : 0.0f;
  }

  f32x16 acc[2][CB];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[h][c][v] = 0.0f;

  const int64_t b0 = (int64_t)blockIdx.y * slab_blocks;
  const int64_t b1 = b0 + slab_blocks < blocks ? b0 + slab_blocks : blocks;
  for (int64_t b = b0; b < b1; b += kMfmaStage) {
    const int count = (int)(b1 - b < kMfmaStage ? b1 - b : kMfmaStage);
    __syncthreads();
    for (int k = wave * 1024; k < count * kBytes; k += (kBlock / kWave) * 1024)
      load_to_lds(packed + b * kBytes + k + lane * 16, image + k);
    // the copies of every wave are in LDS before any wave passes the barrier
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
#pragma unroll 1
    for (int st = 0; st < count * kBlockSteps; ++st) {
      const char* blk = image + (st / kBlockSteps) * kBytes;
      const int s4 = st % kBlockSteps;
      const float4* lp = reinterpret_cast<const float4*>(blk) + 16 * s4;
      const char* ops = blk + kMfmaSlab * 16 + s4 * CB * step_bytes(MODE) + lane * (step_bytes(MODE) / kWave);
      // ---- kernel entries in A-operand layout
      float e[2][8];
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const float4 q = lp[MODE == kModeF32 ? 2 * t + lane / 32 : 8 * (lane / 32) + t];
#pragma unroll
        for (int h = 0; h < 2; ++h) e[h][t] = kernel_entry<float, KIND>(dist2<DIM>(pa[h], q), nullptr);
      }
      // ---- contraction with the packed V operands
      if (MODE == kModeF32) {
#pragma unroll
        for (int c = 0; c < CB; ++c) {
          const float4* src = reinterpret_cast<const float4*>(ops + c * step_bytes(MODE));
          const float4 b0v = src[0], b1v = src[1];
          const float bv[8] = {b0v.x, b0v.y, b0v.z, b0v.w, b1v.x, b1v.y, b1v.z, b1v.w};
#pragma unroll
          for (int t = 0; t < 8; ++t) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
              acc[h][c] = __builtin_amdgcn_mfma_f32_32x32x2f32(e[h][t], bv[t], acc[h][c], 0, 0, 0);
          }
        }
      } else {
        // two entries at a time: one conversion instruction per pair and part
        bf16x8 ahi[2], alo[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int t = 0; t < 8; t += 2) {
            const f32x2 ev = {e[h][t], e[h][t + 1]};
            const bf16x2 hv = __builtin_convertvector(ev, bf16x2);
            ahi[h][t] = hv[0];
            ahi[h][t + 1] = hv[1];
            if (MODE == kModeBf16x3) {
              const uint32_t bits = __builtin_bit_cast(uint32_t, hv);
              const f32x2 rv = {ev[0] - __uint_as_float(bits << 16), ev[1] - __uint_as_float(bits & 0xffff0000u)};
              const bf16x2 lv = __builtin_convertvector(rv, bf16x2);
              alo[h][t] = lv[0];
              alo[h][t + 1] = lv[1];
            }
          }
        // one product per accumulator before the next part: a product waits for
        // the last one on its accumulator
        bf16x8 bhi[CB], blo[CB];
#pragma unroll
        for (int c = 0; c < CB; ++c) {
          bhi[c] = *reinterpret_cast<const bf16x8*>(ops + c * step_bytes(MODE));
          if (MODE == kModeBf16x3) blo[c] = *reinterpret_cast<const bf16x8*>(ops + kPart + c * step_bytes(MODE));
        }
        auto contract = [&](const bf16x8(&av)[2], const bf16x8(&bv)[CB]) {
#pragma unroll
          for (int c = 0; c < CB; ++c)
#pragma unroll
            for (int h = 0; h < 2; ++h)
              acc[h][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[h], bv[c], acc[h][c], 0, 0, 0);
        };
        contract(ahi, bhi);
        if (MODE == kModeBf16x3) {
          contract(ahi, blo);
          contract(alo, bhi);
        }
      }
    }
  }
  // ---- slab partials, in FP32 as accumulated.  32x32 accumulator layout:
  // lane l holds column l%32 and rows 8*(v/4) + 4*(l/32) + v%4, v = 0..15, so
  // four consecutive rows per quarter of the accumulator.
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int c = 0; c < CB; ++c) {
      const int64_t r = c * 32 + (lane % 32);
      if (r >= R) continue;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t i = base + h * 32 + 8 * u + 4 * (lane / 32);
        float* out = part + ((int64_t)blockIdx.y * R + r) * rows + i;
        if (i + 4 <= rows) {
          const f32x4u q = {acc[h][c][4 * u], acc[h][c][4 * u + 1], acc[h][c][4 * u + 2], acc[h][c][4 * u + 3]};
          *reinterpret_cast<f32x4u*>(out) = q;
        } else {
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (i + v < rows) out[v] = acc[h][c][4 * u + v];
        }
      }
    }
}

// ---------------------------------------------------------------------------
// FP64 matrix-core kernel (MPLAK_PREC_F64, kMfma64MinR columns or more, dim <= 4).
//
// A wave owns 32 targets (two 16-row blocks) and all columns of a group of up
// to 64.  For every step of 4 sources a lane evaluates one entry per row block
// in FP64 (coordinate differences and the table exponential, as on the vector
// unit), directly in the A layout of v_mfma_f64_16x16x4_f64, and the matrix
// cores contract it with the step's V operands from LDS.  Each entry is
// evaluated once whatever R (the vector-unit form evaluates it once per 16
// columns and reads every V value of the tile from LDS per source).  The FP64
// matrix rate equals the vector FMA rate on gfx950 and the two do not overlap
// (per 16 columns 224 us at n = 20001, 3-D Gaussian, of which 163 us are the
// products at 78.6 TFLOP/s, on top of 270 us for the entries), so the gain is
// the entries and LDS reads saved.
//
// Sums: 256 sources in the matrix cores' accumulators, then added to the slab's
// sum, as the vector-unit form sums them.  One chain over a slab of thousands
// of sources loses accuracy with its root (relative error, 2-norm, n = 20001:
// 1.7e-15 against 5.9e-16; n = 50000: 3.1e-15 against 6.8e-16).  The second set
// of accumulators leaves two waves per SIMD at 64 columns (n = 20001 1166 us;
// one chain, three waves 1136 us; Matern 1264 and 1261 us) and three at 32 (683 and
// 674 us at four).  At 48 three waves fit with the wave's index in a scalar register,
// so that the staging addresses are scalar too (920 us; two waves 952 us, one
// chain 882 us); at 64 and 32 columns that form is slower (1204 and 703 us).
//
// Row 4 v + r of A takes target 4 r + v of the block, so result v of lane
// 16 r + c is target 4 r + v, column c, and a lane's four results are
// consecutive rows of the partials.

constexpr int kSrc64 = 64;                                 // sources per LDS chunk
constexpr int kTile64 = 32 * (kBlock / kWave);             // 128 targets per workgroup
constexpr int kSteps64 = kSrc64 / 4;
constexpr int kSumChunks64 = 256 / kSrc64;                 // LDS chunks of one inner sum
// resident waves per SIMD (and workgroups per CU) by column blocks: above
constexpr int waves64(int cblocks) { return cblocks == 1 ? 4 : (cblocks <= 3 ? 3 : 2); }

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2u __attribute__((ext_vector_type(2), aligned(8)));

template <int KIND, int DIM, int CB>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(waves64(CB), waves64(CB)))) void mrhs_mfma64_kernel(
    const double* const* __restrict__ points, int64_t row_off, int64_t rows, int64_t col_off, int64_t cols,
    int64_t slab_cols, double scale, int64_t R, const double* __restrict__ V, int64_t ldv, double* __restrict__ part,
    const int32_t* __restrict__ skip) {
  if (skip != nullptr && *skip != 0) return;
  // V operands of a step: CB blocks of 64 lanes (source k = lane / 16, column
  // lane % 16); two doubles of padding spread the staging writes over the banks
  constexpr int kStep = CB * kWave + 2;
  __shared__ double lv[kSteps64 * kStep];
  __shared__ double lp[DIM][kSrc64];
  __shared__ double tab[kExp2Table];
  fill_exp2_table(tab);  // first read after the chunk barrier below
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int w = CB == 3 ? __builtin_amdgcn_readfirstlane(tid / kWave) : tid / kWave;
  const int c16 = lane & 15, r4 = lane >> 4;
  const int64_t base = (int64_t)blockIdx.x * kTile64 + w * 32;

  double p[2][DIM];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    int64_t i = base + 16 * h + 4 * (c16 & 3) + (c16 >> 2);
    if (i >= rows) i = rows - 1;
#pragma unroll
    for (int d = 0; d < DIM; ++d) p[h][d] = points[d][row_off + i] * scale;
  }
  f64x4 acc[2][CB], total[2][CB];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int c = 0; c < CB; ++c) acc[h][c] = total[h][c] = f64x4{0.0, 0.0, 0.0, 0.0};

  const int64_t c0 = (int64_t)blockIdx.y * slab_cols;
  const int64_t c1 = c0 + slab_cols < cols ? c0 + slab_cols : cols;
  int left = kSumChunks64;  // chunks until the inner sum is added to the total
  for (int64_t cb = c0; cb < c1; cb += kSrc64) {
    // lane = source, wave w takes columns w, w + 4, ...: all loads before the
    // barrier, sources and columns past the end are zero
    const int64_t j = cb + lane;
    double v[CB * 4], q = 0.0;
#pragma unroll
    for (int u = 0; u < CB * 4; ++u) {
      const int col = 4 * u + w;
      v[u] = j < c1 && col < R ? V[col * ldv + j] : 0.0;
    }
    if (w < DIM && j < c1) q = points[w][col_off + j] * scale;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < CB * 4; ++u) {
      const int col = 4 * u + w;
      lv[(lane / 4) * kStep + (col / 16) * kWave + (lane % 4) * 16 + col % 16] = v[u];
    }
    if (w < DIM) lp[w][lane] = q;
    __syncthreads();
#pragma unroll 2
    for (int st = 0; st < kSteps64; ++st) {
      double e[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        double s = 0.0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
          const double df = p[h][d] - lp[d][4 * st + r4];
          s = d == 0 ? df * df : fma(df, df, s);
        }
        e[h] = kernel_entry<double, KIND>(s, tab);
      }
#pragma unroll
      for (int c = 0; c < CB; ++c) {
        const double b = lv[st * kStep + c * kWave + lane];
#pragma unroll
        for (int h = 0; h < 2; ++h) acc[h][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(e[h], b, acc[h][c], 0, 0, 0);
      }
    }
    if (--left == 0 || cb + kSrc64 >= c1) {
      left = kSumChunks64;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int c = 0; c < CB; ++c) {
          total[h][c] += acc[h][c];
          acc[h][c] = f64x4{0.0, 0.0, 0.0, 0.0};
        }
    }
  }
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int c = 0; c < CB; ++c) {
      const int64_t r = 16 * c + c16;
      if (r >= R) continue;
      const int64_t i = base + 16 * h + 4 * r4;
      double* out = part + ((int64_t)blockIdx.y * R + r) * rows + i;
      const f64x4 sum = total[h][c];
      const f64x2u lo = {sum[0], sum[1]}, hi = {sum[2], sum[3]};
      if (i + 4 <= rows) {
        *reinterpret_cast<f64x2u*>(out) = lo;
        *reinterpret_cast<f64x2u*>(out + 2) = hi;
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (i + v < rows) out[v] = sum[v];
      }
    }
}

// Y[i + r ldy] = sum over slabs (slab order) + nugget * V at the global
// diagonal.  One row per thread, grid = (row blocks, columns); bound by the
// partials' bandwidth, so kFinishBatch of them are in flight per thread.  FP32
// accumulators leave FP32 partials: the same values as widened ones at half
// the bytes.
constexpr int kFinishBatch = 8;

template <typename PT>
__global__ __launch_bounds__(kBlock) void mrhs_finish_kernel(int64_t rows, int64_t R, int64_t slabs,
                                                             const PT* __restrict__ part, int64_t row_off,
                                                             int64_t col_off, int64_t cols, double nugget,
                                                             const double* __restrict__ V, int64_t ldv,
                                                             double* __restrict__ Y, int64_t ldy,
                                                             const int32_t* __restrict__ skip) {
  if (skip != nullptr && *skip != 0) return;
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= rows) return;
  for (int64_t r = blockIdx.y; r < R; r += gridDim.y) {
    const PT* p = part + r * rows + i;
    double s = (double)p[0];
    for (int64_t k = 1; k < slabs; k += kFinishBatch) {
      PT v[kFinishBatch];
#pragma unroll
      for (int u = 0; u < kFinishBatch; ++u) v[u] = k + u < slabs ? p[(k + u) * R * rows] : PT(0);
#pragma unroll
      for (int u = 0; u < kFinishBatch; ++u)
        if (k + u < slabs) s += (double)v[u];
    }
    const int64_t jd = row_off + i - col_off;
    if (nugget != 0.0 && jd >= 0 && jd < cols) s = fma(nugget, V[r * ldv + jd], s);
    Y[r * ldy + i] = s;
  }
}

// The same where few targets have many slabs, the sum of a row being a chain of
// latencies: 2^shift rows per workgroup, whose other threads are slices k of the
// slabs (k, k + slices, ...); the slices' sums are added in a tree.
template <typename PT>
__global__ __launch_bounds__(kBlock) void mrhs_finish_sliced_kernel(int64_t rows, int64_t R, int64_t slabs, int shift,
                                                                    const PT* __restrict__ part, int64_t row_off,
                                                                    int64_t col_off, int64_t cols, double nugget,
                                                                    const double* __restrict__ V, int64_t ldv,
                                                                    double* __restrict__ Y, int64_t ldy,
                                                                    const int32_t* __restrict__ skip) {
  if (skip != nullptr && *skip != 0) return;
  __shared__ double red[kBlock];
  const int tid = threadIdx.x, slices = kBlock >> shift, slice = tid >> shift;
  const int64_t i = ((int64_t)blockIdx.x << shift) + (tid & ((1 << shift) - 1));
  for (int64_t r = blockIdx.y; r < R; r += gridDim.y) {
    double s = 0.0;
    if (i < rows) {
      const PT* p = part + r * rows + i;
      for (int64_t k = slice; k < slabs; k += kFinishBatch * slices) {
        PT v[kFinishBatch];
#pragma unroll
        for (int u = 0; u < kFinishBatch; ++u) {
          const int64_t q = k + u * slices;
          v[u] = q < slabs ? p[q * R * rows] : PT(0);
        }
#pragma unroll
        for (int u = 0; u < kFinishBatch; ++u)
          if (k + u * slices < slabs) s += (double)v[u];
      }
    }
    red[tid] = s;
    __syncthreads();
    for (int h = kBlock / 2; h >= (1 << shift); h >>= 1) {
      if (tid < h) red[tid] += red[tid + h];
      __syncthreads();
    }
    if (slice == 0 && i < rows) {
      s = red[tid];
      const int64_t jd = row_off + i - col_off;
      if (nugget != 0.0 && jd >= 0 && jd < cols) s = fma(nugget, V[r * ldv + jd], s);
      Y[r * ldy + i] = s;
    }
    __syncthreads();
  }
}

// Rows of a finish workgroup, as a power of two: 256, halved while the launch has
// fewer than 1024 workgroups and a thread more than 32 slabs.  The whole product with one row a thread / so: BF16x3 in 3-D,
// 64 columns, 256 x 300000 421 / 166 us, 200 x 65536 104 / 49 us, 1000 x 20000 58 / 45
// us; FP64, 8 columns, 200 x 65536 51 / 38 us.  Two slices of 32 slabs lose
// (8000 points, FP32, 8 columns: 53 / 57 us).
inline int finish_shift(int64_t rows, int64_t R, int64_t slabs) {
  int shift = 8;
  while (shift > 0 && ((rows + (int64_t(1) << shift) - 1) >> shift) * R < 1024 && slabs > int64_t(32) << (8 - shift)) --shift;
  return shift;
}

template <typename PT>
void launch_finish(const mplak_kernel_desc* d, hipStream_t st, int64_t R, int64_t slabs, const PT* part,
                   const double* V, int64_t ldv, double* Y, int64_t ldy, const int32_t* skip) {
  const int shift = finish_shift(d->row_count, R, slabs);
  const dim3 grid((unsigned)((d->row_count + (int64_t(1) << shift) - 1) >> shift), (unsigned)std::min<int64_t>(R, 65535));
  if (shift == 8)
    hipLaunchKernelGGL(mrhs_finish_kernel<PT>, grid, dim3(kBlock), 0, st, d->row_count, R, slabs, part, d->row_offset,
                       d->col_offset, d->col_count, d->nugget, V, ldv, Y, ldy, skip);
  else
    hipLaunchKernelGGL(mrhs_finish_sliced_kernel<PT>, grid, dim3(kBlock), 0, st, d->row_count, R, slabs, shift, part,
                       d->row_offset, d->col_offset, d->col_count, d->nugget, V, ldv, Y, ldy, skip);
}

// ---------------------------------------------------------------------------
// host-side planning and dispatch

// Fewest columns of the FP64 matrix-core kernel.  Its products are 16 columns
// wide, so up to 8 columns the vector unit's narrower tiles do less work
// (n = 20001, 3-D Gaussian, R = 8: 402 us against 488 us); from 9 the vector
// unit works on 16 as well (R = 12: 611 us against 493 us, R = 64: 2443 us
// against 1169 us; Matern R = 64: 3141 us against 1438 us).
constexpr int64_t kMfma64MinR = 9;

struct MrhsPlan {
  bool mfma;
  int mode;       // MfmaMode when mfma
  bool mfma64;    // FP64 matrix-core kernel
  int rt;         // VALU column tile
  int64_t cblocks;
  Slabs s;
  size_t vpk_bytes, part_bytes;
  int64_t blocks;  // packed source blocks
};

inline int valu_rt(int64_t R) {
  if (R <= 1) return 1;
  if (R <= 2) return 2;
  if (R <= 4) return 4;
  if (R <= 8) return 8;
  return 16;
}

// The kernel of a product, without its slabs.
inline MrhsPlan make_kernel(const mplak_kernel_desc* d, int precision, int64_t R) {
  MrhsPlan p{};
  p.mfma64 = precision == MPLAK_PREC_F64 && R >= kMfma64MinR && d->dim <= 4;
  p.mfma = (precision == MPLAK_PREC_BF16 || precision == MPLAK_PREC_BF16X3 ||
            (precision == MPLAK_PREC_F32 && R >= 16)) && d->dim <= 4;
  return p;
}

inline MrhsPlan make_plan(const mplak_kernel_desc* d, int precision, int64_t R) {
  MrhsPlan p = make_kernel(d, precision, R);
  if (p.mfma64) {
    p.cblocks = (R + 15) / 16;
    p.s = balanced_slabs(d->row_count, d->col_count, kTile64, kSrc64, waves64((int)std::min<int64_t>(p.cblocks, 4)), R);
    p.part_bytes = align_up((size_t)p.s.slabs * (size_t)R * (size_t)d->row_count * sizeof(double), 256);
    return p;
  }
  if (p.mfma) {
    p.mode = precision == MPLAK_PREC_BF16 ? kModeBf16 : (precision == MPLAK_PREC_BF16X3 ? kModeBf16x3 : kModeF32);
    p.cblocks = (R + 31) / 32;
    p.s = balanced_slabs(d->row_count, d->col_count, kMfmaTile, kMfmaSlab, mfma_waves((int)p.cblocks), R, 1, 1.0,
                         kMfmaDrain, longest_fp32_slab(d->row_count, d->col_count));
    p.blocks = (d->col_count + kMfmaSlab - 1) / kMfmaSlab;
    p.vpk_bytes = align_up((size_t)p.blocks * (size_t)block_bytes(p.mode, (int)p.cblocks) + kPackAlign, 256);
  } else {
    p.rt = valu_rt(R);
    const int64_t ctiles = (R + p.rt - 1) / p.rt;
    // a 32-source unit of the double form takes about the chunk's 8 us; a third of
    // that in FP32, three times as long past 3 dimensions (the runtime-dim loop)
    const double weight = d->dim > 3 ? 0.3 : (precision == MPLAK_PREC_F64 ? 1.0 : 3.0);
    p.s = balanced_slabs(d->row_count, d->col_count, kBlock, kValuUnit, 4, R, ctiles, weight);
    p.vpk_bytes = 0;
  }
  p.part_bytes = align_up((size_t)p.s.slabs * (size_t)R * (size_t)d->row_count * (p.mfma ? sizeof(float) : sizeof(double)),
                          256);
  return p;
}

// Columns per launch: the matrix-core kernels hold at most kMfmaGroup.
inline int64_t column_group(const mplak_kernel_desc* d, int precision, int64_t nrhs) {
  const MrhsPlan p = make_kernel(d, precision, nrhs);
  return p.mfma || p.mfma64 ? kMfmaGroup : nrhs;
}

template <typename T, int KIND, int DIM>
void launch_valu_rt(int rt, dim3 grid, hipStream_t st, const mplak_kernel_desc* d, const MrhsPlan& p, double scale,
                    int64_t R, const double* V, int64_t ldv, double* part, const int32_t* skip) {
#define MPLAK_VALU_CASE(RTV)                                                                                \
  case RTV:                                                                                                 \
    hipLaunchKernelGGL((mrhs_valu_kernel<T, KIND, DIM, RTV>), grid, dim3(kBlock), 0, st, d->points, d->dim, \
                       d->row_offset, d->row_count, d->col_offset, d->col_count, p.s.slab_cols, scale, R, V, \
                       ldv, part, skip);                                                                    \
    break;
  switch (rt) {
    MPLAK_VALU_CASE(1)
    MPLAK_VALU_CASE(2)
    MPLAK_VALU_CASE(4)
    MPLAK_VALU_CASE(8)
    default:
      MPLAK_VALU_CASE(16)
  }
#undef MPLAK_VALU_CASE
}

template <typename T, int KIND>
void launch_valu(const mplak_kernel_desc* d, const MrhsPlan& p, hipStream_t st, double scale, int64_t R,
                 const double* V, int64_t ldv, double* part, const int32_t* skip) {
  const dim3 grid((unsigned)p.s.tiles, (unsigned)p.s.slabs, (unsigned)((R + p.rt - 1) / p.rt));
  switch (d->dim) {
    case 1: launch_valu_rt<T, KIND, 1>(p.rt, grid, st, d, p, scale, R, V, ldv, part, skip); break;
    case 2: launch_valu_rt<T, KIND, 2>(p.rt, grid, st, d, p, scale, R, V, ldv, part, skip); break;
    case 3: launch_valu_rt<T, KIND, 3>(p.rt, grid, st, d, p, scale, R, V, ldv, part, skip); break;
    default: launch_valu_rt<T, KIND, 0>(p.rt, grid, st, d, p, scale, R, V, ldv, part, skip); break;
  }
}

template <int KIND, int MODE>
void launch_mfma_mode(const mplak_kernel_desc* d, const MrhsPlan& p, hipStream_t st, double scale, int64_t R,
                      const char* packed, float* part, const int32_t* skip) {
  const dim3 grid((unsigned)p.s.tiles, (unsigned)p.s.slabs);
  auto go = [&](auto cb_tag, auto dim_tag) {
    constexpr int CBV = decltype(cb_tag)::value, DIMV = decltype(dim_tag)::value;
    hipLaunchKernelGGL((mrhs_mfma_kernel<KIND, MODE, CBV, DIMV>), grid, dim3(kBlock), 0, st, d->points, d->row_offset,
                       d->row_count, p.blocks, p.s.slab_cols / kMfmaSlab, scale, R, packed, part, skip);
  };
  auto with_dim = [&](auto cb_tag) {
    switch (d->dim) {
      case 1: go(cb_tag, std::integral_constant<int, 1>{}); break;
      case 2: go(cb_tag, std::integral_constant<int, 2>{}); break;
      case 3: go(cb_tag, std::integral_constant<int, 3>{}); break;
      default: go(cb_tag, std::integral_constant<int, 4>{}); break;
    }
  };
  if (p.cblocks == 1)
    with_dim(std::integral_constant<int, 1>{});
  else
    with_dim(std::integral_constant<int, 2>{});
}

template <int KIND>
void launch_mfma64(const mplak_kernel_desc* d, const MrhsPlan& p, hipStream_t st, double scale, int64_t R,
                   const double* V, int64_t ldv, double* part, const int32_t* skip) {
  const dim3 grid((unsigned)p.s.tiles, (unsigned)p.s.slabs);
  auto go = [&](auto cb_tag, auto dim_tag) {
    constexpr int CBV = decltype(cb_tag)::value, DIMV = decltype(dim_tag)::value;
    hipLaunchKernelGGL((mrhs_mfma64_kernel<KIND, DIMV, CBV>), grid, dim3(kBlock), 0, st, d->points, d->row_offset,
                       d->row_count, d->col_offset, d->col_count, p.s.slab_cols, scale, R, V, ldv, part, skip);
  };
  auto with_dim = [&](auto cb_tag) {
    switch (d->dim) {
      case 1: go(cb_tag, std::integral_constant<int, 1>{}); break;
      case 2: go(cb_tag, std::integral_constant<int, 2>{}); break;
      case 3: go(cb_tag, std::integral_constant<int, 3>{}); break;
      default: go(cb_tag, std::integral_constant<int, 4>{}); break;
    }
  };
  switch (p.cblocks) {
    case 1: with_dim(std::integral_constant<int, 1>{}); break;
    case 2: with_dim(std::integral_constant<int, 2>{}); break;
    case 3: with_dim(std::integral_constant<int, 3>{}); break;
    default: with_dim(std::integral_constant<int, 4>{}); break;
  }
}

template <int KIND>
void launch_mfma(const mplak_kernel_desc* d, const MrhsPlan& p, hipStream_t st, double scale, int64_t R,
                 const char* packed, float* part, const int32_t* skip) {
  if (p.mode == kModeBf16)
    launch_mfma_mode<KIND, kModeBf16>(d, p, st, scale, R, packed, part, skip);
  else if (p.mode == kModeBf16x3)
    launch_mfma_mode<KIND, kModeBf16x3>(d, p, st, scale, R, packed, part, skip);
  else
    launch_mfma_mode<KIND, kModeF32>(d, p, st, scale, R, packed, part, skip);
}

int check_desc(const mplak_kernel_desc* d) {
  if (d == nullptr || d->points == nullptr) return MPLAK_ERR_ARG;
  if (d->dim < 1 || d->dim > kMaxDim) return MPLAK_ERR_ARG;
  if (d->kind != MPLAK_KERNEL_GAUSSIAN && d->kind != MPLAK_KERNEL_MATERN32) return MPLAK_ERR_ARG;
  if (!(d->length_scale > 0.0)) return MPLAK_ERR_ARG;
  if (d->row_count < 0 || d->col_count < 0 || d->row_offset < 0 || d->col_offset < 0) return MPLAK_ERR_ARG;
  return MPLAK_OK;
}

}  // namespace
}  // namespace mplak

using namespace mplak;

extern "C" {

size_t mplak_kernel_mrhs_workspace_bytes(const mplak_kernel_desc* d, int precision, int64_t nrhs) {
  if (check_desc(d) != MPLAK_OK || nrhs <= 0 || d->row_count <= 0 || d->col_count <= 0) return 0;
  // the MFMA paths work on groups of at most kMfmaGroup columns; a narrow
  // last group may take another kernel (and slab count) than the full ones
  const int64_t group = column_group(d, precision, nrhs);
  const MrhsPlan p = make_plan(d, precision, std::min(nrhs, group));
  size_t bytes = p.vpk_bytes + p.part_bytes;
  if (nrhs > group && nrhs % group != 0) {
    const MrhsPlan q = make_plan(d, precision, nrhs % group);
    bytes = std::max(bytes, q.vpk_bytes + q.part_bytes);
  }
  return bytes;
}

int mplak_kernel_mrhs(const mplak_kernel_desc* d, int precision, int64_t nrhs, const double* V, int64_t ldv,
                      double* Y, int64_t ldy, void* work, size_t work_bytes, const int32_t* skip_if,
                      mplak_stream_t s) {
  int st = check_desc(d);
  if (st != MPLAK_OK) return st;
  if (precision < MPLAK_PREC_F64 || precision > MPLAK_PREC_BF16X3) return MPLAK_ERR_ARG;
  if (nrhs < 0) return MPLAK_ERR_ARG;
  if (nrhs == 0 || d->row_count == 0) return MPLAK_OK;
  if (Y == nullptr || ldy < d->row_count) return MPLAK_ERR_ARG;
  if (d->col_count == 0) {
    for (int64_t r = 0; r < nrhs; ++r) {
      st = mplak_fill_f64(Y + r * ldy, d->row_count, 0.0, s);
      if (st != MPLAK_OK) return st;
    }
    return MPLAK_OK;
  }
  if (V == nullptr || ldv < d->col_count) return MPLAK_ERR_ARG;
  if (work == nullptr || work_bytes < mplak_kernel_mrhs_workspace_bytes(d, precision, nrhs)) return MPLAK_ERR_WORKSPACE;
  hipStream_t hs = as_stream(s);
  const double scale = coord_scale(d->kind, d->length_scale);
  const int64_t group = column_group(d, precision, nrhs);
  for (int64_t r0 = 0; r0 < nrhs; r0 += group) {
    const int64_t R = std::min(group, nrhs - r0);
    const MrhsPlan p = make_plan(d, precision, R);
    const double* Vg = V + r0 * ldv;
    double* Yg = Y + r0 * ldy;
    char* w = static_cast<char*>(work);
    char* packed = reinterpret_cast<char*>(align_up(reinterpret_cast<uintptr_t>(w), kPackAlign));
    double* part = reinterpret_cast<double*>(w + p.vpk_bytes);
    float* part32 = reinterpret_cast<float*>(part);
    if (p.mfma) {
      hipLaunchKernelGGL(pack_kernel, dim3((unsigned)std::min<int64_t>(p.blocks, 8192)), dim3(kBlock), 0, hs, d->points,
                         d->dim, d->col_offset, scale, Vg, ldv, R, d->col_count, p.blocks, (int)p.cblocks, p.mode, packed);
      st = launch_status();
      if (st != MPLAK_OK) return st;
      if (d->kind == MPLAK_KERNEL_GAUSSIAN)
        launch_mfma<MPLAK_KERNEL_GAUSSIAN>(d, p, hs, scale, R, packed, part32, skip_if);
      else
        launch_mfma<MPLAK_KERNEL_MATERN32>(d, p, hs, scale, R, packed, part32, skip_if);
    } else if (p.mfma64) {
      if (d->kind == MPLAK_KERNEL_GAUSSIAN)
        launch_mfma64<MPLAK_KERNEL_GAUSSIAN>(d, p, hs, scale, R, Vg, ldv, part, skip_if);
      else
        launch_mfma64<MPLAK_KERNEL_MATERN32>(d, p, hs, scale, R, Vg, ldv, part, skip_if);
    } else {
      if (precision == MPLAK_PREC_F64) {
        if (d->kind == MPLAK_KERNEL_GAUSSIAN)
          launch_valu<double, MPLAK_KERNEL_GAUSSIAN>(d, p, hs, scale, R, Vg, ldv, part, skip_if);
        else
          launch_valu<double, MPLAK_KERNEL_MATERN32>(d, p, hs, scale, R, Vg, ldv, part, skip_if);
      } else {
        if (d->kind == MPLAK_KERNEL_GAUSSIAN)
          launch_valu<float, MPLAK_KERNEL_GAUSSIAN>(d, p, hs, scale, R, Vg, ldv, part, skip_if);
        else
          launch_valu<float, MPLAK_KERNEL_MATERN32>(d, p, hs, scale, R, Vg, ldv, part, skip_if);
      }
    }
    st = launch_status();
    if (st != MPLAK_OK) return st;
    if (p.mfma)
      launch_finish(d, hs, R, p.s.slabs, part32, Vg, ldv, Yg, ldy, skip_if);
    else
      launch_finish(d, hs, R, p.s.slabs, part, Vg, ldv, Yg, ldy, skip_if);
    st = launch_status();
    if (st != MPLAK_OK) return st;
  }
  return MPLAK_OK;
}

}  // extern "C"
