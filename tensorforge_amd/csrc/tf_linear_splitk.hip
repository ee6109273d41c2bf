// Decode-shaped linear layers on MFMA for up to 64 rows.  This file holds
//   * tf_linear_partials / tf_linear_partials_sum -- split-K slices with
//     operands loaded in the MFMA operand layout (below);
//   * tf_linear_stream -- the same products (or a one-slice rounded output)
//     with both operands staged through LDS by whole-row loads;
//   * tf_linear_swiglu -- its form for the stacked gate|up weight with the
//     SwiGLU in the epilogue;
//   * tf_linear_kstream / tf_linear_kswiglu -- K split over a workgroup's
//     wavefronts, each on its own ring of direct-to-LDS loads, for the
//     projections of a decode step.
//
// Split-K form:
//   partials[s][m][n] = sum over k in slice s of x[m][k] * w[n][k]   (fp32)
// and the row sum y[m][n] = round(sum_s partials[s][m][n]).
//
// At decode batch sizes a projection streams its weight matrix once (each
// element is used M <= 64 times) and is HBM-bound; what a library GEMM
// tiled for large M lacks is parallelism -- a 2048 x 2048 weight in 64 x 64
// output tiles is 32 workgroups.  Here blockIdx.x is a 64-column tile and
// blockIdx.y one of S slices of K, so a launch has (N / 64) * S workgroups
// each streaming a 64-row slab of w that is K / S long.  Inside a workgroup
// the four wavefronts split the slice's 32-wide k-steps between them and
// each accumulates the whole 64 x 64 tile (4 row tiles x 4 column tiles of
// v_mfma_f32_16x16x32), so a wavefront reads as many bytes of x as of w (x
// is small and stays in L2; a 16-column tiling would read x four times as
// often as w).  Up to four k-steps of loads (w and x) are issued together.
// The four wavefront tiles are summed once in LDS and stored as the
// slice's fp32 partial; the reduction over the S slices is left to the
// consumer of y (tf_linear_partials_sum here, or a fused consumer), so the
// launch needs no atomics, counters or second pass of its own.
//
// MFMA v_mfma_f32_16x16x32 (bf16 / f16):
//   A = x rows:  lane (l16, q4) holds x[16 mt + l16][k + 8 q4 .. +8]
//   B = w rows:  lane (l16, q4) holds w[n0 + 16 nt + l16][k + 8 q4 .. +8]
//   C:           lane (l16, q4), register r holds y[16 mt + 4 q4 + r][n0 + 16 nt + l16]
//
// Reference semantics: torch.nn.functional.linear(x, w) without bias (fp32
// accumulation, one rounding to the storage type), the nn.Linear
// projections of tensorforge/model/layers.py:88-95, 144-146 as the decode
// step calls them (tensorforge/runtime/decode_bucket.py:441-447, 470,
// 500-505).
#include "tf_common.hpp"

#include <atomic>
#include <type_traits>

namespace tf {
namespace {

template <typename T>
struct SplitMma;

template <>
struct SplitMma<__bf16> {
  typedef __bf16 vec8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ f32x4 mma(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};

template <>
struct SplitMma<_Float16> {
  typedef _Float16 vec8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ f32x4 mma(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

constexpr int kSplitWaves = 4;    // wavefronts per workgroup
constexpr int kSplitCols = 64;    // output columns per workgroup
constexpr int kSplitUnroll = 4;   // k-steps of loads in flight per wavefront

template <typename T, int MT>
__global__ void __launch_bounds__(kSplitWaves * 64)
linear_partials_kernel(const T *__restrict__ x, int64_t x_stride, const T *__restrict__ w,
                       int64_t w_stride, float *__restrict__ partials, int32_t m, int32_t n,
                       int32_t k, int32_t k_per_split) {
  using M = SplitMma<T>;
  using vec8 = typename M::vec8;
  constexpr int NT = kSplitCols / 16;
  constexpr int kItems = MT * NT * 4 * 64;  // floats of one wavefront's tile
  extern __shared__ __attribute__((aligned(16))) float tile_sums[];  // [waves][kItems]
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15;
  const int q4 = lane >> 4;
  const int32_t n0 = blockIdx.x * kSplitCols;
  const int32_t split = blockIdx.y;
  const int32_t s0 = split * k_per_split;
  const int32_t s1 = min(s0 + k_per_split, k);
  // k-steps of the slice, dealt to the wavefronts in contiguous runs.
  const int32_t steps = (s1 - s0) / 32;
  const int32_t per_wave = (steps + kSplitWaves - 1) / kSplitWaves;
  const int32_t k0 = s0 + 32 * min(wave * per_wave, steps);
  const int32_t k1 = s0 + 32 * min((wave + 1) * per_wave, steps);

  const T *wrow[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
    wrow[nt] = w + static_cast<int64_t>(min(n0 + 16 * nt + l16, n - 1)) * w_stride + 8 * q4;
  const T *xrow[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    xrow[mt] = x + static_cast<int64_t>(min(16 * mt + l16, m - 1)) * x_stride + 8 * q4;

  f32x4 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Batches of kSplitUnroll k-steps: every load of a batch is issued before
  // its MFMAs; steps past k1 load the batch's first step again and are
  // zeroed, so the loads stay unconditional.
  for (int32_t kk = k0; kk < k1; kk += 32 * kSplitUnroll) {
    vec8 wb[kSplitUnroll][NT];
    vec8 xa[kSplitUnroll][MT];
#pragma unroll
    for (int u = 0; u < kSplitUnroll; ++u) {
      const int32_t ku = kk + 32 * u < k1 ? kk + 32 * u : kk;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) wb[u][nt] = *reinterpret_cast<const vec8 *>(wrow[nt] + ku);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) xa[u][mt] = *reinterpret_cast<const vec8 *>(xrow[mt] + ku);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kSplitUnroll; ++u) {
      if (kk + 32 * u >= k1) break;  // uniform
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = M::mma(xa[u][mt], wb[u][nt], acc[mt][nt]);
    }
  }

  // Sum the wavefront tiles: item (mt, nt, r, lane).
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        tile_sums[wave * kItems + ((mt * NT + nt) * 4 + r) * 64 + lane] = acc[mt][nt][r];
  __syncthreads();
  float *out = partials + static_cast<int64_t>(split) * m * n;
  for (int item = threadIdx.x; item < kItems; item += blockDim.x) {
    float sum = 0.f;
#pragma unroll
    for (int wv = 0; wv < kSplitWaves; ++wv) sum += tile_sums[wv * kItems + item];
    const int il = item & 63;
    const int r = (item >> 6) & 3;
    const int tile = item >> 8;
    const int mt = tile / NT;
    const int nt = tile - mt * NT;
    const int32_t row = 16 * mt + 4 * (il >> 4) + r;
    const int32_t col = n0 + 16 * nt + (il & 15);
    if (row < m && col < n) out[static_cast<int64_t>(row) * n + col] = sum;
  }
}

// ---------------------------------------------------------------------------
// Weight-streaming form (tf_linear_stream).  A load in the MFMA operand
// layout (lane (l16, q4) reading 16 bytes of row l16) touches 16 rows x half
// a 128-byte line, and a compute unit issues such loads at <= 34 GB/s even
// when they hit L2; whole-row loads run at ~85 GB/s from L2 and stream HBM
// ~10% faster.  Here a workgroup stages 256-wide k chunks of x (16 MT rows)
// and of its 64 weight rows in LDS with whole-row loads (32 threads per
// 512-byte row piece), with the next two chunks' loads in flight in
// registers while the MFMAs read the current one, and each wavefront owns
// 16 output columns over the whole slice -- no cross-wavefront sum.  LDS
// rows are 512 bytes with their 16-byte pieces permuted by
// (piece ^ (row & 15)), so the 16 rows an operand read touches at one k
// fall in distinct banks.
// ---------------------------------------------------------------------------
constexpr int kStreamCols = 64;    // output columns per workgroup (4 wavefronts x 16)
constexpr int kStreamChunk = 256;  // k per LDS chunk (one 512-byte row)

__device__ __forceinline__ int stream_lds_offset(int row, int piece) {
  return row * kStreamChunk + ((piece ^ (row & 15)) << 3);
}

// SWIGLU: the weight stacks gate rows [0, n) over up rows [n, 2n) and the
// workgroup covers 32 output columns j: wavefronts 0-1 compute the gate
// columns and 2-3 the matching up columns, which reach 0-1 through LDS; the
// output is round(swiglu_act(round(g), round(u))), the SwiGLU of the
// rounded projection.
template <typename T, int MT, bool SWIGLU>
__global__ void __launch_bounds__(256)
linear_stream_kernel(const T *__restrict__ x, int64_t x_stride, const T *__restrict__ w,
                     int64_t w_stride, T *__restrict__ y, int64_t y_stride,
                     float *__restrict__ partials, int32_t m, int32_t n, int32_t k,
                     int32_t k_per_split) {
  using M = SplitMma<T>;
  using vec8 = typename M::vec8;
  constexpr int XR = 16 * MT;
  constexpr int kLoadsX = XR / 8;           // 16-byte loads per thread per chunk
  constexpr int kLoadsW = kStreamCols / 8;
  extern __shared__ __attribute__((aligned(16))) unsigned char stream_smem[];
  T *xl = reinterpret_cast<T *>(stream_smem);  // [XR][256], swizzled pieces
  T *wl = xl + XR * kStreamChunk;              // [64][256]

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15;
  const int q4 = lane >> 4;
  const int32_t n0 = blockIdx.x * (SWIGLU ? kStreamCols / 2 : kStreamCols);
  const int32_t split = blockIdx.y;
  const int32_t s0 = split * k_per_split;
  const int32_t s1 = min(s0 + k_per_split, k);
  // Staging map: thread t loads piece t % 32 of row 8 i + t / 32.
  const int lrow = tid >> 5;
  const int lpiece = tid & 31;

  const T *xsrc[kLoadsX];
#pragma unroll
  for (int i = 0; i < kLoadsX; ++i)
    xsrc[i] = x + static_cast<int64_t>(min(8 * i + lrow, m - 1)) * x_stride + 8 * lpiece;
  const T *wsrc[kLoadsW];
#pragma unroll
  for (int i = 0; i < kLoadsW; ++i) {
    const int tr = 8 * i + lrow;  // tile row
    const int64_t row = SWIGLU ? (tr < 32 ? 0 : n) + min(n0 + (tr & 31), n - 1)
                               : min(n0 + tr, n - 1);
    wsrc[i] = w + row * w_stride + 8 * lpiece;
  }

  // Two register sets: while the MFMAs read chunk c from LDS, the loads of
  // chunks c + 1 and c + 2 are in flight (128 KB per workgroup at MT = 4).
  vec8 xa[kLoadsX], wa[kLoadsW], xb[kLoadsX], wb[kLoadsW];
  // Pieces past K (only in a last, partial chunk) read the row's first
  // piece instead; pieces past the slice but inside K are read and unused.
  auto load_chunk = [&](int32_t kk, vec8(&xr)[kLoadsX], vec8(&wr)[kLoadsW]) {
    const int32_t c = kk + 8 * lpiece < k ? kk : -8 * lpiece;
#pragma unroll
    for (int i = 0; i < kLoadsX; ++i) xr[i] = *reinterpret_cast<const vec8 *>(xsrc[i] + c);
#pragma unroll
    for (int i = 0; i < kLoadsW; ++i) wr[i] = *reinterpret_cast<const vec8 *>(wsrc[i] + c);
  };
  auto stage_chunk = [&](const vec8(&xr)[kLoadsX], const vec8(&wr)[kLoadsW]) {
    __syncthreads();  // the previous chunk's operand reads are done
#pragma unroll
    for (int i = 0; i < kLoadsX; ++i)
      *reinterpret_cast<vec8 *>(xl + stream_lds_offset(8 * i + lrow, lpiece)) = xr[i];
#pragma unroll
    for (int i = 0; i < kLoadsW; ++i)
      *reinterpret_cast<vec8 *>(wl + stream_lds_offset(8 * i + lrow, lpiece)) = wr[i];
    __syncthreads();
  };

  f32x4 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto compute_chunk = [&](int32_t kk) {
    const int32_t steps = min(kStreamChunk, s1 - kk) >> 5;
#pragma unroll
    for (int st = 0; st < kStreamChunk / 32; ++st) {
      if (st >= steps) break;  // uniform
      const int piece = 4 * st + q4;
      const vec8 b = *reinterpret_cast<const vec8 *>(wl + stream_lds_offset(16 * wave + l16, piece));
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        acc[mt] = M::mma(*reinterpret_cast<const vec8 *>(xl + stream_lds_offset(16 * mt + l16, piece)),
                         b, acc[mt]);
    }
  };

  constexpr int32_t C = kStreamChunk;
  load_chunk(s0, xa, wa);
  if (s0 + C < s1) load_chunk(s0 + C, xb, wb);
  for (int32_t kk = s0; kk < s1; kk += 2 * C) {
    stage_chunk(xa, wa);
    if (kk + 2 * C < s1) load_chunk(kk + 2 * C, xa, wa);
    compute_chunk(kk);
    if (kk + C >= s1) break;
    stage_chunk(xb, wb);
    if (kk + 3 * C < s1) load_chunk(kk + 3 * C, xb, wb);
    compute_chunk(kk + C);
  }

  // C layout: lane (l16, q4), register r holds y[16 mt + 4 q4 + r][n0 + 16 wave + l16].
  if constexpr (SWIGLU) {
    float *up = reinterpret_cast<float *>(stream_smem);  // [2 waves][MT * 4][64 lanes]
    __syncthreads();  // the last chunk's operand reads are done
    if (wave >= 2) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          up[((wave - 2) * MT * 4 + mt * 4 + r) * 64 + lane] = to_float(from_float<T>(acc[mt][r]));
    }
    __syncthreads();
    const int32_t col = n0 + 16 * wave + l16;
    if (wave >= 2 || col >= n) return;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int32_t row = 16 * mt + 4 * q4 + r;
        if (row >= m) continue;
        const float g = to_float(from_float<T>(acc[mt][r]));
        const float u = up[(wave * MT * 4 + mt * 4 + r) * 64 + lane];
        y[static_cast<int64_t>(row) * y_stride + col] = from_float<T>(swiglu_act(g, u));
      }
    return;
  }
  const int32_t col = n0 + 16 * wave + l16;
  if (col >= n) return;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int32_t row = 16 * mt + 4 * q4 + r;
      if (row >= m) continue;
      if (partials)
        partials[(static_cast<int64_t>(split) * m + row) * n + col] = acc[mt][r];
      else
        y[static_cast<int64_t>(row) * y_stride + col] = from_float<T>(acc[mt][r]);
    }
}

// ---------------------------------------------------------------------------
// K-split form of the weight stream (the projections of a decode step, the
// gate|up + SwiGLU launch included): a workgroup owns a BM x WR tile of
// products over all of K, and its four wavefronts take a quarter of K each.
// A wavefront keeps its own ring of STAGES 64-wide chunks (128-byte row
// pieces) of the tile's x and weight rows in LDS, filled by direct-to-LDS
// loads, and waits only for its own loads: no staging registers and no
// barrier before the four tiles meet once in LDS.
//
// What bounds it is the rate at which a compute unit takes lines it has not
// in its 32 KB L1: about 53 B/ns, from one chunk in flight per wavefront to
// nine and with the products left out, so the time of a weight of a few MB is
// 2.2 us plus (BM + WR) rows of K at that rate, per unit (qkv and o at 64
// rows: 7.1 and 5.9 us).  Larger ones add the memory's time: gate|up's 46 MB
// are 8.6 us at the copy rate.
// Against register-staged chunks of the same quarters (us, MI355X, bf16,
// weights cycled through 2 GB) at 64 / 33 / 17 / 4 rows:
//   qkv + norm (2560 x 2048)              8.1 / 6.9 / 6.8 / 5.6 -> 7.5 / 6.2 / 6.1 / 4.8
//   o + residual (2048 x 2048)            6.5 / 6.2 / 4.9 / 4.8 -> 6.0 / 5.7 / 4.4 / 4.3
//   gate|up + norm + SwiGLU (11264 x 2048) 15.8 / 14.6 / 12.5 / 11.4 -> 13.9 / 11.6 / 10.3 / 9.4
//   down + residual (2048 x 5632)         12.7 / 11.9 / 8.4 / 8.3 -> 12.0 / 9.9 / 7.7 / 7.3
//   4096 x 14336 + residual               38.5 / 33.0 / 25.7 / 21.9 -> 37.2 / 30.8 / 23.7 / 19.4
// ---------------------------------------------------------------------------
// Epilogues of the K-split kernel.
//   kEpiPlain     y = round(sum)
//   kEpiNorm      y = round(rsqrt(mean_k(x[r][k]^2) + eps) * sum): the
//                 RMSNorm of x's rows applied to the product, for a weight
//                 whose columns carry the norm's gain (w'[n][k] = w[n][k] g[k]);
//                 each workgroup sees all of K, so the row sums of squares
//                 come from the x operands it feeds the MFMAs anyway
//   kEpiResidual  y = round(round(sum) + residual[r][n]): the projection
//                 added to the residual stream, rounded as a separate add is
enum KstreamEpi : int { kEpiPlain = 0, kEpiNorm = 1, kEpiResidual = 2 };
struct KstreamParams {
  const void *x;
  const void *w;
  void *y;
  const void *residual;
  int64_t x_stride;
  int64_t w_stride;
  int64_t y_stride;
  int64_t residual_stride;
  float eps;
  int32_t m;
  int32_t n;           // output columns
  int32_t k;
  int32_t tiles_n;
  int32_t row_blocks;  // of BM rows
  int32_t stream;      // weights by nontemporal loads
};

constexpr int kKsWaves = 4;
constexpr int kKsChunk = 64;      // k per ring buffer
constexpr int kKsRowBytes = 128;  // bytes of a chunk row
constexpr int kKsXcds = 8;
constexpr int32_t kKsUnits = 256;  // compute units

// Chunks of a ring: what fits 80 KB (two workgroups per compute unit where
// the grid has that many), at least two.
constexpr int ks_stages(int rows) {
  const int fit = 80 * 1024 / (kKsWaves * rows * kKsRowBytes);
  return fit < 2 ? 2 : (fit > 5 ? 5 : fit);
}

// SWIGLU: the weight stacks gate rows [0, n) over up rows [n, 2n); a tile's
// WR weight rows are WR / 2 gate rows and the same up rows, and the output is
// round(swiglu_act(round(g), round(u))) (g and u scaled by the row's norm
// first under kEpiNorm).
template <typename T, int BM, int WR, bool SWIGLU, int EPI>
__global__ void __launch_bounds__(64 * kKsWaves)
linear_kstream_kernel(KstreamParams p) {
  using M = SplitMma<T>;
  using vec8 = typename M::vec8;
  static_assert(!(SWIGLU && EPI == kEpiResidual), "the residual epilogue has no SwiGLU form");
  constexpr int STAGES = ks_stages(BM + WR);
  constexpr int MT = BM / 16, NT = WR / 16;
  constexpr int OC = SWIGLU ? WR / 2 : WR;     // output columns
  constexpr int kLoads = (BM + WR) / 8;        // load instructions of a chunk: 8 rows each
  constexpr int kStageBytes = (BM + WR) * kKsRowBytes;
  constexpr int kSumRow = WR + 4;              // floats; spreads a store's four rows over the banks
  static_assert(BM % 16 == 0 && WR % 16 == 0 && OC % 8 == 0, "tile");
  static_assert(kLoads * STAGES <= 63, "vmcnt range");
  static_assert(BM * kSumRow * 4 <= STAGES * kStageBytes, "tile sums exceed the staging LDS");
  extern __shared__ __attribute__((aligned(1024))) unsigned char kstream_smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15;
  const int q4 = lane >> 4;
  // The row blocks of a column tile are consecutive workgroups of one
  // compute die (id % 8), so its weights come to that die's L2 once.
  const int32_t group = static_cast<int32_t>(blockIdx.x) / (kKsXcds * p.row_blocks);
  const int32_t in = static_cast<int32_t>(blockIdx.x) - group * kKsXcds * p.row_blocks;
  const int32_t tn = group * kKsXcds + in % kKsXcds;
  if (tn >= p.tiles_n) return;
  const int32_t m0 = in / kKsXcds * BM;
  const int32_t n0 = tn * OC;

  // This wavefront's quarter of K, in whole k-steps of 32.  Of a last chunk of
  // 32 the upper four pieces read the lower ones again and its second k-step
  // is left out.
  const int32_t k_per_wave = (p.k / 32 + kKsWaves - 1) / kKsWaves * 32;
  const int32_t k0 = min(wave * k_per_wave, p.k);
  const int32_t k1 = min(k0 + k_per_wave, p.k);
  const int32_t chunks = (k1 - k0 + kKsChunk - 1) / kKsChunk;
  const int32_t half = (k1 - k0) % kKsChunk != 0 ? chunks - 1 : -1;

  // Load i: rows 8 i .. +8 of the chunk, x rows first, the 16-byte piece q of
  // row r at q ^ (r & 7) so that the lanes of an operand read fall in distinct
  // banks.  Rows past the matrix read its last row and are not stored.
  const int lrow = lane >> 3;
  const int piece = (lane & 7) ^ lrow;
  const unsigned char *src[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int64_t at = static_cast<int64_t>(k0) * 2 + 16 * piece;
    if (8 * i < BM) {
      src[i] = static_cast<const unsigned char *>(p.x) + min(m0 + 8 * i + lrow, p.m - 1) * p.x_stride * 2 + at;
    } else {
      const bool up = SWIGLU && 8 * i - BM >= OC;
      const int64_t row = min(n0 + 8 * i - BM - (up ? OC : 0) + lrow, p.n - 1) + (up ? static_cast<int64_t>(p.n) : 0);
      src[i] = static_cast<const unsigned char *>(p.w) + row * p.w_stride * 2 + at;
    }
  }
  unsigned char *ring = kstream_smem + wave * (STAGES * kStageBytes);
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) unsigned char *)ring));
  const int64_t back = piece >= 4 ? -64 : 0;
  // Chunks are loaded in order; src moves on with them.
  auto load = [&](int32_t c, int32_t stage) {
    const int64_t shift = c == half ? back : 0;
    auto each = [&](auto stream_tag) {
#pragma unroll
      for (int i = 0; i < kLoads; ++i) {
        const uint32_t at = __builtin_amdgcn_readfirstlane(lds0 + static_cast<uint32_t>(stage * kStageBytes + i * 1024));
        if (8 * i < BM)
          load_lds16(src[i] + shift, at);
        else
          load_lds16<decltype(stream_tag)::value>(src[i] + shift, at);
        src[i] += kKsRowBytes;
      }
    };
    if (p.stream)  // uniform
      each(std::true_type{});
    else
      each(std::false_type{});
  };

  f32x4 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  // kEpiNorm: this lane's sums of squares of the x operands it feeds the
  // MFMAs (row 16 mt + l16, eight elements of every k-step in range), taken
  // from the operand registers so they cost no load and overlap the MFMAs.
  float ssq[EPI == kEpiNorm ? MT : 1];
#pragma unroll
  for (int i = 0; i < (EPI == kEpiNorm ? MT : 1); ++i) ssq[i] = 0.f;

  // Chunk c, with FLIGHT chunks loaded after it; LOAD: its buffer then takes
  // chunk c + STAGES (all operands are in registers before the load is issued).
  int32_t stage = 0;
  int32_t c = 0;
  auto step = [&](auto flight_tag, auto load_tag) {
    constexpr int FLIGHT = decltype(flight_tag)::value;
    constexpr bool LOAD = decltype(load_tag)::value;
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(kLoads * FLIGHT) : "memory");
    vec8 a[2][MT], b[2][NT];
    const unsigned char *at = ring + stage * kStageBytes + l16 * kKsRowBytes;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int pc = 16 * ((4 * s + q4) ^ (l16 & 7));
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) a[s][mt] = *reinterpret_cast<const vec8 *>(at + 16 * mt * kKsRowBytes + pc);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) b[s][nt] = *reinterpret_cast<const vec8 *>(at + (BM + 16 * nt) * kKsRowBytes + pc);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
    if constexpr (LOAD) load(c + STAGES, stage);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (s == 1 && c == half) break;  // uniform
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = M::mma(a[s][mt], b[s][nt], acc[mt][nt]);
        if constexpr (EPI == kEpiNorm) ssq[mt] = dot8<T>(a[s][mt], a[s][mt], ssq[mt]);
      }
    }
    stage = stage + 1 == STAGES ? 0 : stage + 1;
    ++c;
  };
  using Yes = std::true_type;
  using No = std::false_type;
#pragma unroll
  for (int i = 0; i < STAGES; ++i)
    if (i < chunks) load(i, i);  // uniform
  while (c + STAGES < chunks) step(std::integral_constant<int, STAGES - 1>{}, Yes{});
  // At most STAGES chunks are left, all in flight.
  if constexpr (STAGES >= 5)
    if (chunks - c >= 5) step(std::integral_constant<int, 4>{}, No{});
  if constexpr (STAGES >= 4)
    if (chunks - c >= 4) step(std::integral_constant<int, 3>{}, No{});
  if constexpr (STAGES >= 3)
    if (chunks - c >= 3) step(std::integral_constant<int, 2>{}, No{});
  if (chunks - c >= 2) step(std::integral_constant<int, 1>{}, No{});
  if (chunks - c >= 1) step(std::integral_constant<int, 0>{}, No{});

  // Sum the four wavefronts' tiles in order: tile row r, weight row j at
  // sums[wave][r][j].
  float *sums = reinterpret_cast<float *>(kstream_smem);
  float *ssq_rows = sums + kKsWaves * BM * kSumRow;  // [4 waves][BM]
  __syncthreads();  // every wavefront's loads have landed and its operand reads are done
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        sums[(wave * BM + 16 * mt + 4 * q4 + r) * kSumRow + 16 * nt + l16] = acc[mt][nt][r];
    if constexpr (EPI == kEpiNorm) {
      float v = ssq[mt];
      v += __shfl_xor(v, 16, 64);  // the four lanes (l16, q4) of row 16 mt + l16
      v += __shfl_xor(v, 32, 64);
      if (q4 == 0) ssq_rows[wave * BM + 16 * mt + l16] = v;
    }
  }
  __syncthreads();
  for (int it = threadIdx.x; it < BM * OC; it += 64 * kKsWaves) {
    const int r = it / OC;
    const int j = it - r * OC;
    const int32_t row = m0 + r;
    const int32_t col = n0 + j;
    if (row >= p.m || col >= p.n) continue;
    float sum = 0.f, sumu = 0.f;
#pragma unroll
    for (int wv = 0; wv < kKsWaves; ++wv) {
      sum += sums[(wv * BM + r) * kSumRow + j];
      if constexpr (SWIGLU) sumu += sums[(wv * BM + r) * kSumRow + OC + j];
    }
    if constexpr (EPI == kEpiNorm) {
      const float sq = ((ssq_rows[r] + ssq_rows[BM + r]) + ssq_rows[2 * BM + r]) + ssq_rows[3 * BM + r];
      const float scale = rsqrtf(sq / static_cast<float>(p.k) + p.eps);
      sum *= scale;
      sumu *= scale;
    }
    T out;
    if constexpr (SWIGLU)
      out = from_float<T>(swiglu_act(to_float(from_float<T>(sum)), to_float(from_float<T>(sumu))));
    else if constexpr (EPI == kEpiResidual)
      out = from_float<T>(to_float(from_float<T>(sum)) +
                          to_float(static_cast<const T *>(p.residual)[static_cast<int64_t>(row) * p.residual_stride + col]));
    else
      out = from_float<T>(sum);
    static_cast<T *>(p.y)[static_cast<int64_t>(row) * p.y_stride + col] = out;
  }
}

template <typename T, int BM, int WR, bool SWIGLU, int EPI>
void launch_kstream(KstreamParams p, hipStream_t stream) {
  constexpr int cols = SWIGLU ? WR / 2 : WR;
  constexpr int staging = kKsWaves * ks_stages(BM + WR) * (BM + WR) * kKsRowBytes;
  constexpr int sums = kKsWaves * BM * (WR + 4) * 4 + kKsWaves * BM * 4;
  constexpr int lds = staging > sums ? staging : sums;
  p.tiles_n = (p.n + cols - 1) / cols;
  p.row_blocks = (p.m + BM - 1) / BM;
  auto kernel = &linear_kstream_kernel<T, BM, WR, SWIGLU, EPI>;
  if (lds > 64 * 1024) {
    // Raise the kernel's dynamic LDS limit once per device (a failure shows
    // up as a launch error).
    constexpr int kMaxDevices = 64;
    static std::atomic<bool> raised[kMaxDevices];
    int device = 0;
    if (hipGetDevice(&device) == hipSuccess && device >= 0 && device < kMaxDevices &&
        !raised[device].load(std::memory_order_acquire)) {
      if (hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess)
        raised[device].store(true, std::memory_order_release);
    }
  }
  const unsigned grid = static_cast<unsigned>((p.tiles_n + kKsXcds - 1) / kKsXcds * kKsXcds * p.row_blocks);
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * kKsWaves), lds, stream, p);
}

// The tile of a call: BM in 16..64 rows and WR in 16..48 weight rows (32..64
// with SwiGLU, half of them up rows), and whether its weights stream past the
// caches.  A compute unit reads ceil(workgroups / 256) x (BM + WR) rows of K
// at 53 B/ns whatever the tile, so the fewest rows win; then, since each row
// block reads the weights and blocks of long rows do not keep together in L2,
// the fewest blocks above kKsShortK (4096 x 4096 at 17 rows: one block 8.3 us,
// two 12.0), then the larger grid (qkv at 64 rows: 216 workgroups in four
// blocks 7.4 us, 160 in two 7.8).
// Nontemporal weights (TinyLlama's qkv at 4 rows 5.3 -> 4.7 us, gate|up 10.7
// -> 9.5) need whole lines per row piece (rows of 1984 bytes: 3.7 -> 4.3) and
// weights that would not stay in the caches anyway (1536 x 1536 at 33 rows
// 4.7 -> 5.1), and they come from memory again for a row block that falls out
// of step with the others: long rows and a last block of few rows, which runs
// ahead (2048 x 5632 at 17 rows 7.9 -> 8.9 us, at 33 rows 10.0 -> 12.3; in
// full blocks, 32 and 64 rows, 9.6 -> 9.2 and 12.5 -> 12.2).
// Over 1 to 64 rows of 39 weights of 0.1 to 268 MB the choice is 1.3% slower
// than the best of 24 forms.  Every form sums a product in the same order, so
// the choice changes no bit.
constexpr int64_t kKsCached = 6000000;  // bytes of weights up to which loads stay temporal
constexpr int32_t kKsShortK = 2048;     // K up to which row blocks keep together

template <typename T, bool SWIGLU, int EPI>
void launch_kstream_tile(KstreamParams p, hipStream_t stream) {
  constexpr int kFirst = SWIGLU ? 32 : 16;
  const int64_t w_rows = SWIGLU ? 2 * static_cast<int64_t>(p.n) : p.n;
  // Each further row block: a tenth of the weights' time at 8 TB/s.
  const float block_us = p.k <= kKsShortK ? 0.f : 0.1f * static_cast<float>(w_rows * p.k) * 2.f / 8e6f;
  int bm = 16, wr = kFirst;
  float best = 0.f;
  int64_t best_grid = 0;
  for (int cm = 16; cm <= 64 && cm < p.m + 16; cm += 16)
    for (int cw = kFirst; cw < kFirst + 48; cw += 16) {
      const int64_t blocks = (p.m + cm - 1) / cm;
      const int64_t grid = blocks * ((w_rows + cw - 1) / cw);
      const int64_t rows = (grid + kKsUnits - 1) / kKsUnits * (cm + cw);
      const float cost = static_cast<float>(rows * p.k) * 2.f / 53e3f + block_us * static_cast<float>(blocks - 1);
      if (best_grid == 0 || cost < best || (cost == best && grid > best_grid)) {
        best = cost;
        best_grid = grid;
        bm = cm;
        wr = cw;
      }
    }
  const uintptr_t lines = reinterpret_cast<uintptr_t>(p.w) | static_cast<uintptr_t>(p.w_stride * 2);
  p.stream = lines % kKsRowBytes == 0 && w_rows * p.k * 2 >= kKsCached &&
             (p.m <= bm || p.k <= kKsShortK || p.m % bm == 0);
#define TF_KSTREAM_CASE(BM)                                                                        \
  if (bm == BM) {                                                                                  \
    if (wr == kFirst) return launch_kstream<T, BM, kFirst, SWIGLU, EPI>(p, stream);                \
    if (wr == kFirst + 16) return launch_kstream<T, BM, kFirst + 16, SWIGLU, EPI>(p, stream);      \
    return launch_kstream<T, BM, kFirst + 32, SWIGLU, EPI>(p, stream);                             \
  }
  TF_KSTREAM_CASE(16)
  TF_KSTREAM_CASE(32)
  TF_KSTREAM_CASE(48)
  TF_KSTREAM_CASE(64)
#undef TF_KSTREAM_CASE
}

template <typename T, int MT, bool SWIGLU>
void launch_stream(const void *x, int64_t x_stride, const void *w, int64_t w_stride, void *y,
                   int64_t y_stride, float *partials, int32_t m, int32_t n, int32_t k,
                   int32_t splits, int32_t k_per_split, hipStream_t stream) {
  const size_t lds = static_cast<size_t>(16 * MT + kStreamCols) * kStreamChunk * sizeof(T);
  const int32_t cols = SWIGLU ? kStreamCols / 2 : kStreamCols;
  hipLaunchKernelGGL((linear_stream_kernel<T, MT, SWIGLU>),
                     dim3((n + cols - 1) / cols, splits), dim3(256), lds, stream,
                     static_cast<const T *>(x), x_stride, static_cast<const T *>(w), w_stride,
                     static_cast<T *>(y), y_stride, partials, m, n, k, k_per_split);
}

template <typename T, bool SWIGLU>
void launch_stream_mt(const void *x, int64_t x_stride, const void *w, int64_t w_stride, void *y,
                      int64_t y_stride, float *partials, int32_t m, int32_t n, int32_t k,
                      int32_t splits, int32_t k_per_split, hipStream_t stream) {
#define TF_STREAM_CASE(MT)                                                                   \
  launch_stream<T, MT, SWIGLU>(x, x_stride, w, w_stride, y, y_stride, partials, m, n, k,    \
                               splits, k_per_split, stream)
  switch ((m + 15) / 16) {
    case 1: TF_STREAM_CASE(1); break;
    case 2: TF_STREAM_CASE(2); break;
    case 3: TF_STREAM_CASE(3); break;
    default: TF_STREAM_CASE(4); break;
  }
#undef TF_STREAM_CASE
}

// y[m][n] = round(sum_s partials[s][m][n]), four columns per thread.
template <typename T>
__global__ void __launch_bounds__(256)
partials_sum_kernel(const float *__restrict__ partials, int32_t splits, int32_t m, int32_t n,
                    T *__restrict__ y, int64_t y_stride) {
  const int64_t quads = static_cast<int64_t>(m) * (n / 4);
  const int64_t plane = static_cast<int64_t>(m) * n;
  for (int64_t q = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; q < quads;
       q += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int32_t row = static_cast<int32_t>(q / (n / 4));
    const int32_t col = 4 * static_cast<int32_t>(q - static_cast<int64_t>(row) * (n / 4));
    const float *src = partials + static_cast<int64_t>(row) * n + col;
    f32x4 s = *reinterpret_cast<const f32x4 *>(src);
    for (int32_t sp = 1; sp < splits; ++sp) s += *reinterpret_cast<const f32x4 *>(src + sp * plane);
    typedef T t4 __attribute__((ext_vector_type(4)));
    const t4 v = {from_float<T>(s[0]), from_float<T>(s[1]), from_float<T>(s[2]),
                  from_float<T>(s[3])};
    *reinterpret_cast<t4 *>(y + static_cast<int64_t>(row) * y_stride + col) = v;
  }
}

template <typename T, int MT>
void launch_partials(const void *x, int64_t x_stride, const void *w, int64_t w_stride,
                     float *partials, int32_t m, int32_t n, int32_t k, int32_t splits,
                     int32_t k_per_split, hipStream_t stream) {
  const size_t lds = static_cast<size_t>(kSplitWaves) * MT * (kSplitCols / 16) * 4 * 64 *
                     sizeof(float);
  hipLaunchKernelGGL((linear_partials_kernel<T, MT>),
                     dim3((n + kSplitCols - 1) / kSplitCols, splits), dim3(kSplitWaves * 64), lds,
                     stream, static_cast<const T *>(x), x_stride, static_cast<const T *>(w),
                     w_stride, partials, m, n, k, k_per_split);
}

template <typename T>
void launch_partials_mt(const void *x, int64_t x_stride, const void *w, int64_t w_stride,
                        float *partials, int32_t m, int32_t n, int32_t k, int32_t splits,
                        int32_t k_per_split, hipStream_t stream) {
  switch ((m + 15) / 16) {
    case 1: launch_partials<T, 1>(x, x_stride, w, w_stride, partials, m, n, k, splits, k_per_split, stream); break;
    case 2: launch_partials<T, 2>(x, x_stride, w, w_stride, partials, m, n, k, splits, k_per_split, stream); break;
    case 3: launch_partials<T, 3>(x, x_stride, w, w_stride, partials, m, n, k, splits, k_per_split, stream); break;
    default: launch_partials<T, 4>(x, x_stride, w, w_stride, partials, m, n, k, splits, k_per_split, stream); break;
  }
}

}  // namespace
}  // namespace tf

extern "C" int32_t tf_linear_partials(const void *x, int64_t x_row_stride, const void *weight,
                                      int64_t weight_row_stride, float *partials, int32_t m,
                                      int32_t n, int32_t k, int32_t splits, int32_t dtype,
                                      void *stream) {
  using namespace tf;
  clear_error();
  if (dtype != TF_DTYPE_FLOAT16 && dtype != TF_DTYPE_BFLOAT16)
    return fail(TF_ERROR_UNSUPPORTED, "linear_partials supports fp16 and bf16");
  if (m < 0 || n < 0 || k < 0) return fail(TF_ERROR_INVALID_ARGUMENT, "sizes must be non-negative");
  if (m > 64) return fail(TF_ERROR_UNSUPPORTED, "linear_partials supports at most 64 rows");
  if (k % 32 != 0 || k == 0)
    return fail(TF_ERROR_UNSUPPORTED, "linear_partials needs K to be a positive multiple of 32");
  if (splits < 1 || splits > k / 32)
    return fail(TF_ERROR_INVALID_ARGUMENT, "splits must be in [1, K / 32]");
  if (x_row_stride < k || weight_row_stride < k)
    return fail(TF_ERROR_INVALID_ARGUMENT, "row strides are shorter than the rows");
  if (n > 65535 * tf::kSplitCols || splits > 65535)
    return fail(TF_ERROR_UNSUPPORTED, "grid too large");
  if (m == 0 || n == 0) return TF_SUCCESS;
  if (!x || !weight || !partials) return fail(TF_ERROR_INVALID_ARGUMENT, "null tensor pointer");
  const uintptr_t align = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(weight) |
                          static_cast<uintptr_t>(x_row_stride * 2) |
                          static_cast<uintptr_t>(weight_row_stride * 2);
  if (align % 16 != 0)
    return fail(TF_ERROR_UNSUPPORTED, "linear_partials needs 16-byte aligned x and weight rows");
  // Slices of whole k-steps; every slice is non-empty.
  const int32_t steps = k / 32;
  const int32_t k_per_split = ((steps + splits - 1) / splits) * 32;
  const int32_t used = (k + k_per_split - 1) / k_per_split;
  if (used != splits)
    return fail(TF_ERROR_INVALID_ARGUMENT, "splits must divide K / 32 into non-empty slices");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == TF_DTYPE_BFLOAT16)
    launch_partials_mt<__bf16>(x, x_row_stride, weight, weight_row_stride, partials, m, n, k,
                               splits, k_per_split, s);
  else
    launch_partials_mt<_Float16>(x, x_row_stride, weight, weight_row_stride, partials, m, n, k,
                                 splits, k_per_split, s);
  return check_launch("linear_partials");
}

extern "C" int32_t tf_linear_partials_sum(const float *partials, int32_t splits, int32_t m,
                                          int32_t n, void *y, int64_t y_row_stride,
                                          int32_t dtype, void *stream) {
  using namespace tf;
  clear_error();
  if (!valid_dtype(dtype)) return fail(TF_ERROR_INVALID_ARGUMENT, "unsupported dtype code");
  if (dtype == TF_DTYPE_FLOAT32)
    return fail(TF_ERROR_UNSUPPORTED, "linear_partials_sum writes fp16 or bf16");
  if (m < 0 || n < 0 || splits < 1) return fail(TF_ERROR_INVALID_ARGUMENT, "invalid sizes");
  if (n % 4 != 0 || y_row_stride % 4 != 0)
    return fail(TF_ERROR_UNSUPPORTED, "linear_partials_sum needs N and the row stride to be multiples of 4");
  if (y_row_stride < n) return fail(TF_ERROR_INVALID_ARGUMENT, "row stride is shorter than the rows");
  if (m == 0 || n == 0) return TF_SUCCESS;
  if (!partials || !y) return fail(TF_ERROR_INVALID_ARGUMENT, "null tensor pointer");
  if ((reinterpret_cast<uintptr_t>(partials) | reinterpret_cast<uintptr_t>(y)) % 16 != 0)
    return fail(TF_ERROR_UNSUPPORTED, "linear_partials_sum needs 16-byte aligned buffers");
  const int64_t quads = static_cast<int64_t>(m) * (n / 4);
  const int64_t blocks = (quads + 255) / 256;
  const dim3 grid(static_cast<unsigned>(blocks < 2048 ? blocks : 2048));
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == TF_DTYPE_BFLOAT16)
    hipLaunchKernelGGL(partials_sum_kernel<__bf16>, grid, dim3(256), 0, s, partials, splits, m, n,
                       static_cast<__bf16 *>(y), y_row_stride);
  else
    hipLaunchKernelGGL(partials_sum_kernel<_Float16>, grid, dim3(256), 0, s, partials, splits, m,
                       n, static_cast<_Float16 *>(y), y_row_stride);
  return check_launch("linear_partials_sum");
}

namespace tf {
namespace {

int32_t linear_stream_entry(const void *x, int64_t x_row_stride, const void *weight,
                            int64_t weight_row_stride, void *y, int64_t y_row_stride,
                            float *partials, int32_t m, int32_t n, int32_t k, int32_t splits,
                            int32_t dtype, void *stream, bool swiglu, const char *name) {
  clear_error();
  if (dtype != TF_DTYPE_FLOAT16 && dtype != TF_DTYPE_BFLOAT16)
    return fail(TF_ERROR_UNSUPPORTED, "linear_stream supports fp16 and bf16");
  if (m < 0 || n < 0 || k < 0) return fail(TF_ERROR_INVALID_ARGUMENT, "sizes must be non-negative");
  if (m > 64) return fail(TF_ERROR_UNSUPPORTED, "linear_stream supports at most 64 rows");
  if (k % 32 != 0 || k == 0)
    return fail(TF_ERROR_UNSUPPORTED, "linear_stream needs K to be a positive multiple of 32");
  if (splits < 1 || splits > k / 32)
    return fail(TF_ERROR_INVALID_ARGUMENT, "splits must be in [1, K / 32]");
  if (!partials && splits != 1)
    return fail(TF_ERROR_INVALID_ARGUMENT, "several K slices need a partials buffer");
  if (x_row_stride < k || weight_row_stride < k || (!partials && y_row_stride < n))
    return fail(TF_ERROR_INVALID_ARGUMENT, "row strides are shorter than the rows");
  if (n > 65535 * (kStreamCols / 2) || splits > 65535)
    return fail(TF_ERROR_UNSUPPORTED, "grid too large");
  if (m == 0 || n == 0) return TF_SUCCESS;
  if (!x || !weight || (!partials && !y))
    return fail(TF_ERROR_INVALID_ARGUMENT, "null tensor pointer");
  const uintptr_t align = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(weight) |
                          static_cast<uintptr_t>(x_row_stride * 2) |
                          static_cast<uintptr_t>(weight_row_stride * 2);
  if (align % 16 != 0)
    return fail(TF_ERROR_UNSUPPORTED, "linear_stream needs 16-byte aligned x and weight rows");
  const int32_t steps = k / 32;
  const int32_t k_per_split = ((steps + splits - 1) / splits) * 32;
  if ((k + k_per_split - 1) / k_per_split != splits)
    return fail(TF_ERROR_INVALID_ARGUMENT, "splits must divide K / 32 into non-empty slices");
  hipStream_t s = static_cast<hipStream_t>(stream);
#define TF_STREAM_LAUNCH(T, G)                                                                \
  launch_stream_mt<T, G>(x, x_row_stride, weight, weight_row_stride, y, y_row_stride, partials, \
                         m, n, k, splits, k_per_split, s)
  if (dtype == TF_DTYPE_BFLOAT16) {
    if (swiglu) TF_STREAM_LAUNCH(__bf16, true); else TF_STREAM_LAUNCH(__bf16, false);
  } else {
    if (swiglu) TF_STREAM_LAUNCH(_Float16, true); else TF_STREAM_LAUNCH(_Float16, false);
  }
#undef TF_STREAM_LAUNCH
  return check_launch(name);
}

}  // namespace
}  // namespace tf

extern "C" int32_t tf_linear_stream(const void *x, int64_t x_row_stride, const void *weight,
                                    int64_t weight_row_stride, void *y, int64_t y_row_stride,
                                    float *partials, int32_t m, int32_t n, int32_t k,
                                    int32_t splits, int32_t dtype, void *stream) {
  return tf::linear_stream_entry(x, x_row_stride, weight, weight_row_stride, y, y_row_stride,
                                 partials, m, n, k, splits, dtype, stream, false,
                                 "linear_stream");
}

extern "C" int32_t tf_linear_swiglu(const void *x, int64_t x_row_stride, const void *gate_up_weight,
                                    int64_t weight_row_stride, void *y, int64_t y_row_stride,
                                    int32_t m, int32_t intermediate, int32_t k, int32_t dtype,
                                    void *stream) {
  return tf::linear_stream_entry(x, x_row_stride, gate_up_weight, weight_row_stride, y,
                                 y_row_stride, nullptr, m, intermediate, k, 1, dtype, stream,
                                 true, "linear_swiglu");
}

namespace tf {
namespace {

int32_t kstream_entry(const void *x, int64_t x_row_stride, const void *weight,
                      int64_t weight_row_stride, void *y, int64_t y_row_stride, int32_t m,
                      int32_t n, int32_t k, int32_t dtype, void *stream, bool swiglu, int epi,
                      float eps, const void *residual, int64_t residual_row_stride,
                      const char *name) {
  clear_error();
  if (dtype != TF_DTYPE_FLOAT16 && dtype != TF_DTYPE_BFLOAT16)
    return fail(TF_ERROR_UNSUPPORTED, "linear_kstream supports fp16 and bf16");
  if (m < 0 || n < 0 || k < 0) return fail(TF_ERROR_INVALID_ARGUMENT, "sizes must be non-negative");
  if (m > 64) return fail(TF_ERROR_UNSUPPORTED, "linear_kstream supports at most 64 rows");
  if (k % 32 != 0 || k == 0)
    return fail(TF_ERROR_UNSUPPORTED, "linear_kstream needs K to be a positive multiple of 32");
  if (x_row_stride < k || weight_row_stride < k || y_row_stride < n)
    return fail(TF_ERROR_INVALID_ARGUMENT, "row strides are shorter than the rows");
  if (epi == kEpiNorm && !(eps > 0.f)) return fail(TF_ERROR_INVALID_ARGUMENT, "eps must be positive");
  if (epi == kEpiResidual && residual_row_stride < n)
    return fail(TF_ERROR_INVALID_ARGUMENT, "residual row stride is shorter than the rows");
  if (n > 65535 * 16) return fail(TF_ERROR_UNSUPPORTED, "grid too large");
  if (m == 0 || n == 0) return TF_SUCCESS;
  if (!x || !weight || !y || (epi == kEpiResidual && !residual))
    return fail(TF_ERROR_INVALID_ARGUMENT, "null tensor pointer");
  const uintptr_t align = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(weight) |
                          static_cast<uintptr_t>(x_row_stride * 2) |
                          static_cast<uintptr_t>(weight_row_stride * 2);
  if (align % 16 != 0)
    return fail(TF_ERROR_UNSUPPORTED, "linear_kstream needs 16-byte aligned x and weight rows");
  hipStream_t s = static_cast<hipStream_t>(stream);
  KstreamParams p;
  p.x = x;
  p.w = weight;
  p.y = y;
  p.residual = residual;
  p.x_stride = x_row_stride;
  p.w_stride = weight_row_stride;
  p.y_stride = y_row_stride;
  p.residual_stride = residual_row_stride;
  p.eps = eps;
  p.m = m;
  p.n = n;
  p.k = k;
  p.tiles_n = p.row_blocks = p.stream = 0;
#define TF_KSTREAM_LAUNCH(T)                                          \
  do {                                                                \
    if (swiglu && epi == kEpiNorm)                                    \
      launch_kstream_tile<T, true, kEpiNorm>(p, s);                   \
    else if (swiglu)                                                  \
      launch_kstream_tile<T, true, kEpiPlain>(p, s);                  \
    else if (epi == kEpiNorm)                                         \
      launch_kstream_tile<T, false, kEpiNorm>(p, s);                  \
    else if (epi == kEpiResidual)                                     \
      launch_kstream_tile<T, false, kEpiResidual>(p, s);              \
    else                                                              \
      launch_kstream_tile<T, false, kEpiPlain>(p, s);                 \
  } while (0)
  if (dtype == TF_DTYPE_BFLOAT16)
    TF_KSTREAM_LAUNCH(__bf16);
  else
    TF_KSTREAM_LAUNCH(_Float16);
#undef TF_KSTREAM_LAUNCH
  return check_launch(name);
}

}  // namespace
}  // namespace tf

extern "C" int32_t tf_linear_kstream(const void *x, int64_t x_row_stride, const void *weight,
                                     int64_t weight_row_stride, void *y, int64_t y_row_stride,
                                     int32_t m, int32_t n, int32_t k, int32_t dtype, void *stream) {
  return tf::kstream_entry(x, x_row_stride, weight, weight_row_stride, y, y_row_stride, m, n, k,
                           dtype, stream, false, tf::kEpiPlain, 0.f, nullptr, 0, "linear_kstream");
}

extern "C" int32_t tf_linear_kstream_norm(const void *x, int64_t x_row_stride,
                                          const void *weight, int64_t weight_row_stride, void *y,
                                          int64_t y_row_stride, int32_t m, int32_t n, int32_t k,
                                          float eps, int32_t dtype, void *stream) {
  return tf::kstream_entry(x, x_row_stride, weight, weight_row_stride, y, y_row_stride, m, n, k,
                           dtype, stream, false, tf::kEpiNorm, eps, nullptr, 0,
                           "linear_kstream_norm");
}

extern "C" int32_t tf_linear_kstream_residual(const void *x, int64_t x_row_stride,
                                              const void *weight, int64_t weight_row_stride,
                                              const void *residual, int64_t residual_row_stride,
                                              void *y, int64_t y_row_stride, int32_t m, int32_t n,
                                              int32_t k, int32_t dtype, void *stream) {
  return tf::kstream_entry(x, x_row_stride, weight, weight_row_stride, y, y_row_stride, m, n, k,
                           dtype, stream, false, tf::kEpiResidual, 0.f, residual,
                           residual_row_stride, "linear_kstream_residual");
}

extern "C" int32_t tf_linear_kswiglu(const void *x, int64_t x_row_stride,
                                     const void *gate_up_weight, int64_t weight_row_stride,
                                     void *y, int64_t y_row_stride, int32_t m,
                                     int32_t intermediate, int32_t k, int32_t dtype,
                                     void *stream) {
  return tf::kstream_entry(x, x_row_stride, gate_up_weight, weight_row_stride, y, y_row_stride,
                           m, intermediate, k, dtype, stream, true, tf::kEpiPlain, 0.f, nullptr, 0,
                           "linear_kswiglu");
}

extern "C" int32_t tf_linear_kswiglu_norm(const void *x, int64_t x_row_stride,
                                          const void *gate_up_weight, int64_t weight_row_stride,
                                          void *y, int64_t y_row_stride, int32_t m,
                                          int32_t intermediate, int32_t k, float eps,
                                          int32_t dtype, void *stream) {
  return tf::kstream_entry(x, x_row_stride, gate_up_weight, weight_row_stride, y, y_row_stride,
                           m, intermediate, k, dtype, stream, true, tf::kEpiNorm, eps, nullptr, 0,
                           "linear_kswiglu_norm");
}
