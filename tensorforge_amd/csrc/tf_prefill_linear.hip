// Linear layers of prefill on MFMA: y[m][n] = x[m][k] . w[n][k]^T for the
// packed prompt rows of a prefill (65 to many thousand), bf16 / fp16
// storage, fp32 accumulation.
//
// A workgroup computes a BM x BN tile of y.  K is walked in 64-wide chunks
// (128-byte row pieces of x and w) held in a ring of STAGES LDS buffers that
// direct-to-LDS loads fill: no staging registers, STAGES - 1 chunks in flight
// while one is multiplied, and one barrier per chunk.  A load instruction of
// a wavefront writes 1024 consecutive LDS bytes (8 rows), so the 16-byte
// pieces of a row are permuted on the global side: piece p of row r sits at
// p ^ (r & 7), and the eight lanes that an operand read serves at a time
// (rows l16, one piece) fall in distinct banks.
//
// MFMA v_mfma_f32_16x16x32 (bf16 / f16) with w as the A operand:
//   A = w rows:  lane (l16, q4) holds w[n + l16][k + 8 q4 .. +8]
//   B = x rows:  lane (l16, q4) holds x[m + l16][k + 8 q4 .. +8]
//   C:           lane (l16, q4), register r holds y[m + l16][n + 4 q4 + r]
// so a lane stores four consecutive columns of one row, and a SwiGLU lane
// holds the gate and the up product of its columns.
//
// Output forms (EPI):
//   kOutRounded  y = round(sum)
//   kOutPartials fp32 slice sums partials[split][m][n] of a K split over the
//                grid (for calls whose tiles leave the chip idle); the
//                consumer adds the slices in order and rounds once
//                (residual_rms_norm_partials, linear_partials_sum)
//   kOutSwiglu   w stacks gate rows [0, n) over up rows [n, 2n):
//                y = round(swiglu_act(round(g), round(u))), the activation of
//                the rounded projection
//
// Reference semantics: the nn.Linear projections of prefill,
// tensorforge/model/layers.py:88-95, 144-158 as runtime/prefill.py:90-135
// calls them.
#include <atomic>
#include <type_traits>

#include "tf_common.hpp"

namespace tf {
namespace {

template <typename T>
struct PlMma;

template <>
struct PlMma<__bf16> {
  typedef __bf16 vec8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ f32x4 mma(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};

template <>
struct PlMma<_Float16> {
  typedef _Float16 vec8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ f32x4 mma(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

enum PlOut : int { kOutRounded = 0, kOutPartials = 1, kOutSwiglu = 2 };

struct PlParams {
  const void *x;
  const void *w;
  void *y;
  float *partials;
  int64_t x_stride;
  int64_t w_stride;
  int64_t y_stride;
  int32_t m;
  int32_t n;           // output columns
  int32_t k_chunks;    // 64-wide chunks of K
  int32_t tiles_m;
  int32_t tiles_n;
  int32_t splits;
};

constexpr int kPlChunk = 64;      // k per LDS buffer
constexpr int kPlRowBytes = 128;  // bytes of a chunk row
constexpr int kPlXcds = 8;
constexpr int kPlBand = 8;        // row tiles of one band of the tile order

// Tile of workgroup `id`: the ids a compute die is dealt (id % 8) take
// consecutive tiles of an order that walks bands of kPlBand row tiles, rows
// fastest, so the tiles a die computes together share their w columns and
// x rows in its L2.
__device__ __forceinline__ void pl_tile(const PlParams &p, int32_t id, int32_t &tm, int32_t &tn,
                                        int32_t &split) {
  const int32_t total = p.tiles_m * p.tiles_n * p.splits;
  const int32_t each = total / kPlXcds, more = total % kPlXcds;
  const int32_t xcd = id % kPlXcds, at = id / kPlXcds;
  int32_t t = (xcd < more ? xcd * (each + 1) : more * (each + 1) + (xcd - more) * each) + at;
  const int32_t plane = p.tiles_m * p.tiles_n;
  split = t / plane;
  t -= split * plane;
  const int32_t band = t / (kPlBand * p.tiles_n);
  const int32_t rows = min(kPlBand, p.tiles_m - band * kPlBand);
  t -= band * kPlBand * p.tiles_n;
  tn = t / rows;
  tm = band * kPlBand + (t - tn * rows);
}

// Every load but the newest `N` of this wavefront has landed and its LDS reads
// are done; then the workgroup barrier, so that holds for every wavefront.
template <int N>
__device__ __forceinline__ void pl_wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N) : "memory");
}

template <typename T, int BM, int BN, int WM, int WN, int STAGES, int EPI>
__global__ void __launch_bounds__(64 * WM * WN)
prefill_linear_kernel(PlParams p) {
  using M = PlMma<T>;
  using vec8 = typename M::vec8;
  constexpr int kWaves = WM * WN;
  constexpr int TM = BM / WM, TN = BN / WN;  // a wavefront's tile
  constexpr int MT = TM / 16, NT = TN / 16;
  constexpr int kGroups = (BM + BN) / 8;     // 8-row load groups of a chunk
  constexpr int kLoads = kGroups / kWaves;   // of a wavefront
  constexpr int kStageBytes = (BM + BN) * kPlRowBytes;
  static_assert(kGroups % kWaves == 0 && TM % 16 == 0 && TN % 16 == 0, "tile split");
  static_assert(EPI != kOutSwiglu || NT % 2 == 0, "gate and up blocks pair up");
  static_assert(kLoads * (STAGES - 1) <= 63, "vmcnt range");
  // Two operand sets where they fit the 256 registers of two wavefronts per
  // SIMD (eight wavefronts) beside the accumulators.
  constexpr bool kTwoSets = kWaves <= 4 || MT * NT * 4 + 8 * (MT + NT) <= 230;
  extern __shared__ __attribute__((aligned(1024))) unsigned char pl_smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15;
  const int q4 = lane >> 4;
  const int wm = wave / WN, wn = wave % WN;
  int32_t tm, tn, split;
  pl_tile(p, blockIdx.x, tm, tn, split);
  const int32_t m0 = tm * BM;
  const int32_t n0 = tn * (EPI == kOutSwiglu ? BN / 2 : BN);
  const int32_t c0 = split * p.k_chunks / p.splits;
  const int32_t chunks = (split + 1) * p.k_chunks / p.splits - c0;

  // Load group i of this wavefront: rows 8 g .. +8 of the chunk, x rows
  // first.  Rows past the matrix read its last row and are not stored.
  const unsigned char *base[kLoads];
  uint32_t voffset[kLoads];
  const int lrow = lane >> 3;
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int g = wave + kWaves * i;  // uniform
    const uint32_t piece = 16u * static_cast<uint32_t>((lane & 7) ^ lrow);
    if (g < BM / 8) {
      const int32_t row = min(8 * g + lrow, p.m - 1 - m0);
      base[i] = static_cast<const unsigned char *>(p.x) +
                (static_cast<int64_t>(m0) * p.x_stride + static_cast<int64_t>(c0) * kPlChunk) * 2;
      voffset[i] = static_cast<uint32_t>(row) * static_cast<uint32_t>(p.x_stride * 2) + piece;
    } else {
      const int tr = 8 * (g - BM / 8) + lrow;  // tile row of w
      int64_t first = n0;                      // uniform
      int32_t row;
      if constexpr (EPI == kOutSwiglu) {
        // A wavefront's TN tile rows: TN / 2 gate columns, then the same up
        // columns.  A load group lies in one of the two.
        const int wt = tr / TN, rr = tr % TN;
        const int32_t col = min(n0 + wt * (TN / 2) + rr % (TN / 2), p.n - 1);
        if (__builtin_amdgcn_readfirstlane(rr / (TN / 2)) != 0) first += p.n;
        row = col - n0;
      } else {
        row = min(n0 + tr, p.n - 1) - n0;
      }
      base[i] = static_cast<const unsigned char *>(p.w) +
                (first * p.w_stride + static_cast<int64_t>(c0) * kPlChunk) * 2;
      voffset[i] = static_cast<uint32_t>(row) * static_cast<uint32_t>(p.w_stride * 2) + piece;
    }
  }
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) unsigned char *)pl_smem));
  // Load i of chunk c into its buffer.
  auto load_one = [&](int32_t c, int32_t stage, int i) {
    const uint32_t at = lds0 + static_cast<uint32_t>(stage * kStageBytes + wave * 1024);
    load_lds16(base[i] + static_cast<int64_t>(c) * kPlRowBytes, voffset[i],
               __builtin_amdgcn_readfirstlane(at + static_cast<uint32_t>(i * kWaves * 1024)));
  };

  f32x4 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Operands of the two 32-wide k-steps of a chunk: while one set is
  // multiplied the other is read from LDS.
  struct Operands {
    vec8 a[NT], b[MT];
  };
  Operands first, second;
  auto read = [&](Operands &f, int32_t stage, int s) {
    const unsigned char *xa = pl_smem + stage * kStageBytes + (wm * TM + l16) * kPlRowBytes;
    const unsigned char *wa = pl_smem + stage * kStageBytes + (BM + wn * TN + l16) * kPlRowBytes;
    const int piece = 16 * ((4 * s + q4) ^ (l16 & 7));
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) f.a[nt] = *reinterpret_cast<const vec8 *>(wa + nt * 16 * kPlRowBytes + piece);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) f.b[mt] = *reinterpret_cast<const vec8 *>(xa + mt * 16 * kPlRowBytes + piece);
  };
  auto multiply_row = [&](const Operands &f, int mt) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = M::mma(f.a[nt], f.b[mt], acc[mt][nt]);
  };
  // One chunk.  With two operand sets its second operands are read under the
  // first products; then the barrier, past which the next chunk has landed
  // and every wavefront holds this chunk in registers, so its buffer takes
  // chunk c + STAGES (LOAD) while the second products run and the next
  // chunk's first operands are read.  With one set the barrier follows both
  // products.  FLIGHT chunks beyond the next may stay in flight.
  int32_t stage = 0;  // buffer of chunk c
  auto step = [&](int32_t c, auto flight_tag, auto load_tag) {
    constexpr int FLIGHT = decltype(flight_tag)::value;
    constexpr bool LOAD = decltype(load_tag)::value;
    const int32_t next = stage + 1 == STAGES ? 0 : stage + 1;
    Operands &late = kTwoSets ? second : first;
    if constexpr (kTwoSets) read(second, stage, 1);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) multiply_row(first, mt);
    if constexpr (!kTwoSets) read(first, stage, 1);
    pl_wait_barrier<kLoads * FLIGHT>();
    if constexpr (kTwoSets) read(first, next, 0);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      if constexpr (LOAD) {
        // Loads spread over the products, which hide their issue.
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = mt * kLoads / MT; i < (mt + 1) * kLoads / MT; ++i) load_one(c + STAGES, stage, i);
        __builtin_amdgcn_sched_barrier(0);
      }
      multiply_row(late, mt);
    }
    if constexpr (!kTwoSets) read(first, next, 0);
    stage = next;
  };
  using Yes = std::true_type;
  using No = std::false_type;
  // The host checks chunks >= STAGES.
#pragma unroll
  for (int c = 0; c < STAGES; ++c)
#pragma unroll
    for (int i = 0; i < kLoads; ++i) load_one(c, c, i);
  pl_wait_barrier<kLoads *(STAGES - 1)>();
  read(first, 0, 0);
  int32_t c = 0;
  for (; c + STAGES < chunks; ++c) step(c, std::integral_constant<int, STAGES - 2>{}, Yes{});
  if constexpr (STAGES >= 4) step(c++, std::integral_constant<int, 2>{}, No{});
  if constexpr (STAGES >= 3) step(c++, std::integral_constant<int, 1>{}, No{});
  step(c++, std::integral_constant<int, 0>{}, No{});
  if constexpr (kTwoSets) read(second, stage, 1);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) multiply_row(first, mt);
  if constexpr (!kTwoSets) read(first, stage, 1);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) multiply_row(kTwoSets ? second : first, mt);

  // Lane (l16, q4) holds row 16 mt + l16, columns 16 nt + 4 q4 .. +4.
  typedef T t4 __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int32_t row = m0 + wm * TM + 16 * mt + l16;
    if (row >= p.m) continue;
    if constexpr (EPI == kOutSwiglu) {
      T *yrow = static_cast<T *>(p.y) + static_cast<int64_t>(row) * p.y_stride;
#pragma unroll
      for (int nt = 0; nt < NT / 2; ++nt) {
        const int32_t col = n0 + wn * (TN / 2) + 16 * nt + 4 * q4;
        t4 out;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          out[r] = from_float<T>(swiglu_act(to_float(from_float<T>(acc[mt][nt][r])),
                                            to_float(from_float<T>(acc[mt][nt + NT / 2][r]))));
        if (col < p.n) *reinterpret_cast<t4 *>(yrow + col) = out;  // n % 4 == 0
      }
    } else {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int32_t col = n0 + wn * TN + 16 * nt + 4 * q4;
        if (col >= p.n) continue;
        if constexpr (EPI == kOutPartials) {
          *reinterpret_cast<f32x4 *>(p.partials + (static_cast<int64_t>(split) * p.m + row) * p.n + col) =
              acc[mt][nt];
        } else {
          const t4 out = {from_float<T>(acc[mt][nt][0]), from_float<T>(acc[mt][nt][1]),
                          from_float<T>(acc[mt][nt][2]), from_float<T>(acc[mt][nt][3])};
          *reinterpret_cast<t4 *>(static_cast<T *>(p.y) + static_cast<int64_t>(row) * p.y_stride + col) = out;
        }
      }
    }
  }
}

template <typename T, int BM, int BN, int WM, int WN, int STAGES, int EPI>
int32_t launch_prefill_linear(PlParams p, hipStream_t stream) {
  constexpr int cols = EPI == kOutSwiglu ? BN / 2 : BN;
  constexpr int lds = STAGES * (BM + BN) * kPlRowBytes;
  p.tiles_m = (p.m + BM - 1) / BM;
  p.tiles_n = (p.n + cols - 1) / cols;
  auto kernel = &prefill_linear_kernel<T, BM, BN, WM, WN, STAGES, EPI>;
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
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(p.tiles_m * p.tiles_n * p.splits)),
                     dim3(64 * WM * WN), lds, stream, p);
  return check_launch("prefill_linear");
}

// The tiles, and the time a 64-wide chunk of K takes a workgroup of each when
// every compute unit has one.  pick_tile charges a call
//   5 us + ceil(workgroups / 256) x chunks per slice x that time
// plus, for K slices, 0.8 us and the slices' bytes at 8 TB/s for their reader,
// and takes the cheapest (tile, slices).  The times are fitted to a sweep of
// TinyLlama's four projections at 72 to 8058 rows on MI355X, over which the
// choice is 1.6% slower than the best of 18 tiles and up to 4 slices (worst:
// 1.2x).  Against the library GEMM (plus the SwiGLU launch for gate|up):
// 271 rows qkv 11.9 -> 8.8 us, o 11.4 -> 8.3, gate|up 33.0 -> 26.7, down
// 27.7 -> 16.3; 1500 rows 21.8 -> 21.2, 19.3 -> 17.4, 84.7 -> 67.3,
// 46.4 -> 43.4; 8058 rows gate|up 405 -> 329 (o 50.1 -> 60.5, down 122 -> 139,
// and qkv at 4096 rows 43.0 -> 54.3, at 6000 47.9 -> 58.1: above 2048 rows the
// callers keep the library for those three).
// A workgroup is bound by the latency of its loads in flight (up to 147 KB)
// at few rows, and by the products at many: at 8058 rows the 256 x 256 tile
// runs at 1.18 PFLOP/s, 1.6 with every row aliased to one (the clock under
// this load is about 1.9 GHz).
struct PlTile {
  int32_t bm, bn, stages;
  float chunk_us;
};
constexpr PlTile kPlTiles[] = {
    {64, 64, 4, 0.185f},   {96, 64, 3, 0.252f},   {128, 64, 3, 0.319f},  {96, 128, 4, 0.437f},
    {128, 128, 4, 0.538f}, {96, 192, 4, 0.574f},  {128, 192, 3, 0.775f}, {128, 256, 3, 0.851f},
    {256, 256, 2, 1.569f}, {256, 320, 2, 1.808f},
};
constexpr int kPlTileCount = sizeof(kPlTiles) / sizeof(kPlTiles[0]);
constexpr int32_t kPlMaxSplits = 4;
constexpr int32_t kPlUnits = 256;  // compute units

// Whether every one of `splits` slices (slice s: chunks [s C / S, (s + 1) C / S))
// fills a ring of `stages`.
bool slices_fill(int32_t chunks, int32_t splits, int32_t stages) { return chunks / splits >= stages; }

// Tile (an index of kPlTiles, -1 if none fits) and cost of a call over w_rows
// weight rows in `splits` slices.
int32_t pick_tile(int32_t m, int32_t w_rows, int32_t chunks, int32_t splits, float &cost) {
  int32_t best = -1;
  cost = 0.f;
  for (int32_t t = 0; t < kPlTileCount; ++t) {
    const PlTile &tile = kPlTiles[t];
    if (!slices_fill(chunks, splits, tile.stages)) continue;
    const int64_t groups = static_cast<int64_t>((m + tile.bm - 1) / tile.bm) *
                           ((w_rows + tile.bn - 1) / tile.bn) * splits;
    float c = 5.f + static_cast<float>((groups + kPlUnits - 1) / kPlUnits) *
                        static_cast<float>((chunks + splits - 1) / splits) * tile.chunk_us;
    if (splits > 1)
      c += 0.8f + static_cast<float>(splits) * static_cast<float>(m) * static_cast<float>(w_rows) * 4.f / 8e6f;
    if (best < 0 || c < cost) {
      best = t;
      cost = c;
    }
  }
  return best;
}

template <typename T, int EPI>
int32_t launch_prefill_linear_tile(const PlParams &p, int32_t tile, hipStream_t stream) {
  switch (tile) {
    case 0: return launch_prefill_linear<T, 64, 64, 2, 2, 4, EPI>(p, stream);
    case 1: return launch_prefill_linear<T, 96, 64, 2, 2, 3, EPI>(p, stream);
    case 2: return launch_prefill_linear<T, 128, 64, 2, 2, 3, EPI>(p, stream);
    case 3: return launch_prefill_linear<T, 96, 128, 2, 2, 4, EPI>(p, stream);
    case 4: return launch_prefill_linear<T, 128, 128, 2, 2, 4, EPI>(p, stream);
    case 5: return launch_prefill_linear<T, 96, 192, 2, 2, 4, EPI>(p, stream);
    case 6: return launch_prefill_linear<T, 128, 192, 2, 2, 3, EPI>(p, stream);
    case 7: return launch_prefill_linear<T, 128, 256, 2, 4, 3, EPI>(p, stream);
    case 8: return launch_prefill_linear<T, 256, 256, 2, 4, 2, EPI>(p, stream);
    default: return launch_prefill_linear<T, 256, 320, 4, 2, 2, EPI>(p, stream);
  }
}

template <typename T>
int32_t launch_prefill_linear_out(const PlParams &p, bool swiglu, int32_t tile, hipStream_t stream) {
  if (swiglu) return launch_prefill_linear_tile<T, kOutSwiglu>(p, tile, stream);
  if (p.partials) return launch_prefill_linear_tile<T, kOutPartials>(p, tile, stream);
  return launch_prefill_linear_tile<T, kOutRounded>(p, tile, stream);
}

}  // namespace
}  // namespace tf

extern "C" int32_t tf_prefill_linear_splits(int32_t m, int32_t n, int32_t k) {
  using namespace tf;
  if (m <= 0 || n <= 0 || k <= 0 || k % kPlChunk != 0) return 0;
  int32_t best = 0;
  float best_cost = 0.f;
  for (int32_t splits = 1; splits <= kPlMaxSplits; ++splits) {
    float cost;
    if (pick_tile(m, n, k / kPlChunk, splits, cost) < 0) continue;
    if (best == 0 || cost < best_cost) {
      best = splits;
      best_cost = cost;
    }
  }
  return best;
}

extern "C" int32_t tf_prefill_linear(const void *x, int64_t x_row_stride, const void *weight,
                                     int64_t weight_row_stride, void *y, int64_t y_row_stride,
                                     float *partials, int32_t m, int32_t n, int32_t k,
                                     int32_t splits, int32_t swiglu, int32_t tile, int32_t dtype,
                                     void *stream) {
  using namespace tf;
  clear_error();
  if (dtype != TF_DTYPE_FLOAT16 && dtype != TF_DTYPE_BFLOAT16)
    return fail(TF_ERROR_UNSUPPORTED, "prefill_linear supports fp16 and bf16");
  if (m < 0 || n < 0 || k < 0) return fail(TF_ERROR_INVALID_ARGUMENT, "sizes must be non-negative");
  if (k == 0 || k % kPlChunk != 0)
    return fail(TF_ERROR_UNSUPPORTED, "prefill_linear needs K to be a positive multiple of 64");
  if (n % 4 != 0) return fail(TF_ERROR_UNSUPPORTED, "prefill_linear needs N to be a multiple of 4");
  if (splits < 1 || splits > k / kPlChunk || splits > 64)
    return fail(TF_ERROR_INVALID_ARGUMENT, "splits must be in [1, min(64, K / 64)]");
  if (!partials && splits != 1)
    return fail(TF_ERROR_INVALID_ARGUMENT, "several K slices need a partials buffer");
  if (partials && swiglu) return fail(TF_ERROR_UNSUPPORTED, "the SwiGLU form has no K slices");
  if (x_row_stride < k || weight_row_stride < k || (!partials && y_row_stride < n))
    return fail(TF_ERROR_INVALID_ARGUMENT, "row strides are shorter than the rows");
  if (tile < 0 || tile > kPlTileCount) return fail(TF_ERROR_INVALID_ARGUMENT, "unknown tile");
  if (m == 0 || n == 0) return TF_SUCCESS;
  if (!x || !weight || (!partials && !y))
    return fail(TF_ERROR_INVALID_ARGUMENT, "null tensor pointer");
  const uintptr_t rows = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(weight) |
                         reinterpret_cast<uintptr_t>(partials) |
                         static_cast<uintptr_t>(x_row_stride * 2) |
                         static_cast<uintptr_t>(weight_row_stride * 2);
  if (rows % 16 != 0 ||
      (!partials && (reinterpret_cast<uintptr_t>(y) | static_cast<uintptr_t>(y_row_stride * 2)) % 8 != 0))
    return fail(TF_ERROR_UNSUPPORTED,
                "prefill_linear needs 16-byte aligned x, weight and partials rows and 8-byte aligned y rows");
  // A lane addresses its row of a tile (at most 320 rows) with 32 bits.
  if (x_row_stride > (1 << 21) || weight_row_stride > (1 << 21) || k > (1 << 21) || n > (1 << 27) || m > (1 << 27))
    return fail(TF_ERROR_UNSUPPORTED, "prefill_linear rows are too long");
  const int32_t chunks = k / kPlChunk;
  const int32_t w_rows = swiglu ? 2 * n : n;
  int32_t chosen = tile - 1;
  if (tile == 0) {
    float cost;
    chosen = pick_tile(m, w_rows, chunks, splits, cost);
  }
  if (chosen < 0 || !slices_fill(chunks, splits, kPlTiles[chosen].stages))
    return fail(TF_ERROR_UNSUPPORTED, "prefill_linear needs K slices that fill its load ring");
  const int64_t groups = static_cast<int64_t>((m + kPlTiles[chosen].bm - 1) / kPlTiles[chosen].bm) *
                         ((w_rows + kPlTiles[chosen].bn - 1) / kPlTiles[chosen].bn) * splits;
  if (groups > 0x7fffff) return fail(TF_ERROR_UNSUPPORTED, "grid too large");
  PlParams p;
  p.x = x;
  p.w = weight;
  p.y = y;
  p.partials = partials;
  p.x_stride = x_row_stride;
  p.w_stride = weight_row_stride;
  p.y_stride = y_row_stride;
  p.m = m;
  p.n = n;
  p.k_chunks = chunks;
  p.tiles_m = p.tiles_n = 0;
  p.splits = splits;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == TF_DTYPE_BFLOAT16)
    return launch_prefill_linear_out<__bf16>(p, swiglu != 0, chosen, s);
  return launch_prefill_linear_out<_Float16>(p, swiglu != 0, chosen, s);
}
