// Causal GQA attention of packed prompts (prefill) on MFMA.
//
// The prompts of a prefill batch are packed into one token stream with no
// padding: token rows q [T, Hq * D], k [T, Hkv * D], v [T, Hkv * D] (row
// strides in elements, so v can be a column slice of the fused QKV rows).
// A work item is a 64-token query block of one prompt: its tokens
// [b0, b0 + 64) attend causally to the prompt's tokens [s, min(b0 + 64, e)),
// where [s, e) is the prompt's token range.  The host lists the blocks
// (block start, prompt start, prompt end), heaviest first.
//
// One workgroup of four wavefronts per (block, kv head, group of QH query
// heads of that kv head); wavefront w serves the block's 16-token tile
// [b0 + 16 w, +16) for the QH heads.  The keys are walked in 64-token
// chunks that direct-to-LDS loads bring into a ring of buffers (no staging
// registers or LDS stores), so a chunk's bytes serve 64 query tokens x QH
// heads and there is one barrier per 64 keys.
//   scores  v_mfma_f32_16x16x32 with the K chunk (16 tokens x 32 dims per
//           tile, read from LDS in the A-operand layout) and the head's
//           query tile as the B operand: lane (l16, q4), register r holds
//           S[key token t0 + 16 j + 4 q4 + r][query token i0 + l16], so the
//           online softmax of a query token is lane-local across q4 lanes;
//   P.V     P converted to the storage type is already the B operand; V^T
//           (A operand) is read from the chunk staged token-major with
//           ds_read_b64_tr_b16, once per chunk for all QH heads.
// The kernel is bound by the softmax's vector work, not by the products: per
// 16 x 32 scores of a wavefront 8 products (128 cycles at D 64) against some
// 40 vector instructions, 8 of them exponentials.  So the running maximum is
// not looked for: the weights are computed against the last one, and only
// where one of them exceeds 2^8 (which the maximum over the weights, needing
// no NaN quieting, shows) is the maximum raised and the chunk's weights
// computed again.  Softmax in base 2, fp32 accumulation, one rounding of the
// output.
//
// MI355X: 19 prompts of 8,058 tokens at 32/4 heads, D 64 92.5 -> 52.5 us (673
// TFLOP/s of causal attention), 4096 + 2051 + 777 tokens at 32/8, D 128 311
// -> 193 us (917), one prompt of 271 9.9 -> 6.0 us, 64 prompts of 20 7.3 -> 7.6,
// against 32-key chunks staged through registers with the maximum looked for in
// every chunk.
//
// Reference semantics: the causal scaled-dot-product attention of prefill,
// tensorforge/runtime/prefill.py:84-88 (causal mask over the padded
// prompts) and :109-118 (torch SDPA with enable_gqa), here without padding.
#include <type_traits>

#include "tf_common.hpp"

namespace tf {
namespace {

constexpr float kPrefillLog2e = 1.4426950408889634f;
constexpr float kPrefillNegInf = -__builtin_huge_valf();
constexpr int kPrefillTile = 16;   // query tokens per wavefront
constexpr int kPrefillWaves = 4;   // wavefronts per workgroup
constexpr int kPrefillBlock = kPrefillTile * kPrefillWaves;  // query tokens per work item
constexpr int kPrefillChunk = 64;  // key tokens per LDS buffer
constexpr float kPrefillFloor = -3e38f;  // running maximum before the first key
constexpr float kPrefillMost = 256.f;    // weight that makes the maximum rise
constexpr int kPrefillXcds = 8;
// Workgroups from which a wavefront serves two heads.
constexpr int64_t prefill_pairs(int head_dim) { return head_dim >= 128 ? 500 : (head_dim >= 64 ? 600 : 1200); }

template <typename T>
struct PrefillMfma;

template <>
struct PrefillMfma<__bf16> {
  typedef __bf16 vec8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ f32x4 mma(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};

template <>
struct PrefillMfma<_Float16> {
  typedef _Float16 vec8 __attribute__((ext_vector_type(8)));
  static __device__ __forceinline__ f32x4 mma(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

typedef short pf_i16x4 __attribute__((ext_vector_type(4)));
typedef short pf_i16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) pf_i16x4 pf_lds_i16x4;

struct PrefillParams {
  const void *q;
  const void *k;
  const void *v;
  void *out;
  const int32_t *tiles;  // [ntiles][3]: query start, prompt start, prompt end
  int64_t q_stride;
  int64_t k_stride;
  int64_t v_stride;
  int64_t out_stride;
  int32_t query_heads;
  int32_t kv_heads;
  int32_t group;
  float scale_log2;
};

// This wavefront's loads have landed, its LDS reads are done, and so for every
// wavefront of the workgroup.
__device__ __forceinline__ void prefill_wait_barrier() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" : : : "memory");
}

template <typename T, int D, int QH>
__global__ void __launch_bounds__(64 * kPrefillWaves)
prefill_attention_kernel(PrefillParams p) {
  using M = PrefillMfma<T>;
  using vec8 = typename M::vec8;
  constexpr int KS = D / 32;
  constexpr int NB = D / 16;
  // LDS rows are 2 D bytes with their 16-byte pieces permuted: piece q of row
  // r sits at q ^ swizzle(r), which changes every R = 128 / D rows (one
  // 256-byte span of the 64 banks), so the 16 lanes of an operand read (rows
  // 16 j .. +15, one piece each) cover the banks once.
  constexpr int kPieces = D / 8;
  constexpr int kRowsPer256 = D >= 128 ? 1 : 128 / D;
  constexpr int kRowBytes = 2 * D;
  constexpr int kBufBytes = kPrefillChunk * kRowBytes;  // K or V of a chunk
  constexpr int kSub = D <= 64 ? 64 : 32;  // keys whose operands are held at once
  __shared__ __attribute__((aligned(1024))) unsigned char ring[2][2][kBufBytes];
  auto swizzle = [](int row) { return (row / kRowsPer256) & (kPieces - 1); };

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int l16 = lane & 15;
  const int q4 = lane >> 4;
  // The blocks come heaviest first, every head group of a block before the
  // next block.  The dies are dealt workgroups round-robin; where the head
  // groups are a multiple of the dies, each die takes neighbouring groups,
  // which share a kv head's K and V in its L2.
  const int32_t groups = p.group / QH;
  const int32_t per_block = p.kv_heads * groups;
  const int32_t block = static_cast<int32_t>(blockIdx.x) / per_block;
  int32_t hg = static_cast<int32_t>(blockIdx.x) - block * per_block;
  if (per_block % kPrefillXcds == 0)
    hg = (hg % kPrefillXcds) * (per_block / kPrefillXcds) + hg / kPrefillXcds;
  const int32_t *tile = p.tiles + 3 * static_cast<int64_t>(block);
  const int32_t b0 = tile[0];
  const int32_t s = tile[1];
  const int32_t e = tile[2];
  const int32_t kvh = hg / groups;
  const int32_t h0 = kvh * p.group + (hg - kvh * groups) * QH;
  // Keys of the block [s, kend_blk); this wavefront's tile [i0, i0 + 16)
  // needs [s, kend) (none when the tile starts past the prompt).
  const int32_t kend_blk = min(b0 + kPrefillBlock, e);
  const int32_t i0 = b0 + kPrefillTile * wave;
  const int32_t kend = min(i0 + kPrefillTile, e);
  const int32_t qt = i0 + l16;  // this lane's query token (column)
  const bool q_ok = qt < e;
  const int32_t nch = (kend_blk - s + kPrefillChunk - 1) / kPrefillChunk;
  const int32_t my_nch = i0 < e ? (kend - s + kPrefillChunk - 1) / kPrefillChunk : 0;

  // Chunk loads: an instruction fills 1024 bytes (kRowsPerLoad rows) of a
  // buffer; this wavefront's first half are of K, the rest of V.  Rows past
  // the block's keys read its last key: their scores are masked.
  constexpr int kLoads = D / 16;  // per wavefront and chunk
  constexpr int kRowsPerLoad = 1024 / kRowBytes;
  const int lrow = lane / kPieces;
  const int64_t strides[2] = {p.k_stride, p.v_stride};
  const unsigned char *bases[2];
  bases[0] = reinterpret_cast<const unsigned char *>(static_cast<const T *>(p.k) +
                                                     static_cast<int64_t>(s) * p.k_stride + static_cast<int64_t>(kvh) * D);
  bases[1] = reinterpret_cast<const unsigned char *>(static_cast<const T *>(p.v) +
                                                     static_cast<int64_t>(s) * p.v_stride + static_cast<int64_t>(kvh) * D);
  int64_t row_off[kLoads];  // bytes of this lane's piece from the chunk's first row
  auto offset_of = [&](int i, int32_t last) {
    const int row = kRowsPerLoad * (wave + kPrefillWaves * (i % (kLoads / 2))) + lrow;
    const int piece = (lane & (kPieces - 1)) ^ swizzle(row);
    return (static_cast<int64_t>(min(row, last)) * strides[i / (kLoads / 2)]) * 2 + 16 * piece;
  };
#pragma unroll
  for (int i = 0; i < kLoads; ++i) row_off[i] = offset_of(i, kPrefillChunk);
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) unsigned char *)&ring[0][0][0]));
  auto load_chunk = [&](int32_t c, int32_t stage) {
    const int32_t last = kend_blk - s - kPrefillChunk * c - 1;  // last valid row of the chunk
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int kv = i / (kLoads / 2);
      const unsigned char *from = bases[kv] + static_cast<int64_t>(kPrefillChunk * c) * strides[kv] * 2;
      int64_t off = row_off[i];
      if (last < kPrefillChunk - 1) off = offset_of(i, last);  // uniform
      const uint32_t at = lds0 + static_cast<uint32_t>((2 * stage + kv) * kBufBytes) +
                          1024u * static_cast<uint32_t>(wave + kPrefillWaves * (i % (kLoads / 2)));
      load_lds16(from + off, __builtin_amdgcn_readfirstlane(at));
    }
  };
  load_chunk(0, 0);

  vec8 qf[QH][KS];  // B operand: q[token i0 + l16][head h0 + hq][32 ks + 8 q4 .. +8]
  {
    const T *qrow = static_cast<const T *>(p.q) + static_cast<int64_t>(q_ok ? qt : s) * p.q_stride;
#pragma unroll
    for (int hq = 0; hq < QH; ++hq)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const vec8 x = *reinterpret_cast<const vec8 *>(qrow + static_cast<int64_t>(h0 + hq) * D + 32 * ks + 8 * q4);
        qf[hq][ks] = q_ok ? x : vec8{};
      }
  }
  // LDS offsets of this lane's operand reads within a buffer (rows 16 apart
  // share their permutation).
  int k_at[KS], v_at[NB];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) k_at[ks] = l16 * kRowBytes + 16 * ((4 * ks + q4) ^ swizzle(l16));
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    const int row = 4 * q4 + (l16 >> 2);
    v_at[n] = row * kRowBytes + 16 * ((2 * n + ((l16 & 3) >> 1)) ^ swizzle(row)) + 8 * (l16 & 1);
  }

  f32x4 acc[QH][NB];
  float m_run[QH], l_run[QH];
#pragma unroll
  for (int hq = 0; hq < QH; ++hq) {
    m_run[hq] = kPrefillFloor;
    l_run[hq] = 0.f;
#pragma unroll
    for (int n = 0; n < NB; ++n) acc[hq][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // Keys [t0 + k0, t0 + k0 + KEYS) of the chunk at t0.
  auto compute = [&](int32_t t0, const unsigned char *kb, const unsigned char *vb, int k0, auto keys_tag) {
    constexpr int KEYS = decltype(keys_tag)::value;
    constexpr int J = KEYS / 16;
    vec8 kf[J][KS];
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        kf[j][ks] = *reinterpret_cast<const vec8 *>(kb + k_at[ks] + (k0 + 16 * j) * kRowBytes);
    // Causal mask: needed when some key of the step lies past the tile's
    // first query token (a query's own token bounds its keys in the prompt).
    const bool masked = t0 + k0 + KEYS - 1 > i0;
    const int32_t limit = qt - t0 - k0 - 4 * q4;  // key 16 j + r (of q4 = 0) is seen up to this
    vec8 pf[QH][J / 2];
    // Every head's scores and weights before any of the rare paths below, so
    // the heads' products and exponentials interleave.
    float sc[QH][4 * J], pr[QH][4 * J];
#pragma unroll
    for (int hq = 0; hq < QH; ++hq)
#pragma unroll
      for (int j = 0; j < J; ++j) {
        f32x4 acc_s = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) acc_s = M::mma(kf[j][ks], qf[hq][ks], acc_s);
#pragma unroll
        for (int r = 0; r < 4; ++r) sc[hq][4 * j + r] = acc_s[r];
      }
    if (masked) {
      int32_t seen = limit;
      asm volatile("" : "+v"(seen));  // keeps the comparisons inside the branch
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int hq = 0; hq < QH; ++hq)
            if (16 * j + r > seen) sc[hq][4 * j + r] = kPrefillNegInf;
    }
    auto weights = [&](int hq) {
#pragma unroll
      for (int i = 0; i < 4 * J; ++i)
        pr[hq][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[hq][i], p.scale_log2, -m_run[hq]));
    };
    bool raise = t0 + k0 == s;  // uniform; the first keys raise the maxima in any case
    if (!raise) {
      float top = 0.f;
#pragma unroll
      for (int hq = 0; hq < QH; ++hq) {
        weights(hq);
#pragma unroll
        for (int i = 0; i < 4 * J; i += 2) top = fmaxf(fmaxf(pr[hq][i], pr[hq][i + 1]), top);
      }
      raise = __ballot(top > kPrefillMost) != 0;
    }
    if (raise) {
#pragma unroll
      for (int hq = 0; hq < QH; ++hq) {
        float mx = sc[hq][0] * p.scale_log2;
#pragma unroll
        for (int i = 1; i < 4 * J; ++i) mx = fmaxf(mx, sc[hq][i] * p.scale_log2);
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float m_new = fmaxf(m_run[hq], mx);
        const float alpha = __builtin_amdgcn_exp2f(m_run[hq] - m_new);
        m_run[hq] = m_new;
        l_run[hq] *= alpha;
#pragma unroll
        for (int n = 0; n < NB; ++n) acc[hq][n] *= alpha;
        weights(hq);
      }
    }
#pragma unroll
    for (int hq = 0; hq < QH; ++hq) {
      float sum[4] = {pr[hq][0], pr[hq][1], pr[hq][2], pr[hq][3]};
#pragma unroll
      for (int i = 0; i < 4 * J; ++i) {
        if (i >= 4) sum[i & 3] += pr[hq][i];
        pf[hq][i >> 3][i & 7] = static_cast<T>(pr[hq][i]);
      }
      l_run[hq] += (sum[0] + sum[1]) + (sum[2] + sum[3]);
    }
#pragma unroll
    for (int h = 0; h < J / 2; ++h) {
      // A step of 32 keys past the tile's own is left out: all its weights
      // are 0, but 0 times a value that is not finite is not.
      if (h > 0 && t0 + k0 + 32 * h >= kend) break;  // wavefront-uniform
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        const unsigned char *rd = vb + v_at[n] + (k0 + 32 * h) * kRowBytes;
        const pf_i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((pf_lds_i16x4 *)rd);
        const pf_i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((pf_lds_i16x4 *)(rd + 16 * kRowBytes));
        const vec8 vt = __builtin_bit_cast(vec8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
        for (int hq = 0; hq < QH; ++hq) acc[hq][n] = M::mma(vt, pf[hq][h], acc[hq][n]);
      }
    }
  };

  // Chunk c waits for its loads; past the barrier every wavefront is done with
  // chunk c - 1, whose buffer takes chunk c + 1.
  using Keys32 = std::integral_constant<int, 32>;
  using Keys64 = std::integral_constant<int, 64>;
  for (int32_t c = 0; c < nch; ++c) {
    prefill_wait_barrier();
    if (c + 1 < nch) load_chunk(c + 1, (c + 1) & 1);
    if (c >= my_nch) continue;  // wavefront-uniform, as all below
    const unsigned char *kb = ring[c & 1][0];
    const unsigned char *vb = ring[c & 1][1];
    const int32_t t0 = s + kPrefillChunk * c;
    const bool whole = kend - t0 > 32;  // the second half has keys of the tile
    if constexpr (kSub == 32) {
      compute(t0, kb, vb, 0, Keys32{});
      if (whole) compute(t0, kb, vb, 32, Keys32{});
    } else if constexpr (QH > 1) {
      compute(t0, kb, vb, 0, Keys64{});
    } else {
      // A form for half a chunk: a third of a short prompt's work.  With
      // several heads its registers cost more (8,058 tokens at 32/4 heads, D
      // 64: 57 -> 64 us).
      if (whole)
        compute(t0, kb, vb, 0, Keys64{});
      else
        compute(t0, kb, vb, 0, Keys32{});
    }
  }

  // Lane-partial sums -> per-column sums; write the query tokens of the prompt.
  if (!q_ok) return;
  T *orow = static_cast<T *>(p.out) + static_cast<int64_t>(qt) * p.out_stride;
  typedef T t4 __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int hq = 0; hq < QH; ++hq) {
    float l = l_run[hq];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    // A query sees a key, so l is 0 only where every score is -inf: then 0 / 0,
    // the NaN of a softmax over nothing.
    const float inv = 1.f / l;
    T *dst = orow + static_cast<int64_t>(h0 + hq) * D;
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      const t4 o = {from_float<T>(acc[hq][n][0] * inv), from_float<T>(acc[hq][n][1] * inv),
                    from_float<T>(acc[hq][n][2] * inv), from_float<T>(acc[hq][n][3] * inv)};
      *reinterpret_cast<t4 *>(dst + 16 * n + 4 * q4) = o;
    }
  }
}

template <typename T, int D, int QH>
int32_t launch_prefill(const PrefillParams &p, int32_t ntiles, hipStream_t stream) {
  // A launch counts its threads in 32 bits.
  const int64_t grid = static_cast<int64_t>(ntiles) * p.kv_heads * (p.group / QH);
  if (grid * (64 * kPrefillWaves) > 0xffffffffll) return fail(TF_ERROR_UNSUPPORTED, "grid too large");
  hipLaunchKernelGGL((prefill_attention_kernel<T, D, QH>), dim3(static_cast<unsigned>(grid)),
                     dim3(64 * kPrefillWaves), 0, stream, p);
  return check_launch("prefill_attention");
}

template <typename T, int D>
int32_t launch_prefill_qh(const PrefillParams &p, int32_t ntiles, int32_t heads_per_wave,
                       hipStream_t stream) {
  // Query heads per wavefront (a power of two dividing the group): as asked,
  // else one where two would leave fewer than prefill_pairs workgroups -- a
  // call then waits for its longest chain of chunks, which one head shortens
  // -- and two otherwise, which read each chunk's operands half as often.
  // MI355X, us with one / two heads: D 64 at 16/1 heads 4096 tokens (512
  // pairs) 61.9 / 65.6, 19 prompts of 8,058 tokens at 32/4 (2176) 61.3 / 52.8;
  // D 128 at 32/8 1000 tokens (256) 22.1 / 26.0, at 16/2 8 x 500 (512) 21.2 /
  // 19.7; D 32 at 8/2 the 8,058 tokens (544) 20.6 / 25.4, 128 x 130 tokens
  // (1536) 16.3 / 11.0.  At most 4 at head_dim 128, for registers.
  constexpr int kMax = D >= 128 ? 4 : 8;
  const int64_t pairs = static_cast<int64_t>(ntiles) * p.kv_heads * ((p.group + 1) / 2);
  int32_t qh = heads_per_wave > 0 ? heads_per_wave : (pairs >= prefill_pairs(D) ? 2 : 1);
  if (qh > kMax) qh = kMax;
  if (qh > p.group) qh = p.group;
  switch (qh) {
    case 1: return launch_prefill<T, D, 1>(p, ntiles, stream);
    case 2: return launch_prefill<T, D, 2>(p, ntiles, stream);
    case 4: return launch_prefill<T, D, 4>(p, ntiles, stream);
    default: return launch_prefill<T, D, kMax>(p, ntiles, stream);
  }
}

template <typename T>
int32_t launch_prefill_dim(const PrefillParams &p, int32_t head_dim, int32_t ntiles,
                           int32_t heads_per_wave, hipStream_t stream) {
  switch (head_dim) {
    case 32: return launch_prefill_qh<T, 32>(p, ntiles, heads_per_wave, stream);
    case 64: return launch_prefill_qh<T, 64>(p, ntiles, heads_per_wave, stream);
    default: return launch_prefill_qh<T, 128>(p, ntiles, heads_per_wave, stream);
  }
}

}  // namespace
}  // namespace tf

extern "C" int32_t tf_prefill_attention(const void *q, int64_t q_row_stride, const void *k,
                                        int64_t k_row_stride, const void *v,
                                        int64_t v_row_stride, void *output,
                                        int64_t output_row_stride, const int32_t *tiles,
                                        int32_t num_tiles, int32_t query_heads, int32_t kv_heads,
                                        int32_t head_dim, float scale,
                                        int32_t heads_per_wave, int32_t dtype, void *stream) {
  using namespace tf;
  clear_error();
  if (dtype != TF_DTYPE_FLOAT16 && dtype != TF_DTYPE_BFLOAT16)
    return fail(TF_ERROR_UNSUPPORTED, "prefill attention supports fp16 and bf16");
  if (head_dim != 32 && head_dim != 64 && head_dim != 128)
    return fail(TF_ERROR_UNSUPPORTED, "prefill attention supports head_dim 32, 64 and 128");
  if (query_heads <= 0 || kv_heads <= 0 || query_heads % kv_heads != 0)
    return fail(TF_ERROR_INVALID_ARGUMENT, "query heads must be a positive multiple of kv heads");
  const int32_t group = query_heads / kv_heads;
  if (group > 16 || (group & (group - 1)) != 0)
    return fail(TF_ERROR_UNSUPPORTED, "prefill attention supports groups of 1, 2, 4, 8 or 16");
  if (heads_per_wave < 0 || heads_per_wave > 8 || (heads_per_wave & (heads_per_wave - 1)) != 0)
    return fail(TF_ERROR_INVALID_ARGUMENT, "heads_per_wave must be 0 or a power of two <= 8");
  if (num_tiles < 0 || num_tiles > 0x7fffffff / 3)
    return fail(TF_ERROR_INVALID_ARGUMENT, "invalid tile count");
  if (q_row_stride < static_cast<int64_t>(query_heads) * head_dim ||
      output_row_stride < static_cast<int64_t>(query_heads) * head_dim ||
      k_row_stride < static_cast<int64_t>(kv_heads) * head_dim ||
      v_row_stride < static_cast<int64_t>(kv_heads) * head_dim)
    return fail(TF_ERROR_INVALID_ARGUMENT, "row strides are shorter than the rows");
  if (num_tiles == 0) return TF_SUCCESS;
  if (!q || !k || !v || !output || !tiles)
    return fail(TF_ERROR_INVALID_ARGUMENT, "null tensor pointer");
  const uintptr_t align = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) |
                          reinterpret_cast<uintptr_t>(v) | reinterpret_cast<uintptr_t>(output) |
                          static_cast<uintptr_t>(q_row_stride * 2) |
                          static_cast<uintptr_t>(k_row_stride * 2) |
                          static_cast<uintptr_t>(v_row_stride * 2) |
                          static_cast<uintptr_t>(output_row_stride * 2);
  if (align % 16 != 0)
    return fail(TF_ERROR_UNSUPPORTED, "prefill attention needs 16-byte aligned rows");
  if (static_cast<int64_t>(kv_heads) * group > 65535) return fail(TF_ERROR_UNSUPPORTED, "grid too large");
  PrefillParams p;
  p.q = q;
  p.k = k;
  p.v = v;
  p.out = output;
  p.tiles = tiles;
  p.q_stride = q_row_stride;
  p.k_stride = k_row_stride;
  p.v_stride = v_row_stride;
  p.out_stride = output_row_stride;
  p.query_heads = query_heads;
  p.kv_heads = kv_heads;
  p.group = group;
  p.scale_log2 = scale * kPrefillLog2e;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == TF_DTYPE_BFLOAT16)
    return launch_prefill_dim<__bf16>(p, head_dim, num_tiles, heads_per_wave, s);
  return launch_prefill_dim<_Float16>(p, head_dim, num_tiles, heads_per_wave, s);
}
