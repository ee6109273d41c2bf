// Fused RoPE + paged KV append: one launch per layer turns the fused QKV
// projection of a batch of tokens (one per decode lane, or a packed set of
// prompts) into the rotated query and writes the rotated key and the value
// of every active token into its cache page; optionally also the rotated key
// densely (prefill attention reads it).
//
// Input row b of `qkv` holds [q heads | k heads | v heads], head_dim each.
// RoPE uses the half-split rotation with per-dimension cos/sin tables
// indexed by the lane's position:
//   out[j]     = x[j] cos[j]     - x[j+D/2] sin[j]
//   out[j+D/2] = x[j+D/2] cos[j+D/2] + x[j] sin[j+D/2]        (j < D/2)
// computed in fp32 and rounded once to the storage type.
//
// Reference semantics this one launch replaces:
//   RoPE on q and k       tensorforge/model/layers.py:33-69
//                         (apply_batched_rotary_embedding, :57-69)
//   cache write           tensorforge/runtime/decode_bucket.py:448-458 ->
//                         tensorforge/kernels/triton_cache.py:23-63
//                         (masked lanes store nothing)
//   the .contiguous() copies of q, k and v at decode_bucket.py:449-450, 460
//   prefill RoPE + append runtime/prefill.py:99-115 (apply_rotary_embedding,
//                         then one write_layer per request)
#include <type_traits>

#include "tf_common.hpp"

namespace tf {
namespace {

// One workgroup per lane.  Threads walk the (Hq + Hkv) * D/2 rotation pairs
// (consecutive threads take consecutive j, so loads and stores coalesce),
// then the Hkv * D value elements.
template <typename T>
__global__ void __launch_bounds__(256)
rope_kv_append_kernel(const T *__restrict__ qkv, int64_t row_stride,
                      const int64_t *__restrict__ positions, const T *__restrict__ cos_table,
                      const T *__restrict__ sin_table, int32_t table_rows,
                      T *__restrict__ query_out, T *__restrict__ key_out,
                      T *__restrict__ key_cache,
                      T *__restrict__ value_cache, const int32_t *__restrict__ physical_blocks,
                      const int32_t *__restrict__ block_offsets,
                      const int32_t *__restrict__ active_mask, int32_t query_heads,
                      int32_t kv_heads, int32_t head_dim, int32_t num_blocks,
                      int32_t block_size) {
  const int64_t b = blockIdx.x;
  const int32_t half = head_dim >> 1;
  int64_t pos = positions[b];
  // The host validates positions; clamping keeps a bad one inside the table.
  pos = pos < 0 ? 0 : (pos >= table_rows ? table_rows - 1 : pos);
  const T *row = qkv + b * row_stride;
  const T *cs = cos_table + pos * head_dim;
  const T *sn = sin_table + pos * head_dim;
  const int32_t page = physical_blocks[b];
  const int32_t offset = block_offsets[b];
  const bool store = active_mask[b] != 0 && page >= 0 && page < num_blocks && offset >= 0 &&
                     offset < block_size;
  const int64_t row_elems = static_cast<int64_t>(kv_heads) * head_dim;
  const int64_t slot = static_cast<int64_t>(page) * block_size + offset;
  T *q_row = query_out + b * static_cast<int64_t>(query_heads) * head_dim;

  const int32_t pairs = (query_heads + kv_heads) * half;
  for (int32_t i = threadIdx.x; i < pairs; i += blockDim.x) {
    const int32_t head = i / half;
    const int32_t j = i - head * half;
    const T *src = row + static_cast<int64_t>(head) * head_dim;
    const float x1 = to_float(src[j]);
    const float x2 = to_float(src[j + half]);
    const float o1 = rope_lo(x1, x2, to_float(cs[j]), to_float(sn[j]));
    const float o2 = rope_hi(x1, x2, to_float(cs[j + half]), to_float(sn[j + half]));
    const T r1 = from_float<T>(o1);
    const T r2 = from_float<T>(o2);
    if (head < query_heads) {
      T *dst = q_row + static_cast<int64_t>(head) * head_dim;
      dst[j] = r1;
      dst[j + half] = r2;
    } else {
      const int64_t kh = static_cast<int64_t>(head - query_heads) * head_dim;
      if (store) {
        T *dst = key_cache + slot * row_elems + kh;
        dst[j] = r1;
        dst[j + half] = r2;
      }
      if (key_out) {
        T *dst = key_out + b * row_elems + kh;
        dst[j] = r1;
        dst[j + half] = r2;
      }
    }
  }
  if (store) {
    const T *v = row + static_cast<int64_t>(query_heads + kv_heads) * head_dim;
    T *dst = value_cache + slot * row_elems;
    for (int32_t i = threadIdx.x; i < row_elems; i += blockDim.x) dst[i] = v[i];
  }
}

// The same work in 16-byte vectors, for tables, rows and caches that allow
// them.  A thread owns one item of a token: VEC rotation pairs of a q or k
// head (the vectors at j and j + D/2), or two vectors of the value row.  The
// items of consecutive tokens are dealt to consecutive threads across the
// whole grid, so no lane idles at any head count.  PARTIALS reads the row
// from the fp32 slice sums of a K-split projection instead (planes of
// row_stride x batch floats), added in slice order and rounded once -- the
// projection's own rounding -- and then also writes the value rows densely.
//
// HBM-bound: 8,058 tokens at 32/4 heads, D 64, bf16 with the dense keys (87
// MB) took 23.5 us with 2-byte accesses and one workgroup per token.
template <typename T>
struct RopeParams {
  const T *qkv;
  const float *partials;
  int32_t splits;
  int64_t plane;
  int64_t row_stride;
  const int64_t *positions;
  const T *cos_table;
  const T *sin_table;
  int32_t table_rows;
  T *query_out;
  T *key_out;
  T *value_out;
  T *key_cache;
  T *value_cache;
  const int32_t *physical_blocks;
  const int32_t *block_offsets;
  const int32_t *active_mask;
  int32_t batch;
  int32_t query_heads;
  int32_t kv_heads;
  int32_t head_dim;
  int32_t num_blocks;
  int32_t block_size;
};

template <typename T, bool PARTIALS>
__global__ void __launch_bounds__(256)
rope_kv_append_vec_kernel(RopeParams<T> p) {
  constexpr int VEC = 16 / sizeof(T);
  struct alignas(16) Vec {
    T v[VEC];
  };
  const uint32_t half = static_cast<uint32_t>(p.head_dim) >> 1;
  const uint32_t pieces = half / VEC;  // items per head
  const uint32_t rotated = static_cast<uint32_t>(p.query_heads + p.kv_heads) * pieces;
  const uint32_t items = rotated + static_cast<uint32_t>(p.kv_heads) * pieces;
  const uint32_t at = blockIdx.x * 256u + threadIdx.x;
  const uint32_t b = at / items;
  if (b >= static_cast<uint32_t>(p.batch)) return;
  const uint32_t item = at - b * items;
  const int32_t page = p.physical_blocks[b];
  const int32_t offset = p.block_offsets[b];
  const bool store = p.active_mask[b] != 0 && page >= 0 && page < p.num_blocks && offset >= 0 &&
                     offset < p.block_size;
  const int64_t row_elems = static_cast<int64_t>(p.kv_heads) * p.head_dim;
  const int64_t slot = (static_cast<int64_t>(page) * p.block_size + offset) * row_elems;
  // VEC elements of the token's row.
  auto load = [&](uint32_t e) -> Vec {
    if constexpr (PARTIALS) {
      const float *src = p.partials + static_cast<int64_t>(b) * p.row_stride + e;
      float sum[VEC];
#pragma unroll
      for (int i = 0; i < VEC; ++i) sum[i] = 0.f;
      for (int32_t s = 0; s < p.splits; ++s) {
#pragma unroll
        for (int q = 0; q < VEC / 4; ++q) {
          const f32x4 x = *reinterpret_cast<const f32x4 *>(src + s * p.plane + 4 * q);
#pragma unroll
          for (int i = 0; i < 4; ++i) sum[4 * q + i] += x[i];
        }
      }
      Vec out;
#pragma unroll
      for (int i = 0; i < VEC; ++i) out.v[i] = from_float<T>(sum[i]);
      return out;
    } else {
      return *reinterpret_cast<const Vec *>(p.qkv + static_cast<int64_t>(b) * p.row_stride + e);
    }
  };
  if (item >= rotated) {
    const uint32_t e = (item - rotated) * 2 * VEC;  // of the value row
    const uint32_t first = static_cast<uint32_t>(p.query_heads + p.kv_heads) * p.head_dim + e;
    const Vec v0 = load(first), v1 = load(first + VEC);
    if (store) {
      *reinterpret_cast<Vec *>(p.value_cache + slot + e) = v0;
      *reinterpret_cast<Vec *>(p.value_cache + slot + e + VEC) = v1;
    }
    if (p.value_out) {
      T *dst = p.value_out + static_cast<int64_t>(b) * row_elems + e;
      *reinterpret_cast<Vec *>(dst) = v0;
      *reinterpret_cast<Vec *>(dst + VEC) = v1;
    }
    return;
  }
  int64_t pos = p.positions[b];
  // The host validates positions; clamping keeps a bad one inside the table.
  pos = pos < 0 ? 0 : (pos >= p.table_rows ? p.table_rows - 1 : pos);
  const uint32_t head = item / pieces;
  const uint32_t j = (item - head * pieces) * VEC;
  const uint32_t e = head * p.head_dim + j;
  const Vec x1 = load(e), x2 = load(e + half);
  const T *cs = p.cos_table + pos * p.head_dim + j;
  const T *sn = p.sin_table + pos * p.head_dim + j;
  const Vec c1 = *reinterpret_cast<const Vec *>(cs), c2 = *reinterpret_cast<const Vec *>(cs + half);
  const Vec s1 = *reinterpret_cast<const Vec *>(sn), s2 = *reinterpret_cast<const Vec *>(sn + half);
  Vec r1, r2;
#pragma unroll
  for (int i = 0; i < VEC; ++i) {
    const float a = to_float(x1.v[i]), c = to_float(x2.v[i]);
    r1.v[i] = from_float<T>(rope_lo(a, c, to_float(c1.v[i]), to_float(s1.v[i])));
    r2.v[i] = from_float<T>(rope_hi(a, c, to_float(c2.v[i]), to_float(s2.v[i])));
  }
  if (head < static_cast<uint32_t>(p.query_heads)) {
    T *dst = p.query_out + static_cast<int64_t>(b) * p.query_heads * p.head_dim + e;
    *reinterpret_cast<Vec *>(dst) = r1;
    *reinterpret_cast<Vec *>(dst + half) = r2;
    return;
  }
  const uint32_t ke = e - static_cast<uint32_t>(p.query_heads) * p.head_dim;
  if (store) {
    T *dst = p.key_cache + slot + ke;
    *reinterpret_cast<Vec *>(dst) = r1;
    *reinterpret_cast<Vec *>(dst + half) = r2;
  }
  if (p.key_out) {
    T *dst = p.key_out + static_cast<int64_t>(b) * row_elems + ke;
    *reinterpret_cast<Vec *>(dst) = r1;
    *reinterpret_cast<Vec *>(dst + half) = r2;
  }
}

// Whether every vector of the call starts on 16 bytes: head halves, rows,
// tables, caches and outputs; and the grid's thread index fits 32 bits.
template <typename T>
bool rope_vectors(const RopeParams<T> &p) {
  constexpr int VEC = 16 / sizeof(T);
  const int32_t half = p.head_dim / 2;
  uintptr_t at = reinterpret_cast<uintptr_t>(p.cos_table) | reinterpret_cast<uintptr_t>(p.sin_table) |
                 reinterpret_cast<uintptr_t>(p.query_out) | reinterpret_cast<uintptr_t>(p.key_out) |
                 reinterpret_cast<uintptr_t>(p.value_out) | reinterpret_cast<uintptr_t>(p.key_cache) |
                 reinterpret_cast<uintptr_t>(p.value_cache);
  at |= p.partials ? reinterpret_cast<uintptr_t>(p.partials) | static_cast<uintptr_t>(p.row_stride * 4)
                   : reinterpret_cast<uintptr_t>(p.qkv) | static_cast<uintptr_t>(p.row_stride * sizeof(T));
  const int64_t threads = static_cast<int64_t>(p.batch) * (p.query_heads + 2 * static_cast<int64_t>(p.kv_heads)) * half;
  return half % VEC == 0 && at % 16 == 0 && threads < (int64_t{1} << 31);
}

// A token that is one pass of a workgroup, few of them: the elementwise kernel
// reads its page, position and flags by scalar loads and divides by nothing
// (8/2 heads, D 32, bf16: 64 tokens 3.0 us against 3.5; 2048 tokens 4.3
// against 3.9; of several passes, 32/4 heads, D 64, 64 tokens 4.1 against 3.4).
template <typename T>
bool rope_narrow(const RopeParams<T> &p) {
  return p.batch <= 512 && (p.query_heads + p.kv_heads) * static_cast<int64_t>(p.head_dim / 2) <= 256;
}

template <typename T, bool PARTIALS>
void launch_rope_vec(const RopeParams<T> &p, hipStream_t stream) {
  constexpr int VEC = 16 / sizeof(T);
  const uint32_t items = static_cast<uint32_t>(p.query_heads + 2 * p.kv_heads) *
                         (static_cast<uint32_t>(p.head_dim) / (2 * VEC));
  const uint32_t blocks = (items * static_cast<uint32_t>(p.batch) + 255) / 256;
  hipLaunchKernelGGL((rope_kv_append_vec_kernel<T, PARTIALS>), dim3(blocks), dim3(256), 0, stream, p);
}

}  // namespace
}  // namespace tf

extern "C" int32_t tf_rope_kv_append(
    const void *qkv, int64_t qkv_row_stride, const int64_t *positions, const void *cos_table,
    const void *sin_table, int32_t table_rows, void *query_out, void *key_out, void *key_cache,
    void *value_cache, const int32_t *physical_blocks, const int32_t *block_offsets,
    const int32_t *active_mask, int32_t batch, int32_t query_heads, int32_t kv_heads,
    int32_t head_dim, int32_t num_blocks, int32_t block_size, int32_t dtype, void *stream) {
  using namespace tf;
  clear_error();
  if (!valid_dtype(dtype)) return fail(TF_ERROR_INVALID_ARGUMENT, "unsupported dtype code");
  if (batch < 0) return fail(TF_ERROR_INVALID_ARGUMENT, "batch must be non-negative");
  if (query_heads <= 0 || kv_heads <= 0 || head_dim <= 0 || (head_dim & 1) || num_blocks <= 0 ||
      block_size <= 0 || table_rows <= 0)
    return fail(TF_ERROR_INVALID_ARGUMENT,
                "heads, blocks and table rows must be positive and head_dim even");
  if (query_heads % kv_heads)
    return fail(TF_ERROR_INVALID_ARGUMENT, "query_heads must be a multiple of kv_heads");
  if (qkv_row_stride < static_cast<int64_t>(query_heads + 2 * kv_heads) * head_dim)
    return fail(TF_ERROR_INVALID_ARGUMENT, "qkv row stride is shorter than the q, k, v heads");
  if (batch == 0) return TF_SUCCESS;
  if (!qkv || !positions || !cos_table || !sin_table || !query_out || !key_cache || !value_cache ||
      !physical_blocks || !block_offsets || !active_mask)
    return fail(TF_ERROR_INVALID_ARGUMENT, "null tensor pointer");
  const dim3 grid(static_cast<unsigned>(batch));
  const dim3 block(256);
  hipStream_t s = static_cast<hipStream_t>(stream);
#define TF_ROPE_LAUNCH(T)                                                                     \
  do {                                                                                        \
    const RopeParams<T> p{static_cast<const T *>(qkv), nullptr, 0, 0, qkv_row_stride, positions, \
                          static_cast<const T *>(cos_table), static_cast<const T *>(sin_table),   \
                          table_rows, static_cast<T *>(query_out), static_cast<T *>(key_out),     \
                          nullptr, static_cast<T *>(key_cache), static_cast<T *>(value_cache),    \
                          physical_blocks, block_offsets, active_mask, batch, query_heads,        \
                          kv_heads, head_dim, num_blocks, block_size};                            \
    if (rope_vectors(p) && !rope_narrow(p)) {                                                 \
      launch_rope_vec<T, false>(p, s);                                                        \
      break;                                                                                  \
    }                                                                                         \
    hipLaunchKernelGGL((rope_kv_append_kernel<T>), grid, block, 0, s,                        \
                       p.qkv, qkv_row_stride, positions, p.cos_table, p.sin_table, table_rows, \
                       p.query_out, p.key_out, p.key_cache, p.value_cache, physical_blocks,   \
                       block_offsets, active_mask, query_heads, kv_heads, head_dim, num_blocks, \
                       block_size);                                                           \
  } while (0)
  switch (dtype) {
    case TF_DTYPE_FLOAT32: TF_ROPE_LAUNCH(float); break;
    case TF_DTYPE_FLOAT16: TF_ROPE_LAUNCH(_Float16); break;
    default: TF_ROPE_LAUNCH(__bf16); break;
  }
#undef TF_ROPE_LAUNCH
  return check_launch("rope_kv_append");
}

extern "C" int32_t tf_rope_kv_append_partials(
    const float *partials, int32_t splits, const int64_t *positions, const void *cos_table,
    const void *sin_table, int32_t table_rows, void *query_out, void *key_out, void *value_out,
    void *key_cache, void *value_cache, const int32_t *physical_blocks,
    const int32_t *block_offsets, const int32_t *active_mask, int32_t batch, int32_t query_heads,
    int32_t kv_heads, int32_t head_dim, int32_t num_blocks, int32_t block_size, int32_t dtype,
    void *stream) {
  using namespace tf;
  clear_error();
  if (dtype != TF_DTYPE_FLOAT16 && dtype != TF_DTYPE_BFLOAT16)
    return fail(TF_ERROR_UNSUPPORTED, "rope_kv_append_partials supports fp16 and bf16");
  if (batch < 0 || splits < 1) return fail(TF_ERROR_INVALID_ARGUMENT, "invalid sizes");
  if (query_heads <= 0 || kv_heads <= 0 || head_dim <= 0 || (head_dim & 1) || num_blocks <= 0 ||
      block_size <= 0 || table_rows <= 0)
    return fail(TF_ERROR_INVALID_ARGUMENT,
                "heads, blocks and table rows must be positive and head_dim even");
  if (query_heads % kv_heads)
    return fail(TF_ERROR_INVALID_ARGUMENT, "query_heads must be a multiple of kv_heads");
  if (batch == 0) return TF_SUCCESS;
  if (!partials || !positions || !cos_table || !sin_table || !query_out || !key_out || !value_out ||
      !key_cache || !value_cache || !physical_blocks || !block_offsets || !active_mask)
    return fail(TF_ERROR_INVALID_ARGUMENT, "null tensor pointer");
  const int64_t row = static_cast<int64_t>(query_heads + 2 * kv_heads) * head_dim;
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto launch = [&](auto *out) -> int32_t {
    using T = std::remove_pointer_t<decltype(out)>;
    const RopeParams<T> p{nullptr, partials, splits, row * batch, row, positions,
                          static_cast<const T *>(cos_table), static_cast<const T *>(sin_table),
                          table_rows, out, static_cast<T *>(key_out), static_cast<T *>(value_out),
                          static_cast<T *>(key_cache), static_cast<T *>(value_cache),
                          physical_blocks, block_offsets, active_mask, batch, query_heads,
                          kv_heads, head_dim, num_blocks, block_size};
    if (!rope_vectors(p))
      return fail(TF_ERROR_UNSUPPORTED,
                  "rope_kv_append_partials needs head_dim % 16 == 0 and 16-byte aligned buffers");
    launch_rope_vec<T, true>(p, s);
    return check_launch("rope_kv_append_partials");
  };
  if (dtype == TF_DTYPE_BFLOAT16) return launch(static_cast<__bf16 *>(query_out));
  return launch(static_cast<_Float16 *>(query_out));
}
