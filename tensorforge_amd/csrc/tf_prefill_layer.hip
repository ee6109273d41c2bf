// One decoder layer of a packed prefill as one call.
//
// The launches are those of the single entry points; what this saves is the
// host's side of them.  A prompt of a few hundred tokens spends 60 to 75 us
// of device time per TinyLlama layer on eight launches, and calling them one
// by one from Python costs the host about 90 us per layer, so the call was
// bound by the host.
//
// Reference semantics: the layer loop of tensorforge/runtime/prefill.py:90-135.
#include "tf_common.hpp"

namespace tf {
namespace {

// y = x . w^T: slice sums into `partials` where that is faster and they fit
// (returns their count), else rounded into `y` (returns 1); 0 on failure
// (`status` set).
int32_t project(const tf_prefill_layer_args &a, const void *x, const void *w, void *y, int32_t n,
                int32_t k, int32_t &status, void *stream) {
  int32_t splits = tf_prefill_linear_splits(a.tokens, n, k);
  if (splits > 1 && static_cast<int64_t>(splits) * a.tokens * n > a.partial_floats) splits = 1;
  const bool sliced = splits > 1;
  status = tf_prefill_linear(x, k, w, k, sliced ? nullptr : y, sliced ? 0 : n,
                             sliced ? a.partials : nullptr, a.tokens, n, k, sliced ? splits : 1, 0, 0,
                             a.dtype, stream);
  return status ? 0 : (sliced ? splits : 1);
}

// residual_out = residual + projection, h = RMSNorm of it.
int32_t add_norm(const tf_prefill_layer_args &a, int32_t splits, const void *residual,
                 const void *norm, void *residual_out, void *stream) {
  if (splits > 1)
    return tf_residual_rms_norm_partials(a.partials, splits, residual, norm, residual_out, a.h,
                                         a.tokens, a.hidden, a.eps, a.dtype, stream);
  return tf_residual_rms_norm(a.rows, residual, norm, residual_out, a.h, a.tokens, a.hidden, a.eps,
                              a.dtype, stream);
}

}  // namespace
}  // namespace tf

extern "C" int32_t tf_prefill_layer(const tf_prefill_layer_args *args, void *stream) {
  using namespace tf;
  clear_error();
  if (!args) return fail(TF_ERROR_INVALID_ARGUMENT, "null arguments");
  const tf_prefill_layer_args &a = *args;
  if (a.tokens < 0 || a.hidden <= 0 || a.intermediate <= 0 || a.query_heads <= 0 || a.kv_heads <= 0 ||
      a.head_dim <= 0)
    return fail(TF_ERROR_INVALID_ARGUMENT, "prefill layer sizes must be positive");
  if (a.tokens == 0) return TF_SUCCESS;
  const int64_t q_width = static_cast<int64_t>(a.query_heads) * a.head_dim;
  const int64_t kv_width = static_cast<int64_t>(a.kv_heads) * a.head_dim;
  if (q_width + 2 * kv_width > (1 << 27) || a.hidden > 16384 || a.intermediate > (1 << 26))
    return fail(TF_ERROR_UNSUPPORTED, "prefill layer rows are too long");
  if (!a.h || !a.residual || !a.second_residual || !a.rows || !a.query || !a.key || !a.value ||
      !a.context || !a.act || (a.partial_floats > 0 && !a.partials))
    return fail(TF_ERROR_INVALID_ARGUMENT, "null buffer");
  const int32_t qkv_width = static_cast<int32_t>(q_width + 2 * kv_width);
  const int32_t o_k = static_cast<int32_t>(q_width);
  int32_t status = 0;

  int32_t splits = project(a, a.h, a.qkv_weight, a.rows, qkv_width, a.hidden, status, stream);
  if (status) return status;
  const char *rows = static_cast<const char *>(a.rows);
  const void *value = a.value;
  int64_t value_stride = kv_width;
  if (splits > 1) {
    status = tf_rope_kv_append_partials(a.partials, splits, a.positions, a.cos_table, a.sin_table,
                                        a.table_rows, a.query, a.key, a.value, a.key_cache,
                                        a.value_cache, a.physical_blocks, a.block_offsets,
                                        a.active_mask, a.tokens, a.query_heads, a.kv_heads,
                                        a.head_dim, a.num_blocks, a.block_size, a.dtype, stream);
  } else {
    status = tf_rope_kv_append(a.rows, qkv_width, a.positions, a.cos_table, a.sin_table, a.table_rows,
                               a.query, a.key, a.key_cache, a.value_cache, a.physical_blocks,
                               a.block_offsets, a.active_mask, a.tokens, a.query_heads, a.kv_heads,
                               a.head_dim, a.num_blocks, a.block_size, a.dtype, stream);
    value = rows + (q_width + kv_width) * dtype_size(a.dtype);
    value_stride = qkv_width;
  }
  if (status) return status;
  status = tf_prefill_attention(a.query, q_width, a.key, kv_width, value, value_stride, a.context,
                                q_width, a.tiles, a.num_tiles, a.query_heads, a.kv_heads, a.head_dim,
                                a.scale, 0, a.dtype, stream);
  if (status) return status;
  splits = project(a, a.context, a.o_weight, a.rows, a.hidden, o_k, status, stream);
  if (status) return status;
  status = add_norm(a, splits, a.residual, a.post_norm, a.second_residual, stream);
  if (status) return status;
  status = tf_prefill_linear(a.h, a.hidden, a.gate_up_weight, a.hidden, a.act, a.intermediate, nullptr,
                             a.tokens, a.intermediate, a.hidden, 1, 1, 0, a.dtype, stream);
  if (status) return status;
  splits = project(a, a.act, a.down_weight, a.rows, a.hidden, a.intermediate, status, stream);
  if (status) return status;
  return add_norm(a, splits, a.second_residual, a.next_norm, a.residual, stream);
}
