// The per-op forward of the whole layer stack as one call: LayerNorm, then per
// layer QKV projection, attention (over the projection, or over the KV cache
// after appending to it), output projection, residual LayerNorm, FFN, residual
// LayerNorm -- the sequence of torch_transformer_benchmark.py:1092-1148 --
// with every intermediate in one caller workspace.
//
// Why a native sequence: issued one by one from Python a launch cost 11.7 us
// of host time (wrapper, allocation, argument conversion) against kernels of
// 3 to 10 us, so every forward of less than about 10 us of GPU work per
// launch ran at the host's pace.  From here a launch costs the runtime's own
// 2 to 3 us.
#include <algorithm>

#include "common.h"
#include "../../include/xblock.h"

namespace xb {

// Byte offsets of the intermediates, each from a 256-byte boundary.  hidden
// (the FFN activation) takes the place of qkv and ctx, which are dead by then.
struct StackLayout {
  int64_t residual, residual2, norm, update, qkv, ctx, hidden, vt, decode, bytes;
};

// A few rows (decode steps): LayerNorm in the prologue of the product that
// follows it (xb_norm_linear), which needs a second residual buffer.
static bool norm_in_products(int64_t rows, int d, int ffn) {
  return xb_select_norm_linear(rows, 3 * d, d) == XB_OK && xb_select_norm_linear(rows, ffn, d) == XB_OK;
}

static int64_t aligned_up(int64_t n) { return (n + 255) / 256 * 256; }

// cache_start < 0: no KV cache.
static int stack_layout(int32_t batch, int64_t seq_len, int32_t heads, int32_t head_dim, int32_t ffn_dim,
                        int attention_variant, int64_t cache_start, StackLayout* out) {
  if (batch < 0 || seq_len < 0 || heads <= 0 || head_dim <= 0 || ffn_dim <= 0) return XB_ERR_BAD_SIZE;
  const int64_t rows = (int64_t)batch * seq_len, d = (int64_t)heads * head_dim;
  if (rows > 0x7fffffffLL || 3 * d > 0x7fffffffLL) return XB_ERR_BAD_SIZE;
  StackLayout l;
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t p = at;
    at += aligned_up(bytes);
    return p;
  };
  l.residual = take(rows * d * 4);
  l.residual2 = take(norm_in_products(rows, (int)d, ffn_dim) ? rows * d * 4 : 0);
  l.norm = take(rows * d * 2);
  l.update = take(rows * d * 2);
  l.qkv = take(rows * 3 * d * 2);
  l.ctx = take(rows * d * 2);
  l.hidden = l.qkv;
  at = std::max(at, aligned_up(l.hidden + rows * ffn_dim * 2));
  const bool vt = cache_start < 0 && attention_variant == XB_ATTN_PINGPONG_VT;
  l.vt = take(vt ? (int64_t)batch * d * xb_vt_row_stride(seq_len) * 2 : 0);
  int64_t decode = 0;
  if (cache_start > 0) {
    decode = xb_attention_kv_cache_workspace_bytes(batch, seq_len, heads, head_dim, cache_start);
    if (decode < 0) return (int)decode;
  }
  l.decode = take(decode);
  l.bytes = at;
  *out = l;
  return XB_OK;
}

}  // namespace xb

using namespace xb;

extern "C" int64_t xb_stack_workspace_bytes(int32_t batch, int64_t seq_len, int32_t heads, int32_t head_dim,
                                            int32_t ffn_dim, int attention_variant, int64_t cache_start) {
  StackLayout l;
  const int bad = stack_layout(batch, seq_len, heads, head_dim, ffn_dim, attention_variant, cache_start, &l);
  return bad ? bad : l.bytes;
}

extern "C" int xb_stack_forward(const xb_stack* st, const float* x, float* y, const uint8_t* token_valid,
                                int32_t batch, int64_t seq_len, int qkv_variant, int out_variant,
                                int ffn_in_variant, int ffn_out_variant, int attention_variant,
                                void* const* caches, int64_t cache_start, int64_t cache_capacity,
                                void* workspace, int64_t workspace_bytes, void* stream) {
  if (!st || st->layers <= 0) return XB_ERR_BAD_SIZE;
  const bool cached = caches != nullptr;
  if (cached && (cache_start < 0 || token_valid != nullptr || !st->causal)) return XB_ERR_BAD_SIZE;
  const int heads = st->heads, hd = st->head_dim;
  StackLayout l;
  int e = stack_layout(batch, seq_len, heads, hd, st->ffn_dim, attention_variant, cached ? cache_start : -1, &l);
  if (e) return e;
  const int64_t rows = (int64_t)batch * seq_len;
  if (rows == 0) return XB_OK;
  if (!st->blocks || !x || !y || !workspace) return XB_ERR_NULL_POINTER;
  if (workspace_bytes < l.bytes) return XB_ERR_WORKSPACE;
  if ((uintptr_t)workspace & 15u) return XB_ERR_MISALIGNED;
  const int d = heads * hd, f = st->ffn_dim;
  char* ws = static_cast<char*>(workspace);
  float* residual = reinterpret_cast<float*>(ws + l.residual);
  void *norm = ws + l.norm, *update = ws + l.update, *qkv = ws + l.qkv, *ctx = ws + l.ctx, *hidden = ws + l.hidden;
  void *vt = ws + l.vt, *decode = ws + l.decode;
  const bool transposed_v = !cached && attention_variant == XB_ATTN_PINGPONG_VT;

  const xb_block* b = st->blocks;
  bool row_blocks = true;
  for (int i = 0; i < st->layers; ++i) row_blocks = row_blocks && b[i].packed != nullptr;
  // Append (unless the projection did) and attend: layer i's context from qkv.
  auto attend = [&](int i, bool appended) -> int {
    const float scale = st->blocks[i].scale;
    if (cached) {
      const int bad = appended ? XB_OK
                               : xb_kv_cache_append(qkv, caches[2 * i], caches[2 * i + 1], batch, seq_len, heads, hd,
                                                    cache_start, cache_capacity, stream);
      if (bad) return bad;
      if (cache_start > 0)
        return xb_attention_kv_cache(qkv, caches[2 * i], caches[2 * i + 1], ctx, batch, seq_len, heads, hd,
                                     cache_start, cache_capacity, scale, decode, l.bytes - l.decode, stream);
    }
    return xb_attention_v(qkv, ctx, token_valid, batch, seq_len, heads, hd, scale, st->causal, attention_variant, stream);
  };
  if (row_blocks) {
    // The residual stream alternates between its buffer and the place of
    // norm and update, which this path does not use.
    float* streams[2] = {residual, static_cast<float*>(norm)};
    const float* in = x;
    e = xb_row_block(st, -1, x, nullptr, nullptr, qkv, nullptr, nullptr, rows, stream);
    for (int i = 0; i < st->layers && !e; ++i) {
      e = attend(i, false);
      if (!e) e = xb_row_block(st, i, in, ctx, streams[i & 1], qkv, y, token_valid, rows, stream);
      in = streams[i & 1];
    }
    return e;
  }
  // The few-row kernel gives the bits of every tile, but only AUTO or its own
  // variant asks for it.
  auto any = [](int v) { return v == XB_VARIANT_AUTO || v == XB_LINEAR_ROWS; };
  // Nor does it take the unaligned inputs that some widths' LayerNorms do.
  uintptr_t vectors = (uintptr_t)x;
  for (int i = 0; i < st->layers; ++i) {
    if (b[i].norm1_affine) vectors |= (uintptr_t)b[i].norm1_g | (uintptr_t)b[i].norm1_b;
    if (b[i].norm2_affine) vectors |= (uintptr_t)b[i].norm2_g | (uintptr_t)b[i].norm2_b;
  }
  const bool aligned = (vectors & 15u) == 0;
  if (aligned && norm_in_products(rows, d, f) && any(qkv_variant) && any(ffn_in_variant) && !transposed_v) {
    float* streams[2] = {residual, reinterpret_cast<float*>(ws + l.residual2)};
    const float* in = x;
    const void* upd = nullptr;
    for (int i = 0; i < st->layers && !e; ++i, ++b) {
      // x + update of the layer before (layer 0: x itself) -> streams[0]; then + the attention's -> streams[1].
      e = xb_norm_linear(in, upd, b->norm1_g, b->norm1_b, b->norm1_eps, b->norm1_affine, upd ? streams[0] : nullptr,
                         b->qkv_w, b->qkv_b, qkv, rows, 3 * d, d, XB_EPI_BIAS, cached ? caches[2 * i] : nullptr,
                         cached ? caches[2 * i + 1] : nullptr, heads, seq_len, cache_start, cache_capacity, stream);
      if (upd) in = streams[0];
      if (!e) e = attend(i, cached);
      if (!e) e = xb_linear_v(ctx, b->out_w, b->out_b, update, rows, d, d, XB_EPI_BIAS, out_variant, stream);
      if (!e)
        e = xb_norm_linear(in, update, b->norm2_g, b->norm2_b, b->norm2_eps, b->norm2_affine, streams[1], b->ffn_in_w,
                           b->ffn_in_b, hidden, rows, f, d, XB_EPI_BIAS_GELU, nullptr, nullptr, 0, 1, 0, 0, stream);
      in = streams[1];
      if (!e) e = xb_linear_v(hidden, b->ffn_out_w, b->ffn_out_b, update, rows, d, f, XB_EPI_BIAS, ffn_out_variant, stream);
      upd = update;
    }
    if (e) return e;
    return xb_residual_layernorm_masked(in, update, XB_F16, st->final_g, st->final_b, nullptr, y, XB_F32, rows, d,
                                        st->final_eps, st->final_affine, token_valid,
                                        token_valid ? XB_MASK_OUTPUT : 0, stream);
  }
  e = xb_layernorm(x, b->norm1_g, b->norm1_b, norm, XB_F16, rows, d, b->norm1_eps, b->norm1_affine, stream);
  const float* res_in = x;
  for (int i = 0; i < st->layers && !e; ++i, ++b) {
    if (transposed_v) {
      e = xb_linear_qkv_vt(norm, b->qkv_w, b->qkv_b, qkv, vt, batch, seq_len, heads, hd, d, qkv_variant, stream);
      if (!e) e = xb_attention_causal_vt(qkv, vt, ctx, batch, seq_len, heads, hd, b->scale, stream);
    } else {
      e = xb_linear_v(norm, b->qkv_w, b->qkv_b, qkv, rows, 3 * d, d, XB_EPI_BIAS, qkv_variant, stream);
      if (!e) e = attend(i, false);
    }
    if (!e) e = xb_linear_v(ctx, b->out_w, b->out_b, update, rows, d, d, XB_EPI_BIAS, out_variant, stream);
    if (!e)
      e = xb_residual_layernorm(res_in, update, XB_F16, b->norm2_g, b->norm2_b, residual, norm, XB_F16, rows, d,
                                b->norm2_eps, b->norm2_affine, stream);
    if (!e) e = xb_linear_v(norm, b->ffn_in_w, b->ffn_in_b, hidden, rows, f, d, XB_EPI_BIAS_GELU, ffn_in_variant, stream);
    if (!e) e = xb_linear_v(hidden, b->ffn_out_w, b->ffn_out_b, update, rows, d, f, XB_EPI_BIAS, ffn_out_variant, stream);
    if (!e && i + 1 < st->layers)
      e = xb_residual_layernorm(residual, update, XB_F16, b[1].norm1_g, b[1].norm1_b, residual, norm, XB_F16, rows, d,
                                b[1].norm1_eps, b[1].norm1_affine, stream);
    res_in = residual;
  }
  if (e) return e;
  return xb_residual_layernorm_masked(residual, update, XB_F16, st->final_g, st->final_b, nullptr, y, XB_F32, rows, d,
                                      st->final_eps, st->final_affine, token_valid,
                                      token_valid ? XB_MASK_OUTPUT : 0, stream);
}
