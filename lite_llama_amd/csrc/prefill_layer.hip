// A decoder layer of an unquantised llama-shaped model over the tokens of a short prefill (at most 192), issued by ONE host call.
//
// Bound by the host: the launches of such a layer (seven; eight where the rotation has one of its own) take 28 - 60 us, and each of them cost 16 - 24 us of interpreter time to prepare (a prompt of
// 37 tokens through 12 layers of 896: 2290 us, of which the GPU worked 670).  The launches are the eager route's own, in its order and with
// its arithmetic: norm, q|k|v, rotation + cache scatter + attention, o as split-K partials that the next norm adds up, gate|up with the
// activation in its epilogue, down as partials.  (The eager route asks the library for q|k|v and o; here they stay on the narrow kernel or
// the row-group loop and on the split-K engine: 5 - 9 us each against 8, without 24 us of the library's host side.)
// These engines take 64 rows: more go through them in parts of equal size, whose weights the Infinity Cache
// holds between them, if the layer's are no more than 100 MB.  us, eager -> here: 12 layers of 896 / 4864, 37 tokens 2290 -> 790 (519 since: fewer checks, the rotation in the attention's launch, plans told apart early), 100 2850 -> 1090, 200
// (four parts) 2790 -> 1530; 4 layers of 1536 / 8960 (94 MB each), 64 tokens 850 -> 374, 100 1020 -> 616, 180 1034 -> 858, 256 1025 -> 1096.
#include "common.h"

int fa_rope_launch(void* out, const void* qkv, int64_t row, const void* cos_t, const void* sin_t, int64_t cos_b_stride, int64_t cos_s_stride,
                   int64_t sin_b_stride, int64_t sin_s_stride, void* pool, int64_t pool_stride_t, int64_t pool_stride_h, const void* select_index,
                   int select_width, const void* starts, int start_width, const void* lens, int len_width, int64_t prompts, int64_t max_len,
                   int64_t tokens, int64_t seq_len, int heads, int kv_heads, int d, float sm_scale, int dtype, int cs_dtype, hipStream_t st);

extern "C" int ll_prefill_layer16(void* residual, void* x, int planes_in, float* planes, void* qkv, void* attn, void* act, const void* norm1,
                                  const void* norm2, float eps, const void* w_qkv, const void* b_qkv, const void* w_o, const void* w_gate_up,
                                  const void* w_down, const void* cos_t, const void* sin_t, int64_t cos_b_stride, int64_t cos_s_stride,
                                  int64_t sin_b_stride, int64_t sin_s_stride, void* pool, int64_t pool_stride_t, int64_t pool_stride_h,
                                  const void* select_index, int select_width, const void* starts, int start_width, const void* lens,
                                  int len_width, int64_t prompts, int64_t max_len, int64_t tokens, int64_t seq_len, int64_t hidden, int heads,
                                  int kv_heads, int head_dim, int64_t inter, float sm_scale, int dtype, int cs_dtype, int max_splits, void* stream) {
  if (dtype != LL_F16 && dtype != LL_BF16) return LL_ERR_DTYPE;
  if (tokens < 1 || tokens > 192 || hidden < 1 || heads < 1 || kv_heads < 1 || head_dim < 1 || inter < 1 || prompts < 1 || seq_len < 1 || planes_in < 0)
    return LL_ERR_SHAPE;
  if (!residual || !x || !planes || !qkv || !attn || !act || !norm1 || !norm2 || !w_qkv || !w_o || !w_gate_up || !w_down || !cos_t || !sin_t ||
      !pool || !select_index || !starts || !lens)
    return LL_ERR_ARG;
  const int64_t q_size = (int64_t)heads * head_dim, row = q_size + 2 * (int64_t)kv_heads * head_dim;
  const int wfmt = dtype == LL_F16 ? 4 : 5;
  const int64_t parts = (tokens + 63) / 64, part = (tokens + parts - 1) / parts, last = tokens - (parts - 1) * part;
  // all of it or nothing: what one of the launches would decline is the caller's to run
  const int o_planes = ll_dense_partials_count(part, hidden, q_size, wfmt, max_splits);
  const int down_planes = ll_dense_partials_count(part, hidden, inter, wfmt, max_splits);
  for (const int64_t m : {part, last})
    if (m < 1 || !ll_dense16_rows_supported(m, row, hidden, 0) || !ll_dense16_rows_supported(m, 2 * inter, hidden, 1) ||
        ll_dense_partials_count(m, hidden, q_size, wfmt, max_splits) != o_planes ||
        ll_dense_partials_count(m, hidden, inter, wfmt, max_splits) != down_planes)
      return 0;
  if (o_planes < 1 || down_planes < 1 || o_planes > 12 || down_planes > 12 || hidden % 8 || hidden > 8192 || head_dim % 8 || q_size % 8 || inter % 8)
    return 0;
  if (parts > 1 && (row + q_size + 3 * inter) * hidden * 2 > 100000000) return 0;
  for (const void* p : {(const void*)residual, (const void*)x, (const void*)planes, (const void*)qkv, (const void*)attn, (const void*)act,
                        norm1, norm2, w_qkv, b_qkv, w_o, w_gate_up, w_down})
    if (!ll_aligned16(p)) return 0;
  auto rows = [](void* base, int64_t at, int64_t width) { return (void*)((char*)base + at * width * 2); };
  auto sums = [&](int64_t i) { return planes + i * part * hidden * max_splits; };
  void* k = rows(qkv, 1, q_size);
  void* v = rows(qkv, 1, q_size + (int64_t)kv_heads * head_dim);
  int r = LL_OK;
#define LL_TRY(CALL)           \
  do {                         \
    r = (CALL);                \
    if (r != LL_OK) return r;  \
  } while (0)
  if (planes_in == 0) LL_TRY(ll_skip_rmsnorm(x, residual, nullptr, norm1, tokens, hidden, eps, dtype, stream));
  for (int64_t i = 0, at = 0; i < parts; ++i, at += part) {
    const int64_t m = i + 1 < parts ? part : last;
    if (planes_in > 0)
      LL_TRY(ll_skip_rmsnorm_partials(rows(x, at, hidden), sums(i), planes_in, rows(residual, at, hidden), norm1, m, hidden, eps, dtype, stream));
    if (ll_dense16_narrow_wins(m, row, hidden))
      LL_TRY(ll_dense16_narrow_matmul(rows(qkv, at, row), rows(x, at, hidden), w_qkv, b_qkv, m, row, hidden, hidden, hidden, dtype, stream));
    else LL_TRY(ll_dense16_rows_matmul(rows(qkv, at, row), rows(x, at, hidden), w_qkv, b_qkv, m, row, hidden, hidden, hidden, dtype, 0, stream));
  }
  r = fa_rope_launch(attn, qkv, row, cos_t, sin_t, cos_b_stride, cos_s_stride, sin_b_stride, sin_s_stride, pool, pool_stride_t, pool_stride_h, select_index,
                     select_width, starts, start_width, lens, len_width, prompts, max_len, tokens, seq_len, heads, kv_heads, head_dim, sm_scale, dtype,
                     cs_dtype, (hipStream_t)stream);
  if (r < 0) return r;
  if (r == 0) {
    LL_TRY(ll_rope_kv_update(qkv, k, cos_t, sin_t, pool, select_index, tokens, heads, kv_heads, head_dim, row, row, seq_len, cos_b_stride,
                             cos_s_stride, sin_b_stride, sin_s_stride, pool_stride_t, pool_stride_h, dtype, cs_dtype, select_width, nullptr, stream));
    LL_TRY(ll_flash_attention_nopad(attn, qkv, k, v, starts, lens, (int)prompts, heads, kv_heads, head_dim, max_len, sm_scale, row, head_dim, row,
                                    head_dim, row, head_dim, q_size, head_dim, dtype, start_width, len_width, stream));
  }
  for (int64_t i = 0, at = 0; i < parts; ++i, at += part) {
    const int64_t m = i + 1 < parts ? part : last;
    r = ll_dense_partials(sums(i), rows(attn, at, q_size), w_o, nullptr, m, hidden, q_size, 1, q_size, wfmt, q_size, q_size, 0, 0, max_splits, stream);
    if (r != o_planes) return r < 0 ? r : LL_ERR_SHAPE;
    LL_TRY(ll_skip_rmsnorm_partials(rows(x, at, hidden), sums(i), o_planes, rows(residual, at, hidden), norm2, m, hidden, eps, dtype, stream));
    LL_TRY(ll_dense16_rows_matmul(rows(act, at, inter), rows(x, at, hidden), w_gate_up, nullptr, m, 2 * inter, hidden, hidden, hidden, dtype, 1, stream));
    r = ll_dense_partials(sums(i), rows(act, at, inter), w_down, nullptr, m, hidden, inter, 1, inter, wfmt, inter, inter, 0, 0, max_splits, stream);
    if (r != down_planes) return r < 0 ? r : LL_ERR_SHAPE;
  }
#undef LL_TRY
  return down_planes;
}
