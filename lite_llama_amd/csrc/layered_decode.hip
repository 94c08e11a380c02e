// One call per layer for a step of decoded tokens: the launches of a layer whose norms sit on its sublayers' results (mixer, then a dense or a
// routed feed-forward), issued one after the other from here.  The kernels, their order and their operands are those of the single entries; what is
// gone is the interpreter between two launches -- some 8 us a launch, 10 launches a layer, where a decoded token's kernels take 5 - 15 us each.  us
// of host time per step of 6 decoded tokens, four layers of 3072 (attention beside a state-space mixer, a fixed decay, two gated ones; a dense and three
// routed feed-forwards), single calls -> this: 880 -> 470; the step 920 -> 620, bound by its kernels
//
// The arguments are two arrays, LayeredDecode's fields in their order (addresses and integers alike as int64) and the floats; scratch is one block,
// whose size the first entry returns (0: a part of the layer is not served here, and nothing was launched: the caller makes the single calls).
#include <stdlib.h>

#include "common.h"

extern "C" int64_t ll_dense16_partial_words(int64_t m, int64_t n, int64_t k);

namespace {

struct DecodeLinear {   // [n][k], rows dense
  const void *w, *bias;
  int64_t n, k;
};

struct LayeredDecode {
  int64_t dtype, tokens, seqs, width, longest_context;
  const int32_t *tok_seq, *tok_pos, *select, *seq_start, *seq_first_pos, *seq_slot, *seq_parity, *token_table;
  int64_t tt_stride;
  // the residual, and what is still to enter it (first: the rows that open the stack, nothing pending)
  float* x;
  const void *first, *y;
  int64_t parts;
  const void* shared;
  const float* shared_scale;
  const void *y_bias, *post_w;
  // mixer: 0 attention beside a state-space branch, 1 a fixed decay per head, 2 a decay per key entry
  int64_t mixer;
  DecodeLinear in, low, out;
  int64_t heads, qk_heads, dk, dv;   // of the recurrence
  float* state;
  const void *decay, *decay_bias;    // 1: fp32 [heads], -; 2: -, [heads dk]
  const void* out_norm;
  int64_t out_norm_len, out_norm_parts;
  // 0 only
  int64_t a_heads, a_kv, a_dk, a_dv, window, pairs;
  const void *q_norm, *k_norm;
  const float* freq;
  void *k_cache, *v_cache;
  const void *conv_w, *conv_bias;
  int64_t conv_channels, conv_taps;
  void* conv_state;
  int64_t conv_half;
  const void *dt_bias, *a_log, *skip;
  // feed-forward: 0 none, 1 dense, 2 routed
  int64_t mlp;
  const void* mixer_post_w;   // norm of the mixer's result
  DecodeLinear up, down;      // 1
  int64_t ff;
  const void *router, *correction;   // 2
  int64_t outputs, identity, top, scoring, experts;
  const void *gate_up, *expert_down;
  int64_t clamped;
  void *rows, *result;        // the feed-forward's input rows (2: they may ride on); what the layer leaves
  float* own;
};
struct LayeredDecodeFloats {
  double eps, value_scale, branch_scale, attn_scale, q_scale, inv_tau, limit;
};

enum Route { NOT_SERVED = 0, NARROW, ROWS, SPLIT };

// the route that such a projection takes on its own (quantization/methods.py), of rows that begin at multiples of x_ld
Route linear_route(const DecodeLinear& l, int64_t m, int64_t x_ld) {
  const int64_t n = l.n, k = l.k;
  if (x_ld % 8 || k % 8 || !ll_aligned16(l.w) || (reinterpret_cast<uintptr_t>(l.bias) & 7u)) return NOT_SERVED;
  if (ll_dense16_narrow_wins(m, n, k)) return getenv("LL_DENSE16_NARROW_OFF") ? NOT_SERVED : NARROW;
  if (x_ld != k) return NOT_SERVED;
  const int route = ll_dense16_route(m, n, k);
  if (route & (LL_ROUTE_ROWS | LL_ROUTE_ROWS_NARROWER)) return getenv("LL_DENSE16_ROWS_OFF") || !ll_dense16_rows_supported(m, n, k, 0) ? NOT_SERVED : ROWS;
  if ((route & LL_ROUTE_SPLIT) && k % 64 == 0 && n % 4 == 0 && ll_dense16_partial_words(m, n, k) > 0 && !getenv("LL_DENSE16_OFF")) return SPLIT;
  return NOT_SERVED;
}

// Both passes walk the same code: the first (no base) counts the scratch and finds what is not served, the second launches.
struct Walk {
  const LayeredDecode& a;
  const LayeredDecodeFloats& f;
  unsigned char* base;
  void* stream;
  int64_t used = 0;
  int status = LL_OK;   // > 0: not served
  bool live() const { return base != nullptr; }
  template <class T>
  T* take(int64_t count) {
    T* p = live() ? reinterpret_cast<T*>(base + used) : nullptr;
    used += (count * (int64_t)sizeof(T) + 255) / 256 * 256;
    return p;
  }
  bool ok(int rc) {
    if (rc != LL_OK && status == LL_OK) status = rc;
    return status == LL_OK;
  }
  void refuse() {
    if (status == LL_OK) status = 1;
  }
  void linear(const DecodeLinear& l, const uint16_t* x, int64_t x_ld, void* out) {
    const Route r = linear_route(l, a.tokens, x_ld);
    if (r == NOT_SERVED) return refuse();
    float* planes = r == SPLIT ? take<float>(ll_dense16_partial_words(a.tokens, l.n, l.k)) : nullptr;
    if (!live() || status != LL_OK) return;
    const int dt = (int)a.dtype;
    if (r == NARROW) ok(ll_dense16_narrow_matmul(out, x, l.w, l.bias, a.tokens, l.n, l.k, x_ld, l.k, dt, stream));
    else if (r == ROWS) ok(ll_dense16_rows_matmul(out, x, l.w, l.bias, a.tokens, l.n, l.k, x_ld, l.k, dt, 0, stream));
    else {
      const int rc = ll_dense16_matmul(out, x, l.w, l.bias, a.tokens, l.n, l.k, x_ld, l.k, dt, planes, stream);
      ok(rc == 1 ? LL_OK : rc < 0 ? rc : LL_ERR_ARG);
    }
  }
  void scan(const uint16_t* q, const uint16_t* k, const uint16_t* v, int64_t ld, int kind, const void* gate, const void* dt, int64_t dt_ld, float* o) {
    if (!ll_linear_scan_supported(a.dk, a.dv) ||
        ll_linear_scan_walk_floats(a.tokens, a.seqs, a.heads, a.dk, a.dv, a.heads / a.qk_heads, kind, 1) != 0)
      return refuse();
    if (!live() || status != LL_OK) return;
    ok(ll_linear_scan(q, ld, k, ld, v, ld, a.heads, a.dk, a.dv, a.heads / a.qk_heads, kind, kind == 0 ? 1 : 0, kind == 1 ? (float)f.q_scale : 1.0f,
                      (const float*)a.decay, gate, gate ? a.heads * a.dk : 0, a.decay_bias, kind == 1 ? (float)f.inv_tau : 1.0f, dt, dt_ld, a.dt_bias,
                      a.a_log, a.skip, o, a.seqs, a.seq_start, a.seq_first_pos, a.seq_slot, a.state, nullptr, a.tokens, 1, (int)a.dtype, stream));
  }
  void out_norm(uint16_t* out, int64_t out_ld, const float* o, const uint16_t* gate, int64_t gate_ld, int kind, int gate_first, float scale) {
    if (live() && status == LL_OK)
      ok(ll_gated_out_norm(out, out_ld, o, gate, gate_ld, kind, gate_first, a.out_norm, a.out_norm_len, (float)f.eps, scale, a.tokens, a.heads * a.dv,
                           a.out_norm_parts, (int)a.dtype, stream));
  }
  void norm(void* h, const void* y, int64_t parts, const void* shared, const float* shared_scale, const void* y_bias, const void* post_w) {
    if (live() && status == LL_OK)
      ok(ll_gated_group_norm(a.x, a.x, h, y, parts, shared, shared_scale, nullptr, 0, nullptr, post_w, nullptr, a.tokens, a.width, 1, (float)f.eps,
                             y_bias, (int)a.dtype, stream));
  }

  void mixer(const uint16_t* h, void* out) {
    const int64_t n = a.tokens, v = a.heads * a.dv, qk = a.qk_heads * a.dk, ld = a.in.n;
    uint16_t* rows = take<uint16_t>(n * ld);
    linear(a.in, h, a.width, rows);
    float* o = take<float>(n * v);
    if (a.mixer == 0) {
      const int64_t aw = a.a_heads * a.a_dv, q_cols = (a.a_heads + a.a_kv) * a.a_dk + a.a_kv * a.a_dv, mixed_ld = aw + v;
      const int64_t z_off = q_cols, conv_off = z_off + v, dt_off = conv_off + a.conv_channels;
      if (!ll_ragged_attention_mfma_supported(a.a_dk, a.a_dv, (int)a.dtype) || (a.a_kv * a.a_dk) % 8 || (a.a_kv * a.a_dv) % 8 ||
          !ll_aligned16(a.k_cache) || !ll_aligned16(a.v_cache) || a.longest_context < 1 || getenv("LL_RAGGED_ATTN_VALU"))
        return refuse();
      const int64_t partition = ll_ragged_attention_partition(), parts = (a.longest_context + partition - 1) / partition;
      uint16_t* q = take<uint16_t>(n * a.a_heads * a.a_dk);
      float* partials = parts > 1 ? take<float>(n * a.a_heads * parts * (2 + a.a_dv)) : nullptr;
      uint16_t* mixed = take<uint16_t>(n * mixed_ld);
      uint16_t* ubc = take<uint16_t>(n * a.conv_channels);
      if (live() && status == LL_OK) {
        ok(ll_rownorm_rope_cache(rows, ld, a.q_norm, a.k_norm, (float)f.eps, a.freq, a.pairs, (float)f.value_scale, a.tok_pos, a.select, q, a.k_cache,
                                 a.v_cache, n, a.a_heads, a.a_kv, a.a_dk, a.a_dv, (int)a.dtype, stream)) &&
            ok(ll_ragged_attention_mfma(q, a.k_cache, a.v_cache, a.token_table, a.tt_stride, a.seq_slot, a.seq_start, a.seq_first_pos, nullptr,
                                        (float)f.attn_scale, mixed, n, a.seqs, 1, a.longest_context, 1, partials, a.a_heads, a.a_kv, a.a_dk, a.a_dv,
                                        a.a_kv * a.a_dk, a.a_kv * a.a_dv, a.window, 0, mixed_ld, 0.0f, nullptr, 0, nullptr, 0, (int)a.dtype, stream)) &&
            ok(ll_conv_act(ubc, a.conv_channels, rows + conv_off, ld, a.conv_w, a.conv_bias, a.conv_channels, a.conv_taps, a.conv_state, a.conv_half,
                           a.tok_seq, a.tok_pos, a.seq_start, a.seq_first_pos, a.seq_slot, a.seq_parity, n, 1, (int)a.dtype, stream));
      }
      // u | B | C: values, keys, queries
      scan(ubc + v + qk, ubc + v, ubc, a.conv_channels, 2, nullptr, rows + dt_off, ld, o);
      out_norm(mixed + aw, mixed_ld, o, rows + z_off, ld, 1, 1, (float)f.branch_scale);
      linear(a.out, mixed, mixed_ld, out);
      return;
    }
    uint16_t* normed = take<uint16_t>(n * v);
    uint16_t* logits = nullptr;
    if (a.mixer == 2) {
      logits = take<uint16_t>(n * a.low.n);
      if (linear_route(a.low, n, ld) != NARROW || (2 * qk + 2 * v) % 8) return refuse();   // (the columns are read where they are)
      linear(a.low, rows + 2 * qk + 2 * v, ld, logits);
    }
    scan(rows, rows + qk, rows + 2 * qk, ld, a.mixer == 2 ? 1 : 0, logits, nullptr, 0, o);
    out_norm(normed, v, o, rows + 2 * qk + v, ld, a.mixer == 2 ? 1 : 2, 0, 1.0f);
    linear(a.out, normed, v, out);
  }

  void feed_forward(const uint16_t* h) {
    const int64_t n = a.tokens, ff = a.ff;
    if (a.mlp == 1) {
      uint16_t* rows = take<uint16_t>(n * 2 * ff);
      uint16_t* act = take<uint16_t>(n * ff);
      linear(a.up, h, a.width, rows);
      if (live() && status == LL_OK) ok(ll_glu_act(act, ff, rows, 2 * ff, rows + ff, 2 * ff, n, ff, 0, 0.0f, 1.0f, (int)a.dtype, stream));
      linear(a.down, act, ff, a.result);
      return;
    }
    const int64_t slots = n * a.top, block = ll_moe_rows_block(slots, a.experts, a.width, ff, (int)a.dtype);
    const int skipped = a.identity > 0;
    if (a.experts > 8192) return refuse();   // (skipped slots' zeros: the caller's)
    const int64_t padded = slots + (a.experts + skipped) * (block - 1), blocks = (padded + block - 1) / block;
    int32_t* ids = take<int32_t>(slots);
    float* weights = take<float>(slots);
    float* logits = take<float>(n * a.outputs);
    int32_t* counts = take<int32_t>(a.experts);
    int32_t* sorted = take<int32_t>(padded);
    int32_t* owner = take<int32_t>(blocks);
    int32_t* post = take<int32_t>(1);
    uint16_t* act = take<uint16_t>(slots * ff);
    if (!live() || status != LL_OK) return;
    const int dt = (int)a.dtype;
    ok(ll_group_router_sorted(h, a.width, a.router, nullptr, n, a.width, a.outputs, a.top, 1, 1, 1.0f, (int)a.scoring, ids, weights, a.own, logits,
                              a.correction, a.identity, a.experts, block, skipped, counts, sorted, owner, post, dt, stream)) &&
        ok(ll_moe_rows_gemm(h, a.width, a.top, a.gate_up, 2 * ff * a.width, a.width, ff, a.clamped ? 2 : 1, nullptr, act, ff, sorted, owner, post, slots,
                            a.experts, block, a.clamped ? (float)f.limit : 0.0f, dt, stream)) &&
        ok(ll_moe_rows_gemm(act, ff, 1, a.expert_down, a.width * ff, ff, a.width, 0, weights, a.result, a.width, sorted, owner, post, slots, a.experts,
                            block, 0.0f, dt, stream));
  }

  void run() {
    const int64_t n = a.tokens;
    const uint16_t* h = (const uint16_t*)a.first;
    if (!h) {
      uint16_t* own = take<uint16_t>(n * a.width);
      norm(own, a.y, a.parts, a.shared, a.shared_scale, a.y_bias, a.post_w);
      h = own;
    }
    uint16_t* mixed = a.mlp ? take<uint16_t>(n * a.width) : (uint16_t*)a.result;
    mixer(h, mixed);
    if (!a.mlp || status != LL_OK) return;
    norm(a.rows, mixed, 1, nullptr, nullptr, nullptr, a.mixer_post_w);
    feed_forward((const uint16_t*)a.rows);
  }
};

bool readable(const int64_t* args, int64_t count, const double* floats, int64_t float_count) {
  static_assert(sizeof(LayeredDecode) % sizeof(int64_t) == 0 && sizeof(void*) == sizeof(int64_t), "eight bytes a field");
  if (!args || !floats || count * (int64_t)sizeof(int64_t) != (int64_t)sizeof(LayeredDecode) ||
      float_count * (int64_t)sizeof(double) != (int64_t)sizeof(LayeredDecodeFloats))
    return false;
  const LayeredDecode& a = *reinterpret_cast<const LayeredDecode*>(args);
  return (a.dtype == LL_F16 || a.dtype == LL_BF16) && a.tokens >= 1 && a.tokens <= 64 && a.seqs == a.tokens && a.mixer >= 0 && a.mixer <= 2 &&
         a.mlp >= 0 && a.mlp <= 2 && a.qk_heads >= 1 && a.heads % a.qk_heads == 0 && a.width >= 8 && a.width % 8 == 0 &&
         ll_aligned16(a.first);   // (what the first product reads; all other rows are this file's own)
}

}  // namespace

// bytes of scratch for such a layer, or 0: not served (LL_NO_LAYER_CALLS in the environment: none is)
extern "C" int64_t ll_layered_decode_bytes(const int64_t* args, int64_t count, const double* floats, int64_t float_count) {
  if (!readable(args, count, floats, float_count) || getenv("LL_NO_LAYER_CALLS")) return 0;
  Walk w{*reinterpret_cast<const LayeredDecode*>(args), *reinterpret_cast<const LayeredDecodeFloats*>(floats), nullptr, nullptr};
  w.run();
  return w.status == LL_OK ? w.used : 0;
}

// scratch: 256-byte aligned, as many bytes as ll_layered_decode_bytes returned for the same arguments
extern "C" int ll_layered_decode(const int64_t* args, int64_t count, const double* floats, int64_t float_count, void* scratch, int64_t bytes,
                                 void* stream) {
  if (!readable(args, count, floats, float_count)) return LL_ERR_SHAPE;
  const int64_t need = ll_layered_decode_bytes(args, count, floats, float_count);
  if (need == 0 || bytes < need) return LL_ERR_SHAPE;
  const LayeredDecode& a = *reinterpret_cast<const LayeredDecode*>(args);
  if (!scratch || (reinterpret_cast<uintptr_t>(scratch) & 255u) || !a.x || !a.result || (!a.first && (!a.y || !a.post_w)) || (a.mlp && !a.rows)) return LL_ERR_ARG;
  Walk w{a, *reinterpret_cast<const LayeredDecodeFloats*>(floats), (unsigned char*)scratch, stream};
  w.run();
  return w.status > 0 ? LL_ERR_ARG : w.status;
}
