// Mixture of experts with a SIGMOID router over expert groups, for 16-bit and 32-bit storage dtypes (the softmax-router fp16
// path of moe.hip stays as it is):
//
//   ll_group_router   logits = W_router h in fp32, scores = sigmoid(logits); the experts form `group_count` equal groups of
//                     neighbours, a group's score is the sum of its two best scores, only the best `group_keep` groups stay
//                     eligible; the `top` best eligible experts are chosen, their scores divided by their sum (+ 1e-20) and
//                     multiplied by `route_scale`.  One more row of weights may give a per-token sigmoid scale (for a shared
//                     expert).  Up to 512 rows of router weights in one launch (a workgroup forms its tokens' logits and selects), more
//                     in two: the logits as an 8 x 8 register-tiled product per wave, then one wave per token.  Selection by ranks (ties:
//                     the lower index first), so slot k of a token holds its k-th best expert.
//   ll_moe_sort       slots (token, k) sorted by expert, every expert's run padded to the row-block size with a sentinel:
//                     sorted_ids / block_expert / num_post as in moe_align_block_size.  Deterministic: no atomics.
//   ll_moe_rows_gemm  the grouped products over sorted row blocks: act = silu(a Wg_e^T) * (a Wu_e^T) (gate and up rows
//                     stacked in one matrix per expert), out = (a W_e^T) * slot weight, or act = relu((slot weight * a) W_e^T)^2 (experts
//                     without a gate whose weight multiplies their INPUT), fp32 accumulation.  MFMA form for
//                     16-bit storage with contraction widths that are multiples of 8, a plain tiled form otherwise.
#include <type_traits>

#include "common.h"
#include "moe_stream.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

namespace {

template <int DT>
__device__ __forceinline__ float ldv(const void* p, int64_t i) {
  if constexpr (DT == LL_F32) return ((const float*)p)[i];
  else return to_f32<DT>(((const uint16_t*)p)[i]);
}
template <int DT>
__device__ __forceinline__ void stv(void* p, int64_t i, float v) {
  if constexpr (DT == LL_F32) ((float*)p)[i] = v;
  else ((uint16_t*)p)[i] = from_f32<DT>(v);
}

__device__ __forceinline__ float sigmoid_exact(float v) { return 1.0f / (1.0f + expf(-v)); }

// what one row block of the grouped products does with its sums: 0 times the slot's weight, 1 a gated pair (glu_pair), 2 the square
// of relu of the sum times the slot's weight (the weight multiplies the expert's input: the sum is linear in it)
template <int MODE>
__device__ __forceinline__ float slot_value(float sum, float weight) {
  const float v = sum * weight;
  if constexpr (MODE == 2) {
    const float r = fmaxf(v, 0.f);
    return r * r;
  }
  return v;
}

// the gated pair of an expert's first product.  limit < 0: silu(g) u; else the clamped form g' sigmoid(1.702 g') (u' + 1) with
// g' = min(g, limit), u' = clamp(u, -limit, limit)
template <int DT>
__device__ __forceinline__ float glu_pair(float g, float u, float limit) {
  if (limit >= 0.f) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit) + 1.0f;
    return g * (DT == LL_F32 ? sigmoid_exact(1.702f * g) : ll_sigmoidf(1.702f * g)) * u;
  }
  return g * (DT == LL_F32 ? sigmoid_exact(g) : ll_sigmoidf(g)) * u;
}

// ------------------------------------------------------------------------------------------------------------------------
// router, first launch: logits [n][experts (+ 1)] = h W^T in fp32.  A wave owns 8 tokens x 8 weight rows (x 2 rows for steps of
// a few tokens, where more and shorter waves matter more than reuse) and walks the width
// in pieces (16 bytes where rows are aligned): 16 piece loads feed 64 x VEC fused multiply-adds, so a weight row is fetched
// once per 8 tokens and a token row once per 8 experts.  A token's logit does not depend on which other tokens ride along:
// every lane sums ITS pieces in order, then the lanes are added in a fixed order.
// ------------------------------------------------------------------------------------------------------------------------
template <int DT, int VEC>
__device__ __forceinline__ void load_piece(const void* p, int64_t at, float (&o)[VEC]) {
  if constexpr (VEC == 1) {
    o[0] = ldv<DT>(p, at);
  } else if constexpr (DT == LL_F32) {
    const f32x4 v = *reinterpret_cast<const f32x4*>((const float*)p + at);
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = v[i];
  } else {
    const U16x8 v = *reinterpret_cast<const U16x8*>((const uint16_t*)p + at);
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] = to_f32<DT>(v.v[i]);
  }
}

template <int DT, int VEC, int EW>
__global__ __launch_bounds__(256) void router_logits_kernel(const void* __restrict__ h, int64_t h_ld, const void* __restrict__ w_router,
                                                            const void* __restrict__ w_extra, int width, int experts, int rows,
                                                            float* __restrict__ logits, int64_t n) {
  constexpr int TW = 8;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t t0 = (int64_t)blockIdx.x * TW;
  const int e0 = (blockIdx.y * 4 + wave) * EW;
  if (e0 >= rows) return;   // (wave-uniform; no workgroup barrier below)
  int64_t hat[TW];
  const void* wp[EW];
  int64_t wat[EW];
#pragma unroll
  for (int i = 0; i < TW; ++i) hat[i] = (t0 + i < n ? t0 + i : n - 1) * h_ld;
#pragma unroll
  for (int j = 0; j < EW; ++j) {
    const int e = e0 + j < rows ? e0 + j : rows - 1;
    wp[j] = e < experts ? w_router : w_extra;
    wat[j] = e < experts ? (int64_t)e * width : 0;
  }
  float acc[TW][EW];
#pragma unroll
  for (int i = 0; i < TW; ++i)
#pragma unroll
    for (int j = 0; j < EW; ++j) acc[i][j] = 0.f;
  for (int p = lane * VEC; p < width; p += 64 * VEC) {
    float hv[TW][VEC];
#pragma unroll
    for (int i = 0; i < TW; ++i) load_piece<DT, VEC>(h, hat[i] + p, hv[i]);
#pragma unroll
    for (int j = 0; j < EW; ++j) {
      float wv[VEC];
      load_piece<DT, VEC>(wp[j], wat[j] + p, wv);
#pragma unroll
      for (int i = 0; i < TW; ++i)
#pragma unroll
        for (int k = 0; k < VEC; ++k) acc[i][j] += hv[i][k] * wv[k];
    }
  }
#pragma unroll
  for (int i = 0; i < TW; ++i)
#pragma unroll
    for (int j = 0; j < EW; ++j) {
      const float v = wave_sum(acc[i][j]);
      if (lane == 0 && t0 + i < n && e0 + j < rows) logits[(t0 + i) * rows + e0 + j] = v;
    }
}

// The choice of one token's experts from its logits, by one wave (`lane` of 64; LDS operations of a wave complete in order, so its lanes need no
// barrier between them).  LDS per token: scores [E], group score [G], group kept [G], chosen scores [top], and for SCORING 2 plain scores [E]
// (4096 experts, 4096 groups and 64 slots stay below the 64 KB of a launch).  SCORING 0: sigmoid scores, weights = chosen / sum; 1: the logits themselves rank the experts (no groups) and the weights are
// the softmax over the chosen logits alone; 2: scores = softmax over ALL logits (no groups), the experts are ranked by score + correction[e],
// the weights are the chosen scores themselves (not renormalised); the last `identity` experts have no weights of their own -- a slot that
// chose one keeps its id (>= experts - identity, which the sort by expert never places) and its score is added to extra_scale[t], the factor
// of the token's own input row; 3: sigmoid scores as in 0, but the weights are the chosen scores themselves (not renormalised); 4: scores =
// softmax over ALL logits, a group's score is its largest, weights = chosen / sum
struct SelectArgs {
  int rows, experts, top, group_count, group_keep, identity;
  float route_scale;
  int32_t* ids;
  float* weights;
  float* extra_scale;
  const void* correction;
};
__host__ __device__ static inline size_t select_floats(int scoring, int experts, int group_count, int top) {
  return (size_t)(scoring == 2 ? 2 : 1) * experts + 2 * group_count + top;
}

__device__ __forceinline__ void select_settle() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), lane));
}

// ... where neither groups nor many slots are asked for: a lane holds the scores of EL experts in registers, and the best is taken `top` times.
// Ranking every expert against every other takes experts^2 / 64 compares per token (68 experts: some 600 vector instructions, of which this needs
// some 250); sums in the same order, the same choices.  (A NaN ranks behind every number here, so that every slot gets an expert.)  us of router and
// sort in a graph, ranks -> this: 34 rows, top 4, 32 tokens 13.6 -> 13.1, 3264 33.0 -> 31.9; 68 rows, top 8, 32 tokens 18.5 -> 16.1, 3264 70.3 -> 66.7
constexpr int kSmallTop = 16;

template <int SCORING, int DT, int EL>
__device__ __forceinline__ void select_small(const SelectArgs& p, const float* z, int64_t t, int lane) {
  const int experts = p.experts, top = p.top;
  float zv[EL], shift[EL], plain[EL], score[EL];
#pragma unroll
  for (int i = 0; i < EL; ++i) {
    const int e = lane + 64 * i < experts ? lane + 64 * i : experts - 1;
    zv[i] = z[e];
    shift[i] = SCORING == 2 && p.correction ? ldv<DT>(p.correction, e) : 0.f;
  }
  float extra = 0.f;
  if (SCORING != 2 && p.extra_scale) extra = z[p.rows - 1];
  if constexpr (SCORING == 2 || SCORING == 4) {
    float top_z = zv[0];   // (a clamped lane repeats the last expert's)
#pragma unroll
    for (int i = 1; i < EL; ++i) top_z = fmaxf(top_z, zv[i]);
    top_z = wave_max(top_z);
    float total = 0.f;
#pragma unroll
    for (int i = 0; i < EL; ++i) {
      plain[i] = expf(zv[i] - top_z);
      const float term = lane + 64 * i < experts ? plain[i] : 0.f;   // (in index order, eight at a time: the last ones past the end add zeros)
      for (int e = 0; e < 64 && e + 64 * i < experts; e += 8)
#pragma unroll
        for (int j = 0; j < 8; ++j) total += lane_value(term, e + j);
    }
#pragma unroll
    for (int i = 0; i < EL; ++i) {
      plain[i] /= total;
      score[i] = SCORING == 2 && p.correction ? plain[i] + shift[i] : plain[i];
    }
  } else {
#pragma unroll
    for (int i = 0; i < EL; ++i) plain[i] = score[i] = SCORING == 1 ? zv[i] : sigmoid_exact(zv[i]);
  }
  if (SCORING != 2 && p.rows > experts && lane == 0) p.extra_scale[t] = sigmoid_exact(extra);
  bool left[EL];
#pragma unroll
  for (int i = 0; i < EL; ++i) left[i] = lane + 64 * i < experts;
  int id = 0;
  float own = 0.f, mine = 0.f, sum = 0.f, first = 0.f;   // lane k: slot k's expert and score; sums in the slots' order
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
#pragma unroll
    for (int i = 0; i < EL; ++i) best = left[i] ? fmaxf(best, score[i]) : best;
    best = wave_max(best);
    unsigned long long mask[EL];
#pragma unroll
    for (int i = 0; i < EL; ++i) mask[i] = __ballot(left[i] && score[i] == best);
    bool any = mask[0] != 0;
#pragma unroll
    for (int i = 1; i < EL; ++i) any = any || mask[i] != 0;
    if (!any) {   // only NaN is left
#pragma unroll
      for (int i = 0; i < EL; ++i) mask[i] = __ballot(left[i]);
    }
    int e = 0;
    float value = 0.f;
#pragma unroll
    for (int i = EL - 1; i >= 0; --i) {
      if (mask[i]) {
        const int l = __ffsll(mask[i]) - 1;
        e = l + 64 * i;
        value = lane_value(plain[i], l);
      }
    }
#pragma unroll
    for (int i = 0; i < EL; ++i) left[i] = left[i] && e != lane + 64 * i;
    if (SCORING == 2) own += e >= experts - p.identity ? value : 0.f;
    else if (SCORING == 1) {
      first = k == 0 ? value : first;
      value = expf(value - first);
      sum += value;
    } else sum += value;
    id = lane == k ? e : id;
    mine = lane == k ? value : mine;
  }
  if (SCORING == 2 && p.extra_scale && lane == 0) p.extra_scale[t] = own * p.route_scale;
  if (lane < top) {
    p.ids[t * top + lane] = id;
    p.weights[t * top + lane] = (SCORING == 1 ? mine / sum : SCORING == 2 || SCORING == 3 ? mine : mine / (sum + 1e-20f)) * p.route_scale;
  }
}

template <int SCORING, int DT>
__device__ __forceinline__ void select_token(const SelectArgs& p, const float* z, int64_t t, float* lds, int lane) {
  const int experts = p.experts, top = p.top;
  if (p.group_count == 1 && experts <= 128 && top <= kSmallTop) {
    if (experts <= 64) select_small<SCORING, DT, 1>(p, z, t, lane);
    else select_small<SCORING, DT, 2>(p, z, t, lane);
    return;
  }
  float* score = lds;
  float* gscore = score + experts;
  float* gkeep = gscore + p.group_count;
  float* chosen = gkeep + p.group_count;
  float* plain = SCORING == 2 ? chosen + top : score;
  if constexpr (SCORING == 2 || SCORING == 4) {
    // softmax over all experts: every lane adds the exponentials in index order (one value for the whole wave)
    float top_z = -INFINITY;
    for (int e = lane; e < experts; e += 64) top_z = fmaxf(top_z, z[e]);
    top_z = wave_max(top_z);
    for (int e = lane; e < experts; e += 64) plain[e] = expf(z[e] - top_z);
    float shift[2] = {0.f, 0.f};   // (the first 128 experts' corrections are requested before they are needed)
    if (SCORING == 2 && p.correction)
#pragma unroll
      for (int i = 0; i < 2; ++i) shift[i] = ldv<DT>(p.correction, lane + 64 * i < experts ? lane + 64 * i : 0);
    select_settle();
    float total = 0.f;
#pragma unroll 8
    for (int e = 0; e < experts; ++e) total += plain[e];   // (eight LDS reads on their way at a time)
    select_settle();
    for (int e = lane; e < experts; e += 64) {
      const float sc = plain[e] / total;
      plain[e] = sc;
      score[e] = SCORING == 2 && p.correction ? sc + (e < 64 ? shift[0] : e < 128 ? shift[1] : ldv<DT>(p.correction, e)) : sc;
    }
    if (SCORING == 4 && p.extra_scale)
      for (int e = experts + lane; e < p.rows; e += 64) p.extra_scale[t] = sigmoid_exact(z[e]);
  } else {
    for (int e = lane; e < p.rows; e += 64) {
      if (e < experts) score[e] = SCORING == 1 ? z[e] : sigmoid_exact(z[e]);
      else p.extra_scale[t] = sigmoid_exact(z[e]);
    }
  }
  select_settle();
  if constexpr (SCORING == 2) {
    auto place = [&](int e, int rank) {
      if (e < experts && rank < top) {
        p.ids[t * top + rank] = e;
        chosen[rank] = e >= experts - p.identity ? plain[e] : 0.f;   // (what the token's own row is scaled by)
        p.weights[t * top + rank] = plain[e] * p.route_scale;
      }
    };
    int e0 = lane;
    for (; e0 - lane + 64 < experts; e0 += 128) {   // two experts of a lane at a time
      const int e1 = e0 + 64;
      const float mine0 = score[e0], mine1 = score[e1 < experts ? e1 : 0];
      int rank0 = 0, rank1 = 0;
#pragma unroll 8
      for (int o = 0; o < experts; ++o) {
        const float sc = score[o];
        rank0 += (sc > mine0 || (sc == mine0 && o < e0)) ? 1 : 0;
        rank1 += (sc > mine1 || (sc == mine1 && o < e1)) ? 1 : 0;
      }
      place(e0, rank0);
      place(e1, rank1);
    }
    if (e0 - lane < experts) {
      const float mine = score[e0 < experts ? e0 : 0];
      int rank = 0;
#pragma unroll 8
      for (int o = 0; o < experts; ++o) {
        const float sc = score[o];
        rank += (sc > mine || (sc == mine && o < e0)) ? 1 : 0;
      }
      place(e0, rank);
    }
    select_settle();
    if (p.extra_scale) {                      // slots in rank order: the same sum whatever lane found which slot
      float own = 0.f;
#pragma unroll 8
      for (int k = 0; k < top; ++k) own += chosen[k];
      if (lane == 0) p.extra_scale[t] = own * p.route_scale;
    }
    return;
  }
  const int per = experts / p.group_count;
  for (int g = lane; g < p.group_count; g += 64) {
    float b1 = -INFINITY, b2 = -INFINITY;   // the two largest of the group
    for (int j = 0; j < per; ++j) {
      const float s = score[g * per + j];
      if (s > b1) { b2 = b1; b1 = s; }
      else if (s > b2) b2 = s;
    }
    gscore[g] = SCORING != 4 && per > 1 ? b1 + b2 : b1;
  }
  select_settle();
  for (int g = lane; g < p.group_count; g += 64) {
    const float mine = gscore[g];
    int rank = 0;
    for (int o = 0; o < p.group_count; ++o) {
      const float s = gscore[o];
      rank += (s > mine || (s == mine && o < g)) ? 1 : 0;
    }
    gkeep[g] = rank < p.group_keep ? 1.0f : 0.0f;
  }
  select_settle();
  for (int e = lane; e < experts; e += 64) {
    if (gkeep[e / per] == 0.0f) continue;
    const float mine = score[e];
    int rank = 0;
#pragma unroll 8
    for (int o = 0; o < experts; ++o) {
      const float s = score[o];
      rank += (gkeep[o / per] != 0.0f && (s > mine || (s == mine && o < e))) ? 1 : 0;
    }
    if (rank < top) {
      p.ids[t * top + rank] = e;
      chosen[rank] = mine;
    }
  }
  select_settle();
  float sum = 0.f;
  if constexpr (SCORING == 1) {   // chosen[0] is the largest: exp(z - z_max) summed in slot order by every lane
    for (int k = 0; k < top; ++k) sum += expf(chosen[k] - chosen[0]);
    for (int k = lane; k < top; k += 64) p.weights[t * top + k] = expf(chosen[k] - chosen[0]) / sum * p.route_scale;
  } else if constexpr (SCORING == 3) {
    for (int k = lane; k < top; k += 64) p.weights[t * top + k] = chosen[k] * p.route_scale;
  } else {
    for (int k = 0; k < top; ++k) sum += chosen[k];
    for (int k = lane; k < top; k += 64) p.weights[t * top + k] = chosen[k] / (sum + 1e-20f) * p.route_scale;
  }
}

// router of many experts, second launch: a wave per token over its logits
template <int SCORING, int DT>
__global__ __launch_bounds__(64) void group_select_kernel(const float* __restrict__ logits, const SelectArgs p) {
  extern __shared__ float lds[];
  select_token<SCORING, DT>(p, logits + (int64_t)blockIdx.x * p.rows, blockIdx.x, lds, threadIdx.x);
}

// ------------------------------------------------------------------------------------------------------------------------
// router in one launch (up to kRouterRows rows of weights): a workgroup of eight waves per TW tokens.  A wave owns an eighth of the rows, five at
// a time, and sums as the form above does (lanes' pieces in order, then the lanes in a fixed order: the same bits; 16-bit products are
// exact in fp32, so fused multiply-adds round where product and sum did); the logits meet in LDS and the first TW waves choose.
// Bound by its launch, one trip for the weights (L2: 140 KB per workgroup) and the chain of the choice.  us, logits and choice in two launches ->
// here, 34 rows of 2048, top 4: 1 token 12.9 -> 7.6, 262 14.4 -> 9.1, 512 24.5 -> 9.3, 3264
// 44 -> 23; 68 rows of 3072, top 8: 32 tokens 22.9 -> 12.9, 512 37 -> 21, 3264 85 -> 54 (three pieces of the width at a time on sixteen waves spill: 20).
// ------------------------------------------------------------------------------------------------------------------------
constexpr int kRouterRows = 512;

template <int SCORING, int DT, int VEC, int TW, int NW>
__global__ __launch_bounds__(64 * NW) void router_kernel(const void* __restrict__ h, int64_t h_ld, const void* __restrict__ w_router,
                                                     const void* __restrict__ w_extra, int width, int64_t n, const SelectArgs p) {
  constexpr int EW = 5, PU = TW > 1 ? 1 : NW == 8 ? 4 : 2;   // rows of weights and pieces of the width that are requested together
  extern __shared__ float lds[];                // [TW][rows] logits, then what select_token wants, TW times
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int64_t t0 = (int64_t)blockIdx.x * TW;
  const int rows = p.rows, share = (rows + NW - 1) / NW, from = wave * share, to = from + share < rows ? from + share : rows;
  int64_t hat[TW];
#pragma unroll
  for (int i = 0; i < TW; ++i) hat[i] = (t0 + i < n ? t0 + i : n - 1) * h_ld;
  for (int e0 = from; e0 < to; e0 += EW) {
    const void* wp[EW];
    int64_t wat[EW];
#pragma unroll
    for (int j = 0; j < EW; ++j) {
      const int e = e0 + j < to ? e0 + j : to - 1;
      wp[j] = e < p.experts ? w_router : w_extra;
      wat[j] = e < p.experts ? (int64_t)e * width : 0;
    }
    float acc[TW][EW];
#pragma unroll
    for (int i = 0; i < TW; ++i)
#pragma unroll
      for (int j = 0; j < EW; ++j) acc[i][j] = 0.f;
    for (int p0 = lane * VEC; p0 < width; p0 += 64 * VEC * PU) {
      float hv[PU][TW][VEC], wv[PU][EW][VEC];
#pragma unroll
      for (int u = 0; u < PU; ++u) {
        const int at = p0 + u * 64 * VEC;
        const bool in = at < width;
#pragma unroll
        for (int i = 0; i < TW; ++i) {
          load_piece<DT, VEC>(h, hat[i] + (in ? at : p0), hv[u][i]);
          if (!in)
#pragma unroll
            for (int k = 0; k < VEC; ++k) hv[u][i][k] = 0.f;
        }
#pragma unroll
        for (int j = 0; j < EW; ++j) {
          load_piece<DT, VEC>(wp[j], wat[j] + (in ? at : p0), wv[u][j]);
          if (!in)
#pragma unroll
            for (int k = 0; k < VEC; ++k) wv[u][j][k] = 0.f;
        }
      }
#pragma unroll
      for (int u = 0; u < PU; ++u)
#pragma unroll
        for (int j = 0; j < EW; ++j)
#pragma unroll
          for (int i = 0; i < TW; ++i)
#pragma unroll
            for (int k = 0; k < VEC; ++k) {
              if constexpr (DT == LL_F32) acc[i][j] += hv[u][i][k] * wv[u][j][k];
              else acc[i][j] = __builtin_fmaf(hv[u][i][k], wv[u][j][k], acc[i][j]);
            }
    }
#pragma unroll
    for (int i = 0; i < TW; ++i)
#pragma unroll
      for (int j = 0; j < EW; ++j) {
        const float v = wave_sum(acc[i][j]);
        if (lane == 0 && e0 + j < to) lds[i * rows + e0 + j] = v;
      }
  }
  __syncthreads();
  if (wave < TW && t0 + wave < n) {
    const int64_t each = (int64_t)select_floats(SCORING, p.experts, p.group_count, p.top);
    select_token<SCORING, DT>(p, lds + wave * rows, t0 + wave, lds + TW * rows + wave * each, lane);
  }
}

// ------------------------------------------------------------------------------------------------------------------------
// sort by expert.  Up to kSortExperts experts one launch, a workgroup per expert: it counts every expert in front of its own in LDS (its run's
// start), each wave the own expert's slots of its share of the step, then every wave places its share behind the earlier ones --
// two passes over the ids, no barrier inside them.  With `skipped`, a last workgroup places the slots that no expert serves
// (ids outside 0 .. experts - 1) in a run of their own whose blocks name expert -1: their rows of the result are zeros.  Bound by its
// launch and a few trips to memory; us, count and place in two launches -> here: 128 slots 10.4 -> 5.5, 13 056 slots 36 -> 11.8
// ------------------------------------------------------------------------------------------------------------------------
constexpr int kSortExperts = 8192;
constexpr int kSortWaves = 16;   // most waves of a workgroup

// hist: LDS [experts], counts of the experts in front of this workgroup's
__device__ __forceinline__ void sort_expert(const int32_t* ids, int num_slots, int experts, int block_m, int skipped, int* hist,
                                            int32_t* __restrict__ counts, int32_t* __restrict__ sorted, int32_t* __restrict__ block_expert,
                                            int32_t* __restrict__ num_post) {
  __shared__ int part[kSortWaves], start[kSortWaves];
  const int e = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, threads = blockDim.x, waves = threads >> 6;
  for (int i = tid; i < e; i += threads) hist[i] = 0;
  __syncthreads();
  const int share = (num_slots + waves - 1) / waves, lo = wave * share, hi = lo + share < num_slots ? lo + share : num_slots;
  auto mine = [&](int id) { return e < experts ? id == e : (id < 0 || id >= experts); };
  int own = 0;
#pragma unroll 4
  for (int i = lo + lane; i < hi; i += 64) {
    const int id = ids[i];
    own += mine(id) ? 1 : 0;
    if (id >= 0 && id < e && id < experts) atomicAdd(&hist[id], 1);
  }
  for (int off = 32; off > 0; off >>= 1) own += __shfl_xor(own, off);
  if (lane == 0) part[wave] = own;
  __syncthreads();
  int base = 0;
  for (int o = tid; o < e; o += threads) base += (hist[o] + block_m - 1) / block_m * block_m;
  for (int off = 32; off > 0; off >>= 1) base += __shfl_xor(base, off);
  if (lane == 0) start[wave] = base;
  __syncthreads();
  base = 0;
  int total = 0;
  for (int w = 0; w < waves; ++w) {
    base += start[w];
    total += part[w];
  }
  const int padded = (total + block_m - 1) / block_m * block_m;
  int at = base;
  for (int w = 0; w < wave; ++w) at += part[w];
#pragma unroll 4
  for (int i0 = lo; i0 < hi; i0 += 64) {
    const int i = i0 + lane;
    const bool hit = i < hi && mine(ids[i]);
    const unsigned long long mask = __ballot(hit);
    if (hit) sorted[at + __popcll(mask & ((1ull << lane) - 1ull))] = i;
    at += __popcll(mask);
  }
  for (int i = total + tid; i < padded; i += threads) sorted[base + i] = num_slots;
  for (int b = tid; b < padded / block_m; b += threads) block_expert[base / block_m + b] = e < experts ? e : -1;
  if (tid == 0) {
    if (e < experts) counts[e] = total;
    if (e == experts - 1 + skipped) num_post[0] = base + padded;
  }
}

__global__ __launch_bounds__(1024) void moe_sort_kernel(const int32_t* __restrict__ ids, int num_slots, int experts, int block_m, int skipped,
                                                       int32_t* __restrict__ counts, int32_t* __restrict__ sorted,
                                                       int32_t* __restrict__ block_expert, int32_t* __restrict__ num_post) {
  extern __shared__ int hist[];
  sort_expert(ids, num_slots, experts, block_m, skipped, hist, counts, sorted, block_expert, num_post);
}

// ------------------------------------------------------------------------------------------------------------------------
// router and sort of few tokens (up to kRouteTokens): the logits by a wave per token and two rows, all over the chip, then ONE launch in which
// each expert's workgroup chooses for every token by itself (the choices stay in LDS; the first workgroup writes them out) and sorts its slots.
// In a workgroup per token as above the weights come through one CU each, 20 - 25 KB/us where they are not in its L2: at few tokens
// that, and not the choice, was the launch's time.  Sums in router_kernel's order: the same bits.
// ------------------------------------------------------------------------------------------------------------------------
constexpr int kRouteTokens = 16;

template <int DT, int VEC>
__global__ __launch_bounds__(64) void route_logits_kernel(const void* __restrict__ h, int64_t h_ld, const void* __restrict__ w_router,
                                                          const void* __restrict__ w_extra, int width, int experts, int rows,
                                                          float* __restrict__ logits) {
  constexpr int EW = 2, PU = 8;   // rows of weights; pieces of the width that are requested together
  const int lane = threadIdx.x, e0 = blockIdx.x * EW;
  const int64_t hat = (int64_t)blockIdx.y * h_ld;
  const void* wp[EW];
  int64_t wat[EW];
#pragma unroll
  for (int j = 0; j < EW; ++j) {
    const int e = e0 + j < rows ? e0 + j : rows - 1;
    wp[j] = e < experts ? w_router : w_extra;
    wat[j] = e < experts ? (int64_t)e * width : 0;
  }
  float acc[EW] = {};
  for (int p0 = lane * VEC; p0 < width; p0 += 64 * VEC * PU) {
    float hv[PU][VEC], wv[PU][EW][VEC];
#pragma unroll
    for (int u = 0; u < PU; ++u) {
      const int at = p0 + u * 64 * VEC;
      const bool in = at < width;
#pragma unroll
      for (int j = 0; j < EW; ++j) load_piece<DT, VEC>(wp[j], wat[j] + (in ? at : p0), wv[u][j]);
      load_piece<DT, VEC>(h, hat + (in ? at : p0), hv[u]);
#pragma unroll
      for (int k = 0; k < VEC; ++k) {
        hv[u][k] = in ? hv[u][k] : 0.f;
#pragma unroll
        for (int j = 0; j < EW; ++j) wv[u][j][k] = in ? wv[u][j][k] : 0.f;
      }
    }
#pragma unroll
    for (int u = 0; u < PU; ++u)
#pragma unroll
      for (int j = 0; j < EW; ++j)
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
          if constexpr (DT == LL_F32) acc[j] += hv[u][k] * wv[u][j][k];
          else acc[j] = __builtin_fmaf(hv[u][k], wv[u][j][k], acc[j]);
        }
  }
#pragma unroll
  for (int j = 0; j < EW; ++j) {
    const float v = wave_sum(acc[j]);
    if (lane == 0 && e0 + j < rows) logits[(int64_t)blockIdx.y * rows + e0 + j] = v;
  }
}

// sorted_experts: those with weights (ids beyond them are identity experts); LDS: hist [sorted_experts], the choices' ids and weights [n top] and
// extra [n], then what select_token wants, once per wave
template <int SCORING, int DT>
__global__ __launch_bounds__(1024) void route_sort_kernel(const float* __restrict__ logits, const SelectArgs p, int n, int sorted_experts, int block_m,
                                                          int skipped, int32_t* __restrict__ counts, int32_t* __restrict__ sorted,
                                                          int32_t* __restrict__ block_expert, int32_t* __restrict__ num_post) {
  extern __shared__ int route_lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), waves = (int)blockDim.x >> 6;
  const int slots = n * p.top;
  int32_t* ids = route_lds + sorted_experts;
  float* weights = (float*)(ids + slots);
  float* extra = weights + slots;
  float* scratch = extra + n + (size_t)wave * select_floats(SCORING, p.experts, p.group_count, p.top);
  SelectArgs q = p;
  q.ids = ids;
  q.weights = weights;
  q.extra_scale = p.extra_scale ? extra : nullptr;
  for (int i = threadIdx.x; i < slots; i += blockDim.x) {   // (a slot that NaN logits leave without an expert is one that no expert serves)
    ids[i] = -1;
    weights[i] = 0.f;
  }
  __syncthreads();
  for (int t = wave; t < n; t += waves) {
    select_token<SCORING, DT>(q, logits + (int64_t)t * p.rows, t, scratch, lane);
    select_settle();   // (the next token's scores take this one's place)
  }
  __syncthreads();
  if (blockIdx.x == 0) {
    for (int i = threadIdx.x; i < slots; i += blockDim.x) {
      p.ids[i] = ids[i];
      p.weights[i] = weights[i];
    }
    if (p.extra_scale)
      for (int i = threadIdx.x; i < n; i += blockDim.x) p.extra_scale[i] = extra[i];
  }
  sort_expert(ids, slots, sorted_experts, block_m, skipped, route_lds, counts, sorted, block_expert, num_post);
}

// more experts: a workgroup per expert, twice (count, then place)
__global__ __launch_bounds__(256) void moe_count_kernel(const int32_t* __restrict__ ids, int num_slots, int32_t* __restrict__ counts) {
  __shared__ int part[4];
  const int e = blockIdx.x, tid = threadIdx.x;
  int c = 0;
  for (int i = tid; i < num_slots; i += 256) c += ids[i] == e ? 1 : 0;
  for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
  if ((tid & 63) == 0) part[tid >> 6] = c;
  __syncthreads();
  if (tid == 0) counts[e] = part[0] + part[1] + part[2] + part[3];
}

__global__ __launch_bounds__(256) void moe_place_kernel(const int32_t* __restrict__ ids, int num_slots, int experts, int block_m,
                                                        const int32_t* __restrict__ counts, int32_t* __restrict__ sorted,
                                                        int32_t* __restrict__ block_expert, int32_t* __restrict__ num_post) {
  __shared__ int wtot[4];
  const int e = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int base = 0;
  for (int o = 0; o < e; ++o) base += (counts[o] + block_m - 1) / block_m * block_m;
  const int mine = counts[e];
  const int padded = (mine + block_m - 1) / block_m * block_m;
  int running = 0;
  for (int at = 0; at < num_slots; at += 256) {
    const int i = at + tid;
    const bool hit = i < num_slots && ids[i] == e;
    const unsigned long long mask = __ballot(hit);
    const int before = __popcll(mask & ((1ull << lane) - 1ull));
    __syncthreads();   // (the previous round's totals have been read)
    if (lane == 0) wtot[wave] = __popcll(mask);
    __syncthreads();
    int off = running;
    for (int w = 0; w < wave; ++w) off += wtot[w];
    if (hit) sorted[base + off + before] = i;
    running += wtot[0] + wtot[1] + wtot[2] + wtot[3];
  }
  for (int i = mine + tid; i < padded; i += 256) sorted[base + i] = num_slots;
  for (int b = tid; b < padded / block_m; b += 256) block_expert[base / block_m + b] = e;
  if (e == experts - 1 && tid == 0) num_post[0] = base + padded;
}

// ------------------------------------------------------------------------------------------------------------------------
// grouped products, plain tiled form: 32 sorted rows x 64 columns per workgroup, 32 contraction entries per pass
// ------------------------------------------------------------------------------------------------------------------------
template <int DT, int MODE>
__global__ __launch_bounds__(256) void moe_rows_gemm_kernel(const void* __restrict__ a, int64_t a_ld, int a_div,
                                                            const void* __restrict__ w, int64_t w_stride_e, int K, int N,
                                                            const float* __restrict__ slot_weight, void* __restrict__ out,
                                                            int64_t out_ld, const int32_t* __restrict__ sorted,
                                                            const int32_t* __restrict__ block_expert,
                                                            const int32_t* __restrict__ num_post, int num_slots, float glu_limit, int shift) {
  constexpr bool GLU = MODE == 1;
  constexpr int BM = 32, BN = 64, BK = 32;
  __shared__ float As[BM][BK + 1];
  __shared__ int rows[BM];
  // (sorted in blocks of 32 << shift rows.  The first 32 rows of all blocks, then the next of all: where one row tile per block is in use, neighbours in
  // the grid, which go to different XCDs, all have work -- in the rows' own order every fourth had, on two XCDs of eight: 32 tokens of 8 experts each,
  // 128 experts of 1024 / 132 in 16 bits 71 us with blocks of 32 rows, 140 with blocks of 128, 61 so)
  const int blocks = (int)(gridDim.x >> shift), block = (((int)blockIdx.x % blocks) << shift) + (int)blockIdx.x / blocks;
  if (block * BM >= num_post[0]) return;
  const int e = block_expert[block >> shift];
  if (sorted[block * BM] >= num_slots) return;
  if (e < 0) {   // slots that no expert serves: zeros (of the last product; nothing reads the first one's)
    if (GLU) return;
    for (int i = threadIdx.x; i < BM * BN; i += 256) {
      const int slot = sorted[block * BM + i / BN], c = blockIdx.y * BN + i % BN;
      if (slot < num_slots && c < N) stv<DT>(out, (int64_t)slot * out_ld + c, 0.f);
    }
    return;
  }
  const int tid = threadIdx.x, tx = tid & 63, ty = tid >> 6;
  if (tid < BM) rows[tid] = sorted[block * BM + tid];
  const int col = blockIdx.y * BN + tx;
  const bool colok = col < N;
  const int64_t wg_at = (int64_t)e * w_stride_e + (int64_t)col * K;
  const int64_t wu_at = (int64_t)e * w_stride_e + (int64_t)(N + col) * K;
  float acc_g[8], acc_u[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) acc_g[r] = acc_u[r] = 0.f;
  for (int k0 = 0; k0 < K; k0 += BK) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < BM * BK / 256; ++u) {
      const int idx = tid + 256 * u, r = idx / BK, kk = idx - r * BK;
      const int slot = rows[r];
      As[r][kk] = (slot < num_slots && k0 + kk < K) ? ldv<DT>(a, (int64_t)(slot / a_div) * a_ld + k0 + kk) : 0.f;
    }
    __syncthreads();
    if (colok) {
      const int kn = K - k0 < BK ? K - k0 : BK;
      for (int kk = 0; kk < kn; ++kk) {
        const float wg = ldv<DT>(w, wg_at + k0 + kk);
        const float wu = GLU ? ldv<DT>(w, wu_at + k0 + kk) : 0.f;
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          const float av = As[ty * 8 + r][kk];
          acc_g[r] += av * wg;
          if (GLU) acc_u[r] += av * wu;
        }
      }
    }
  }
  if (!colok) return;
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const int slot = rows[ty * 8 + r];
    if (slot >= num_slots) continue;
    float v;
    if (GLU) {
      v = glu_pair<DT>(acc_g[r], acc_u[r], glu_limit);
    } else {
      v = slot_value<MODE>(acc_g[r], slot_weight ? slot_weight[slot] : 1.0f);
    }
    stv<DT>(out, (int64_t)slot * out_ld + col, v);
  }
}

struct alignas(16) Q4 {
  uint32_t x, y, z, w;
};

// ------------------------------------------------------------------------------------------------------------------------
// grouped products, LDS-tiled MFMA form for blocks of 128 sorted rows: a workgroup of four waves owns a block's rows x 128 weight rows
// (gate|up: 64 output columns, their gate rows and up rows) and walks the contraction in steps of 64.
//   * Both tiles go global -> LDS by LDS-DMA as 128-byte row pieces, slot s of row r at s ^ ((r >> 1) & 7) (through the source address):
//     fragment reads are bank-conflict free.  Weights sit three steps deep, rows two (80 KB: two workgroups per CU): 32 KB of weights of
//     a CU are always on their way, which is what streaming them from memory needs.  One barrier per step.
//   * Row tiles without a slot are not multiplied; wave (wr, wc) owns row tiles wr and wr + 2 (of 32 rows) and two weight tiles, so that
//     a half-full block still keeps every matrix core busy.
//   * Tiles are dealt to the XCDs in contiguous ranges of the tiles that exist (num_post, a device value), four blocks side by side under
//     one weight tile: blocks of one expert read it from the XCD's own L2.
// us for both products, 32 experts of 2048 / 704 with 384 / 706 rows each: 362 / 602 with one buffer filled through registers and two barriers
// per step, 254 / 427 with a step's requests in front of its products (0.48 PFLOP/s: two operand tiles per 128 x 128 results through L2); at 70 rows
// each 95 us, of which the weights alone need 55.  With the requests between the products, from 32-bit offsets, before -> now: 32 experts of 2048 / 704,
// 1500 tokens with 4 experts each 146 -> 137, 3100 236 -> 209, 4096 280 -> 243; 64 of 3072 / 512 with 8 each, 1500 tokens 335 -> 291, 4096 627 -> 577;
// up to 1000 tokens of either as before (the weights' stream).
// ------------------------------------------------------------------------------------------------------------------------
__device__ const uint32_t moe_zeros[4] __attribute__((aligned(16))) = {0, 0, 0, 0};   // what pieces behind the contraction's end read

// 64 lanes x 16 bytes from per-lane addresses to 1 KB of LDS at byte `dst` (counted by vmcnt, which the compiler does not see)
__device__ __forceinline__ void dma16(uint32_t dst, const void* src) {
  dst = __builtin_amdgcn_readfirstlane(dst);
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "s"(dst), "v"(src) : "memory");
}
// ... from a wave-uniform address and 32-bit offsets
__device__ __forceinline__ void dma16(uint32_t dst, const void* base, uint32_t off) {
  dst = __builtin_amdgcn_readfirstlane(dst);
  const uint64_t at = (uint64_t)base;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)at), hi = __builtin_amdgcn_readfirstlane((uint32_t)(at >> 32));   // (each back in 32 bits)
  base = (const void*)(((uint64_t)hi << 32) | lo);
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "s"(dst), "v"(off), "s"(base) : "memory");
}
template <int DT>
__device__ __forceinline__ f32x16 mfma32(const Q4& a, const Q4& b, f32x16 c) {
  if constexpr (DT == LL_F16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

template <int DT, int MODE, bool FAR>
__global__ __launch_bounds__(256, 2) void moe_rows_gemm_tiled_kernel(const uint16_t* __restrict__ a, int64_t a_ld, int a_div,
                                                                     const uint16_t* __restrict__ w, int64_t w_stride_e, int K, int N,
                                                                     const float* __restrict__ slot_weight, uint16_t* __restrict__ out,
                                                                     int64_t out_ld, const int32_t* __restrict__ sorted,
                                                                     const int32_t* __restrict__ block_expert,
                                                                     const int32_t* __restrict__ num_post, int num_slots, float glu_limit,
                                                                     int tiles_n, int wide, int few, int sure) {
  constexpr bool GLU = MODE == 1;
  constexpr int CW = GLU ? 64 : 128, TILE = 128 * 128;   // output columns; bytes of a stage's operand
  extern __shared__ __attribute__((aligned(16))) unsigned char tile_lds[];   // rows x 2, weights x 3
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave & 1, wc = wave >> 1, tl = lane & 31, h = lane >> 5;
  int block, nt;
  if (few > 0) {   // (`few` blocks at most: every tile has its place in the grid, and nothing below waits for num_post)
    nt = (int)blockIdx.x / few;
    block = (int)blockIdx.x - nt * few;
    if (block >= sure && block * 128 >= num_post[0]) return;   // (the lists reach that far only if a run of skipped slots does)
  } else {
    const int blocks = num_post[0] / 128;
    const int total = blocks * tiles_n;   // (below 2^31: checked on the host for the largest count)
    const int xcd = blockIdx.x & 7;
    const int first = (int)((int64_t)total * xcd / 8), last = (int)((int64_t)total * (xcd + 1) / 8);
    const int at = first + (int)(blockIdx.x >> 3);
    if (at >= last) return;
    const int per = 4 * tiles_n, g4 = at / per, in4 = at - g4 * per;
    const int side = blocks - 4 * g4 < 4 ? blocks - 4 * g4 : 4;
    nt = in4 / side;
    block = 4 * g4 + (in4 - nt * side);
  }
  const int n0 = nt * CW;
  const int32_t* srt = sorted + (int64_t)block * 128;
  int e = block_expert[block], own[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) own[j] = srt[(wave * 4 + j) * 8 + (lane >> 3)];
  if (few > 0) {
    int post = num_post[0];
    asm volatile("" : "+s"(post), "+s"(e), "+v"(own[0]), "+v"(own[1]), "+v"(own[2]), "+v"(own[3]));   // (requested together)
    if (block * 128 >= post) return;   // (nothing was sorted there: no address has been made of it yet)
  }
  if (e < 0) {   // slots that no expert serves: zeros (of the last product; nothing reads the first one's)
    if (GLU) return;
    for (int i = tid; i < 128 * CW; i += 256) {
      const int slot = srt[i / CW], c = n0 + i % CW;
      if (slot < num_slots && c < N) out[(int64_t)slot * out_ld + c] = 0;
    }
    return;
  }
  // what this thread requests of a step: row (and weight row) 8 (4 wave + j) + lane / 8, one swizzled 16-byte piece of it: offsets from the
  // operand's (the expert's) first byte, in 32 bits where the host has seen that they fit
  using Off = std::conditional_t<FAR, uint64_t, uint32_t>;
  const char* abase = (const char*)a;
  const char* wbase = (const char*)(w + (int64_t)e * w_stride_e);
  Off aoff[4], woff[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = (wave * 4 + j) * 8 + (lane >> 3), piece = ((lane & 7) ^ ((r >> 1) & 7)) * 16;
    const int slot = own[j];   // (rows without a slot read row 0, columns >= N the last: they feed only unstored results)
    aoff[j] = (slot < num_slots ? (Off)(slot / a_div) : (Off)0) * (Off)(a_ld * 2) + piece;
    int col = GLU ? n0 + (r & 63) : n0 + r;
    col = col < N ? col : N - 1;
    woff[j] = (Off)(GLU && r >= 64 ? (Off)N + col : (Off)col) * ((Off)K * 2) + piece;
  }
  // request j of step s; the pieces of a last, partial step that lie behind the contraction read zeros, and so do steps behind the last one
  const int whole = K / 64;
  auto get = [&](uint32_t dst, const char* base, Off off, int j, int s, bool inside) {
    if (inside || s < whole) {
      if constexpr (FAR) dma16(dst, base + (int64_t)s * 128 + off);
      else dma16(dst, base + (int64_t)s * 128, off);
    } else {
      const int r = (wave * 4 + j) * 8 + (lane >> 3), piece = ((lane & 7) ^ ((r >> 1) & 7)) * 8;
      dma16(dst, s * 64 + piece < K ? base + (int64_t)s * 128 + off : (const char*)moe_zeros);
    }
  };
  auto get_a = [&](int s, int j, bool inside) { get((uint32_t)((s & 1) * TILE + (wave * 4 + j) * 1024), abase, aoff[j], j, s, inside); };
  auto get_w = [&](int s, int j, int buf, bool inside) {
    get((uint32_t)((2 + buf) * TILE + (wave * 4 + j) * 1024), wbase, woff[j], j, s, inside);
  };
  const bool act0 = srt[32 * wr] < num_slots, act1 = srt[32 * (wr + 2)] < num_slots;   // (an expert's empty rows stand last)
  f32x16 acc[2][2];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[m][j][r] = 0.f;
  const int sw = (tl >> 1) & 7;
  const unsigned char* arow = tile_lds + (32 * wr + tl) * 128;
  const unsigned char* wrow0 = tile_lds + 2 * TILE + ((GLU ? 32 * wc : 64 * wc) + tl) * 128;
  const int wrow1 = (GLU ? 64 : 32) * 128;
#pragma unroll
  for (int j = 0; j < 4; ++j) get_a(0, j, false);
#pragma unroll
  for (int j = 0; j < 4; ++j) get_w(0, j, 0, false);
#pragma unroll
  for (int j = 0; j < 4; ++j) get_w(1, j, 1, false);
  const int steps = (K + 63) / 64;
  // A step in four quarters of 16 columns: the fragments of the next quarter are read and two of the eight requests are issued between the products
  // of this one (a request occupies its wave for some 80 cycles: in front of the step's fragments, as they were, eight of them kept the
  // matrix cores waiting for longer than the products take).  MI: row tiles of this wave that hold a slot
  auto walk = [&](auto tag) {
    constexpr int MI = decltype(tag)::value;
    int buf = 0;
    auto step = [&](int s, auto inside) {   // (inside: what the step requests lies in whole steps)
      constexpr bool IN = decltype(inside)::value;
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0x0074);   // all but the last four requests (the weights of step s + 1); own fragment reads
      __builtin_amdgcn_s_barrier();
      const unsigned char* ap = arow + (s & 1) * TILE;
      const unsigned char* wp = wrow0 + buf * TILE;
      const int wbuf = buf == 0 ? 2 : buf - 1;   // (the buffer step s - 1 has been read from)
      Q4 wf[2][2], af[2][2];
      auto read = [&](int q) {
        const int o = ((2 * q + h) ^ sw) * 16;
        if constexpr (MI > 0) {
          wf[q & 1][0] = *reinterpret_cast<const Q4*>(wp + o);
          af[q & 1][0] = *reinterpret_cast<const Q4*>(ap + o);
          wf[q & 1][1] = *reinterpret_cast<const Q4*>(wp + wrow1 + o);
          if constexpr (MI > 1) af[q & 1][1] = *reinterpret_cast<const Q4*>(ap + 64 * 128 + o);
        }
      };
      read(0);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (q < 3) read(q + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 2; ++i) {   // (the rows' four requests in front of the weights': the wait above counts on it)
          if constexpr (MI > 0) {
            acc[0][i] = mfma32<DT>(wf[q & 1][i], af[q & 1][0], acc[0][i]);
            if constexpr (MI > 1) acc[1][i] = mfma32<DT>(wf[q & 1][i], af[q & 1][1], acc[1][i]);
          }
          __builtin_amdgcn_sched_barrier(0);
          if (q < 2) get_a(s + 1, 2 * q + i, IN);
          else get_w(s + 2, 2 * (q - 2) + i, wbuf, IN);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      buf = buf == 2 ? 0 : buf + 1;
    };
    int s = 0;
    for (; s + 2 < whole; ++s) step(s, std::true_type{});
    for (; s < steps; ++s) step(s, std::false_type{});
  };
  if (!act0) walk(std::integral_constant<int, 0>{});
  else if (!act1) walk(std::integral_constant<int, 1>{});
  else walk(std::integral_constant<int, 2>{});
  __builtin_amdgcn_s_waitcnt(0x0070);   // (requests past the end have landed before the LDS is given back)
  if (!act0) return;
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const int slot = srt[32 * (wr + 2 * m) + tl];
    if (slot >= num_slots) continue;
    const float weight = !GLU && slot_weight ? slot_weight[slot] : 1.0f;
    uint16_t* orow = out + (int64_t)slot * out_ld;
#pragma unroll
    for (int j = 0; j < (GLU ? 1 : 2); ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {   // result 4 q + i of the lane: weight row 8 q + 4 h + i of the tile
        const int col = n0 + (GLU ? 32 * wc : 64 * wc + 32 * j) + 8 * q + 4 * h;
        uint16_t y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float v = acc[m][j][4 * q + i];
          y[i] = from_f32<DT>(GLU ? glu_pair<DT>(v, acc[m][1][4 * q + i], glu_limit) : slot_value<MODE>(v, weight));
        }
        if (wide) {
          if (col < N) *reinterpret_cast<uint2*>(orow + col) = uint2{(uint32_t)y[0] | (uint32_t)y[1] << 16, (uint32_t)y[2] | (uint32_t)y[3] << 16};
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (col + i < N) orow[col + i] = y[i];
        }
      }
  }
}

}  // namespace

#define LL_BY_DTYPE(dtype, CALL)             \
  do {                                       \
    if (dtype == LL_F16) { CALL(LL_F16); }   \
    else if (dtype == LL_BF16) { CALL(LL_BF16); } \
    else { CALL(LL_F32); }                   \
  } while (0)

struct RouterCall {
  SelectArgs p;
  size_t each;   // floats of LDS for one token's choice
  bool aligned;
};

static int router_call(RouterCall& c, const void* h, int64_t h_ld, const void* w_router, const void* w_extra, int64_t n, int64_t width,
                       int64_t experts, int64_t top, int64_t group_count, int64_t group_keep, float route_scale, int scoring, int32_t* ids,
                       float* weights, float* extra_scale, float* logits, const void* correction, int64_t identity, int dtype) {
  if (dtype != LL_F16 && dtype != LL_BF16 && dtype != LL_F32) return LL_ERR_DTYPE;
  if (scoring == 2 && (group_count != 1 || w_extra || identity < 0 || identity > experts || (identity > 0 && !extra_scale)))
    return LL_ERR_SHAPE;
  if (scoring != 2 && (correction || identity)) return LL_ERR_SHAPE;
  if (n < 0 || width < 1 || h_ld < width || experts < 1 || experts > 4096 || top < 1 || top > experts || top > 64 || group_count < 1 ||
      experts % group_count || group_keep < 1 || group_keep > group_count || group_keep * (experts / group_count) < top ||
      scoring < 0 || scoring > 4 || (scoring == 1 && group_count != 1))
    return LL_ERR_SHAPE;
  if (n > 0 && (!h || !w_router || !ids || !weights || !logits || (w_extra && !extra_scale))) return LL_ERR_ARG;
  const int rows = (int)experts + (w_extra ? 1 : 0);
  const int vec = dtype == LL_F32 ? 4 : 8;
  c.aligned = width % vec == 0 && h_ld % vec == 0 && ll_aligned16(h) && ll_aligned16(w_router) && (!w_extra || ll_aligned16(w_extra));
  c.p = SelectArgs{rows, (int)experts, (int)top, (int)group_count, (int)group_keep, (int)identity, route_scale, ids, weights, extra_scale, correction};
  c.each = select_floats(scoring, (int)experts, (int)group_count, (int)top);
  return LL_OK;
}

// logits: fp32 scratch [n][experts + (w_extra ? 1 : 0)], written where the router takes two launches (more than kRouterRows rows)
extern "C" int ll_group_router(const void* h, int64_t h_ld, const void* w_router, const void* w_extra, int64_t n, int64_t width,
                               int64_t experts, int64_t top, int64_t group_count, int64_t group_keep, float route_scale, int scoring,
                               int32_t* ids, float* weights, float* extra_scale, float* logits, const void* correction, int64_t identity,
                               int dtype, void* stream) {
  RouterCall c;
  const int bad = router_call(c, h, h_ld, w_router, w_extra, n, width, experts, top, group_count, group_keep, route_scale, scoring, ids, weights,
                              extra_scale, logits, correction, identity, dtype);
  if (bad || n == 0) return bad;
  const SelectArgs& p = c.p;
  const int rows = p.rows;
  const size_t each = c.each;
  const bool aligned = c.aligned;
  hipStream_t st = (hipStream_t)stream;
  if (rows <= kRouterRows) {
    const int tw = n > 256 ? 4 : 1, nw = tw == 1 && rows > 40 ? 16 : 8;   // tokens per workgroup; waves
    const dim3 grid((unsigned)((n + tw - 1) / tw));
    const size_t lds = sizeof(float) * tw * (rows + each);
#define LL_R(S, DT, V, T, W) router_kernel<S, DT, V, T, W><<<grid, 64 * W, lds, st>>>(h, h_ld, w_router, w_extra, (int)width, n, p)
#define LL_RT(S, DT, V) do { if (tw == 4) LL_R(S, DT, V, 4, 8); else if (nw == 16) LL_R(S, DT, V, 1, 16); else LL_R(S, DT, V, 1, 8); } while (0)
#define LL_RV(S, DT, V) do { if (aligned) LL_RT(S, DT, V); else LL_RT(S, DT, 1); } while (0)
#define LL_RS(DT, V)                                                                                                                  \
  do {                                                                                                                                \
    if (scoring == 0) LL_RV(0, DT, V); else if (scoring == 1) LL_RV(1, DT, V); else if (scoring == 2) LL_RV(2, DT, V);                \
    else if (scoring == 3) LL_RV(3, DT, V); else LL_RV(4, DT, V);                                                                     \
  } while (0)
    if (dtype == LL_F32) LL_RS(LL_F32, 4); else if (dtype == LL_F16) LL_RS(LL_F16, 8); else LL_RS(LL_BF16, 8);
#undef LL_RS
#undef LL_RV
#undef LL_RT
#undef LL_R
    return LL_LAUNCH_CHECK();
  }
  const int ew = n >= 512 ? 8 : 2;   // weight rows per wave
  const dim3 grid((unsigned)((n + 7) / 8), (unsigned)((rows + 4 * ew - 1) / (4 * ew)));
#define LL_RL_ARGS h, h_ld, w_router, w_extra, (int)width, (int)experts, rows, logits, n
#define LL_RL(DT, V)                                                                         \
  if (ew == 8) router_logits_kernel<DT, V, 8><<<grid, 256, 0, st>>>(LL_RL_ARGS);             \
  else router_logits_kernel<DT, V, 2><<<grid, 256, 0, st>>>(LL_RL_ARGS)
  if (!aligned) {
#define CALL(DT) LL_RL(DT, 1)
    LL_BY_DTYPE(dtype, CALL);
#undef CALL
  } else if (dtype == LL_F32) {
    LL_RL(LL_F32, 4);
  } else if (dtype == LL_F16) {
    LL_RL(LL_F16, 8);
  } else {
    LL_RL(LL_BF16, 8);
  }
#undef LL_RL
#undef LL_RL_ARGS
  const size_t lds = sizeof(float) * each;
#define LL_GS(S, DT) group_select_kernel<S, DT><<<dim3((unsigned)n), 64, lds, st>>>(logits, p)
  if (scoring == 2) {
#define CALL(DT) LL_GS(2, DT)
    LL_BY_DTYPE(dtype, CALL);
#undef CALL
  } else if (scoring == 1) LL_GS(1, LL_F32);
  else if (scoring == 4) LL_GS(4, LL_F32);
  else if (scoring == 3) LL_GS(3, LL_F32);
  else LL_GS(0, LL_F32);
#undef LL_GS
  return LL_LAUNCH_CHECK();
}

// rows per sorted block: 128 (the LDS-tiled form) where a 16-bit matrix-core product applies to either contraction, else 32.  At any number of
// rows: a form of one wave per 32 rows x 32 columns straight from memory, which it replaced, was slower down to a few decoded tokens (both
// products, us, that form -> this one: 64 experts of 3072 / 512, 6 tokens with 8 experts each 123 -> 98, 32 163 -> 134, 128 196 -> 145, 800
// 559 -> 200; 32 experts of 2048 / 704, 32 tokens with 4 each 81 -> 74, 600 205 -> 95)
extern "C" int64_t ll_moe_rows_block(int64_t num_slots, int64_t experts, int64_t width, int64_t ff, int dtype) {
  (void)num_slots;
  (void)experts;
  return dtype != LL_F32 && (width % 8 == 0 || ff % 8 == 0) ? 128 : 32;
}

// counts: int32 scratch [experts].  sorted [num_slots + experts * (block - 1)], block_expert [ceil(that / block)], num_post [1]
static int moe_sort(const int32_t* ids, int64_t num_slots, int64_t experts, int64_t block, int skipped, int32_t* counts, int32_t* sorted,
                    int32_t* block_expert, int32_t* num_post, void* stream) {
  if (num_slots < 0 || experts < 1 || experts > 65535 || (block != 32 && block != 128) || num_slots + experts * block >= (1ll << 31))
    return LL_ERR_SHAPE;
  if (!ids || !counts || !sorted || !block_expert || !num_post) return LL_ERR_ARG;
  hipStream_t st = (hipStream_t)stream;
  if (experts <= kSortExperts) {
    moe_sort_kernel<<<dim3((unsigned)(experts + skipped)), num_slots >= 2048 ? 1024 : 256, sizeof(int) * (size_t)experts, st>>>(
        ids, (int)num_slots, (int)experts, (int)block, skipped, counts, sorted, block_expert, num_post);
    return LL_LAUNCH_CHECK();
  }
  if (skipped) return LL_ERR_SHAPE;
  moe_count_kernel<<<dim3((unsigned)experts), 256, 0, st>>>(ids, (int)num_slots, counts);
  moe_place_kernel<<<dim3((unsigned)experts), 256, 0, st>>>(ids, (int)num_slots, (int)experts, (int)block, counts, sorted,
                                                            block_expert, num_post);
  return LL_LAUNCH_CHECK();
}

extern "C" int ll_moe_sort(const int32_t* ids, int64_t num_slots, int64_t experts, int64_t block, int32_t* counts, int32_t* sorted,
                           int32_t* block_expert, int32_t* num_post, void* stream) {
  return moe_sort(ids, num_slots, experts, block, 0, counts, sorted, block_expert, num_post, stream);
}

// ... and the slots whose id is no expert's in blocks of their own behind them (expert -1): sorted and block_expert for experts + 1 runs
extern "C" int ll_moe_sort_skipped(const int32_t* ids, int64_t num_slots, int64_t experts, int64_t block, int32_t* counts, int32_t* sorted,
                                   int32_t* block_expert, int32_t* num_post, void* stream) {
  return moe_sort(ids, num_slots, experts, block, 1, counts, sorted, block_expert, num_post, stream);
}

// ll_group_router, and its choices sorted as ll_moe_sort (`skipped`: ll_moe_sort_skipped) sorts them: `sorted_experts` experts in blocks of `block`
extern "C" int ll_group_router_sorted(const void* h, int64_t h_ld, const void* w_router, const void* w_extra, int64_t n, int64_t width,
                                      int64_t experts, int64_t top, int64_t group_count, int64_t group_keep, float route_scale, int scoring,
                                      int32_t* ids, float* weights, float* extra_scale, float* logits, const void* correction, int64_t identity,
                                      int64_t sorted_experts, int64_t block, int skipped, int32_t* counts, int32_t* sorted,
                                      int32_t* block_expert, int32_t* num_post, int dtype, void* stream) {
  RouterCall c;
  const int bad = router_call(c, h, h_ld, w_router, w_extra, n, width, experts, top, group_count, group_keep, route_scale, scoring, ids, weights,
                              extra_scale, logits, correction, identity, dtype);
  if (bad) return bad;
  const int rows = c.p.rows;
  const size_t lds = sizeof(float) * (sorted_experts + 2 * n * top + n + 16 * c.each);
  // us of router and sort in a graph, weights not in L2, workgroups per token and per expert -> here: 34 rows of 2048, top 4: 1 token 12.8 -> 9.5,
  // 4 13.3 -> 9.8, 8 13.6 -> 10.4, 16 13.2 -> 12.3, 24 13.1 -> 13.2 (every workgroup chooses for every token); 68 rows of 3072, top 8: 1 15.9 -> 11.1,
  // 4 16.5 -> 11.6, 8 16.5 -> 12.3, 16 16.5 -> 15.1, 24 16.3 -> 16.7
  if (n < 1 || n > kRouteTokens || rows > kRouterRows || sorted_experts < 1 || sorted_experts > experts || (block != 32 && block != 128) ||
      lds + 2 * sizeof(int) * kSortWaves > 65536) {   // (a launch has 64 KB unasked, with what the sort holds of its own)
    const int rc = ll_group_router(h, h_ld, w_router, w_extra, n, width, experts, top, group_count, group_keep, route_scale, scoring, ids, weights,
                                   extra_scale, logits, correction, identity, dtype, stream);
    return rc ? rc : moe_sort(ids, n * top, sorted_experts, block, skipped ? 1 : 0, counts, sorted, block_expert, num_post, stream);
  }
  if (!counts || !sorted || !block_expert || !num_post) return LL_ERR_ARG;
  if (scoring != 2 && !w_extra) c.p.extra_scale = nullptr;   // (no row of weights makes it: left as it is, as ll_group_router leaves it)
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)((rows + 1) / 2), (unsigned)n);
#define LL_RL(DT, V) route_logits_kernel<DT, V><<<grid, 64, 0, st>>>(h, h_ld, w_router, w_extra, (int)width, (int)experts, rows, logits)
  if (!c.aligned) {
#define CALL(DT) LL_RL(DT, 1)
    LL_BY_DTYPE(dtype, CALL);
#undef CALL
  } else if (dtype == LL_F32) {
    LL_RL(LL_F32, 4);
  } else if (dtype == LL_F16) {
    LL_RL(LL_F16, 8);
  } else {
    LL_RL(LL_BF16, 8);
  }
#undef LL_RL
  const unsigned threads = n <= 4 ? 256 : n <= 8 ? 512 : 1024;   // a wave per token
#define LL_GS(S, DT)                                                                                                                          \
  route_sort_kernel<S, DT><<<dim3((unsigned)(sorted_experts + (skipped ? 1 : 0))), threads, lds, st>>>(logits, c.p, (int)n, (int)sorted_experts, \
                                                                                                     (int)block, skipped ? 1 : 0, counts, sorted, \
                                                                                                     block_expert, num_post)
  if (scoring == 2) {
#define CALL(DT) LL_GS(2, DT)
    LL_BY_DTYPE(dtype, CALL);
#undef CALL
  } else if (scoring == 1) LL_GS(1, LL_F32);
  else if (scoring == 4) LL_GS(4, LL_F32);
  else if (scoring == 3) LL_GS(3, LL_F32);
  else LL_GS(0, LL_F32);
#undef LL_GS
  return LL_LAUNCH_CHECK();
}

// glu != 0: w [experts][2 N][K] (gate rows, then up rows), out[slot][N] = silu(a_row Wg^T) * (a_row Wu^T) with a_row =
// a[slot / a_div] (glu == 2: the clamped pair g' sigmoid(1.702 g') (u' + 1), g' = min(g, limit), u' = clamp(u, +-limit)); glu == 0: w [experts][N][K], out[slot][N] = (a[slot / a_div] W^T) * slot_weight[slot] (NULL: 1).
// glu == 3: w [experts][N][K], out[slot][N] = relu(slot_weight[slot] (a[slot / a_div] W^T))^2: an expert without a gate whose weight
// multiplies its input.
extern "C" int ll_moe_rows_gemm(const void* a, int64_t a_ld, int64_t a_div, const void* w, int64_t w_stride_e, int64_t K, int64_t N,
                                int glu, const float* slot_weight, void* out, int64_t out_ld, const int32_t* sorted,
                                const int32_t* block_expert, const int32_t* num_post, int64_t num_slots, int64_t experts,
                                int64_t block, float limit, int dtype, void* stream) {
  if (dtype != LL_F16 && dtype != LL_BF16 && dtype != LL_F32) return LL_ERR_DTYPE;
  if (glu < 0 || glu > 3 || (glu == 2 && !(limit >= 0.f))) return LL_ERR_SHAPE;
  const int mode = glu == 3 ? 2 : glu ? 1 : 0;   // (which epilogue; 1: gate and up rows)
  const float glu_limit = glu == 2 ? limit : -1.0f;
  if (num_slots < 0 || K < 1 || N < 1 || a_div < 1 || a_ld < K || out_ld < N || w_stride_e < (mode == 1 ? 2 : 1) * N * K || experts < 1 ||
      (block != 32 && block != 128))
    return LL_ERR_SHAPE;
  if (num_slots == 0) return LL_OK;
  if (!a || !w || !out || !sorted || !block_expert || !num_post) return LL_ERR_ARG;
  const int64_t most = (num_slots + (experts + 1) * (block - 1)) / block;   // blocks (a run of skipped slots may stand behind the experts')
  hipStream_t st = (hipStream_t)stream;
  static const bool no_mfma = getenv("LL_MOE_ROWS_VALU") != nullptr;   // A/B knob, read once
  const bool mfma = !no_mfma && dtype != LL_F32 && K % 8 == 0 && a_ld % 8 == 0 && w_stride_e % 8 == 0 && ll_aligned16(a) && ll_aligned16(w);
  if (block == 128 && mfma) {
    if (num_slots <= 36 * experts && num_slots < (1ll << 30) && N <= (1 << 24) && K <= (1 << 24)) {   // few rows per expert: the weights as one stream per CU (moe_stream.hip: figures)
      const int form = mode == 1 ? MS_GLU : mode == 2 ? MS_RELU2 : MS_SCALED;
      MoeStreamParams t{};
      t.out = (uint16_t*)out; t.a = (const uint16_t*)a; t.w = (const unsigned char*)w; t.weight32 = mode == 1 ? nullptr : slot_weight;
      t.sorted = sorted; t.block_expert = block_expert; t.num_post = num_post;
      t.a_ld = a_ld; t.out_ld = out_ld; t.w_stride_e = w_stride_e * 2; t.w_stride_n = K * 2; t.K = (int)K; t.N = (int)N;
      t.num_slots = (int)num_slots; t.a_div = (int)a_div; t.block_m = (int)block; t.limit = glu_limit;
      t.safe = (int)(num_slots + experts * (block - 1));
      if (moe_stream_wants(t, MS_W16, form, dtype, experts, experts)) return moe_stream_launch(t, MS_W16, form, dtype, experts, st);
    }
    const int64_t tiles_n = (N + (mode == 1 ? 63 : 127)) / (mode == 1 ? 64 : 128), max_tiles = most * tiles_n;
    if (max_tiles > 0x7ffffff0ll) return LL_ERR_SHAPE;
    // a few tiles are their chain of loads: the grid names them (8 experts of 1024 / 512, one token 26.4 -> 25.6 us for both products).  More: ranges
    // of the tiles that exist, one per XCD (32 of 3072 / 512, 64 tokens: 65 us, 77 where the grid named 272)
    const int few = max_tiles <= 128 ? (int)most : 0;
    const unsigned grid = (unsigned)(few ? max_tiles : (max_tiles + 7) / 8 * 8 + 8);   // (a range of an XCD may hold one tile more than an eighth)
    const int wide = N % 4 == 0 && out_ld % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & 7u) == 0;
    constexpr int bytes = 5 * 128 * 128;
    // rows and one expert's weights within 32-bit offsets, as all but the very largest are
    const bool near = (num_slots / a_div + 1) * a_ld * 2 < (1ll << 32) && (mode == 1 ? 2 : 1) * N * K * 2 < (1ll << 32);
    int dev = 0;
    (void)hipGetDevice(&dev);
#define CALL_F(DT, G, FAR)                                                                                                         \
  do {                                                                                                                            \
    static bool attr[16] = {false};                                                                                               \
    if (dev >= 0 && dev < 16 && !attr[dev]) {                                                                                     \
      (void)hipFuncSetAttribute((const void*)moe_rows_gemm_tiled_kernel<DT, G, FAR>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes); \
      attr[dev] = true;                                                                                                           \
    }                                                                                                                             \
    moe_rows_gemm_tiled_kernel<DT, G, FAR><<<dim3(grid), 256, bytes, st>>>((const uint16_t*)a, a_ld, (int)a_div, (const uint16_t*)w,   \
                                                                      w_stride_e, (int)K, (int)N, slot_weight, (uint16_t*)out, out_ld, \
                                                                      sorted, block_expert, num_post, (int)num_slots, glu_limit, \
                                                                      (int)tiles_n, wide, few, (int)((num_slots + experts * 127) / 128)); \
  } while (0)
#define CALL_T(DT, G)             \
  if (near) CALL_F(DT, G, false); \
  else CALL_F(DT, G, true)
    if (dtype == LL_F16) { if (mode == 1) { CALL_T(LL_F16, 1); } else if (mode == 2) { CALL_T(LL_F16, 2); } else { CALL_T(LL_F16, 0); } }
    else { if (mode == 1) { CALL_T(LL_BF16, 1); } else if (mode == 2) { CALL_T(LL_BF16, 2); } else { CALL_T(LL_BF16, 0); } }
#undef CALL_T
#undef CALL_F
    return LL_LAUNCH_CHECK();
  }
  const int64_t max_blocks = most * (block / 32);   // (the plain form takes either order)
  const dim3 grid((unsigned)max_blocks, (unsigned)((N + 63) / 64));
#define CALL_P(DT, G)                                                                                                        \
  moe_rows_gemm_kernel<DT, G><<<grid, 256, 0, st>>>(a, a_ld, (int)a_div, w, w_stride_e, (int)K, (int)N, slot_weight, out, out_ld, sorted, \
                                                    block_expert, num_post, (int)num_slots, glu_limit, block == 128 ? 2 : 0)
#define CALL(DT)                        \
  if (mode == 1) CALL_P(DT, 1);         \
  else if (mode == 2) CALL_P(DT, 2);    \
  else CALL_P(DT, 0)
  LL_BY_DTYPE(dtype, CALL);
#undef CALL
#undef CALL_P
  return LL_LAUNCH_CHECK();
}
