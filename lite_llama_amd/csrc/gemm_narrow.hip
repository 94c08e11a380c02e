// F.linear of up to 64 rows over an unquantised fp16 / bf16 weight [N][K] of a few thousand rows: the narrow projections of a decoded token, whose
// weights (up to about 25 MB) are too short a stream for a persistent loop (gemm_w16_rows.hip wants a 32-row group per CU) and too short to pay
// a finishing launch for split-K planes.
//   * A workgroup owns 16 (or 32) weight rows and ALL of K; its waves deal the contraction out in units of 128 entries and add their sums up
//     in LDS, in wave order: finished outputs in one launch, a row's sums in an order that depends on K alone -- and for K > 1024 on whether
//     there are more than 32 rows, which ll_dense16_narrow_wins leaves to other routes.
//   * Fragments come straight from memory, 64 bytes of 16 rows per load (256 bytes of them, a whole row's unit per quarter wave, took 9 - 25 %
//     longer); the next unit's weights are requested before this one is multiplied.
// Bound by its launch, two trips to memory and the activations, which every workgroup reads from L2: bf16 2048 x 2048 1 row 5.6 us, 32 rows 8.9 (the
// library 11.2 at either, split-K planes + finish 7.9 / 10.1); 2048 x 4096, 16 rows 10.9 (14.1), 32 14.6 (11.4); 8192 x 2048, 16 rows 11.9 (the
// row-group loop 12.8); 896 x 896, 64 rows 6.8 (8.1); 1024 x 16, 32 rows 2.4 (3.8); 3072 x 3072, 16 rows 9.5 (12.4), 32 12.2 (10.8); 5120 x 3072, 1
// row 13.3 (13.2): ll_dense16_narrow_wins.
#include "common.h"

typedef __bf16 nr_bf16x8 __attribute__((ext_vector_type(8)));

struct NarrowParams {
  uint16_t* out;
  const uint16_t* x;
  const uint16_t* w;
  const uint16_t* bias;
  int m, n, k, units;
  int64_t x_stride, w_stride;
};

template <int DT>
__device__ __forceinline__ f32x4 nr_mfma(const i32x4& a, const i32x4& b, f32x4 c) {
  if constexpr (DT == LL_F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(nr_bf16x8, a), __builtin_bit_cast(nr_bf16x8, b), c, 0, 0, 0);
}

// MT: 16-row parts of the activations; RG: 16-row groups of the weights; NW: waves
template <int DT, int MT, int RG, int NW>
__global__ __launch_bounds__(64 * NW) void narrow_kernel(const NarrowParams p) {
  __shared__ __attribute__((aligned(16))) f32x4 sums[NW * RG * MT * 64];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int n0 = (int)blockIdx.x * 16 * RG;
  const uint16_t* wp[RG];
  const uint16_t* xp[MT];
#pragma unroll
  for (int g = 0; g < RG; ++g) {
    const int row = n0 + 16 * g + r < p.n ? n0 + 16 * g + r : p.n - 1;   // (rows behind N feed results that are not stored)
    wp[g] = p.w + (int64_t)row * p.w_stride + 8 * q;
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int row = 16 * t + r < p.m ? 16 * t + r : p.m - 1;
    xp[t] = p.x + (int64_t)row * p.x_stride + 8 * q;
  }
  f32x4 acc[RG][MT];
#pragma unroll
  for (int g = 0; g < RG; ++g)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[g][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr i32x4 ZERO = {0, 0, 0, 0};
  i32x4 wn[RG][4];
  auto get_w = [&](int u) {
#pragma unroll
    for (int g = 0; g < RG; ++g)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = u * 128 + 32 * j + 8 * q;
        wn[g][j] = k < p.k ? __builtin_nontemporal_load(reinterpret_cast<const i32x4*>(wp[g] + u * 128 + 32 * j)) : ZERO;
      }
  };
  if (wv < p.units) get_w(wv);
  for (int u = wv; u < p.units; u += NW) {
    i32x4 w[RG][4], x[MT][4];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = u * 128 + 32 * j + 8 * q;
        x[t][j] = k < p.k ? *reinterpret_cast<const i32x4*>(xp[t] + u * 128 + 32 * j) : ZERO;
      }
#pragma unroll
    for (int g = 0; g < RG; ++g)
#pragma unroll
      for (int j = 0; j < 4; ++j) w[g][j] = wn[g][j];
    if (u + NW < p.units) get_w(u + NW);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int g = 0; g < RG; ++g)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[g][t] = nr_mfma<DT>(w[g][j], x[t][j], acc[g][t]);
  }
#pragma unroll
  for (int g = 0; g < RG; ++g)
#pragma unroll
    for (int t = 0; t < MT; ++t) sums[((wv * RG + g) * MT + t) * 64 + lane] = acc[g][t];
  __syncthreads();
  const int used = p.units < NW ? p.units : NW;
  for (int i = tid; i < RG * MT * 64; i += 64 * NW) {   // lane (row of the part, q): outputs 4 q .. 4 q + 3 of the group
    const int g = i / (MT * 64), t = i / 64 % MT, l = i & 63;
    f32x4 s = sums[i];
    for (int v = 1; v < used; ++v) {
      const f32x4 o = sums[v * RG * MT * 64 + i];
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] += o[e];
    }
    const int row = 16 * t + (l & 15), col = n0 + 16 * g + 4 * (l >> 4);
    if (row >= p.m || col >= p.n) continue;
    uint16_t* to = p.out + (int64_t)row * p.n + col;
    if (p.n % 4 == 0) {
      if (p.bias) {
        const uint2 b = *reinterpret_cast<const uint2*>(p.bias + col);
        s[0] += to_f32<DT>((uint16_t)(b.x & 0xffffu));
        s[1] += to_f32<DT>((uint16_t)(b.x >> 16));
        s[2] += to_f32<DT>((uint16_t)(b.y & 0xffffu));
        s[3] += to_f32<DT>((uint16_t)(b.y >> 16));
      }
      uint16_t o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = from_f32<DT>(s[e]);
      *reinterpret_cast<uint2*>(to) = uint2{(uint32_t)o[0] | (uint32_t)o[1] << 16, (uint32_t)o[2] | (uint32_t)o[3] << 16};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (col + e < p.n) to[e] = from_f32<DT>(p.bias ? s[e] + to_f32<DT>(p.bias[col + e]) : s[e]);
    }
  }
}

extern "C" int ll_dense16_narrow_supported(int64_t m, int64_t n, int64_t k) {
  return m >= 1 && m <= 64 && n >= 1 && n < (1 << 24) && k >= 8 && k % 8 == 0 && k < (1 << 24) ? 1 : 0;
}

// Where it is the faster route (figures above): short contractions at any of its row counts, longer ones for a few rows.
extern "C" int ll_dense16_narrow_wins(int64_t m, int64_t n, int64_t k) {
  if (!ll_dense16_narrow_supported(m, n, k)) return 0;
  if (k <= 1024) return n <= 2048 ? 1 : m <= 16 && n <= 8192;
  if (k <= 2048 && n <= 2048) return m <= 32;
  return m <= 16 && ((k <= 2048 && n <= 8192) || (k <= 4096 && n * k <= 10000000));
}

// out [m][n] = x [m][k] @ w [n][k]^T (+ bias); rows of x and w 16-byte aligned (strides in elements, multiples of 8)
extern "C" int ll_dense16_narrow_matmul(void* out, const void* x, const void* w, const void* bias, int64_t m, int64_t n, int64_t k,
                                        int64_t x_stride_m, int64_t w_stride_n, int dtype, void* stream) {
  if (dtype != LL_F16 && dtype != LL_BF16) return LL_ERR_DTYPE;
  if (m == 0) return LL_OK;
  if (!ll_dense16_narrow_supported(m, n, k) || x_stride_m < k || w_stride_n < k || x_stride_m % 8 || w_stride_n % 8) return LL_ERR_SHAPE;
  if (!out || !x || !w || !ll_aligned16(x) || !ll_aligned16(w) || (reinterpret_cast<uintptr_t>(out) & 7u) || (reinterpret_cast<uintptr_t>(bias) & 7u))
    return LL_ERR_ARG;
  NarrowParams p{(uint16_t*)out, (const uint16_t*)x, (const uint16_t*)w, (const uint16_t*)bias, (int)m, (int)n, (int)k, (int)((k + 127) / 128),
                 x_stride_m, w_stride_n};
  // 32 weight rows per workgroup where 16 each would be more than a workgroup per CU: the activations are read half as often
  const int rg = n > 16 * 256 ? 2 : 1, mt = m <= 16 ? 1 : m <= 32 ? 2 : 4, nw = p.units > 8 && mt < 4 ? 16 : 8;
  const unsigned grid = (unsigned)((n + 16 * rg - 1) / (16 * rg));
  hipStream_t st = (hipStream_t)stream;
#define NR_GO(DT, MT, RG, NW) narrow_kernel<DT, MT, RG, NW><<<dim3(grid), 64 * NW, 0, st>>>(p)
#define NR_NW(DT, MT, RG) do { if (nw == 16) NR_GO(DT, MT, RG, (MT < 4 ? 16 : 8)); else NR_GO(DT, MT, RG, 8); } while (0)
#define NR_RG(DT, MT) do { if (rg == 2) NR_NW(DT, MT, 2); else NR_NW(DT, MT, 1); } while (0)
#define NR_DT(DT) do { if (mt == 1) NR_RG(DT, 1); else if (mt == 2) NR_RG(DT, 2); else NR_RG(DT, 4); } while (0)
  if (dtype == LL_F16) NR_DT(LL_F16);
  else NR_DT(LL_BF16);
#undef NR_DT
#undef NR_RG
#undef NR_NW
#undef NR_GO
  return LL_LAUNCH_CHECK();
}
