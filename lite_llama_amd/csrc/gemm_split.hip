// Split-K projections of at most 64 rows over ROW-MAJOR weights (fp8 e4m3 / int8 with block scales, int8 x int8, fp16, bf16) that leave their
// sums as planes [slice][m][n] for the next launch.  References: lite_llama/kernels/quantization/w8a16.py:28-207, w8a8.py:28-217,
// models/quantization/methods/unquantized.py:21-22.
//   * A workgroup, at most one per CU, owns GROUPS x 32 weight rows and a slice of the contraction; slices of a tile stand apart by all tiles,
//     so the CUs of an XCD share few slices of the activations.
//   * Four LOADER waves bring units of 128 bytes of every weight row (whole lines, non-temporal) and the same columns of the activations into a
//     ring of LDS slots by LDS-DMA, up to 11 units ahead: most shares are on their way at once.  16-byte slot s of a row stands at
//     s ^ ((row >> 1) & 7) (activations in 256-byte rows: s ^ (row & 15)), through the SOURCE address: fragment reads are conflict free.
//   * One CONSUMER wave per row group runs the unit's MFMAs 32x32x16 (int8 x int8 32x32x32) from LDS fragments.
//   * The sums pass through the idle ring and leave as whole lines.
// Bound by the ramp of a launch (about 3 us), then by what a CU can take in, about 27 KB/us.  us, the kernel that parks one 16 KB chunk per workgroup in
// registers -> here, the same bits (calls that follow each other over 0.7 GB of weights): 1536 x 8960 bf16, 27 rows 14.6 -> 8.6, 64 rows 17.7 -> 9.8; 1536 x
// 1536 4.8 -> 4.0; 896 x 4864 fp16, 37 rows 10.6 -> 5.7; 4096 x 4096, 64 rows 13.6 -> 11.4, x 14336, one row 27.6 -> 21.7; int8 x int8, 30 rows 4096 x 14336 17.2 -> 12.5, 6144 x 4096 8.9 -> 8.0; fp8, 64 rows 5120
// x 2048 10.0 -> 8.8, 4096 x 14336 27.6 -> 20.1.  In slices of its own choice, whose sums round otherwise, the bf16 and fp8 products take up to 0.9 us
// less.  Weights requested straight into registers, as the packed int4 words are: fp8, 5 rows 2048 x 4096 6.1 -> 5.0 (a lane's piece of a row is half a
// line there; gemm_short_dense.hip has the small 8-bit ones).
#include "common.h"
#include "gemm_w4_common.h"
#include "gemm_w8_common.h"

namespace {

typedef __bf16 sk_bf16x8 __attribute__((ext_vector_type(8)));

constexpr int SK_FP8 = 1, SK_I8 = 2, SK_I8I8 = 3, SK_F16 = 4, SK_BF16 = 5;

// row groups that a tile of a format may have (a consumer wave each; eight leave a ring of three or four)
constexpr int SK_MOST_GROUPS = 8;
constexpr bool sk_tile(int wfmt, int groups) { return groups == 1 || groups == 2 || groups == 4 || (wfmt != SK_I8I8 && (groups == 3 || groups == 8)); }

template <int WF, int MT, int GROUPS>
struct SkLds {
  static constexpr bool W8A16 = WF == SK_FP8 || WF == SK_I8;
  static constexpr int KB = 128;                    // bytes of a weight row per unit
  static constexpr int XKB = W8A16 ? 256 : 128;     // bytes of an activation row per unit
  static constexpr int W_BYTES = GROUPS * 32 * KB, X_BYTES = MT * 32 * XKB, SLOT = W_BYTES + X_BYTES;
  static constexpr int FIT = 160 * 1024 / SLOT, R = FIT < 12 ? FIT : 12;
  static constexpr int THREADS = 64 * (GROUPS + 4);
  static constexpr int WOPS = GROUPS, XOPS = X_BYTES / 4096, OPS = WOPS + XOPS;   // LDS-DMA operations per loader wave and unit
  static constexpr int OSTR = GROUPS * 32 + 4;      // words per row of the finished sums
  static constexpr int BYTES = R * SLOT;
  static constexpr int SUMS = MT * 32 * OSTR * 4;   // bytes of the tile's sums
  static_assert(SUMS <= BYTES && (R - 1) * OPS <= 63, "ring");
};

struct SkParams {
  void* part;
  const unsigned char* x;
  const unsigned char* w;
  const float* scales;
  int64_t n, x_stride, w_stride;   // (strides in bytes)
  int64_t s_stride_n, s_stride_k;
  int m, group_n, group_k;
  int tiles, total, cap;           // items = slice * tiles + tile; workgroup b takes item (b % 8) * cap + b / 8
  int units, each;                 // slice s owns units [s * each, + each) of them
};

template <int N>
__device__ __forceinline__ void sk_wait_units(int k) {  // at most k units of N operations each may still be in flight
  switch (k) {
    case 0: v3_vmcnt<0>(); break;
    case 1: v3_vmcnt<N>(); break;
    case 2: v3_vmcnt<2 * N>(); break;
    case 3: v3_vmcnt<3 * N>(); break;
    case 4: v3_vmcnt<4 * N>(); break;
    case 5: v3_vmcnt<(5 * N < 63 ? 5 * N : 63)>(); break;
    case 6: v3_vmcnt<(6 * N < 63 ? 6 * N : 63)>(); break;
    case 7: v3_vmcnt<(7 * N < 63 ? 7 * N : 63)>(); break;
    case 8: v3_vmcnt<(8 * N < 63 ? 8 * N : 63)>(); break;
    case 9: v3_vmcnt<(9 * N < 63 ? 9 * N : 63)>(); break;
    default: v3_vmcnt<(10 * N < 63 ? 10 * N : 63)>(); break;
  }
}

template <int WF, int MT, int GROUPS>
__global__ __launch_bounds__((SkLds<WF, MT, GROUPS>::THREADS)) void split_kernel(const SkParams p) {
  using LD = SkLds<WF, MT, GROUPS>;
  constexpr bool W8A16 = LD::W8A16, I8A = WF == SK_I8I8;
  constexpr int R = LD::R, XKB = LD::XKB, XPER = 1024 / XKB, XS = XKB / 16;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int item = ((int)blockIdx.x & 7) * p.cap + ((int)blockIdx.x >> 3);
  if ((int)blockIdx.x >> 3 >= p.cap || item >= p.total) return;
  const int slice = item / p.tiles, tile = item - slice * p.tiles;
  const int u0 = slice * p.each, units = p.units - u0 < p.each ? p.units - u0 : p.each;
  const int64_t row0 = (int64_t)tile * GROUPS * 32;

  if (wv >= GROUPS) {
    // ======================================== loaders ======================================== //
    const int L = wv - GROUPS;
    uint32_t woff[LD::WOPS], xoff[LD::XOPS];
#pragma unroll
    for (int j = 0; j < LD::WOPS; ++j) {
      const int r = (L * LD::WOPS + j) * 8 + (lane >> 3);
      woff[j] = (uint32_t)(r * p.w_stride) + (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) * 16);
    }
#pragma unroll
    for (int j = 0; j < LD::XOPS; ++j) {
      int r = (L * LD::XOPS + j) * XPER + lane / XS;
      const int slot = (lane % XS) ^ (W8A16 ? r & 15 : (r >> 1) & 7);
      if (r >= p.m) r = p.m - 1;  // rows >= M feed only sums that are not stored
      xoff[j] = (uint32_t)(r * p.x_stride) + (uint32_t)(slot * 16);
    }
    const unsigned char* wb = p.w + row0 * p.w_stride + (int64_t)u0 * LD::KB;
    const unsigned char* xb = p.x + (int64_t)u0 * XKB;
    int issued = 0;
    uint32_t dst = 0;
    auto issue = [&]() {
#pragma unroll
      for (int j = 0; j < LD::WOPS; ++j) v3_dma16<true>(dst + (L * LD::WOPS + j) * 1024, wb, woff[j]);
#pragma unroll
      for (int j = 0; j < LD::XOPS; ++j) v3_dma16<false>(dst + LD::W_BYTES + (L * LD::XOPS + j) * 1024, xb, xoff[j]);
      wb += LD::KB;
      xb += XKB;
      ++issued;
      dst = dst + LD::SLOT == R * LD::SLOT ? 0 : dst + LD::SLOT;
    };
    const int pre = units < R - 1 ? units : R - 1;
    for (int i = 0; i < pre; ++i) issue();
    sk_wait_units<LD::OPS>(issued - 1);
    asm volatile("s_barrier" ::: "memory");  // P0: unit 0 has landed
    for (int u = 0; u < units; ++u) {
      if (issued < units) issue();  // into the slot of unit u - 1, free since the barrier that ended it
      const int need = units < u + 2 ? units : u + 2;
      sk_wait_units<LD::OPS>(issued - need);
      asm volatile("s_barrier" ::: "memory");  // B_u: unit u + 1 has landed
    }
  } else {
    // ======================================= consumers ======================================= //
    const int nl = lane & 31, h = lane >> 5, rg = wv;
    f32x16 accf[MT];
    i32x16 acci[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int e = 0; e < 16; ++e) { accf[mt][e] = 0.f; acci[mt][e] = 0; }
    const unsigned char* wrow = lds + (rg * 32 + nl) * LD::KB;
    const unsigned char* xrow = lds + LD::W_BYTES + nl * XKB;
    const float* srow = nullptr;
    if constexpr (W8A16) srow = p.scales + ((row0 + rg * 32 + nl) / p.group_n) * p.s_stride_n;
    auto scale_at = [&](int u) {  // of this lane's 64 columns of a unit (the last unit's again past it)
      return srow[(int64_t)(((u0 + (u < units ? u : units - 1)) * 128 + h * 64) / p.group_k) * p.s_stride_k];
    };
    float sc = 0.f;
    if constexpr (W8A16) sc = scale_at(0);
    uint32_t slot = 0;
    asm volatile("s_barrier" ::: "memory");  // P0
    for (int u = 0; u < units; ++u) {
      float next = 0.f;
      if constexpr (W8A16) next = scale_at(u + 1);   // on its way under this unit's products
      if constexpr (W8A16) {
        // a lane half holds 64 columns of its row; a product takes eight of either half
        const uint32_t sp = d8_bcast(WF == SK_FP8 ? sc * 256.0f : sc);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const u32x4 wf = *reinterpret_cast<const u32x4*>(wrow + slot + (((4 * h + j) ^ ((nl >> 1) & 7)) * 16));
          u32x4 a, b;
          uint32_t lo, hi;
#define SK_WIDEN(W) if constexpr (WF == SK_FP8) d8_fp8(W, sp, lo, hi); else d8_i8(W, sp, lo, hi);
          SK_WIDEN(wf.x) a.x = lo; a.y = hi;
          SK_WIDEN(wf.y) a.z = lo; a.w = hi;
          SK_WIDEN(wf.z) b.x = lo; b.y = hi;
          SK_WIDEN(wf.w) b.z = lo; b.w = hi;
#undef SK_WIDEN
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            const unsigned char* xb = xrow + slot + mt * 32 * XKB;
            const u32x4 xa = *reinterpret_cast<const u32x4*>(xb + (((8 * h + 2 * j) ^ (nl & 15)) * 16));
            const u32x4 xc = *reinterpret_cast<const u32x4*>(xb + (((8 * h + 2 * j + 1) ^ (nl & 15)) * 16));
            accf[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, xa), accf[mt], 0, 0, 0);
            accf[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, b), __builtin_bit_cast(f16x8, xc), accf[mt], 0, 0, 0);
          }
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const u32x4 wf = *reinterpret_cast<const u32x4*>(wrow + slot + (((2 * j + h) ^ ((nl >> 1) & 7)) * 16));
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            const u32x4 xf = *reinterpret_cast<const u32x4*>(xrow + slot + mt * 32 * XKB + (((2 * j + h) ^ ((nl >> 1) & 7)) * 16));
            if constexpr (WF == SK_F16)
              accf[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, wf), __builtin_bit_cast(f16x8, xf), accf[mt], 0, 0, 0);
            else if constexpr (WF == SK_BF16)
              accf[mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(sk_bf16x8, wf), __builtin_bit_cast(sk_bf16x8, xf), accf[mt], 0, 0, 0);
            else
              acci[mt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, wf), __builtin_bit_cast(i32x4, xf), acci[mt], 0, 0, 0);
          }
        }
      }
      sc = next;
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // B_u: this unit's slot may be filled again
      slot = slot + LD::SLOT == R * LD::SLOT ? 0 : slot + LD::SLOT;
    }
    // the ring is idle: the tile's sums go through it, so that they leave in whole lines.  A lane holds, for row nl (+ 32 mt), the
    // columns 8 g + 4 h .. + 3 of its 32
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        i32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (I8A) v[e] = acci[mt][4 * g + e];
          else v[e] = (int)__float_as_uint(accf[mt][4 * g + e]);
        }
        *reinterpret_cast<i32x4*>(lds + ((mt * 32 + nl) * LD::OSTR + rg * 32 + 8 * g + 4 * h) * 4) = v;
      }
  }
  __syncthreads();
  constexpr int QUADS = GROUPS * 8;
  int32_t* out = (int32_t*)p.part + (int64_t)slice * p.m * p.n + row0;
  for (int i = tid; i < p.m * QUADS; i += LD::THREADS) {
    const int r = i / QUADS, q = i - r * QUADS;
    const unsigned char* from = lds + (r * LD::OSTR + q * 4) * 4;
    *reinterpret_cast<i32x4*>(out + r * p.n + q * 4) = *reinterpret_cast<const i32x4*>(from);
  }
}

int sk_num_cus() {
  static int cus[16] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) return 256;
  if (!cus[dev]) {
    hipDeviceProp_t prop;
    cus[dev] = hipGetDeviceProperties(&prop, dev) == hipSuccess && prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
  }
  return cus[dev];
}

struct SkPlan {
  int groups = 0, slices = 0, each = 0;   // each: units of a slice
};

// Row groups of a tile, slices and their units.  At most a workgroup per CU: two rounds double the ramp.
// Floating sums round in the order they are formed in, and that order is the one of the kernel that parks a chunk per workgroup (gemm_w8_skinny.hip), which has
// the shapes that are not served here: its slices, and within a unit its products -- a call's values do not depend on which of the two runs.  The tile is then the
// narrowest that leaves no CU two.  Whole numbers have one sum: slices as they cost least.  us: a unit of GROUPS row groups at 27 KB/us, its
// activations at 130 KB/us and its barrier, and what a plane costs here and where it is added up.
SkPlan sk_plan(int64_t m, int64_t n, int64_t k, int wfmt, int max_splits) {
  SkPlan best;
  const bool w16 = wfmt == SK_F16 || wfmt == SK_BF16;
  if (wfmt < SK_FP8 || wfmt > SK_BF16 || m < 1 || m > 64 || n < 32 || n % 32 != 0 || max_splits < 1) return best;
  const int64_t row = w16 ? k * 2 : k;
  if (row < 128 || row % 128 != 0 || n >= (1 << 30) || k >= (1 << 24)) return best;
  const int units = (int)(row / 128), cus = sk_num_cus();
  const int64_t rgs = n / 32;
  if (wfmt != SK_I8I8) {
    const int s = d8_splits(n, k, w16 ? 64 : 128, max_splits), each = (units + s - 1) / s, slices = (units + each - 1) / each;
    for (int g = 1; g <= SK_MOST_GROUPS; ++g)
      if (sk_tile(wfmt, g) && rgs % g == 0 && rgs / g * slices <= cus) return SkPlan{g, slices, each};
    return best;
  }
  double least = 1e30;
  for (int g = 4; g >= 1; g /= 2) {
    if (rgs % g) continue;
    for (int s = 1; s <= max_splits && s <= units && rgs / g * s <= cus; ++s) {
      const int each = (units + s - 1) / s;
      const double cost = each * (g * 4.0 / 27 + 4.0 / 130 + 0.05) + 0.15 * s;
      if (cost < least) {
        least = cost;
        best = SkPlan{g, (units + each - 1) / each, each};
      }
    }
  }
  return best;
}

// (shares shorter than the ring take only what they fill: a launch of many KB of LDS starts later)
template <int WF, int MT, int GROUPS>
void sk_go(const SkParams& p, hipStream_t st) {
  using LD = SkLds<WF, MT, GROUPS>;
  static bool attr[16] = {false};
  int dev = 0;
  (void)hipGetDevice(&dev);
  if (dev >= 0 && dev < 16 && !attr[dev]) {
    (void)hipFuncSetAttribute((const void*)split_kernel<WF, MT, GROUPS>, hipFuncAttributeMaxDynamicSharedMemorySize, LD::BYTES);
    attr[dev] = true;
  }
  const int ring = (p.each < LD::R ? p.each : LD::R) * LD::SLOT;
  split_kernel<WF, MT, GROUPS><<<dim3((unsigned)(p.cap * 8)), LD::THREADS, ring > LD::SUMS ? ring : LD::SUMS, st>>>(p);
}

}  // namespace

// planes the launch leaves for (m, n, k, format), alike for any m; 0: not served, the kernel of gemm_w8_skinny.hip runs
int sk_partials_slices(int64_t m, int64_t n, int64_t k, int wfmt, int max_splits) { return sk_plan(m, n, k, wfmt, max_splits).slices; }

// Returns the planes written, 0 where the call is declined, < 0 on a launch error.  Strides in bytes.
int sk_launch(void* out, const void* x, const void* w, const float* scales, int64_t m, int64_t n, int64_t k, int group_n, int64_t group_k,
              int wfmt, int64_t x_stride, int64_t w_stride, int64_t s_stride_n, int64_t s_stride_k, int max_splits, void* stream) {
  const SkPlan pl = sk_plan(m, n, k, wfmt, max_splits);
  if (!pl.slices) return 0;
  if (w_stride % 16 || x_stride % 16 || !ll_aligned16(w) || !ll_aligned16(x) || !ll_aligned16(out)) return 0;
  if (SK_MOST_GROUPS * 32 * w_stride >= (1ll << 31) || m * x_stride >= (1ll << 31)) return 0;
  SkParams p{};
  p.part = out; p.x = (const unsigned char*)x; p.w = (const unsigned char*)w; p.scales = scales;
  p.n = n; p.x_stride = x_stride; p.w_stride = w_stride; p.s_stride_n = s_stride_n; p.s_stride_k = s_stride_k;
  p.m = (int)m; p.group_n = group_n > 0 ? group_n : 1;
  p.group_k = group_k > 0 && group_k < k ? (int)group_k : (int)k;
  p.units = (int)((wfmt == SK_F16 || wfmt == SK_BF16 ? k * 2 : k) / 128);
  p.each = pl.each;
  p.tiles = (int)(n / (32 * pl.groups));
  p.total = p.tiles * pl.slices;
  p.cap = (p.total + 7) / 8;
  hipStream_t st = (hipStream_t)stream;
#define SK_T(WF, MT, G) if constexpr (sk_tile(WF, G)) { if (pl.groups == G) sk_go<WF, MT, G>(p, st); }
#define SK_G(WF, MT) SK_T(WF, MT, 1) SK_T(WF, MT, 2) SK_T(WF, MT, 3) SK_T(WF, MT, 4) SK_T(WF, MT, 8)
#define SK_M(WF) if (m > 32) { SK_G(WF, 2) } else { SK_G(WF, 1) }
  switch (wfmt) {
    case SK_FP8: SK_M(SK_FP8) break;
    case SK_I8: SK_M(SK_I8) break;
    case SK_I8I8: SK_M(SK_I8I8) break;
    case SK_F16: SK_M(SK_F16) break;
    default: SK_M(SK_BF16) break;
  }
#undef SK_M
#undef SK_G
#undef SK_T
  return hipGetLastError() == hipSuccess ? pl.slices : LL_ERR_LAUNCH;
}
