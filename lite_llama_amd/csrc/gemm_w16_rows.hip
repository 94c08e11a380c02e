// Decode-shaped F.linear for UNQUANTISED fp16 / bf16 weights [N][K] (M <= 64 rows): the row-group loop of gemm_w4_v4.hip without
// a dequantiser.  Reference: lite_llama/models/quantization/methods/unquantized.py:21-22 and the lm_head of models/base.py:486-489
// are torch's library GEMM; BASELINE config 2 (Qwen2.5-1.5B bf16, batch 32) has its fused gate|up and the lm_head there.
//   * A workgroup owns a contiguous run of 32-row groups (or, r16_deal, of halves of them; runs differ by at most one) and ALL
//     of K; it walks its run in tiles of up to 4 groups (WIDE: 8), of equal size to within one.  Finished outputs only: no
//     split-K planes, no finish launch, bias or the fused swiglu of a row-interleaved gate|up in the epilogue (the decode engines'
//     epilogue, common.h::ll_silu_mul_f32).
//   * Four LOADERS stream, per unit of 256 (128) bytes of every row, the tile's weight blocks -- 32 KB -- and the activation block into a ring of
//     LDS slots by LDS-DMA: row-major with the 16-byte slots of a row permuted by R16Lds::swizzle, through the per-lane SOURCE
//     address: fragment reads are conflict free; weights non-temporal.  CONSUMERS, one per row group of the tile, run the unit's MFMA
//     32x32x16 from LDS fragments and keep the tile's accumulators (16 x MT registers) for the whole K loop: no cross-wave exchange.
//     The loaders run ahead ACROSS tile boundaries, so a tile's epilogue overlaps the next tile's first units.
//   * Long streams of rows a multiple of 4 KB long: workgroup b begins every tile b steps of 256 bytes into its rows and wraps; int8 streams under 256 MB
//     5 b steps.  All of them beginning at column 0 ask the same few memory channels, and so do runs of a power of two rows whose steps of b keep
//     pace with them.  us for 600 MB, 1 row, all from column 0 -> staggered: K = 2048 113 -> 94, 4096 127 -> 98, 8192 139 -> 124; staggered within
//     an XCD instead, b / 8: 98, 106, 124; K = 3584: 90 -> 91, 37888 rows of it 50 -> 52.  b / 5 b steps: int8 28672 x 4096 23.8 / 23.1, 16384 x 8192 36.3 /
//     25.7; from 256 MB on b and 5 b are within 2 % of each other, either way.  Sums of 16-bit products in another order round otherwise, which travels
//     through all that follows, so 16-bit streams under 256 MB keep the ascending one (in 5 b steps 32 rows of 32768 x 2048 take 25.6 instead of 32.7, 14336 x 4096
//     24.5 instead of 25.6, 28672 x 4096 43 instead of 50); int8 sums are exact, and staggered from 64 MB.
//   * one s_barrier per unit.  Of every row group each loader requests a quarter, and nothing is requested that no one reads: neither groups that a
//     tile lacks nor activations behind the last row; the waits count what was.  (Loaders of one group each, which pointed the requests of
//     groups that were not there at one cached KB so that the count stayed the same, took as long for a tile of one group as for four.  us,
//     then -> here: 32 rows 6144 x 2048 11.6 -> 9.8, 8192 x 2048 11.8 -> 10.0, 11264 x 2048 14.2 -> 12.7, 6 rows 9216 x 3072 18.2 -> 14.1, 64 rows
//     8192 x 2048 14.1 -> 12.7; tiles that are full, as before: 17920 x 1536 13.9, 128256 x 4096 160 (6.6 TB/s).  A higher priority for the
//     loaders' waves gains nothing here.)
#include <stdlib.h>

#include "common.h"
#include "gemm_w4_common.h"

typedef __bf16 r16_bf16x8 __attribute__((ext_vector_type(8)));

// WIDE (more than 32 rows over more than four row groups per CU): tiles of eight groups in units of 128 bytes, so that a fifth of what a CU fetches
// is activations, as with 32 rows, and not a third; 96 KB of weights on their way and not 64.  us, 64 rows, 16-bit: 128256 x 4096 184 -> 167, 152064 x
// 3584 199 -> 192, 37888 x 3584 54 -> 46; int8 128256 x 4096 97 -> 89.  Where the groups are few a tile is not full: 11264 x 2048 15.1 -> 22.3.
template <int MT, bool WIDE>
struct R16Lds {
  static constexpr int GROUPS = WIDE ? 8 : 4;     // row groups of a tile, a consumer each
  static constexpr int THREADS = 64 * (GROUPS + 4);
  static constexpr int KB = WIDE ? 128 : 256;     // bytes of a row per unit
  static constexpr int W_BYTES = GROUPS * 32 * KB;
  static constexpr int X_BYTES = 32 * MT * KB;
  static constexpr int SLOT = W_BYTES + X_BYTES;  // 40 KB; 48 KB (more than 32 rows, four groups)
  static constexpr int R = 160 * 1024 / SLOT;     // 4; 3
  static constexpr int BYTES = R * SLOT;
  // which 16-byte slot of its row a piece stands in: slot ^ swizzle(row), so that the lanes of a fragment read meet all banks
  static __device__ __forceinline__ int swizzle(int row) { return WIDE ? (row >> 1) & 7 : row & 15; }
};

struct R16Params {
  uint16_t* out;
  const uint16_t* x;
  const uint16_t* w;
  const uint16_t* bias;
  int64_t m, n, k, x_stride, w_stride;
  int chunks;        // units of a row: its bytes / R16Lds::KB
  int piece;         // what is dealt out: 32-row groups (2) or halves of them (1)
  int rbase, rrem;   // workgroup b owns pieces [b * rbase + min(b, rrem), + rbase + (b < rrem))
  int stagger;       // workgroup b begins a tile that many times b steps of 256 bytes into its rows
  int epi;           // 0: out[m, n] (+ bias);  1: rows are (gate_j, up_j) pairs -> out[m, n / 2] = silu(gate) * up
  const float* a_scale;  // R16_I8 only: per-token activation scales [m], per-channel weight scales [n] (smoothquant, w8a8.py:118-149)
  const float* w_scale;
};
#define R16_I8 2  // DT code of the int8 x int8 form: x / w are int8 rows of 256 k per chunk, out is fp16

__device__ __forceinline__ void r16_wait(int k) {  // at most k operations may still be in flight
#define R16_C(K) case K: v3_vmcnt<K>(); break;
  switch (k) {
    R16_C(1) R16_C(2) R16_C(3) R16_C(4) R16_C(5) R16_C(6) R16_C(7) R16_C(8) R16_C(9) R16_C(10) R16_C(11) R16_C(12) R16_C(13) R16_C(14) R16_C(15)
    R16_C(16) R16_C(17) R16_C(18) R16_C(19) R16_C(20)
    default: v3_vmcnt<0>(); break;
  }
#undef R16_C
}

template <int MT, int DT, bool WIDE>
__global__ __launch_bounds__((R16Lds<MT, WIDE>::THREADS)) __attribute__((amdgpu_waves_per_eu(WIDE ? 3 : 2, WIDE ? 3 : 2))) void wgemm16_rows_kernel(const R16Params p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  using LD = R16Lds<MT, WIDE>;
  constexpr int R = LD::R, KB = LD::KB, GROUPS = LD::GROUPS;
  constexpr int PER = 1024 / KB, SLOTS = KB / 16;   // rows of an LDS-DMA operation; 16-byte slots of a row
  constexpr int PG = 8 / GROUPS;                    // weight operations per loader wave, unit and row group
  constexpr int XP = LD::X_BYTES / 4096;  // activation operations per loader wave and unit, at most
  static_assert((R - 2) * (8 + XP) <= 20, "the waits");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = (int)blockIdx.x;
  const int lo = (b * p.rbase + (b < p.rrem ? b : p.rrem)) * p.piece;   // in halves of a group, as are the tiles' sizes
  const int cnt = p.rbase + (b < p.rrem ? 1 : 0);
  if (cnt <= 0) return;
  // (tiles of equal size to within one piece: a last tile of a group or two would walk the whole contraction with little on its way)
  const int most = p.piece == 2 ? GROUPS : 2 * GROUPS;
  const int tiles = (cnt + most - 1) / most, tbase = cnt / tiles, trem = cnt - tbase * tiles;
  const int units = tiles * p.chunks;
  const int halves = (int)(p.n >> 4);
  auto sized = [&](int t, int first) {   // tile t's halves (N may end inside the last group)
    const int s = (tbase + (t < trem ? 1 : 0)) * p.piece;
    return first + s < halves ? s : halves - first;
  };

  if (wv >= GROUPS) {
    // ======================================== loaders ======================================== //
    // Of every group each takes a quarter; nothing is requested that no one reads.
    const int L = wv - GROUPS;
    uint32_t woff[PG], xoff[XP];
#pragma unroll
    for (int q = 0; q < PG; ++q) {
      const int r = (4 * q + L) * PER + lane / SLOTS, slot = (lane % SLOTS) ^ LD::swizzle(r);
      woff[q] = (uint32_t)((int64_t)r * p.w_stride * 2 + slot * 16);
    }
#pragma unroll
    for (int j = 0; j < XP; ++j) {
      int64_t r = (4 * j + L) * PER + lane / SLOTS;
      const int slot = (lane % SLOTS) ^ LD::swizzle((int)(r & 31));
      if (r >= p.m) r = p.m - 1;  // rows >= M feed only unstored outputs
      xoff[j] = (uint32_t)(r * p.x_stride * 2 + slot * 16);
    }
    int xops = ((int)p.m - L * PER + 4 * PER - 1) / (4 * PER);   // this wave's activation operations that hold a row
    xops = xops < 0 ? 0 : xops;
    int issued = 0, t = 0, first = lo, size = sized(0, lo), done = 0, c = 0, ops = 0, before = 0;   // operations of the last unit and the one before it
    if (p.stagger) {   // (WIDE units are half as long: two of them per step, so that a row's sum begins at the same column in either form)
      c = b * p.stagger % (p.chunks * KB / 256) * (256 / KB);
    }
    const size_t group = 32 * (size_t)p.w_stride * 2;
    const char* wt = (const char*)p.w + (size_t)lo * (group / 2);   // the tile's rows
    uint32_t dst = 0;
    auto issue = [&]() {
      const char* wb = wt + (size_t)c * KB;
      const char* xb = (const char*)p.x + (size_t)c * KB;
#pragma unroll
      for (int g = 0; g < GROUPS; ++g) {
        if (2 * g + 1 >= size) break;
#pragma unroll
        for (int q = 0; q < PG; ++q) v3_dma16<true>(dst + g * 32 * KB + (4 * q + L) * 1024, wb, woff[q]);
        wb += group;
      }
      if ((size & 1) && (PG == 2 || L < 2)) v3_dma16<true>(dst + (size >> 1) * 32 * KB + L * 1024, wb, woff[0]);   // half a group: its first 16 rows
#pragma unroll
      for (int j = 0; j < XP; ++j) {
        if (j >= xops) break;
        v3_dma16<false>(dst + LD::W_BYTES + (4 * j + L) * 1024, xb, xoff[j]);
      }
      ++issued;
      before = ops;
      ops = (PG == 2 ? size : (size + (L < 2 ? 1 : 0)) >> 1) + xops;
      if (++c == p.chunks) c = 0;
      if (++done == p.chunks) {
        done = 0;
        wt += (size_t)size * (group / 2);
        first += size;
        size = sized(++t, first);
      }
      dst = dst + LD::SLOT == R * LD::SLOT ? 0 : dst + LD::SLOT;
    };
    auto wait = [&](int later) { r16_wait(later <= 0 ? 0 : later == 1 ? ops : ops + before); };   // but for the last `later` units (at most R - 2), all have landed
    const int pre = units < R - 1 ? units : R - 1;
    for (int i = 0; i < pre; ++i) issue();
    wait(issued - 1);  // unit 0 has landed
    asm volatile("s_barrier" ::: "memory");  // P0
    for (int u = 0; u < units; ++u) {
      if (issued < units) issue();  // into the slot of unit u - 1, free since the barrier that ended it
      const int need = units < u + 2 ? units : u + 2;
      wait(issued - need);  // unit u + 1 has landed before the consumers are released into it
      asm volatile("s_barrier" ::: "memory");  // B_u
    }
    return;
  }

  // ======================================= consumers ======================================= //
  const int nl = lane & 31, h = lane >> 5;
  const int wrow = (wv * 32 + nl) * KB;  // this wave's row group of the tile, weight row nl
  constexpr int ODT = DT == R16_I8 ? LL_F16 : DT;  // output / bias storage type
  f32x16 acc[MT];
  i32x16 iacc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int e = 0; e < 16; ++e) { acc[mt][e] = 0.f; iacc[mt][e] = 0; }
  auto swap32 = [](uint32_t& a, uint32_t& bb) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, bb, false, false);
    a = r[0];
    bb = r[1];
  };
  const bool has_bias = p.bias != nullptr;
  int t = 0, first = lo, size = sized(0, lo), c = 0;
  uint32_t slot = 0;
  asm volatile("s_barrier" ::: "memory");  // P0: unit 0 has landed
  for (int u = 0; u < units; ++u) {
    const bool mine = 2 * wv < size, whole = 2 * wv + 1 < size;
    if (mine) {
      const unsigned char* wb = lds + slot + wrow;
      const unsigned char* xb = lds + slot + LD::W_BYTES + nl * KB;
#pragma unroll
      for (int s = 0; s < KB / 32; ++s) {
        const int off = ((2 * s + h) ^ LD::swizzle(nl)) * 16;
        const u32x4 wf = *reinterpret_cast<const u32x4*>(wb + off);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const u32x4 xf = *reinterpret_cast<const u32x4*>(xb + mt * 32 * KB + off);
          if constexpr (DT == LL_F16)
            acc[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, wf), __builtin_bit_cast(f16x8, xf), acc[mt], 0, 0, 0);
          else if constexpr (DT == LL_BF16)
            acc[mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(r16_bf16x8, wf), __builtin_bit_cast(r16_bf16x8, xf), acc[mt], 0, 0, 0);
          else  // 16 int8 per lane and k-step of 32: the same 16-byte slots, exact int32 sums
            iacc[mt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, wf), __builtin_bit_cast(i32x4, xf), iacc[mt], 0, 0, 0);
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // B_u: this unit's slot may be refilled
    slot = slot + LD::SLOT == R * LD::SLOT ? 0 : slot + LD::SLOT;
    if (++c == p.chunks) {
      c = 0;
      if (mine) {
        // a lane holds, for batch row nl (+ 32 mt), the weight rows 8g + 4h .. + 3 of the group: the decode engines' epilogue
        const int64_t ncol = (int64_t)(first + 2 * wv) * 16;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const int64_t mrow = nl + mt * 32;
          const bool row_ok = mrow < p.m, store = row_ok && (whole || h == 0);
          float v[16];
          if constexpr (DT == R16_I8) {
            // (acc.f32 * a_scale[m]) * w_scale[n], each product rounded to fp32 before the next (w8a8.py:118-120): pinned so that
            // the narrowing conversion below cannot be fused into it (common.h::ll_silu_mul_f32 has the story)
            const float as = p.a_scale[row_ok ? mrow : 0];
#pragma unroll
            for (int g = 0; g < 4; ++g) {
              const f32x4 ws = *reinterpret_cast<const f32x4*>(p.w_scale + ncol + 8 * (whole ? g : g & 1) + 4 * h);   // (rows that are not there: any that are)
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                float f = ((float)iacc[mt][4 * g + e] * as) * ws[e];
                asm volatile("" : "+v"(f));
                v[4 * g + e] = f;
              }
            }
          } else {
#pragma unroll
            for (int e = 0; e < 16; ++e) v[e] = acc[mt][e];
          }
          if (has_bias) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
              const uint2 bb = *reinterpret_cast<const uint2*>(p.bias + ncol + 8 * (whole ? g : g & 1) + 4 * h);
              v[4 * g + 0] += to_f32<ODT>((uint16_t)(bb.x & 0xffffu));
              v[4 * g + 1] += to_f32<ODT>((uint16_t)(bb.x >> 16));
              v[4 * g + 2] += to_f32<ODT>((uint16_t)(bb.y & 0xffffu));
              v[4 * g + 3] += to_f32<ODT>((uint16_t)(bb.y >> 16));
            }
          }
          uint32_t lo2[4], hi2[4], sw[4];
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            uint16_t o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              float f = v[4 * g + e];
              asm volatile("" : "+v"(f));
              o[e] = from_f32<ODT>(f);
            }
            lo2[g] = (uint32_t)o[0] | ((uint32_t)o[1] << 16);
            hi2[g] = (uint32_t)o[2] | ((uint32_t)o[3] << 16);
            if (p.epi)  // both outputs rounded to the storage dtype, then silu(g) * u in fp32: swiglu_forward's arithmetic
              sw[g] = (uint32_t)from_f32<ODT>(ll_silu_mul_f32(to_f32<ODT>(o[0]), to_f32<ODT>(o[1]))) |
                      ((uint32_t)from_f32<ODT>(ll_silu_mul_f32(to_f32<ODT>(o[2]), to_f32<ODT>(o[3]))) << 16);
          }
          const int64_t nn = ncol + 16 * h;
          if (p.epi) {
            swap32(sw[0], sw[2]);
            swap32(sw[1], sw[3]);
            if (store) *reinterpret_cast<u32x4*>(p.out + mrow * (p.n >> 1) + (nn >> 1)) = u32x4{sw[0], sw[2], sw[1], sw[3]};
          } else {
            swap32(lo2[0], lo2[2]);
            swap32(hi2[0], hi2[2]);
            swap32(lo2[1], lo2[3]);
            swap32(hi2[1], hi2[3]);
            if (store) {
              *reinterpret_cast<u32x4*>(p.out + mrow * p.n + nn) = u32x4{lo2[0], hi2[0], lo2[2], hi2[2]};
              *reinterpret_cast<u32x4*>(p.out + mrow * p.n + nn + 8) = u32x4{lo2[1], hi2[1], lo2[3], hi2[3]};
            }
          }
#pragma unroll
          for (int e = 0; e < 16; ++e) { acc[mt][e] = 0.f; iacc[mt][e] = 0; }
        }
      }
      first += size;
      size = sized(++t, first);
    }
  }
}

static int r16_num_cus() {
  static int cus[16] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) return 256;
  if (!cus[dev]) {
    hipDeviceProp_t prop;
    cus[dev] = hipGetDeviceProperties(&prop, dev) == hipSuccess && prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
  }
  return cus[dev];
}

// Deals n / 16 halves of 32-row groups out to the CUs: in groups, or in halves where a few workgroups would have a group more than the rest -- they
// take that much longer -- and where rows keep the column that their workgroup begins at.  us, groups -> halves, 6 / 32 rows: 8224 x 2048 11.3 -> 11.0 /
// 12.1 -> 11.7, 9248 x 3072 15.2 -> 14.4 / 17.3 -> 15.9, 9216 x 4096 21.2 -> 20.0 / 22.9 -> 20.9, 17920 x 1536 13.9 -> 13.4 / 14.4 -> 13.9; where more
// than a third of the workgroups has one group more, 11264 x 2048 12.9 -> 13.1 / 13.8 -> 13.6, and below a group per CU, 4096 x 2048 8.9 -> 9.2 /
// 9.2 -> 9.5: groups.  Returns the workgroups.
static int r16_deal(R16Params& p, int* groups) {
  const int cus = r16_num_cus();
  const int64_t halves = p.n / 16, rgs = (halves + 1) / 2;
  const bool few = rgs > cus && rgs % cus > 0 && rgs % cus <= cus / 3;
  p.piece = few && (halves + cus - 1) / cus < (rgs + cus - 1) / cus * 2 && !p.stagger ? 1 : 2;
  const int64_t pieces = p.piece == 1 ? halves : rgs;
  const int grid = (int)(pieces < cus ? pieces : cus);
  p.rbase = (int)(pieces / grid); p.rrem = (int)(pieces % grid);
  *groups = (int)((p.rbase + (p.rrem > 0)) * p.piece + 1) / 2;   // of the fullest workgroup
  return grid;
}

// the row-group loop needs R16Lds::BYTES of LDS per workgroup (160 KB at MT = 1): callers fall back when the device's opt-in
// limit is smaller
static bool r16_lds_fits(int64_t m) {
  static int optin[16] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) return true;  // no device (host-side plan queries): gfx950 assumed
  if (!optin[dev]) {
    int v = 0;
    optin[dev] = hipDeviceGetAttribute(&v, hipDeviceAttributeSharedMemPerBlockOptin, dev) == hipSuccess && v > 0 ? v : 160 * 1024;
  }
  return (m <= 32 ? R16Lds<1, false>::BYTES : R16Lds<2, true>::BYTES) <= optin[dev];   // (the larger of the two for m > 32)
}

extern "C" int ll_dense16_rows_supported(int64_t m, int64_t n, int64_t k, int epilogue) {
  if (m < 1 || m > 64 || n < 32 || n % 16 != 0 || k < 128 || k % 128 != 0) return 0;
  if (epilogue != 0 && epilogue != 1) return 0;
  return r16_lds_fits(m) ? 1 : 0;
}

// The routes of a projection of a few rows (quantization/methods.py, layered_decode.hip), us per launch, hipGraph replays over rotating weights, bf16:
// ROWS, wide outputs on the row-group loop, rows / library / split-K engine: fused gate|up 17920 x 1536 at 32 rows incl. the swiglu 13.4 / 25.2 / 30.9;
//   lm_head 151936 x 1536 at 32 rows 80.6 / 106.4 / 96.9 (5.8 TB/s); 152064 x 3584 at 64 rows 204.8 / 210.9 / 226.8; gate|up 37888 x 3584 fp16 at 64 rows
//   55.7 / 76.0 / 85.3.  It needs about one 32-row group per CU to fill the chip: down 1536 x 8960 35.8 / 21.8 / 20.7.
// ROWS_NARROWER, outputs that end inside a 32-row group, or of too few groups for a CU each.  Rows / library, 1, 8, 32 and 48 rows: 8208 x 1024 5.7 / 8.7,
//   5.8 / 8.8, 6.2 / 11.9, 7.4 / 12.6; 12080 x 3072 15.5 / 21.8, 15.6 / 20.4, 16.1 / 17.9, 17.9 / 19.7; 32752 x 3072 33.8 / 42.7 .. 35.3 / 52.9.  Rows / split-K
//   engine, 1 and 32 rows: 8208 x 4096 15.2 / 18.8, 15.7 / 22.1; 12080 x 14336 58.6 / 72.7, 67.6 / 81.3; 32784 x 8192 88 / 124, 97 / 131; the least at 8192
//   columns, whose rows lie 16 KB apart: 8208 35.6 / 35.0, 37.3 / 39.3 -- and there, above 32 rows, the library is ahead (48 rows of 12080 47.0 / 43.7,
//   5120 columns 29.5 / 30.4, 14336 77 / 86) up to 16 400 outputs (49 / 69).  Of too few groups, short contractions, rows / library: 7168 x 3072 1 row
//   12.3 / 13.1, 32 13.3 / 14.3, 48 16.9 / 19.1; 6176 x 2048 24 rows 8.7 / 12.6, 48 11.3 / 13.0; 4096 x 2048 32 rows 8.4 / 11.6; 4096 x 128 32 rows 3.3 / 4.1;
//   5120 x 1024 32 rows 5.7 / 11.5; on the other side 6144 x 3072 16 rows 12.7 / 12.7, 4096 x 3072 32 rows 12.2 / 11.3, 6144 x 4096 32 rows 16.5 / 16.4.
//   Sums run in the order of columns, as the library's do in most of these shapes above 16 rows; where it or the split-K engine cuts the contraction, 1 - 8 of 10 000
//   results round the other way, and both are equally far from 64 bits (1.66e-3 of their size in bf16).
// SPLIT, long contractions or the widest outputs of up to 32 rows on the split-K engine, engine / library: down 1536 x 8960 20.4 / 21.8, lm_head 151936 x
//   1536 94.9 / 104.1; elsewhere the library is ahead (7 / 9 on small projections, 211 / 230 on the lm_head of 3584 at 64 rows).
extern "C" int ll_dense16_route(int64_t m, int64_t n, int64_t k) {
  if (m < 1 || m > 64) return 0;
  int route = 0;
  if (k % 128 == 0) {
    if (n >= 8192 && n % 32 == 0) route |= LL_ROUTE_ROWS;
    else if (m <= 48 && n % 16 == 0 && ((n >= 8192 && !(m > 32 && k % 8192 == 0 && n < 16384)) || (k <= 3072 && n >= 7168) ||
                                        (k <= 2048 && n >= (m <= 32 ? 4096 : 5120))))
      route |= LL_ROUTE_ROWS_NARROWER;
  }
  if (m <= 32 && (k >= 4096 || n >= 32768)) route |= LL_ROUTE_SPLIT;
  return route;
}

// out [m][n] (epilogue 0, + bias) or [m][n / 2] (epilogue 1: rows of w interleaved (gate_j, up_j)) = x [m][k] @ w [n][k]^T for an
// unquantised fp16 / bf16 weight; m <= 64, n % 16 == 0, k % 128 == 0, rows 16-byte aligned.  Returns LL_OK, or an error code.
extern "C" int ll_dense16_rows_matmul(void* out, const void* x, const void* w, const void* bias, int64_t m, int64_t n, int64_t k,
                                      int64_t x_stride_m, int64_t w_stride_n, int dtype, int epilogue, void* stream) {
  if (dtype != LL_F16 && dtype != LL_BF16) return LL_ERR_DTYPE;
  if (m < 0 || n <= 0 || k <= 0) return LL_ERR_SHAPE;
  if (m == 0) return LL_OK;
  if (!ll_dense16_rows_supported(m, n, k, epilogue) || x_stride_m % 8 != 0 || w_stride_n % 8 != 0) return LL_ERR_SHAPE;
  if (!out || !x || !w || !ll_aligned16(out) || !ll_aligned16(x) || !ll_aligned16(w) || (bias && ((uintptr_t)bias & 7))) return LL_ERR_ARG;
  if ((m - 1) * x_stride_m * 2 + k * 2 >= (1ll << 31) || 32 * w_stride_n * 2 >= (1ll << 31)) return LL_ERR_SHAPE;
  R16Params p{};
  p.out = (uint16_t*)out; p.x = (const uint16_t*)x; p.w = (const uint16_t*)w; p.bias = (const uint16_t*)bias;
  p.m = m; p.n = n; p.k = k; p.x_stride = x_stride_m; p.w_stride = w_stride_n;
  p.stagger = w_stride_n % 2048 == 0 && n * k * 2 >= (1ll << 28);
  p.epi = epilogue;
  int groups = 0;
  const int grid = r16_deal(p, &groups);
  const bool wide = m > 32 && groups > 4;
  p.chunks = (int)(k * 2 / (wide ? 128 : 256));
  hipStream_t st = (hipStream_t)stream;
#define R16_GO(MT, DT, WIDE)                                                                                                   \
  {                                                                                                                      \
    static bool attr_[16] = {false}; /* per device */                                                   \
    int dev_ = 0;                                                                                                        \
    (void)hipGetDevice(&dev_);                                                                                           \
    if (dev_ >= 0 && dev_ < 16 && !attr_[dev_]) {                                                                        \
      (void)hipFuncSetAttribute((const void*)wgemm16_rows_kernel<MT, DT, WIDE>, hipFuncAttributeMaxDynamicSharedMemorySize, R16Lds<MT, WIDE>::BYTES); \
      attr_[dev_] = true;                                                                                                \
    }                                                                                                                    \
    wgemm16_rows_kernel<MT, DT, WIDE><<<dim3((unsigned)grid), R16Lds<MT, WIDE>::THREADS, R16Lds<MT, WIDE>::BYTES, st>>>(p);                          \
  }
  if (m <= 32) {
    if (dtype == LL_F16) R16_GO(1, LL_F16, false) else R16_GO(1, LL_BF16, false)
  } else if (wide) {
    if (dtype == LL_F16) R16_GO(2, LL_F16, true) else R16_GO(2, LL_BF16, true)
  } else {
    if (dtype == LL_F16) R16_GO(2, LL_F16, false) else R16_GO(2, LL_BF16, false)
  }
#undef R16_GO
  return LL_LAUNCH_CHECK();
}

// smoothquant (W8A8) form: out [m][n] fp16 (epilogue 0, + bias) or [m][n / 2] (epilogue 1: rows of qw interleaved (gate_j, up_j)) =
// fp16(((float)(qa [m][k] int8 @ qw [n][k]^T int32) * a_scale[m]) * w_scale[n] (+ bias)) -- ll_w8a8_matmul's epilogue
// (kernels/quantization/w8a8.py:118-149), exact int32 sums on mfma_i32_32x32x32_i8; then silu(gate) * up on the rounded outputs
// (= ll_w8a8_finish_swiglu).  m <= 64, n % 32 == 0, k % 256 == 0, row strides (bytes) % 16 == 0.
extern "C" int ll_w8a8_rows_supported(int64_t m, int64_t n, int64_t k, int epilogue) {
  return (m >= 1 && m <= 64 && n >= 32 && n % 32 == 0 && k >= 256 && k % 256 == 0 && (epilogue == 0 || epilogue == 1) && r16_lds_fits(m)) ? 1 : 0;
}

extern "C" int ll_w8a8_rows_matmul(void* out, const int8_t* qa, const float* a_scale, const int8_t* qw, const float* w_scale,
                                   const void* bias, int64_t m, int64_t n, int64_t k, int64_t qa_stride_m, int64_t qw_stride_n,
                                   int epilogue, void* stream) {
  if (m < 0 || n <= 0 || k <= 0) return LL_ERR_SHAPE;
  if (m == 0) return LL_OK;
  if (!ll_w8a8_rows_supported(m, n, k, epilogue) || qa_stride_m % 16 != 0 || qw_stride_n % 16 != 0) return LL_ERR_SHAPE;
  if (!out || !qa || !qw || !a_scale || !w_scale || !ll_aligned16(out) || !ll_aligned16(qa) || !ll_aligned16(qw) || !ll_aligned16(w_scale) ||
      (bias && ((uintptr_t)bias & 7)))
    return LL_ERR_ARG;
  if ((m - 1) * qa_stride_m + k >= (1ll << 31) || 32 * qw_stride_n >= (1ll << 31)) return LL_ERR_SHAPE;
  R16Params p{};
  p.out = (uint16_t*)out; p.x = (const uint16_t*)qa; p.w = (const uint16_t*)qw; p.bias = (const uint16_t*)bias;
  p.a_scale = a_scale; p.w_scale = w_scale;
  p.m = m; p.n = n; p.k = k;
  p.x_stride = qa_stride_m / 2; p.w_stride = qw_stride_n / 2;  // the kernel addresses rows in 2-byte units
  p.stagger = qw_stride_n % 4096 || n * k < (1ll << 26) ? 0 : n * k < (1ll << 28) ? 5 : 1;
  p.epi = epilogue;
  int groups = 0;
  const int grid = r16_deal(p, &groups);
  const bool wide = m > 32 && groups > 4;
  p.chunks = (int)(k / (wide ? 128 : 256));
  hipStream_t st = (hipStream_t)stream;
#define R16_GO8(MT, WIDE)                                                                                                      \
  {                                                                                                                      \
    static bool attr_[16] = {false}; /* per device */                                                   \
    int dev_ = 0;                                                                                                        \
    (void)hipGetDevice(&dev_);                                                                                           \
    if (dev_ >= 0 && dev_ < 16 && !attr_[dev_]) {                                                                        \
      (void)hipFuncSetAttribute((const void*)wgemm16_rows_kernel<MT, R16_I8, WIDE>, hipFuncAttributeMaxDynamicSharedMemorySize, R16Lds<MT, WIDE>::BYTES); \
      attr_[dev_] = true;                                                                                                \
    }                                                                                                                    \
    wgemm16_rows_kernel<MT, R16_I8, WIDE><<<dim3((unsigned)grid), R16Lds<MT, WIDE>::THREADS, R16Lds<MT, WIDE>::BYTES, st>>>(p);                      \
  }
  if (m <= 32) R16_GO8(1, false) else if (wide) R16_GO8(2, true) else R16_GO8(2, false)
#undef R16_GO8
  return LL_LAUNCH_CHECK();
}
