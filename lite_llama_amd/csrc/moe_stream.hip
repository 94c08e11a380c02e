// Grouped expert products of a few rows per expert: weights are streamed once, at the rate of memory.
//
//   * Persistent workgroups (one per CU; two where 8-bit weights have to be widened) own contiguous runs of 16-row groups of the weights that
//     the step touches (row groups of all row blocks in order, dealt out to within one) and walk them in tiles of four groups, ALL of the
//     contraction each.  Workgroups of one tile each, which this replaces where few rows meet an expert, come and go six times per CU and pay
//     their chain of dependent loads (block -> expert and slots -> addresses -> weights) every time; here the row lists are read once, and
//     the loads run ahead ACROSS tiles.
//   * Four LOADER waves fill a ring of units by LDS-DMA -- 64 weight rows x 256 bytes, the block's activation rows of the same contraction
//     range (half of their places are skipped where no block of the run fills them), 8-bit weights also their scales.  Four CONSUMER waves,
//     one per row group, multiply from LDS (MFMA 16 x 16 x 32).  16-byte pieces of row r stand at slot ^ (r & 15): fragment reads are free of
//     bank conflicts.  One barrier per unit.
//   * An expert's contraction begins at unit e mod units and wraps: experts whose rows are a power of two long do not all ask the same
//     memory channels, and the order of a sum depends on the expert alone, not on what else rides along.
//   * Bound by memory, the chain in front of the first unit (about 5 us) and, for 8-bit weights, the widening between two barriers: a second
//     workgroup per CU fills those gaps (128 experts of 2048 / 768 in 8-bit floats, 64 tokens with 8 each, both products: 128 us with one
//     workgroup per CU, 117 with two; 16-bit weights gain nothing by it).  Ring depths of 4 to 6 units are alike.
//   us for both products, tiles -> here.  8-bit floats, 128 experts of 2048 / 768, top 8: 1 token 42 -> 24, 8 67 -> 54, 32 120 -> 102, 64
//   137 -> 117 (604 MB: 5.2 TB/s); in pieces of 32 rows (of 16) 200 167 -> 155 (167), 256 178 -> 162 (209), 320 181 -> 168, 400 186 -> 191.  bf16, 34 of 2048 / 704, top 4: 1 token 33 -> 17, 32 tokens 77 -> 58, 128 78 -> 65; 68 of 3072 / 512,
//   top 8: 6 tokens 89 -> 74, 32 156 -> 111 (642 MB), 128 160 -> 126; in pieces of 64 rows 160 tokens 161 -> 131, 262 (31 rows per expert) 165 ->
//   150 (pieces of 32: 185), 34 experts 200 77 -> 73, 300 (35) 78.5 -> 77, 400 (47) 80 -> 85: up to 36 rows per expert in ll_moe_rows_gemm.  ll_moe_gemm has other
//   tiles and lines of its own (moe.hip).
#include <stdlib.h>

#include "gemm_w4_common.h"
#include "moe_stream.h"

namespace {

typedef __bf16 ms_bf16x8 __attribute__((ext_vector_type(8)));

constexpr int MS_LIST = 512, MS_OWN = 8;   // row blocks in all / of one workgroup
constexpr int MS_W_BYTES = 64 * 256;

template <int WF, int MT_>
struct MsLds {
  static constexpr int THREADS = 512;                          // four consumers, four loaders
  static constexpr int PER_CU = WF != MS_W16 && MT_ == 1 ? 2 : 1, RING = PER_CU == 2 ? 3 : 4;
  static constexpr int MT = MT_, ROWS = 16 * MT;               // rows of a piece of a block
  static constexpr int KU = WF == MS_W16 ? 128 : 256;          // contraction entries of a unit
  static constexpr int X_BYTES = ROWS * KU * 2;
  static constexpr int S_BYTES = WF == MS_W16 ? 0 : 64 * 4 * 4;   // scales: [loader][64-column step][16 rows]
  static constexpr int SLOT = MS_W_BYTES + X_BYTES + S_BYTES;
  static constexpr int LIST = RING * SLOT;                  // int32 [MS_LIST]: row block | expert << 16
  static constexpr int OWN = LIST + MS_LIST * 4;   // int32 [MS_OWN]: expert
  static constexpr int SLOTS = OWN + MS_OWN * 4;               // int32 [MS_OWN][ROWS]
  static constexpr int WEIGHTS = SLOTS + MS_OWN * ROWS * 4;    // float [MS_OWN][ROWS]
  static constexpr int COUNTS = WEIGHTS + MS_OWN * ROWS * 4;   // int32 [8], [1]
  static constexpr int BYTES = COUNTS + 48;                    // (nothing static: the ring begins at LDS byte 0)
  static_assert(BYTES * PER_CU <= 160 * 1024, "LDS");
  static constexpr int XOPS = X_BYTES / 4096;                  // activation operations per loader and unit
};

__device__ const uint32_t ms_zeros[4] __attribute__((aligned(16))) = {0, 0, 0, 0};   // what pieces without an entry read

// 64 lanes x 16 bytes from per-lane addresses to LDS at byte `dst`
__device__ __forceinline__ void ms_dma16(uint32_t dst, const void* src) {
  dst = __builtin_amdgcn_readfirstlane(dst);
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "s"(dst), "v"(src) : "memory");
}

template <int OPS>
__device__ __forceinline__ void ms_wait_units(int k) {   // at most k units of OPS operations each may still be in flight
  if (k <= 0) v3_vmcnt<0>();
  else if (k == 1) v3_vmcnt<OPS>();
  else v3_vmcnt<2 * OPS>();
}

// eight 8-bit weights -> fp16, exactly (8-bit floats: times 2^-8; the codes 0x7f and 0xff as 480, as in moe.hip)
template <int WF>
__device__ __forceinline__ u32x4 ms_widen(uint32_t lo, uint32_t hi) {
  u32x4 o;
  if constexpr (WF == MS_INT8) {
    lo ^= 0x80808080u;
    hi ^= 0x80808080u;
    o.x = v3_pk_add(__builtin_amdgcn_perm(0x64646464u, lo, 0x04010400u), 0xE480E480u);
    o.y = v3_pk_add(__builtin_amdgcn_perm(0x64646464u, lo, 0x04030402u), 0xE480E480u);
    o.z = v3_pk_add(__builtin_amdgcn_perm(0x64646464u, hi, 0x04010400u), 0xE480E480u);
    o.w = v3_pk_add(__builtin_amdgcn_perm(0x64646464u, hi, 0x04030402u), 0xE480E480u);
  } else {   // sign, four exponent and three mantissa bits one place down, the sign's copy cleared
    typedef short s16x2 __attribute__((ext_vector_type(2)));
    auto half = [](uint32_t w, uint32_t sel) {
      const s16x2 v = __builtin_bit_cast(s16x2, __builtin_amdgcn_perm(0u, w, sel)) >> 1;
      return __builtin_bit_cast(uint32_t, v) & 0xBFFFBFFFu;
    };
    o.x = half(lo, 0x010C000Cu);
    o.y = half(lo, 0x030C020Cu);
    o.z = half(hi, 0x010C000Cu);
    o.w = half(hi, 0x030C020Cu);
  }
  return o;
}

template <int DT>
__device__ __forceinline__ f32x4 ms_mfma(const u32x4& a, const u32x4& b, f32x4 c) {
  if constexpr (DT == LL_F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ms_bf16x8, a), __builtin_bit_cast(ms_bf16x8, b), c, 0, 0, 0);
}

// the gated pair of fp32 sums (moe_sparse.hip has the same one): limit < 0: silu(g) u; else g' sigmoid(1.702 g') (u' + 1)
__device__ __forceinline__ float ms_glu(float g, float u, float limit) {
  if (limit >= 0.f) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit) + 1.0f;
    return g * ll_sigmoidf(1.702f * g) * u;
  }
  return g * ll_sigmoidf(g) * u;
}

template <int WF, int MT, int MODE, int XOPS>
__device__ __forceinline__ void ms_load(const MoeStreamParams& p, unsigned char* lds, int L, int lane, int lo, int hi, int rgs, int i0, int units, int total) {
  using LD = MsLds<WF, MT>;
  constexpr int KU = LD::KU, EB = WF == MS_W16 ? 2 : 1, ROWS = LD::ROWS;
  constexpr int OPS = 4 + XOPS + (WF == MS_W16 ? 0 : 1);
  const int32_t* experts = reinterpret_cast<const int32_t*>(lds + LD::OWN);
  const int32_t* rows = reinterpret_cast<const int32_t*>(lds + LD::SLOTS);
  const int row_bytes = p.K * EB;
  const char *wbase = nullptr, *sbase = nullptr;   // the expert's matrix and scales
  uint32_t woff[4], xoff[XOPS], soff = 0;          // where this lane's pieces of unit 0 begin
  bool live = false;
  int rg = lo, unit = 0, left = 0, issued = 0;
  uint32_t dst = 0;
  // (piece `at` of row r comes from byte 16 (at ^ (r & 15)) of it)
  auto open = [&]() {   // the tile at row group rg
    const int i = rg / rgs, r0 = rg - i * rgs;
    const int e = __builtin_amdgcn_readfirstlane(experts[i - i0]);
    int groups = rgs - r0 < 4 ? rgs - r0 : 4;
    groups = hi - rg < groups ? hi - rg : groups;
    live = L < groups;
    const int g = r0 + L;
    wbase = (const char*)p.w + (int64_t)e * p.w_stride_e;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = 4 * j + (lane >> 4);
      int row;
      if constexpr (MODE == MS_GLU) {
        row = 8 * g + (r >> 1);
        row = (row < p.N ? row : p.N - 1) + (r & 1 ? p.N : 0);
      } else {
        row = 16 * g + r;
        row = row < p.N ? row : p.N - 1;   // rows behind N feed results that are not stored
      }
      woff[j] = (uint32_t)row * (uint32_t)p.w_stride_n + ((lane & 15) ^ r) * 16;
    }
    const int32_t* own = rows + (i - i0) * ROWS;
#pragma unroll
    for (int j = 0; j < XOPS; ++j) {
      const int at = L + 4 * j;
      const int r = WF == MS_W16 ? 4 * at + (lane >> 4) : 2 * at + (lane >> 5);
      const int slot = own[r];   // (places without a slot read row 0: they feed results that are not stored)
      xoff[j] = (slot < p.num_slots ? (uint32_t)(slot / p.a_div) * (uint32_t)(p.a_ld * 2) : 0u) +
                ((WF == MS_W16 ? (lane & 15) : (lane & 31)) ^ (r & 15)) * 16;
    }
    if constexpr (WF != MS_W16) {
      int row = 16 * g + (lane & 15);
      row = row < p.N ? row : p.N - 1;
      sbase = (const char*)(p.scales + (int64_t)e * p.s_stride_e);
      soff = (uint32_t)(row / (int)p.group_n) * (uint32_t)(p.s_stride_n * 4);
    }
    unit = e % units;
    left = units;
    rg += groups;
  };
  auto issue = [&]() {
    if (left == 0) open();
    const int at = unit * 256, xat = unit * (KU * 2);
    if (at + 256 <= row_bytes) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (live) v3_dma16<true>(dst + (4 * L + j) * 1024, wbase + at, woff[j]);
        else v3_dma16<false>(dst + (4 * L + j) * 1024, ms_zeros, 0u);
      }
#pragma unroll
      for (int j = 0; j < XOPS; ++j) v3_dma16<false>(dst + MS_W_BYTES + (L + 4 * j) * 1024, (const char*)p.a + xat, xoff[j]);
    } else {   // the contraction ends inside the unit: zeros behind it, on both sides
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int piece = ((lane & 15) ^ (4 * j + (lane >> 4))) * 16;
        ms_dma16(dst + (4 * L + j) * 1024, live && at + piece < row_bytes ? wbase + at + woff[j] : (const char*)ms_zeros);
      }
#pragma unroll
      for (int j = 0; j < XOPS; ++j) {
        const int r = WF == MS_W16 ? 4 * (L + 4 * j) + (lane >> 4) : 2 * (L + 4 * j) + (lane >> 5);
        const int piece = ((WF == MS_W16 ? (lane & 15) : (lane & 31)) ^ (r & 15)) * 16;
        ms_dma16(dst + MS_W_BYTES + (L + 4 * j) * 1024, xat + piece < p.K * 2 ? (const char*)p.a + xat + xoff[j] : (const char*)ms_zeros);
      }
    }
    if constexpr (WF != MS_W16) {
      int k = unit * KU + (lane >> 4) * 64;
      k = k < p.K ? k : p.K - 1;
      v3_dma4<false>(dst + MS_W_BYTES + LD::X_BYTES + L * 256, sbase, soff + (uint32_t)(k >> p.k_shift) * (uint32_t)(p.s_stride_k * 4));
    }
    if (++unit == units) unit = 0;
    --left;
    ++issued;
    dst = dst + LD::SLOT == LD::RING * LD::SLOT ? 0 : dst + LD::SLOT;
  };
  const int pre = total < LD::RING - 1 ? total : LD::RING - 1;
  for (int i = 0; i < pre; ++i) issue();
  ms_wait_units<OPS>(issued - 1);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // P0: unit 0 has landed
  for (int u = 0; u < total; ++u) {
    if (issued < total) issue();   // into the slot of unit u - 1, free since the barrier that ended it
    const int need = total < u + 2 ? total : u + 2;
    ms_wait_units<OPS>(issued - need);   // unit u + 1 has landed before the consumers are released into it
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // B_u
  }
}

template <int DT, int WF, int MT, int MODE>
__global__ __launch_bounds__((MsLds<WF, MT>::THREADS)) __attribute__((amdgpu_waves_per_eu(2 * (MsLds<WF, MT>::PER_CU), 2 * (MsLds<WF, MT>::PER_CU)))) void moe_stream_kernel(const MoeStreamParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  using LD = MsLds<WF, MT>;
  constexpr int KU = LD::KU, ROWS = LD::ROWS, THREADS = LD::THREADS;
  constexpr bool PAIRS = MODE == MS_GLU || MODE == MS_GLU_ROUNDED;
  uint32_t* list = reinterpret_cast<uint32_t*>(lds + LD::LIST);
  int32_t* rows = reinterpret_cast<int32_t*>(lds + LD::SLOTS);
  float* weights = reinterpret_cast<float*>(lds + LD::WEIGHTS);
  int* part = reinterpret_cast<int*>(lds + LD::COUNTS);
  int* most_rows = part + 8;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int sub = p.block_m / ROWS;                       // pieces of ROWS rows per block
  const int rgs = MODE == MS_GLU ? (p.N + 7) / 8 : (p.N + 15) / 16;
  const int nout = MODE == MS_GLU_ROUNDED ? p.N / 2 : p.N;
  if (tid == 0) *most_rows = 0;

  // the pieces with a slot, in order (a block's slots stand in front).  Lists are requested before num_post is known, as far as they exist.
  const int cap = (p.safe + ROWS - 1) / ROWS;
  int first = p.num_slots, expert = 0;
  if (tid < cap) {
    first = p.sorted[tid * ROWS];
    expert = p.block_expert[tid / sub];
  }
  int post = p.num_post[0];
  asm volatile("" : "+v"(first), "+v"(expert), "+s"(post));   // (requested together)
  const int pieces = post / ROWS;
  int count = 0, skipped = 0;
  for (int j0 = 0; j0 < pieces; j0 += THREADS) {
    const int j = j0 + tid;
    if ((j0 > 0 || tid >= cap) && j < pieces) {
      first = p.sorted[j * ROWS];
      expert = p.block_expert[j / sub];
    }
    const bool has = j < pieces && first < p.num_slots, in = has && expert >= 0;
    const unsigned long long mask = __ballot(in), none = __ballot(has && expert < 0);
    if (lane == 0) part[wv] = __popcll(mask) | __popcll(none) << 16;
    __syncthreads();
    int at = count, behind = skipped;
    for (int w = 0; w < THREADS / 64; ++w) {
      const int n = part[w];
      if (w < wv) {
        at += n & 0xffff;
        behind += n >> 16;
      }
      count += n & 0xffff;
      skipped += n >> 16;
    }
    const unsigned long long below = (1ull << lane) - 1ull;
    at += __popcll(mask & below);
    behind = MS_LIST - 1 - (behind + __popcll(none & below));
    if (in && at < MS_LIST) list[at] = (uint32_t)j | (uint32_t)expert << 16;
    if (has && expert < 0 && behind >= 0) list[behind] = (uint32_t)j;
    __syncthreads();
  }
  count = __builtin_amdgcn_readfirstlane(count);
  skipped = __builtin_amdgcn_readfirstlane(skipped);
  if constexpr (!PAIRS) {   // slots that no expert serves: zeros (of the last product; nothing reads the first one's)
    for (int t = (int)blockIdx.x; t < skipped * ROWS; t += (int)gridDim.x) {
      const int slot = p.sorted[(int)list[MS_LIST - 1 - t / ROWS] * ROWS + t % ROWS];
      if (slot < p.num_slots)
        for (int c = tid; c < p.N; c += THREADS) p.out[(int64_t)slot * p.out_ld + c] = 0;
    }
  }
  const int64_t total_rg = (int64_t)count * rgs;
  const int b = (int)blockIdx.x, grid = (int)gridDim.x;
  const int lo = (int)(total_rg * b / grid), hi = (int)(total_rg * (b + 1) / grid);
  if (lo >= hi) return;
  const int i0 = lo / rgs, own = (hi - 1) / rgs - i0 + 1;   // row blocks of this run
  if (tid < own) reinterpret_cast<int32_t*>(lds + LD::OWN)[tid] = (int)(list[i0 + tid] >> 16);
  if (tid < own * ROWS) {
    const int slot = p.sorted[(int)(list[i0 + tid / ROWS] & 0xffffu) * ROWS + tid % ROWS];
    rows[tid] = slot;
    if (slot < p.num_slots) atomicMax(most_rows, tid % ROWS + 1);
  }
  __syncthreads();
  const int units = (p.K + KU - 1) / KU;
  int tiles = 0;
  for (int rg = lo; rg < hi; ++tiles) {
    const int r0 = rg % rgs;
    int groups = rgs - r0 < 4 ? rgs - r0 : 4;
    rg += hi - rg < groups ? hi - rg : groups;
  }
  const int total = tiles * units;
  const int full = __builtin_amdgcn_readfirstlane(*most_rows);

  if (wv >= 4) {
    if (full > ROWS / 2) ms_load<WF, MT, MODE, LD::XOPS>(p, lds, wv - 4, lane, lo, hi, rgs, i0, units, total);
    else ms_load<WF, MT, MODE, LD::XOPS / 2>(p, lds, wv - 4, lane, lo, hi, rgs, i0, units, total);
    return;
  }

  // consumers: row group wv of every tile
  for (int i = tid; i < own * ROWS; i += 256) {
    const int slot = rows[i];
    float v = 1.f;
    if (slot < p.num_slots) {
      if (p.weight32) v = p.weight32[slot];
      else if (p.weight16) v = f16_bits_to_f32(p.weight16[slot]);
    }
    weights[i] = v;
  }
  const int r = lane & 15, q = lane >> 4;
  f32x4 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bool wide = ((PAIRS ? 2 : 4) * 2 - 1 & (int)(reinterpret_cast<uintptr_t>(p.out) | (uintptr_t)(p.out_ld * 2))) == 0;
  uint32_t slot_at = 0;
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // P0
  for (int rg = lo; rg < hi;) {
    const int i = rg / rgs, r0 = rg - i * rgs;
    int groups = rgs - r0 < 4 ? rgs - r0 : 4;
    groups = hi - rg < groups ? hi - rg : groups;
    const bool mine = wv < groups;
    for (int u = 0; u < units; ++u) {
      if (mine) {
        const unsigned char* wb = lds + slot_at + wv * 4096 + r * 256;
        const unsigned char* xb = lds + slot_at + MS_W_BYTES + r * (KU * 2);
        // (all fragments of the unit are requested before the first is used: one wave per matrix core waits for LDS once)
        if constexpr (WF == MS_W16) {
          u32x4 wf[4], x[MT][4];
#pragma unroll
          for (int s = 0; s < 4; ++s) wf[s] = *reinterpret_cast<const u32x4*>(wb + ((4 * s + q) ^ r) * 16);
#pragma unroll
          for (int m = 0; m < MT; ++m)
            if (m == 0 || 16 * m < full)
#pragma unroll
              for (int s = 0; s < 4; ++s) x[m][s] = *reinterpret_cast<const u32x4*>(xb + 16 * m * KU * 2 + ((4 * s + q) ^ r) * 16);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int m = 0; m < MT; ++m)
            if (m == 0 || 16 * m < full)
#pragma unroll
              for (int s = 0; s < 4; ++s) acc[m] = ms_mfma<DT>(wf[s], x[m][s], acc[m]);
        } else {
          // a lane's 16 weights of a 64-column step feed two products; the activations' columns are taken in the same order.  The step's
          // sums are multiplied by the scales of their weight rows: a weight enters exactly.
          const float* sb = reinterpret_cast<const float*>(lds + slot_at + MS_W_BYTES + LD::X_BYTES) + wv * 64 + 4 * q;
          u32x4 raw[4], x0[MT][4], x1[MT][4];
          f32x4 sv[4], step[4];
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            raw[t] = *reinterpret_cast<const u32x4*>(wb + ((4 * t + q) ^ r) * 16);
            sv[t] = *reinterpret_cast<const f32x4*>(sb + t * 16);
          }
#pragma unroll
          for (int m = 0; m < MT; ++m)
            if (m == 0 || 16 * m < full)
#pragma unroll
              for (int t = 0; t < 4; ++t) {
                x0[m][t] = *reinterpret_cast<const u32x4*>(xb + 16 * m * KU * 2 + ((8 * t + 2 * q) ^ r) * 16);
                x1[m][t] = *reinterpret_cast<const u32x4*>(xb + 16 * m * KU * 2 + ((8 * t + 2 * q + 1) ^ r) * 16);
              }
          __builtin_amdgcn_sched_barrier(0);
          u32x4 w0[4], w1[4];
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            w0[t] = ms_widen<WF>(raw[t].x, raw[t].y);
            w1[t] = ms_widen<WF>(raw[t].z, raw[t].w);
          }
#pragma unroll
          for (int m = 0; m < MT; ++m)
            if (m == 0 || 16 * m < full) {
#pragma unroll
              for (int t = 0; t < 4; ++t) {
                step[t] = ms_mfma<LL_F16>(w0[t], x0[m][t], f32x4{0.f, 0.f, 0.f, 0.f});
                step[t] = ms_mfma<LL_F16>(w1[t], x1[m][t], step[t]);
              }
#pragma unroll
              for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[m][i] = __builtin_fmaf(step[t][i], sv[t][i], acc[m][i]);
            }
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // B_u: this unit's slot may be refilled
      slot_at = slot_at + LD::SLOT == LD::RING * LD::SLOT ? 0 : slot_at + LD::SLOT;
    }
    if (mine) {
      if constexpr (WF == MS_FP8) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int t = 0; t < 4; ++t) acc[m][t] *= 256.0f;   // (exact: what ms_widen left out)
      }
      // a lane holds weight rows 4 q .. 4 q + 3 of the group for row r (+ 16 m)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int slot = rows[(i - i0) * ROWS + 16 * m + r];
        const float weight = weights[(i - i0) * ROWS + 16 * m + r];
        if (slot < p.num_slots) {
          uint16_t* orow = p.out + (int64_t)slot * p.out_ld;
          if constexpr (PAIRS) {
            uint16_t y[2];
            const int col = (r0 + wv) * 8 + 2 * q;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
              const float g = acc[m][2 * t], v = acc[m][2 * t + 1];
              if constexpr (MODE == MS_GLU_ROUNDED)
                y[t] = from_f32<DT>(ll_silu_mul_f32(to_f32<DT>(from_f32<DT>(g * weight)), to_f32<DT>(from_f32<DT>(v * weight))));
              else
                y[t] = from_f32<DT>(ms_glu(g, v, p.limit));
            }
            if (wide && col + 1 < nout) *reinterpret_cast<uint32_t*>(orow + col) = (uint32_t)y[0] | (uint32_t)y[1] << 16;
            else {
              if (col < nout) orow[col] = y[0];
              if (col + 1 < nout) orow[col + 1] = y[1];
            }
          } else {
            uint16_t y[4];
            const int col = (r0 + wv) * 16 + 4 * q;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              float v = acc[m][t] * weight;
              if constexpr (MODE == MS_RELU2) {
                v = fmaxf(v, 0.f);
                v = v * v;
              }
              y[t] = from_f32<DT>(v);
            }
            if (wide && col + 3 < nout)
              *reinterpret_cast<uint2*>(orow + col) = uint2{(uint32_t)y[0] | (uint32_t)y[1] << 16, (uint32_t)y[2] | (uint32_t)y[3] << 16};
            else
#pragma unroll
              for (int t = 0; t < 4; ++t)
                if (col + t < nout) orow[col + t] = y[t];
          }
        }
      }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    rg += groups;
  }
}

int ms_cus(int* lds) {
  static int cus[16] = {0}, optin[16] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) return 0;
  if (!cus[dev]) {
    int n = 0, v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeSharedMemPerBlockOptin, dev) != hipSuccess) v = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) n = 0;
    optin[dev] = v;
    cus[dev] = n > 0 ? n : 1;
  }
  *lds = optin[dev];
  return cus[dev];
}

int ms_lds(int wfmt, int rows) { return wfmt != MS_W16 ? (rows == 32 ? MsLds<MS_FP8, 2>::BYTES : MsLds<MS_FP8, 1>::BYTES) : rows == 64 ? MsLds<MS_W16, 4>::BYTES : MsLds<MS_W16, 2>::BYTES; }

// rows of a piece.  8-bit weights: 16, or 32 from 9 rows per expert on, beside many experts from 12 on (us, pieces of 16 / 32: 128 experts of 2048 / 768, 10 rows
// 147 / 153, 12 160 / 156, 16 204 / 162; 200 of 2048 / 512, 12 170 / 181, 14 192 / 184; 64 of 2048 / 768, 10 76 / 77, 12 83 / 81; 32, 10 44 / 43, 12 52 / 49; 8,
// 10 28 / 24).  16-bit ones: 32, or 64 from 16 on (128, 16 239 / 240, 24 271 / 265, 32 375 / 282)
int ms_rows(const MoeStreamParams& p, int wfmt, int64_t experts) {
  if (wfmt != MS_W16) return p.num_slots > (experts > 40 ? 12 : 9) * experts && p.block_m % 32 == 0 ? 32 : 16;
  return p.num_slots > 16 * experts && p.block_m % 64 == 0 ? 64 : 32;
}

template <int DT, int WF, int MT, int MODE>
int ms_go(const MoeStreamParams& p, int grid, hipStream_t stream) {
  constexpr int bytes = MsLds<WF, MT>::BYTES;
  static bool attr[16] = {false};
  int dev = 0;
  (void)hipGetDevice(&dev);
  if (dev >= 0 && dev < 16 && !attr[dev]) {
    (void)hipFuncSetAttribute((const void*)moe_stream_kernel<DT, WF, MT, MODE>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    attr[dev] = true;
  }
  moe_stream_kernel<DT, WF, MT, MODE><<<dim3((unsigned)grid * MsLds<WF, MT>::PER_CU), MsLds<WF, MT>::THREADS, bytes, stream>>>(p);
  return LL_LAUNCH_CHECK();
}

}  // namespace

bool moe_stream_wants(const MoeStreamParams& p, int wfmt, int mode, int dtype, int64_t experts, int64_t runs) {
  static const bool off = getenv("LL_MOE_NO_STREAM") != nullptr;   // A/B knob, read once
  if (off || (dtype != LL_F16 && (dtype != LL_BF16 || wfmt != MS_W16)) || experts > 65535 || runs > 65535) return false;
  const int eb = wfmt == MS_W16 ? 2 : 1, rows = ms_rows(p, wfmt, experts);
  if (p.block_m % rows || p.K < 128 || (int64_t)p.K * eb % 16 || p.K > (1 << 24) || p.N < 16 || p.N > (1 << 24) || p.a_ld % 8 ||
      p.w_stride_n % 16 || p.w_stride_e % 16 || !ll_aligned16(p.a) || !ll_aligned16(p.w) || (mode == MS_GLU_ROUNDED && p.N % 2))
    return false;
  if (p.w_stride_n * (mode == MS_GLU ? 2 : 1) * (int64_t)p.N >= (1ll << 32) || ((int64_t)p.num_slots / p.a_div + 1) * p.a_ld * 2 >= (1ll << 32)) return false;
  if (wfmt != MS_W16) {   // (scales of whole 64-column steps, found by a shift)
    const bool one = p.group_k >= p.K;
    if (mode == MS_GLU || p.group_n < 1 || (!one && (p.group_k < 64 || (p.group_k & (p.group_k - 1)))) || p.s_stride_n < 0 || p.s_stride_k < 0 ||
        ((int64_t)p.N * p.s_stride_n + p.K / 64 * p.s_stride_k) * 4 >= (1ll << 32))
      return false;
  }
  int lds = 0;
  const int cus = ms_cus(&lds);
  const int64_t most = ((int64_t)p.num_slots + (runs + 1) * (p.block_m - 1)) / rows + 1;
  const int64_t filled = p.num_slots / rows + runs + 1;   // pieces with a slot
  return cus > 0 && filled <= MS_LIST && filled / cus + 2 <= MS_OWN && most <= 65535 && ms_lds(wfmt, rows) <= lds &&
         (filled + 1) * (((int64_t)p.N + 7) / 8) < (1ll << 30);
}

int moe_stream_launch(const MoeStreamParams& asked, int wfmt, int mode, int dtype, int64_t experts, hipStream_t stream) {
  MoeStreamParams p = asked;
  p.group_n = p.group_n < p.N ? p.group_n : p.N;
  p.k_shift = 31;
  if (wfmt != MS_W16 && p.group_k < p.K)
    for (p.k_shift = 6; (1ll << p.k_shift) < p.group_k; ++p.k_shift) {}
  int lds = 0;
  const int cus = ms_cus(&lds);
#define MS_8(WF, MODE) return ms_rows(p, wfmt, experts) == 32 ? ms_go<LL_F16, WF, 2, MODE>(p, cus, stream) : ms_go<LL_F16, WF, 1, MODE>(p, cus, stream)
  if (wfmt == MS_FP8) {
    if (mode == MS_GLU_ROUNDED) MS_8(MS_FP8, MS_GLU_ROUNDED);
    MS_8(MS_FP8, MS_SCALED);
  }
  if (wfmt == MS_INT8) {
    if (mode == MS_GLU_ROUNDED) MS_8(MS_INT8, MS_GLU_ROUNDED);
    MS_8(MS_INT8, MS_SCALED);
  }
#undef MS_8
  const bool deep = ms_rows(p, wfmt, experts) == 64;
#define MS_W(DT, MODE) return deep ? ms_go<DT, MS_W16, 4, MODE>(p, cus, stream) : ms_go<DT, MS_W16, 2, MODE>(p, cus, stream)
  if (dtype == LL_F16) {
    if (mode == MS_SCALED) MS_W(LL_F16, MS_SCALED);
    if (mode == MS_RELU2) MS_W(LL_F16, MS_RELU2);
    if (mode == MS_GLU) MS_W(LL_F16, MS_GLU);
    MS_W(LL_F16, MS_GLU_ROUNDED);
  }
  if (mode == MS_SCALED) MS_W(LL_BF16, MS_SCALED);
  if (mode == MS_RELU2) MS_W(LL_BF16, MS_RELU2);
  if (mode == MS_GLU) MS_W(LL_BF16, MS_GLU);
#undef MS_W
  return LL_ERR_SHAPE;
}
