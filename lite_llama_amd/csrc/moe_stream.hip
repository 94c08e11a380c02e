// Grouped expert products of a few rows per expert: weights are streamed once, at the rate of memory.
//
//   * Persistent workgroups, one per CU, own contiguous runs of 16-row groups of the weights that the step touches (row groups of all row blocks in
//     order, dealt out to within one) and walk them in tiles of up to eight groups, ALL of the contraction each.  Workgroups of one tile each,
//     which this replaces where few rows meet an expert, come and go six times per CU and pay their chain of dependent loads (block -> expert
//     and slots -> addresses -> weights) every time; here the row lists are read once, and the loads run ahead ACROSS tiles.
//   * Four LOADER waves fill a ring of units by LDS-DMA -- up to 128 weight rows x 256 bytes, the block's activation rows of the same contraction
//     range, 8-bit weights also their scales (one request of a unit where 16 rows share them, eight where not).  Eight CONSUMER waves, one per
//     row group, multiply from LDS (MFMA 16 x 16 x 32).  16-byte pieces of row r stand at slot ^ (r & 15): fragment reads are free of bank
//     conflicts.  One barrier per unit.
//   * The loaders are bound by issuing, so nothing is requested that no one reads -- neither row groups that a tile lacks nor places behind the
//     fullest block's rows: a request of 64 zeros costs what one of weights does -- and a loader's wave goes first (s_setprio: 73.5 / 44.6 us
//     for the two products of 64 tokens below, 71.8 / 42.0 with it).  The waits count what was really requested.
//   * In front of the first unit stand the launch, the lists, their order, the addresses: 5 us, half of it instructions that are met for the first
//     time.  Every loader finds the row blocks by itself, the weights of the first units are requested before any slot is known, and there is no
//     integer division on the way (with them: 1 us more for both products).
//   * An expert's contraction begins at unit e mod units and wraps: experts whose rows are a power of two long do not all ask the same
//     memory channels, and the order of a sum depends on the expert alone, not on what else rides along.
//   * Rows of 128 bytes in units twice as many: 80 / 46 us where these take 72 / 42 (memory answers half lines of 256 bytes worse).  Tiles of four
//     groups, two workgroups per CU for 8-bit weights, which this replaces: the second one of a CU came 10 us late, and a tile of one group
//     took as long as one of four.  us for both products, that -> here: 8-bit floats, 128 experts of 2048 / 768, top 8: 1 token 34 -> 29.9,
//     8 70 -> 65, 32 108 -> 102, 64 124 -> 119 (604 MB: 5.1 TB/s), 128 140 -> 136, 200 169 -> 151, 256 174 -> 155, 320 191 -> 192; bf16, 34 of
//     2048 / 704, top 4: 1 21.2 -> 21.1, 4 42 -> 33, 32 63 -> 59, 128 68 -> 62, 262 81 -> 67; 68 of 3072 / 512, top 8: 1 27.8 -> 29.1 (24 units
//     of two groups in a row: latency), 1 less since tiles of up to two groups have a ring of six instead of four, 6 69 -> 67, 32 119 -> 114, 128 133 -> 124, 262 159 -> 135.
//   Lines against the tiles (before that change; us, tiles -> streams): 8-bit floats, 128 of 2048 / 768: 1 token 42 -> 24, 64 137 -> 117, 320 181 ->
//   168, 400 186 -> 191; bf16, 34 of 2048 / 704, top 4: 1 token 33 -> 17, 128 78 -> 65, 300 (35 rows per expert) 78.5 -> 77, 400 (47) 80 -> 85; 68 of
//   3072 / 512: 262 (31) 165 -> 150: up to 36 rows per expert in ll_moe_rows_gemm.  ll_moe_gemm has other tiles and lines of its own (moe.hip).
#include <stdlib.h>

#include "gemm_w4_common.h"
#include "moe_stream.h"

namespace {

typedef __bf16 ms_bf16x8 __attribute__((ext_vector_type(8)));

constexpr int MS_LIST = 512, MS_OWN = 8;   // row blocks in all / of one workgroup
constexpr int MS_WAVES = 12;               // eight consumers, four loaders
constexpr int MS_KB = 256;                 // bytes of a weight row in a unit

template <int WF, int MT_>
struct MsLds {
  static constexpr int THREADS = MS_WAVES * 64;
  static constexpr int MT = MT_, ROWS = 16 * MT;               // rows of a piece of a block
  static constexpr int KU = WF == MS_W16 ? 128 : 256;          // contraction entries of a unit
  static constexpr int XB = KU * 2;                            // bytes of an activation row per unit
  static constexpr int X_BYTES = ROWS * XB;
  static constexpr int S_BYTES = WF == MS_W16 ? 0 : 8 * 4 * 16 * 4;   // scales: [row group][64-column step][16 rows], or, alike in 16 rows, [row group][step]
  static constexpr int slot(int groups) { return groups * 16 * MS_KB + X_BYTES + S_BYTES; }   // of the ring: three units of eight row groups, four of four, six of two
  static constexpr int ring(int groups) { return groups == 8 ? 3 : groups == 4 ? 4 : 3 * slot(8) < 6 * slot(2) ? 5 : 6; }
  static constexpr int LIST = 3 * slot(8);                  // int32 [MS_LIST]: row block | expert << 16
  static constexpr int SLOTS = LIST + MS_LIST * 4;             // int32 [MS_OWN][ROWS]
  static constexpr int FROM = SLOTS + MS_OWN * ROWS * 4;       // uint32 [MS_OWN][ROWS]: where the slot's activations begin, bytes
  static constexpr int WEIGHTS = FROM + MS_OWN * ROWS * 4;     // float [MS_OWN][ROWS]
  static constexpr int COUNTS = WEIGHTS + MS_OWN * ROWS * 4;   // int32: pieces, skipped, most rows
  static constexpr int BYTES = COUNTS + 16;                    // (nothing static: the ring begins at LDS byte 0)
  static_assert(BYTES <= 160 * 1024, "LDS");
  static constexpr int XOPS = X_BYTES / 4096;                  // activation operations per loader and unit, at most
  static_assert(ring(4) * slot(4) <= LIST && ring(2) * slot(2) <= LIST && 8 + 2 + XOPS <= 24 && 2 * (4 + 1 + XOPS) <= 24 &&
                    (ring(2) - 2) * (2 + (WF != MS_W16) + XOPS) <= 24, "the ring, the waits");
};

__device__ const uint32_t ms_zeros[4] __attribute__((aligned(16))) = {0, 0, 0, 0};   // what pieces without an entry read

// 64 lanes x 16 bytes from per-lane addresses to LDS at byte `dst`
__device__ __forceinline__ void ms_dma16(uint32_t dst, const void* src) {
  dst = __builtin_amdgcn_readfirstlane(dst);
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "s"(dst), "v"(src) : "memory");
}

__device__ __forceinline__ void ms_wait(int k) {   // at most k operations may still be in flight
#define MS_C(K) case K: v3_vmcnt<K>(); break;
  switch (k) {
    MS_C(1) MS_C(2) MS_C(3) MS_C(4) MS_C(5) MS_C(6) MS_C(7) MS_C(8) MS_C(9) MS_C(10) MS_C(11) MS_C(12) MS_C(13) MS_C(14) MS_C(15) MS_C(16) MS_C(17) MS_C(18)
    MS_C(19) MS_C(20) MS_C(21) MS_C(22) MS_C(23) MS_C(24)
    default: v3_vmcnt<0>(); break;
  }
#undef MS_C
}

// A run of row groups in tiles of at most eight groups of one row block, the last two of a segment alike.
struct MsWalk {
  int i, r0, left;   // row block and group in it of the next tile, groups of the run not yet in a tile
  __device__ __forceinline__ int open(int rgs) {   // the next tile's groups: r0 - its groups .. r0 of row block i
    if (r0 == rgs) {
      ++i;
      r0 = 0;
    }
    const int s = rgs - r0 < left ? rgs - r0 : left;
    const int h = s <= 8 ? s : s <= 16 ? (s + 1) >> 1 : 8;
    r0 += h;
    left -= h;
    return h;
  }
};

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

__device__ __forceinline__ int ms_over(int n, double inverse) {   // n / d, exactly: 0 <= n < 2^31, inverse = 1 / d, d < 2^20
  return __builtin_amdgcn_readfirstlane((int)(((double)n + 0.5) * inverse));
}

// GROUPS: the run's tiles have no more row groups than that
template <int WF, int MT, int MODE, int GROUPS>
__device__ __forceinline__ void ms_load(const MoeStreamParams& p, unsigned char* lds, int L, int lane, MsWalk run, int rgs, int i0, int units, int total) {
  using LD = MsLds<WF, MT>;
  constexpr int KU = LD::KU, EB = WF == MS_W16 ? 2 : 1, ROWS = LD::ROWS, XOPS = LD::XOPS, XL = LD::XB / 16;   // lanes of an activation row
  constexpr int RING = LD::ring(GROUPS), W_BYTES = GROUPS * 16 * MS_KB, SLOT = LD::slot(GROUPS);
  constexpr int SOPS = GROUPS == 8 ? 2 : 1;   // requests of a unit's scales, where not all 16 rows share them
  const uint32_t* list = reinterpret_cast<const uint32_t*>(lds + LD::LIST);
  const int32_t* rows = reinterpret_cast<const int32_t*>(lds + LD::FROM);
  const int row_bytes = p.K * EB;
  // ---- weights (and scales) of the next unit.  (piece `at` of row r stands at at ^ (r & 15))
  MsWalk wrun = run;
  const char *wbase = nullptr, *sbase = nullptr;   // the expert's matrix and scales
  uint32_t woff[GROUPS], soff[2] = {0, 0};                      // where this lane's pieces of unit 0 begin
  int wunit = 0, wleft = 0, groups = 0;
  uint32_t wdst = 0;
  auto weights = [&]() {
    if (wleft == 0) {
      groups = wrun.open(rgs);
      const int e = __builtin_amdgcn_readfirstlane((int)(list[wrun.i] >> 16)), r0 = wrun.r0 - groups;
      wbase = (const char*)p.w + (int64_t)e * p.w_stride_e;
#pragma unroll
      for (int j = 0; j < GROUPS; ++j) {
        const int r = 4 * L + (lane >> 4), g = r0 + j;
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
      if constexpr (WF != MS_W16) {
        sbase = (const char*)(p.scales + (int64_t)e * p.s_stride_e);
#pragma unroll
        for (int j = 0; j < SOPS; ++j) {
          int row = p.rows16 ? 16 * (r0 + (lane >> 2)) : 16 * (r0 + 4 * j + L) + (lane & 15);
          row = row < p.N ? row : p.N - 1;
          soff[j] = (uint32_t)(p.n_shift >= 0 ? row >> p.n_shift : row / (int)p.group_n) * (uint32_t)(p.s_stride_n * 4);
        }
      }
      wunit = e - ms_over(e, p.per_unit) * units;
      wleft = units;
    }
    const int at = wunit * MS_KB;
    const bool whole = at + MS_KB <= row_bytes;
    const int piece = ((lane & 15) ^ (4 * L + (lane >> 4))) * 16;
#pragma unroll
    for (int j = 0; j < GROUPS; ++j) {
      const uint32_t dst = wdst + (4 * j + L) * 1024;
      if (j >= groups) break;
      if (whole) v3_dma16<true>(dst, wbase + at, woff[j]);
      else ms_dma16(dst, at + piece < row_bytes ? wbase + at + woff[j] : (const char*)ms_zeros);   // the contraction ends inside the unit: zeros behind it, on both sides
    }
    if constexpr (WF != MS_W16) {
      int k = wunit * KU + (p.rows16 ? lane & 3 : lane >> 4) * 64;
      k = k < p.K ? k : p.K - 1;
#pragma unroll
      for (int j = 0; j < SOPS; ++j)
        if (p.rows16 ? j == 0 && L == 3 : 4 * j + L < groups) v3_dma4<false>(wdst + W_BYTES + LD::X_BYTES + (p.rows16 ? 0 : (4 * j + L) * 256), sbase, soff[j] + (uint32_t)(k >> p.k_shift) * (uint32_t)(p.s_stride_k * 4));
    }
    if (++wunit == units) wunit = 0;
    --wleft;
    wdst = wdst + SLOT == RING * SLOT ? 0 : wdst + SLOT;
  };
  // ---- its activations
  MsWalk xrun = run;
  uint32_t xoff[XOPS];
  int xunit = 0, xleft = 0, xops = 0;
  uint32_t xdst = W_BYTES;
  auto xrow = [&](int j) { return (L + 4 * j) * (64 / XL) + lane / XL; };   // (pieces stand at at ^ (r & 15))
  auto xpiece = [&](int j) { return (uint32_t)(lane % XL ^ (xrow(j) & 15)) * 16; };
  auto activations = [&]() {
    if (xleft == 0) {
      (void)xrun.open(rgs);
      const int32_t* own = rows + (xrun.i - i0) * ROWS;
#pragma unroll
      for (int j = 0; j < XOPS; ++j) {
        xoff[j] = (uint32_t)own[xrow(j)] + xpiece(j);   // (places without a slot read row 0: they feed results that are not stored)
      }
      const int e = __builtin_amdgcn_readfirstlane((int)(list[xrun.i] >> 16));
      xunit = e - ms_over(e, p.per_unit) * units;
      xleft = units;
    }
    const int xat = xunit * LD::XB;
    const bool whole = xat + LD::XB <= p.K * 2;
#pragma unroll
    for (int j = 0; j < XOPS; ++j) {
      const uint32_t dst = xdst + (L + 4 * j) * 1024;
      if (j >= xops) break;
      if (whole) v3_dma16<false>(dst, (const char*)p.a + xat, xoff[j]);
      else ms_dma16(dst, xat + (int)xpiece(j) < p.K * 2 ? (const char*)p.a + xat + xoff[j] : (const char*)ms_zeros);
    }
    if (++xunit == units) xunit = 0;
    --xleft;
    xdst = xdst + SLOT == RING * SLOT + W_BYTES ? W_BYTES : xdst + SLOT;
  };
  __builtin_amdgcn_s_setprio(3);   // (a consumer's arithmetic does not keep a request waiting)
  // the weights of the whole ring are on their way before the slots are known
  const int pre = total < RING - 1 ? total : RING - 1;
  for (int i = 0; i < pre; ++i) weights();
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // slots
  const int full = __builtin_amdgcn_readfirstlane(reinterpret_cast<const int*>(lds + LD::COUNTS)[2]);   // rows of the fullest block of the run
  xops = (full - L * (64 / XL) + 256 / XL - 1) / (256 / XL);   // this wave's requests of a unit that hold any of them
  xops = xops < 0 ? 0 : xops < XOPS ? xops : XOPS;
  for (int i = 0; i < pre; ++i) activations();
  ms_wait((pre - 1) * xops);   // (the activations of the first ring follow all its weights)
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // P0: unit 0 has landed
  int ops[RING - 2];   // requests of the last units, the latest first (of the first ring's: those behind its weights)
#pragma unroll
  for (int i = 0; i < RING - 2; ++i) ops[i] = xops;
  for (int u = 0; u < total; ++u) {
    if (u + RING - 1 < total) {   // into the slot of unit u - 1, free since the barrier that ended it
      weights();
      activations();
#pragma unroll
      for (int i = RING - 3; i > 0; --i) ops[i] = ops[i - 1];
      ops[0] = groups + xops + (WF == MS_W16 ? 0 : p.rows16 ? L == 3 : (groups > L) + (groups > 4 + L));
    }
    // unit u + 1 has landed before the consumers are released into it: behind it are the units that follow it, at most RING - 2
    int later = 0;
#pragma unroll
    for (int i = 0; i < RING - 2; ++i) later += i < total - 2 - u ? ops[i] : 0;
    ms_wait(later);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // B_u
  }
}

template <int DT, int WF, int MT, int MODE>
__global__ __launch_bounds__((MsLds<WF, MT>::THREADS)) __attribute__((amdgpu_waves_per_eu(3, 3))) void moe_stream_kernel(const MoeStreamParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  using LD = MsLds<WF, MT>;
  constexpr int KU = LD::KU, ROWS = LD::ROWS, THREADS = LD::THREADS;
  constexpr bool PAIRS = MODE == MS_GLU || MODE == MS_GLU_ROUNDED;
  uint32_t* list = reinterpret_cast<uint32_t*>(lds + LD::LIST);
  int32_t* rows = reinterpret_cast<int32_t*>(lds + LD::SLOTS);
  float* weights = reinterpret_cast<float*>(lds + LD::WEIGHTS);
  int* counts = reinterpret_cast<int*>(lds + LD::COUNTS);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int sub = p.block_m / ROWS;                       // pieces of ROWS rows per block
  const int rgs = MODE == MS_GLU ? (p.N + 7) / 8 : (p.N + 15) / 16;
  const int nout = MODE == MS_GLU_ROUNDED ? p.N / 2 : p.N;
  const int units = (p.K + KU - 1) / KU;
  const int b = (int)blockIdx.x, grid = (int)gridDim.x;
  int count = 0, skipped = 0;

  // The pieces with a slot, in order (a block's slots stand in front).  Every loader wave finds them for itself -- the same values to the same
  // places -- so that its first request waits for no barrier; lists are requested before num_post is known, as far as they exist.
  if (wv >= 8) {
    constexpr int AHEAD = 4;
    const int cap = (p.safe + ROWS - 1) / ROWS;
    int first[AHEAD], expert[AHEAD];
#pragma unroll
    for (int c = 0; c < AHEAD; ++c) {
      const int j = 64 * c + lane;
      first[c] = p.num_slots;
      expert[c] = 0;
      if (j < cap) {
        first[c] = p.sorted[j * ROWS];
        expert[c] = p.block_expert[sub == 1 ? j : j / sub];
      }
    }
    int post = p.num_post[0];
    asm volatile("" : "+v"(first[0]), "+v"(first[1]), "+v"(first[2]), "+v"(first[3]), "+v"(expert[0]), "+v"(expert[1]), "+v"(expert[2]), "+v"(expert[3]), "+s"(post));   // (requested together)
    const int pieces = post / ROWS;
    auto take = [&](int j, int slot, int e) {
      const bool has = j < pieces && slot < p.num_slots, in = has && e >= 0;
      const unsigned long long mask = __ballot(in), none = __ballot(has && e < 0), below = (1ull << lane) - 1ull;
      const int at = count + __popcll(mask & below), behind = MS_LIST - 1 - (skipped + __popcll(none & below));
      if (in && at < MS_LIST) list[at] = (uint32_t)j | (uint32_t)e << 16;
      if (has && e < 0 && behind >= 0) list[behind] = (uint32_t)j;
      count += __popcll(mask);
      skipped += __popcll(none);
    };
#pragma unroll
    for (int c = 0; c < AHEAD; ++c)
      if (64 * c < pieces) take(64 * c + lane, first[c], expert[c]);
    for (int j = 64 * AHEAD + lane; j - lane < pieces; j += 64) {
      int slot = p.num_slots, e = 0;
      if (j < pieces) {
        slot = p.sorted[j * ROWS];
        e = p.block_expert[sub == 1 ? j : j / sub];
      }
      take(j, slot, e);
    }
    counts[0] = count;
    counts[1] = skipped;
    counts[2] = 0;
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // lists
  if (wv < 8) {
    count = counts[0];
    skipped = counts[1];
  }
  count = __builtin_amdgcn_readfirstlane(count);
  skipped = __builtin_amdgcn_readfirstlane(skipped);
  // Runs to within one row group.  (Divisions by multiplication with what the host hands over: nothing is requested before this is through.)
  const int total_rg = count * rgs, each = ms_over(total_rg, p.per_workgroup), more = total_rg - each * grid;
  int lo = each * b + (b < more ? b : more), hi = lo + each + (b < more ? 1 : 0), i0, own;   // own: row blocks of this run
  const int lg = count > 1 ? 32 - __builtin_clz(count - 1) : 0, per = p.grid_log2 - lg;   // (1 << per workgroups per row block)
  if (each < 8 && count > 0 && per >= 4 && rgs <= (each + 2) << per) {
    // few blocks: runs within one, hardly longer ones -- a run across an end is two tiles, which is twice the time (one token, 4 of 40 experts of
    // 2048 / 712: 25.9 -> 21.9 us for both products; 4 tokens, 16 of 34 of 2048 / 704: 38.3 -> 33.2)
    i0 = b >> per;
    own = i0 < count ? 1 : 0;
    const int w = b & ((1 << per) - 1), part = rgs >> per, rest = rgs & ((1 << per) - 1);
    lo = i0 * rgs + part * w + (w < rest ? w : rest);
    hi = own ? lo + part + (w < rest ? 1 : 0) : lo;
    own = lo < hi ? 1 : 0;
  } else {
    i0 = ms_over(lo, p.per_block);
    own = lo < hi ? ms_over(hi - 1, p.per_block) - i0 + 1 : 0;
  }
  MsWalk run{i0, lo - i0 * rgs, hi - lo};
  const int widest = run.left <= 2 ? 2 : run.left <= 4 ? 4 : 8;   // (row groups of a tile: narrow ones in a ring of more units)
  const int slot_bytes = widest == 2 ? LD::slot(2) : widest == 4 ? LD::slot(4) : LD::slot(8), w_bytes = slot_bytes - LD::X_BYTES - LD::S_BYTES;
  const int ring = widest == 2 ? LD::ring(2) : widest == 4 ? LD::ring(4) : LD::ring(8);
  if (wv >= 8) {
    if (lo >= hi) return;   // (as a whole: the consumers behind their zeros)
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0), for the compiler: it would wait for the lists' registers between the requests
    const int head = rgs - run.r0 < run.left ? rgs - run.r0 : run.left, tail = run.left - head - (own - 2) * rgs;
    const int total = units * ((head + 7) / 8 + (own > 1 ? (own - 2) * ((rgs + 7) / 8) + (tail + 7) / 8 : 0));
    if (widest == 2) ms_load<WF, MT, MODE, 2>(p, lds, wv - 8, lane, run, rgs, i0, units, total);
    else if (widest == 4) ms_load<WF, MT, MODE, 4>(p, lds, wv - 8, lane, run, rgs, i0, units, total);
    else ms_load<WF, MT, MODE, 8>(p, lds, wv - 8, lane, run, rgs, i0, units, total);
    return;
  }

  // consumers: row group wv of every tile
  static_assert(MS_OWN * ROWS <= 512, "a thread per slot");
  int slot = p.num_slots;
  if (tid < own * ROWS) {
    slot = p.sorted[(int)(list[i0 + tid / ROWS] & 0xffffu) * ROWS + tid % ROWS];
    rows[tid] = slot;
    reinterpret_cast<uint32_t*>(lds + LD::FROM)[tid] = slot < p.num_slots ? (uint32_t)(p.a_div == 1 ? slot : slot / p.a_div) * (uint32_t)(p.a_ld * 2) : 0u;
    if (slot < p.num_slots) atomicMax(counts + 2, tid % ROWS + 1);
  }
  if (lo < hi) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // slots
  uint32_t weight_bits = 0;   // (on its way until the first unit has landed)
  if (slot < p.num_slots) {
    if (p.weight32) weight_bits = reinterpret_cast<const uint32_t*>(p.weight32)[slot];
    else if (p.weight16) weight_bits = p.weight16[slot];
  }
  if constexpr (!PAIRS) {   // slots that no expert serves: zeros (of the last product; nothing reads the first one's)
    for (int t = b; t < skipped * ROWS; t += grid) {
      const int slot = p.sorted[(int)list[MS_LIST - 1 - t / ROWS] * ROWS + t % ROWS];
      if (slot < p.num_slots)
        for (int c = tid; c < p.N; c += 512) p.out[(int64_t)slot * p.out_ld + c] = 0;
    }
  }
  if (lo >= hi) return;
  const int full = __builtin_amdgcn_readfirstlane(counts[2]);
  const int r = lane & 15, q = lane >> 4;
  f32x4 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bool wide = ((PAIRS ? 2 : 4) * 2 - 1 & (int)(reinterpret_cast<uintptr_t>(p.out) | (uintptr_t)(p.out_ld * 2))) == 0;
  uint32_t slot_at = 0;
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // P0
  if (tid < own * ROWS) weights[tid] = slot >= p.num_slots ? 1.f : p.weight32 ? __uint_as_float(weight_bits) : p.weight16 ? f16_bits_to_f32((uint16_t)weight_bits) : 1.f;
  while (run.left > 0) {
    const int groups = run.open(rgs), i = run.i, r0 = run.r0 - groups;
    const bool mine = wv < groups;
    for (int u = 0; u < units; ++u) {
      if (mine) {
        const unsigned char* wb = lds + slot_at + wv * 4096 + r * MS_KB;
        const unsigned char* xb = lds + slot_at + w_bytes + r * LD::XB;
        // (all fragments of the unit are requested before the first is used: one wave per matrix core waits for LDS once)
        if constexpr (WF == MS_W16) {
          u32x4 wf[4], x[MT][4];
#pragma unroll
          for (int s = 0; s < 4; ++s) wf[s] = *reinterpret_cast<const u32x4*>(wb + ((4 * s + q) ^ r) * 16);
#pragma unroll
          for (int m = 0; m < MT; ++m)
            if (m == 0 || 16 * m < full)
#pragma unroll
              for (int s = 0; s < 4; ++s) x[m][s] = *reinterpret_cast<const u32x4*>(xb + 16 * m * LD::XB + ((4 * s + q) ^ r) * 16);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int m = 0; m < MT; ++m)
            if (m == 0 || 16 * m < full)
#pragma unroll
              for (int s = 0; s < 4; ++s) acc[m] = ms_mfma<DT>(wf[s], x[m][s], acc[m]);
        } else {
          // a lane's 16 weights of a 64-column step feed two products; the activations' columns are taken in the same order.  The step's
          // sums are multiplied by the scales of their weight rows: a weight enters exactly.
          const float* sb = reinterpret_cast<const float*>(lds + slot_at + w_bytes + LD::X_BYTES) + wv * 64 + 4 * q;
          u32x4 raw[4], x0[MT][4], x1[MT][4];
          f32x4 sv[4], step[4];
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            raw[t] = *reinterpret_cast<const u32x4*>(wb + ((4 * t + q) ^ r) * 16);
          }
          if (p.rows16) {
            const f32x4 alike = *reinterpret_cast<const f32x4*>(lds + slot_at + w_bytes + LD::X_BYTES + wv * 16);
#pragma unroll
            for (int t = 0; t < 4; ++t) sv[t] = f32x4{alike[t], alike[t], alike[t], alike[t]};
          } else {
#pragma unroll
            for (int t = 0; t < 4; ++t) sv[t] = *reinterpret_cast<const f32x4*>(sb + t * 16);
          }
#pragma unroll
          for (int m = 0; m < MT; ++m)
            if (m == 0 || 16 * m < full)
#pragma unroll
              for (int t = 0; t < 4; ++t) {
                x0[m][t] = *reinterpret_cast<const u32x4*>(xb + 16 * m * LD::XB + ((8 * t + 2 * q) ^ r) * 16);
                x1[m][t] = *reinterpret_cast<const u32x4*>(xb + 16 * m * LD::XB + ((8 * t + 2 * q + 1) ^ r) * 16);
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
      slot_at = slot_at + slot_bytes == ring * slot_bytes ? 0 : slot_at + slot_bytes;
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
  moe_stream_kernel<DT, WF, MT, MODE><<<dim3((unsigned)grid), MsLds<WF, MT>::THREADS, bytes, stream>>>(p);
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
  p.rows16 = p.group_n % 16 == 0 || p.group_n >= p.N;
  int lds = 0;
  const int cus = ms_cus(&lds);
  p.n_shift = -1;
  for (int i = 0; i < 31; ++i)
    if (p.group_n == (1ll << i)) p.n_shift = i;
  p.per_workgroup = 1.0 / cus;
  p.per_unit = 1.0 / ((p.K * (wfmt == MS_W16 ? 2 : 1) + MS_KB - 1) / MS_KB);
  for (p.grid_log2 = 0; (2 << p.grid_log2) <= cus; ++p.grid_log2) {}
  p.per_block = 1.0 / (mode == MS_GLU ? (p.N + 7) / 8 : (p.N + 15) / 16);
  p.k_shift = 31;
  if (wfmt != MS_W16 && p.group_k < p.K)
    for (p.k_shift = 6; (1ll << p.k_shift) < p.group_k; ++p.k_shift) {}
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
