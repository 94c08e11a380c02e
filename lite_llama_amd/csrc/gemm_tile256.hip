// GEMMs over int4 / fp8 / int8 weights for MANY rows (prefill): 256 token rows x 256 weight rows per tile, one persistent workgroup
// per CU.  Semantics as the 128-row engines beside it (gemm_w4_prefill.hip, gemm_w8_prefill.hip: a8 w4a16.py:28-207,
// a9 w8a16.py:155-216, a10 w8a8.py:151-217), the same dequantised weights bit for bit and the same epilogues; fp32 / int32 sums over k in
// MFMA order.
//
//   * eight waves of 128 weight x 64 token rows (int8 x int8, which dequantises nothing: four of 128 x 128, whose fragments feed twice as many
//     products); MFMA 32x32 accumulators, weights as operand A, so a lane ends up with consecutive output columns of one token row;
//   * a weight is dequantised ONCE per 256 token rows, by the thread that fetched it, and parked as fp16 in LDS (the 128-row engines
//     dequantise it in every wave's registers, once per 128 rows);
//   * both operands sit in LDS as [256 rows][128 bytes], 16-byte slot s of row r at s ^ ((r >> 1) & 7): fragment reads and the LDS-DMA of the
//     activations (and of int8 weights under int8 activations) are bank-conflict free;
//   * double-buffered, ONE barrier per 64-k step (128 bytes of k), placed in front of the step's LAST quarter: that quarter's fragments
//     are in registers already, so behind the barrier the next step's first fragments are read and the requests of the steps ahead issued
//     under its MFMAs.  At the barrier everything requested before it has to be there;
//   * the steps of a workgroup's tiles are one sequence: the next tile's first steps are requested under this tile's last, its first weights
//     parked before the epilogue (a tile per launch slot instead spent 13 - 27 thousand cycles of 100 - 150 on its ramp and epilogue);
//   * the tiles behind the last full round of the chip are cut along the contraction, a slice per idle CU (SPLIT), and added up by a launch of
//     their own (t2_plan has the rule and what it buys);
//   * tiles are dealt to the 8 XCDs in contiguous ranges of an order that walks 8 row tiles x 4 column tiles together: the 32 CUs of an
//     XCD share 8 + 4 operand tiles through their L2, whatever the number of tiles.
// What bounds it: calls back to back on an otherwise idle card, silu(gate) * up in the epilogue.  8144 x 37888 x 3584 int4: 1.85 ms = 1.19 PFLOP/s
// (the 128-row engine 2.05; the library's fp16 GEMM of this shape, which dequantises nothing, 1.69 = 1.31 PFLOP/s).  Counters: matrix pipes
// busy 69 % of the cycles at 1.49 GHz -- the clock falls as they are kept busier (57 % at 1.73 GHz with four waves).  Without fragment reads
// and requests (MFMAs and dequantisation alone) it reaches 1.43 PFLOP/s.  int8 x int8, 5000 x 28672 x 4096: 505 us = 2.33 POP/s.  fp8
// 8192 x 5120 x 2048 (no activation): 191 us (the 128-row engine 296): 2.5 rounds of tiles.
#include <type_traits>

#include "common.h"
#include "gemm_tile256.h"
#include "gemm_w4_common.h"
#include "gemm_w8_common.h"

// WF: 0 int4 (the decode engines' packed stream), 1 fp8 e4m3, 2 int8 (fp16 activations), 3 int8 x int8.
// MF: 32-row token fragments of a wave: 4 on four waves, 2 on eight.
// GROUPED: expert products over rows sorted by expert (moe.hip: blocks of 256 slots of one expert).
// SPLIT: slices of the contraction of the tiles behind the full rounds, one per workgroup: raw sums -> planes (tile256_finish_kernel).
template <int WF, int MF, bool GROUPED, bool SPLIT>
__global__ __launch_bounds__(1024 / MF) __attribute__((amdgpu_waves_per_eu(4 / MF, 4 / MF))) void tile256_kernel(const T2Params p) {
  constexpr int NWV = 16 / MF;         // waves
  constexpr int XP = 32 / NWV;         // activation pieces per wave and step
  constexpr bool I8A = WF == 3;
  constexpr int OPND = 256 * 128;      // bytes of one operand tile of a step
  constexpr int WT = 2 * OPND;         // LDS: activations of even / odd steps, weights of even / odd steps
  constexpr int BK = I8A ? 128 : 64;   // k per step
  constexpr int NL = (WF == 0 ? 8 : 16) / NWV;  // 16-byte weight pieces per thread and step
  constexpr int NU = NL * (WF == 0 ? 4 : 2);     // 16-byte slots they are dequantised to
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nl = lane & 31, h = lane >> 5;
  int ksteps = (int)(p.k / BK), kfirst = 0;
  auto swz = [](int row, int slot) { return slot ^ ((row >> 1) & 7); };

  // ---- the workgroup's tiles: its XCD's range, every `stride`-th ----
  const int tiles_m = GROUPED ? p.num_post[0] >> 8 : p.tiles_m;
  const int tiles = GROUPED ? tiles_m * p.tiles_n : SPLIT ? p.rest * p.slices : p.full, per = (tiles + 7) >> 3;
  const int stride = (int)gridDim.x >> 3;
  int t = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
  const int tend = ((int)blockIdx.x & 7) * per + per < tiles ? ((int)blockIdx.x & 7) * per + per : tiles;
  if (t >= tend) return;
  auto tile_of = [&](int i, int& m, int& n) {
    const int gsz = 8 * p.tiles_n, g = i / gsz;
    i -= g * gsz;
    const int rows = tiles_m - 8 * g < 8 ? tiles_m - 8 * g : 8;
    n = i / rows;
    m = (8 * g + (i - n * rows)) * 256;
    n *= 256;
  };
  const int item = t;
  if constexpr (SPLIT) {   // items of one slice stand together: the CUs of an XCD read the same columns of the contraction
    const int slice = t / p.rest;
    t = p.full + t - slice * p.rest;
    kfirst = slice * p.slice_steps;
    ksteps = ksteps - kfirst < p.slice_steps ? ksteps - kfirst : p.slice_steps;
  }
  int m0, n0, m1, n1;  // first row / column of the tile that is multiplied, of the one whose steps are requested after it
  tile_of(t, m0, n0);

  // ---- loader roles ----
  // activations: 32 pieces of 8 rows x 128 B, eight per wave; lane -> (row, physical slot), the swizzle in the SOURCE address
  uint32_t xoff[XP];
  // GROUPED: row r of row block m is the slot sorted_ids[m + r] (num_slots: none), its input row slot / top_k.  A tile's slots stand in LDS
  // behind the operands, requested a tile ahead into a ring of three (a wave may still read those of the tile in front of the one another wave
  // has begun): in registers they were spilled, and read from memory where they are used they waited for the stores of the tile before.  us of
  // fused_moe with both products, in registers -> here (with the fragments' addresses formed in the loop and fewer operations per widened fp8
  // weight): fp8, 128 experts of 2048 / 768, top 8, 3000 tokens 497 -> 485, 4096 683 -> 653, 8192 1151 -> 1104; 8 of 4096 / 14336, top 2, 600 tokens
  // 878 -> 825, 4096 3478 -> 3324.  What is left per tile of 12 steps (cycles): 12 500 of epilogue, 9000 until its stores are out, 34 000 of steps.
  constexpr int ST = 4 * OPND;
  const int* slots = reinterpret_cast<const int*>(lds + ST);
  int turn = 0, turn1 = 0;  // where the slots of the tile that is multiplied begin, and those of the tile after it
  auto fetch_slots = [&](int m, int into) {
    if constexpr (GROUPED) {
      if (wv < 4) v3_dma4<false>((uint32_t)(ST + (into + wv * 64) * 4), p.sorted_ids + m, (uint32_t)(wv * 256 + lane * 4));
    }
  };
  auto aim_x = [&](int m) {
#pragma unroll
    for (int j = 0; j < XP; ++j) {
      const int r = (wv * XP + j) * 8 + (lane >> 3);
      if constexpr (GROUPED) {
        const int slot = slots[turn1 + r];
        const uint32_t row = (uint32_t)(slot < p.num_slots ? slot : p.num_slots - 1) / (uint32_t)p.top_k;  // (no slot: feeds only unstored outputs)
        xoff[j] = row * (uint32_t)p.x_stride + swz(r, lane & 7) * 16;
        continue;
      }
      const uint32_t row = m + r < (int)p.m ? m + r : (int)p.m - 1;  // rows >= M feed only unstored outputs
      xoff[j] = row * (uint32_t)p.x_stride + swz(r, lane & 7) * 16;
    }
  };
  // weights: DMA like the activations (int8 x int8), or 16-byte pieces into registers -- int4: 1-KB pieces (row group 2 wv + j, k-half
  // of the step) in stream order; 8-bit: four lanes per row's 64 bytes, piece j = 16 rows
  uint32_t woff[I8A ? XP : NL], soff[NL];
  const unsigned char* wbase = p.w;
  const char* sbase = WF == 0 ? (const char*)p.sp : (const char*)p.scales;
  auto aim_w = [&](int m, int n) {
    if constexpr (GROUPED) {
      const int64_t expert = ((const __attribute__((address_space(4))) int32_t*)p.expert_ids)[m >> 8];  // (a scalar load)
      wbase = p.w + expert * p.w_stride_e;
      sbase = (const char*)p.scales + expert * p.s_stride_e * 4;
    }
    if constexpr (WF == 0) {
      wbase = p.w + (size_t)(n / 128) * p.chunks * 8192;
      sbase = (const char*)p.sp + (size_t)n * 8;
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        const int rg = wv * NL + j;    // 32-row group of the tile
        woff[j] = (uint32_t)((rg >> 2) * p.chunks * 8192 + (rg & 3) * 1024 + lane * 16);
        soff[j] = (uint32_t)((rg * 32 + nl) * 8);
      }
    } else {
#pragma unroll
      for (int j = 0; j < (I8A ? XP : NL); ++j) {
        const int r = I8A ? (wv * XP + j) * 8 + (lane >> 3) : (wv * NL + j) * 16 + (lane >> 2);
        const uint32_t row = n + r < (int)p.n ? n + r : (int)p.n - 1;  // rows >= N feed only unstored outputs
        woff[j] = row * (uint32_t)p.w_stride + (I8A ? swz(r, lane & 7) : lane & 3) * 16;
        if constexpr (!I8A) soff[j] = (row / (uint32_t)p.group_n) * (uint32_t)p.s_stride_n * 4u;
      }
    }
  };
  // where a piece is parked: one base per 16-byte slot; a thread's pieces are 32 (16) rows apart, which leaves the swizzle alone
  constexpr int NP = WF == 0 ? 4 : 2, PSTEP = WF == 0 ? 32 * 128 : 16 * 128;
  unsigned char* pdst[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int r = WF == 0 ? wv * NL * 32 + nl : wv * NL * 16 + (lane >> 2);
    pdst[i] = lds + WT + r * 128 + swz(r, WF == 0 ? h * 4 + i : (lane & 3) * 2 + i) * 16;
  }
  uint32_t magic = 0x64006400u;
  asm volatile("" : "+v"(magic));

  struct WRegs {
    u32x4 w[NL];
    u32x2 s2[NL];
    float s1[NL];
  };
  // Steps are requested in order, one tile's behind the other's: the next tile's first steps are on their way before this tile's last
  // are multiplied.  xk / wk: steps requested of the tile that is aimed at; kin / kg: the scale block of the step requested next.
  int xk = 0, wk = 0, kin = 0;
  int64_t kg = 0;
  if constexpr (SPLIT && WF != 0 && !I8A) {
    const int64_t from = (int64_t)kfirst * 64, block = from / p.group_k;
    kin = (int)(from - block * p.group_k);
    kg = block * p.s_stride_k;
  }
  auto load_w = [&](WRegs& r) {
    if constexpr (I8A) return;
    if (wk == ksteps) {
      wk = kin = 0;
      kg = 0;
      aim_w(m1, n1);
    }
    if constexpr (WF == 0) {
      const int c = (SPLIT ? kfirst + wk : wk) >> 1, kh = wk & 1;   // (slices begin at even steps)
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        r.w[j] = *reinterpret_cast<const u32x4*>(wbase + (size_t)c * 8192 + kh * 4096 + woff[j]);
        r.s2[j] = *reinterpret_cast<const u32x2*>(sbase + (size_t)(c >> p.gshift) * (size_t)p.n * 8 + soff[j]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        r.w[j] = *reinterpret_cast<const u32x4*>(wbase + (size_t)(SPLIT ? kfirst + wk : wk) * 64 + woff[j]);
        r.s1[j] = *reinterpret_cast<const float*>(sbase + kg * 4 + soff[j]);
      }
      kin += 64;
      const bool wrap = kin >= p.group_k;
      kin = wrap ? 0 : kin;
      kg += wrap ? p.s_stride_k : 0;
    }
    ++wk;
  };
  // DMA request j (0 .. 7: activations; 8 .. 15: int8 weights under int8 activations) of a step; request 0 opens the step
  const unsigned char *xb = p.x, *wb = p.w;
  auto issue = [&](int buf, int j) {
    if (j == 0) {
      if (xk == ksteps) {
        xk = 0;
        aim_x(m1);
        if constexpr (I8A) aim_w(m1, n1);
      }
      xb = p.x + (size_t)(SPLIT ? kfirst + xk : xk) * 128;
      if constexpr (I8A) wb = p.w + (size_t)(SPLIT ? kfirst + xk : xk) * 128;
      ++xk;
    }
    if (j < XP) v3_dma16<false>((uint32_t)(buf * OPND + (wv * XP + j) * 1024), xb, xoff[j]);
    else if constexpr (I8A) v3_dma16<false>((uint32_t)(WT + buf * OPND + (wv * XP + j - XP) * 1024), wb, woff[j - XP]);
  };

  // unit u (0 .. 7) of the dequantisation of a step's weights into LDS buffer B: one 16-byte slot
  auto park = [&](const WRegs& r, auto B, int u) {
    constexpr int buf = decltype(B)::value;
    if constexpr (WF == 0) {
      const int j = u >> 2, o = u & 3;  // word o of piece j = k-octet h * 4 + o of its weight row
      *reinterpret_cast<f16x8*>(pdst[o] + buf * OPND + j * PSTEP) = v3_dequant(r.w[j][o], r.s2[j].x, r.s2[j].y, magic);
    } else if constexpr (!I8A) {
      const int q = u >> 1, i = u & 1;
      const uint32_t s = d8_bcast(WF == 1 ? r.s1[q] * 256.0f : r.s1[q]);
      u32x4 o;
      uint32_t a, b;
      if constexpr (WF == 1) d8_fp8(r.w[q][2 * i], s, a, b);
      else d8_i8(r.w[q][2 * i], s, a, b);
      o.x = a; o.y = b;
      if constexpr (WF == 1) d8_fp8(r.w[q][2 * i + 1], s, a, b);
      else d8_i8(r.w[q][2 * i + 1], s, a, b);
      o.z = a; o.w = b;
      *reinterpret_cast<u32x4*>(pdst[i] + buf * OPND + q * PSTEP) = o;
    }
  };

  // ---- consumer geometry: wave (wn, wm) multiplies weight rows wn * 128 .. by token rows wm * 128 .. ----
  constexpr int MP = 8 / MF;  // token parts
  // (waves v and v + 4 share a SIMD: eight waves give it two different token parts, so a grouped tile whose rows end in its first half keeps
  // every SIMD at half its products instead of two SIMDs at all of theirs)
  const int wn = wv / MP, wm = MF == 2 ? (wv + 2 * wn) % MP : wv % MP;
  // per MFMA step kk of a step: 16-byte slot kk * 2 + h (rows nl + a multiple of 32 share the swizzle) = where slot h stands, its bits 5 and 6
  // exchanged by kk
  uint32_t xsrc = (wm * MF * 32 + nl) * 128 + swz(nl, h) * 16, wsrc = WT + (wn * 128 + nl) * 128 + swz(nl, h) * 16;
  i32x4 xf[2][MF], wf[2][4];
  auto read_frag = [&](auto B, int kk, int set, int i) {
    constexpr int buf = decltype(B)::value;
    // in the order in which the MFMAs ask for them: the first weight fragment, the activations, the other weight fragments
    const int w = i == 0 ? 0 : i - MF, x = i - 1;
    if (i == 0 || i > MF) wf[set][w] = *reinterpret_cast<const i32x4*>(lds + (wsrc ^ (kk * 32)) + buf * OPND + w * 4096);
    else xf[set][x] = *reinterpret_cast<const i32x4*>(lds + (xsrc ^ (kk * 32)) + buf * OPND + x * 4096);
  };
  using Acc = typename std::conditional<I8A, i32x16, f32x16>::type;
  Acc acc[4][MF];
  auto mul1 = [&](int set, int i) {
        const int ni = i / MF, mi = i % MF;
        if constexpr (I8A) acc[ni][mi] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf[set][ni], xf[set][mi], acc[ni][mi], 0, 0, 0);
        else
          acc[ni][mi] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, wf[set][ni]), __builtin_bit_cast(f16x8, xf[set][mi]),
                                                             acc[ni][mi], 0, 0, 0);
  };
  using std::integral_constant;
  constexpr integral_constant<int, 0> Q0{};
  constexpr integral_constant<int, 1> Q1{};
  WRegs rA, rB;  // weights of odd / even steps ahead
  if constexpr (GROUPED) {
    fetch_slots(m0, 0);
    __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_s_barrier();
  }
  aim_x(m0);
  aim_w(m0, n0);
  m1 = m0;
  n1 = n0;
  load_w(rB);
#pragma unroll
  for (int j = 0; j < (I8A ? 2 * XP : XP); ++j) issue(0, j);
  load_w(rA);
#pragma unroll
  for (int j = 0; j < (I8A ? XP : XP / 2); ++j) issue(1, j);  // (the rest of step 1: under step 0)
#pragma unroll
  for (int u = 0; u < NU; ++u) park(rB, Q0, u);
  load_w(rB);
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0) (the builtin: the compiler knows the registers are there)
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < 4 + MF; ++i) read_frag(Q0, 0, 0, i);
  // Step ks, in sixteen groups of four MFMAs; what runs beside them is spread evenly (the four waves run in step: what one of them asks
  // for in a row, the other three ask for at the same time).  R = weights of step ks + 1, parked in groups 0 .. 10; those of step ks + 2
  // arrive at this step's barrier, those of ks + 3 replace R.
  constexpr int ND = I8A ? XP / 4 : XP / 8;  // requests per group (0: every second group one)
#define T2_DMA(buf, from)                                                                                \
  if constexpr (ND > 0) { _Pragma("unroll") for (int e = 0; e < ND; ++e) issue(buf, from + (g & 3) * ND + e); }      \
  else if (g % 2 == 0) issue(buf, from + (g & 3) / 2);
#define T2_STEP(R, cur, nxt, MULS)                                                                           \
  /* (GROUPED: the addresses of kk 1 .. 3 are formed where they are used; kept over the loop they were spilled, and every reload waited for \
     all that was requested before it) */                                                                \
  if constexpr (GROUPED) asm volatile("" : "+v"(xsrc), "+v"(wsrc));                                      \
  _Pragma("unroll") for (int g = 0; g < 16; ++g) {                                                       \
    const int q = g >> 2, set = q & 1, i0 = (g & 3) * MF;                                                \
    if (g == 12) {                                                                                       \
      __builtin_amdgcn_s_waitcnt(0x0070);                                                                \
      __builtin_amdgcn_s_barrier();                                                                      \
      __builtin_amdgcn_sched_barrier(0);                                                                 \
    }                                                                                                    \
    if (g == 15) load_w(R);                                                                              \
    if (MULS) mul1(set, i0);                                                                             \
    /* from the barrier on this step's buffer is free (its last fragments were read before it): requests of step ks + 2 -- those \
       of groups 0 .. belong to the step before: ks + 1 */                                              \
    if (g >= 12) { T2_DMA(decltype(cur)::value, 0) }                                                     \
    else if (g < 4) { T2_DMA(decltype(nxt)::value, (I8A ? XP : XP / 2)) }                                \
    constexpr int total = 4 + MF;                                                                        \
    const int fa = (g & 3) * 2 - ((g & 3) == 3 && MF == 2), fb = (g & 3) * 2 + ((g & 3) < 2 || MF == 4 ? 2 : (g & 3) == 2 ? 1 : 0); \
    _Pragma("unroll") for (int f = fa; f < fb && f < total; ++f) {                                       \
      if (q == 3) read_frag(nxt, 0, 0, f);                                                               \
      else if (MULS) read_frag(cur, q + 1, set ^ 1, f);                                                  \
    }                                                                                                    \
    if (NU == 8 && g < 12 && g % 3 != 2) park(R, nxt, g / 3 * 2 + g % 3);                                \
    if (NU == 4 && g < 12 && g % 3 == 0) park(R, nxt, g / 3);                                            \
    if (MULS) { _Pragma("unroll") for (int i = 1; i < MF; ++i) mul1(set, i0 + i); }                              \
    _Pragma("unroll") for (int i = 0; i < MF; ++i) {                                                     \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                                 \
      if (MF == 2 || i % 2 == 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                      \
      if constexpr (!I8A) __builtin_amdgcn_sched_group_barrier(0x002, (WF == 0 ? 4 : 6) * 4 / MF, 0);    \
      if (!I8A && i == MF - 1) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);                        \
    }                                                                                                    \
    __builtin_amdgcn_sched_barrier(0);                                                                   \
  }
  for (;;) {
  const bool more = !SPLIT && t + stride < tend;
  if (more) tile_of(t + stride, m1, n1);  // (else: the same tile's first steps once more, never multiplied)
  turn1 = turn == 512 ? 0 : turn + 256;
  fetch_slots(m1, turn1);
#pragma unroll
  for (int ni = 0; ni < 4; ++ni)
#pragma unroll
    for (int mi = 0; mi < MF; ++mi)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[ni][mi][e] = 0;
  int left = ksteps;
  // (an even number of steps: one exit, or the accumulators' registers do not line up)
  if (!GROUPED || __builtin_amdgcn_readfirstlane(slots[turn + wm * MF * 32]) < p.num_slots) {
    do {
      T2_STEP(rA, Q0, Q1, true)
      T2_STEP(rB, Q1, Q0, true)
      left -= 2;
    } while (left > 0);
  } else {
    do {  // none of the wave's rows has a slot (a block's slots come first): it only feeds the others
      T2_STEP(rA, Q0, Q1, false)
      T2_STEP(rB, Q1, Q0, false)
      left -= 2;
    } while (left > 0);
  }

  if constexpr (SPLIT) {   // 1 KB per wave and store: the finishing launch reads them in the same order
#pragma unroll
    for (int ni = 0; ni < 4; ++ni)
#pragma unroll
      for (int mi = 0; mi < MF; ++mi) {
        asm volatile("" : "+a"(acc[ni][mi]));
        Acc a = acc[ni][mi];
        char* to = (char*)p.planes + ((size_t)item * 64 + (wv * 4 + ni) * MF + mi) * 4096 + lane * 16;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          i32x4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if constexpr (I8A) v[e] = a[4 * g + e];
            else v[e] = (int)__float_as_uint(a[4 * g + e]);
          }
          *reinterpret_cast<i32x4*>(to + g * 1024) = v;
        }
      }
    break;
  }

  // ---- epilogue: a lane holds, for token row m = nl, the weight rows 8 g + 4 h .. + 3 of a 32-row group ----
  auto swap32 = [](uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
  };
  const bool has_bias = !GROUPED && p.bias != nullptr;
  float as[MF];
  f32x4 ws[I8A ? 4 : 1][4];
  uint2 bb[4][4];
  const int nb = n0 + wn * 128 + 4 * h;
  if constexpr (I8A) {
#pragma unroll
    for (int mi = 0; mi < MF; ++mi) {
      const int mrow = m0 + (wm * MF + mi) * 32 + nl;
      as[mi] = p.a_scale[mrow < (int)p.m ? mrow : 0];
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
      ws[i >> 2][i & 3] = *reinterpret_cast<const f32x4*>(p.scales + (nb + (i >> 2) * 32 < (int)p.n ? nb + (i >> 2) * 32 : 4 * h) + 8 * (i & 3));
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) bb[i >> 2][i & 3] = uint2{0, 0};
  if (has_bias) {
#pragma unroll
    for (int i = 0; i < 16; ++i)
      bb[i >> 2][i & 3] = *reinterpret_cast<const uint2*>(p.bias + (nb + (i >> 2) * 32 < (int)p.n ? nb + (i >> 2) * 32 : 4 * h) + 8 * (i & 3));
    // (waited for here: a load that some path leaves unused would be waited for by every step of the loop above)
    __builtin_amdgcn_s_waitcnt(0x0f70);
  }
  float rw[GROUPED ? MF : 1];
  int slot0[GROUPED ? MF : 1];
  if constexpr (GROUPED) {
#pragma unroll
    for (int mi = 0; mi < MF; ++mi) slot0[mi] = slots[turn + (wm * MF + mi) * 32 + nl];
#pragma unroll
    for (int mi = 0; mi < MF; ++mi) rw[mi] = p.topk_w ? f16_bits_to_f32(p.topk_w[slot0[mi] < p.num_slots ? slot0[mi] : 0]) : 1.f;
  }
  if constexpr (I8A || GROUPED) __builtin_amdgcn_s_waitcnt(0x0f70);
#pragma unroll
  for (int ni = 0; ni < 4; ++ni) {
    const int64_t ncol = n0 + wn * 128 + ni * 32;
    const bool col_ok = ncol < p.n;  // (n % 32 == 0: a 32-row group is in or out as a whole)
#pragma unroll
    for (int mi = 0; mi < MF; ++mi) {
      const int64_t mrow = GROUPED ? slot0[mi] : m0 + (wm * MF + mi) * 32 + nl;
      const bool row_ok = GROUPED ? mrow < p.num_slots : mrow < p.m;
      // the tile leaves the accumulation registers here and not earlier: all sixteen at once would spill everything else
      asm volatile("" : "+a"(acc[ni][mi]));
      if (!col_ok) continue;
      float v[16];
      if constexpr (I8A) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[4 * g + e] = ((float)acc[ni][mi][4 * g + e] * as[mi]) * ws[ni][g][e];  // w8a8.py:118-120
          if (p.acc_out && row_ok)
            *reinterpret_cast<i32x4*>(p.acc_out + mrow * p.n + ncol + 8 * g + 4 * h) =
                i32x4{(int)acc[ni][mi][4 * g], (int)acc[ni][mi][4 * g + 1], (int)acc[ni][mi][4 * g + 2], (int)acc[ni][mi][4 * g + 3]};
        }
      } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = acc[ni][mi][e];
      }
      if (has_bias) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          v[4 * g + 0] += f16_bits_to_f32((uint16_t)(bb[ni][g].x & 0xffffu));
          v[4 * g + 1] += f16_bits_to_f32((uint16_t)(bb[ni][g].x >> 16));
          v[4 * g + 2] += f16_bits_to_f32((uint16_t)(bb[ni][g].y & 0xffffu));
          v[4 * g + 3] += f16_bits_to_f32((uint16_t)(bb[ni][g].y >> 16));
        }
      }
      if constexpr (GROUPED) {
        if (p.topk_w) {  // router weight, in fp32 (fused_moe.py:203-205)
#pragma unroll
          for (int e = 0; e < 16; ++e) v[e] *= rw[mi];
        }
      }
      uint32_t lo[4], hi[4], sg[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        uint16_t o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float f = v[4 * g + e];
          asm volatile("" : "+v"(f));  // the fp32 value is rounded ONCE, here (never a fused multiply-convert: see w8a8_fused.hip)
          o[e] = f32_to_f16_bits(f);
        }
        lo[g] = (uint32_t)o[0] | ((uint32_t)o[1] << 16);
        hi[g] = (uint32_t)o[2] | ((uint32_t)o[3] << 16);
        if (p.epi) {  // rows are (gate_j, up_j) pairs: both rounded to fp16, then silu(g) * u in fp32 (the stand-alone kernels' arithmetic)
          const float g0 = f16_bits_to_f32(o[0]), u0 = f16_bits_to_f32(o[1]);
          const float g1 = f16_bits_to_f32(o[2]), u1 = f16_bits_to_f32(o[3]);
          sg[g] = (uint32_t)f32_to_f16_bits(ll_silu_mul_f32(g0, u0)) | ((uint32_t)f32_to_f16_bits(ll_silu_mul_f32(g1, u1)) << 16);
        }
      }
      const int64_t nn = ncol + 16 * h;
      if (p.epi) {
        swap32(sg[0], sg[2]);
        swap32(sg[1], sg[3]);
        if (row_ok) *reinterpret_cast<u32x4*>(p.out + mrow * (p.n >> 1) + (nn >> 1)) = u32x4{sg[0], sg[2], sg[1], sg[3]};
      } else {
        swap32(lo[0], lo[2]);
        swap32(hi[0], hi[2]);
        swap32(lo[1], lo[3]);
        swap32(hi[1], hi[3]);
        if (row_ok) {
          *reinterpret_cast<u32x4*>(p.out + mrow * p.n + nn) = u32x4{lo[0], hi[0], lo[2], hi[2]};
          *reinterpret_cast<u32x4*>(p.out + mrow * p.n + nn + 8) = u32x4{lo[1], hi[1], lo[3], hi[3]};
        }
      }
    }
  }
  if (!more) break;
  t += stride;
  m0 = m1;
  n0 = n1;
  turn = turn1;
  }
#undef T2_STEP
#undef T2_DMA
  __builtin_amdgcn_s_waitcnt(0x0070);  // (the requests past the last tile have landed before the LDS is given back)
}

// Sums of the slices of the tiles behind the full rounds, in slice order, through the epilogue above.  A wave per 32 x 32 results; bound by
// reading the planes (4 TB/s).
template <int WF, int MF>
__global__ __launch_bounds__(256) void tile256_finish_kernel(const T2Params p) {
  constexpr bool I8A = WF == 3;
  const int lane = threadIdx.x & 63, nl = lane & 31, h = lane >> 5;
  const int ti = (int)blockIdx.x >> 4, frag = ((int)blockIdx.x & 15) * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  constexpr int MP = 8 / MF;
  const int mi = frag % MF, ni = frag / MF & 3, wv = frag / (4 * MF);
  const int wn = wv / MP, wm = MF == 2 ? (wv + 2 * wn) % MP : wv % MP;
  int i = p.full + ti;
  const int gsz = 8 * p.tiles_n, g8 = i / gsz;
  i -= g8 * gsz;
  const int rows = p.tiles_m - 8 * g8 < 8 ? p.tiles_m - 8 * g8 : 8, tn = i / rows;
  const int64_t mrow = (int64_t)(8 * g8 + (i - tn * rows)) * 256 + (wm * MF + mi) * 32 + nl;
  const int64_t ncol = (int64_t)tn * 256 + wn * 128 + ni * 32;
  if (ncol >= p.n || mrow - nl >= p.m) return;   // (wave-uniform)
  const char* from = (const char*)p.planes + ((size_t)ti * 64 + frag) * 4096 + lane * 16;
  const size_t plane = (size_t)p.rest * 64 * 4096;
  i32x4 sum[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) sum[g] = *reinterpret_cast<const i32x4*>(from + g * 1024);
  for (int s = 1; s < p.slices; ++s) {
    from += plane;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const i32x4 v = *reinterpret_cast<const i32x4*>(from + g * 1024);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (I8A) sum[g][e] += v[e];
        else sum[g][e] = (int)__float_as_uint(__uint_as_float((uint32_t)sum[g][e]) + __uint_as_float((uint32_t)v[e]));
      }
    }
  }
  const bool row_ok = mrow < p.m;
  const float as = I8A ? p.a_scale[row_ok ? mrow : 0] : 1.f;
  uint32_t lo[4], hi[4], sg[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int64_t col = ncol + 8 * g + 4 * h;
    float v[4];
    if constexpr (I8A) {
      const f32x4 ws = *reinterpret_cast<const f32x4*>(p.scales + col);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = ((float)sum[g][e] * as) * ws[e];
      if (p.acc_out && row_ok) *reinterpret_cast<i32x4*>(p.acc_out + mrow * p.n + col) = sum[g];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = __uint_as_float((uint32_t)sum[g][e]);
    }
    if (p.bias) {
      const uint2 b = *reinterpret_cast<const uint2*>(p.bias + col);
      v[0] += f16_bits_to_f32((uint16_t)(b.x & 0xffffu));
      v[1] += f16_bits_to_f32((uint16_t)(b.x >> 16));
      v[2] += f16_bits_to_f32((uint16_t)(b.y & 0xffffu));
      v[3] += f16_bits_to_f32((uint16_t)(b.y >> 16));
    }
    uint16_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = f32_to_f16_bits(ll_pinned(v[e]));
    lo[g] = (uint32_t)o[0] | ((uint32_t)o[1] << 16);
    hi[g] = (uint32_t)o[2] | ((uint32_t)o[3] << 16);
    if (p.epi)
      sg[g] = (uint32_t)f32_to_f16_bits(ll_silu_mul_f32(f16_bits_to_f32(o[0]), f16_bits_to_f32(o[1]))) |
              ((uint32_t)f32_to_f16_bits(ll_silu_mul_f32(f16_bits_to_f32(o[2]), f16_bits_to_f32(o[3]))) << 16);
  }
  if (!row_ok) return;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int64_t col = ncol + 8 * g + 4 * h;
    if (p.epi) *reinterpret_cast<uint32_t*>(p.out + mrow * (p.n >> 1) + (col >> 1)) = sg[g];
    else *reinterpret_cast<uint2*>(p.out + mrow * p.n + col) = uint2{lo[g], hi[g]};
  }
}

// How the tiles behind the full rounds are shared: `slices` parts of the contraction each (1: not at all), of `steps` 64 (int8 x int8 128)
// columns.  A few tiles alone cost a whole contraction on idle neighbours; shared, 1 / slices of it, the sums' way to memory and back (0.1 us a
// plane) and a launch.  us, whole -> shared, int8 x int8 4096 x 14336: 16 tiles (100 rows) 114 -> 33, 64 121 -> 70, 128 128 -> 115, 272 (4280 rows)
// 291 -> 216; 4096 x 4096, 32 tiles 42 -> 29, 272 96 -> 83; fp8 2048 x 4096, 16 tiles 86 -> 32, 64 89 -> 56; int4 37888 x 3584, 296
// tiles 166 -> 142, but 888 (120 behind three rounds, halves) 366 -> 375: behind full rounds it has to promise more.
struct T2Plan {
  int full, rest, slices, steps;
  double rounds;   // what all tiles cost, in full rounds
};
static T2Plan t2_plan(int64_t m, int64_t n, int64_t k, int wf) {
  const int64_t tiles = ((m + 255) / 256) * ((n + 255) / 256);
  T2Plan r{(int)(tiles / 256 * 256), (int)(tiles % 256), 1, 0, 0.0};
  const int steps = (int)(k / (wf == 3 ? 128 : 64));
  const double step = 1.45, whole = steps * step;   // us
  double best = (r.full > 0 ? 0.8 : 0.95) * whole;
  r.rounds = (double)((tiles + 255) / 256);
  for (int s = 2; s <= 64 && s * r.rest <= 256 && r.rest > 0; ++s) {
    const int each = (steps + 2 * s - 1) / (2 * s) * 2;
    const int parts = (steps + each - 1) / each;
    if (steps - (parts - 1) * each < 8) continue;
    const double cost = each * step + 6.0 + 0.1 * r.rest * parts;
    if (cost >= best) continue;
    best = cost;
    r.slices = parts;
    r.steps = each;
    r.rounds = r.full / 256 + cost / whole;
  }
  return r;
}

extern "C" int64_t ll_tile256_split_bytes(int64_t m, int64_t n, int64_t k, int wf) {
  if (m < 1 || n < 1 || m >= (1ll << 30) || n >= (1ll << 30) || wf < 0 || wf > 3 || !tile256_wants(m, n, k, wf, true)) return 0;
  const T2Plan r = t2_plan(m, n, k, wf);
  return r.slices > 1 ? (int64_t)r.rest * r.slices * 64 * 4096 : 0;
}

// Whether the 256 x 256 tiles take [m, k] x [n, k]^T: an even number of steps, at least eight (the pipeline's reach is four), and shapes at
// which they are the faster engine.  They pay about 3 us once (a ramp of three steps, one workgroup on a CU), and the CUs that the last round
// of tiles leaves idle; the 128-row engines walk groups of 16 x 16 tiles, and pay for columns that end early in one.  us, 128-row engine ->
// here, alone on the GPU:
//   int4   past 16 column tiles: 5120 x 3584, 1024 rows 1.24x, 8192 1.55x; but one round and a sliver of a narrow grid loses (4352 x 3584, 4096
//          rows = 272 tiles 160 -> 173).  Up to 16: 144 .. 256 tiles (3584 x 3584, 4096 rows = 224 1.12x), or more where the last round's idle share
//          is below what the 128-row engine wastes on its 17th .. 32nd column (3584 columns, 10 700 rows = 2.3 rounds 1.12x, 9300 = 2.02 0.96x;
//          4096 x 3584, 7168 rows = 1.75 rounds 1.07x, 6144 = 1.5 0.95x).  Short contractions pay the ramp per tile: k 512 4352 x 2048
//          rows 0.91x, 8192 x 4096 0.86x, k 1024 4096 x 6144 0.87x, 12288 x 2048 0.91x.
//          With their last round shared (t2_plan), few tiles of a long contraction are faster here too (3584 x 18944, 28 tiles 249 -> 80 us, 112 293
//          -> 255; 3584 x 3584, 28 tiles 53 -> 36, 84 57 -> 61), and a sliver behind a full round loses nothing (4608 x 3584, 306 tiles 167 -> 151).
//   8-bit  weights under fp16: any rows past 16 column tiles (5120 x 2048 fp8, 96 rows 1.4x, 8192 1.6x); up to 16 the 128-row engine's one round
//          is as good until k or the rows outgrow it: k 2048, 256 rows 4096 columns 41.4 -> 44.9 (int8), k 3072 1.14x; k 1024, 1024 rows 1.06x (fp8).
//   int8   x int8: 4096 x 512, 65 rows 13.0 -> 16.4; k 3072 1.0x, 4096 1.05x; 256 rows k 1536 1.01x; 28672 x 4096, 5000 rows 1.15x.
int tile256_wants(int64_t m, int64_t n, int64_t k, int wf, bool split) {
  if (k % (wf == 3 ? 256 : 128) != 0 || k < 512) return 0;
  if (m >= (1ll << 30) || n >= (1ll << 30)) return 0;
  const int64_t rows = (m + 255) / 256, cols = (n + 255) / 256, tiles = rows * cols, rounds = (tiles + 255) / 256;
  const T2Plan plan = t2_plan(m, n, k, wf);
  if (wf == 0 && split && plan.slices > 1) {
    if (plan.full > 0) return cols > 16 || plan.rounds * 256 * cols * 20 <= tiles * 16 * 23;
    return plan.rounds * 1.45 * (k / 64) < (cols > 16 ? 1.2 : 0.87) * (k / 64) + 4;   // (us; the 128-row engine's one round)
  } else if (wf == 0) {
    if (cols <= 16) {
      if (tiles < 144 || (tiles > 256 && tiles < 368)) return 0;
      if (tiles > 256 && rounds * 256 * cols * 20 > tiles * 16 * 23) return 0;  // rounds / filled rounds <= 1.15 * 16 / cols
    }
    if (cols > 16 && cols < 20 && tiles > 256 && tiles < 300) return 0;
    if (k < 1024 && cols > 12 && cols < 19) return 0;
    return k >= 2048 || !(cols == 15 || cols == 16 || (cols >= 32 && tiles >= 256));
  }
  if (wf == 3 && n < 256 && k < 2048) return 0;
  if (wf == 3) return cols > 32 || k >= (m <= 128 ? 3072 : m <= 256 ? 1536 : m <= 1024 ? 768 : 512);
  if (cols > 16) {
    if (k >= 1024) return 1;
    return wf == 1 ? k >= 768 || cols < 32 || m <= 1024 : (k >= 768 && m <= 1024) || (m >= 3072 && cols > 18 && cols < 32);
  }
  int64_t least = rows == 1 ? 2560 : rows == 2 ? 2048 : rows <= 8 ? 1024 : cols <= 8 ? 512 : 1024;
  if (cols < 4 && rows <= 8) least = rows <= 2 ? 3072 : 2048;
  return k >= (wf == 2 && least > 512 && rows <= 8 ? least + 512 : least);
}

template <int WF, int MF, bool GROUPED, bool SPLIT>
static int t2_go(const T2Params& p, unsigned grid, hipStream_t st) {
  constexpr int bytes = 4 * 256 * 128 + (GROUPED ? 3 * 256 * 4 : 0);
  static bool attr[16] = {false};
  int dev = 0;
  (void)hipGetDevice(&dev);
  if (dev >= 0 && dev < 16 && !attr[dev]) {
    (void)hipFuncSetAttribute((const void*)tile256_kernel<WF, MF, GROUPED, SPLIT>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    attr[dev] = true;
  }
  tile256_kernel<WF, MF, GROUPED, SPLIT><<<dim3(grid), 1024 / MF, bytes, st>>>(p);
  return hipGetLastError() == hipSuccess ? LL_OK : LL_ERR_LAUNCH;
}

template <int WF, int MF>
static int t2_all(T2Params& p, hipStream_t st) {
  auto grid = [](int64_t tiles) { return (unsigned)((tiles + 7) / 8 < 32 ? (tiles + 7) / 8 * 8 : 256); };  // at most one workgroup per CU
  if (p.full > 0) {
    const int r = t2_go<WF, MF, false, false>(p, grid(p.full), st);
    if (r != LL_OK || p.slices <= 1) return r;
  }
  const int r = t2_go<WF, MF, false, true>(p, grid((int64_t)p.rest * p.slices), st);
  if (r != LL_OK) return r;
  tile256_finish_kernel<WF, MF><<<dim3((unsigned)p.rest * 16), 256, 0, st>>>(p);
  return hipGetLastError() == hipSuccess ? LL_OK : LL_ERR_LAUNCH;
}

int tile256_launch(T2Params& p, int wf, void* planes, int64_t plane_bytes, void* stream) {
  p.tiles_m = (int)((p.m + 255) / 256);
  p.tiles_n = (int)((p.n + 255) / 256);
  const T2Plan r = t2_plan(p.m, p.n, p.k, wf);
  p.slices = 1;
  p.full = p.tiles_m * p.tiles_n;
  if (r.slices > 1 && planes && plane_bytes >= (int64_t)r.rest * r.slices * 64 * 4096 && ll_aligned16(planes)) {
    p.full = r.full; p.rest = r.rest; p.slices = r.slices; p.slice_steps = r.steps; p.planes = planes;
  }
  hipStream_t st = (hipStream_t)stream;
  switch (wf) {
    case 0: return t2_all<0, 2>(p, st);
    case 1: return t2_all<1, 2>(p, st);
    case 2: return t2_all<2, 2>(p, st);
    default: return t2_all<3, 4>(p, st);
  }
}

int tile256_grouped_launch(T2Params& p, int wf, void* stream) {
  p.tiles_n = (int)((p.n + 255) / 256);
  hipStream_t st = (hipStream_t)stream;
  return wf == 1 ? t2_go<1, 2, true, false>(p, 256, st) : t2_go<2, 2, true, false>(p, 256, st);
}
