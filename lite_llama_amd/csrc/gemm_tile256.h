// Host side of the 256 x 256 tiles (gemm_tile256.hip), for the entry points that own the shape and alignment checks.
#pragma once
#include <stdint.h>

struct T2Params {
  uint16_t* out;            // fp16 [M][N] (epi 1: [M][N / 2])
  const unsigned char* x;   // fp16 or int8 [M][K], row stride x_stride BYTES, 16-byte aligned rows
  const unsigned char* w;   // int4: the packed stream; else [N][K] bytes, row stride w_stride
  const void* sp;           // int4: [K / group][N] (s, -z s) fp16 pairs
  const float* scales;      // 8-bit: block scales; int8 x int8: [N]
  const float* a_scale;     // int8 x int8: [M]
  const uint16_t* bias;     // fp16 [N] or nullptr
  int32_t* acc_out;         // int8 x int8: raw sums [M][N] or nullptr
  int64_t m, n, k, x_stride, w_stride, s_stride_n, s_stride_k, group_k;
  int group_n, chunks, gshift, epi;
  int tiles_m, tiles_n;     // (filled by the launch, like the next ones)
  int full, rest, slices, slice_steps;  // tiles that are multiplied whole, tiles behind them in `slices` parts of slice_steps steps
  void* planes;             // their sums
  // expert products (8-bit weights): blocks of 256 sorted slots of one expert, num_post of them in all (a device value)
  const int32_t *sorted_ids, *expert_ids, *num_post;
  const uint16_t* topk_w;   // weight per slot, or nullptr
  int64_t w_stride_e, s_stride_e;
  int num_slots, top_k;
};

// Whether [m, k] x [n, k]^T should take the 256 x 256 tiles; wf as the kernel's (0 int4, 1 fp8, 2 int8, 3 int8 x int8); split: the caller
// brings the ll_tile256_split_bytes() that the last round of tiles is shared through.
int tile256_wants(int64_t m, int64_t n, int64_t k, int wf, bool split = false);
int tile256_launch(T2Params& p, int wf, void* planes, int64_t plane_bytes, void* stream);
int tile256_grouped_launch(T2Params& p, int wf, void* stream);
