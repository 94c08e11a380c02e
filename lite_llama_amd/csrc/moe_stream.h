// Launch of the streaming form of the grouped expert products (moe_stream.hip): what ll_moe_gemm and ll_moe_rows_gemm hand over.
#pragma once
#include "common.h"

enum { MS_W16 = 0, MS_FP8 = 1, MS_INT8 = 2 };   // weights: in the storage type, 8-bit floats, int8 codes (the 8-bit ones with block scales)
enum {
  MS_SCALED = 0,      // out[n] = sum * slot weight
  MS_RELU2 = 1,       // out[n] = relu(sum * slot weight)^2
  MS_GLU = 2,         // gate rows, then up rows: out[j] = glu(gate_j, up_j) of the fp32 sums (limit >= 0: the clamped pair)
  MS_GLU_ROUNDED = 3  // rows are (gate_j, up_j) pairs: both sums * slot weight rounded to the storage type, then silu(g) * u
};

struct MoeStreamParams {
  uint16_t* out;
  const uint16_t* a;
  const unsigned char* w;
  const float* scales;          // 8-bit weights: one per group_n rows x group_k columns
  const float* weight32;        // slot weights, or null: 1
  const uint16_t* weight16;     // ... in fp16 bits
  const int32_t* sorted;
  const int32_t* block_expert;
  const int32_t* num_post;
  int64_t a_ld, out_ld;         // elements
  int64_t w_stride_e, w_stride_n;  // bytes
  int64_t s_stride_e, s_stride_n, s_stride_k, group_n, group_k;
  int K, N;                     // N: weight rows per expert, of MS_GLU the outputs (the expert has 2 N rows)
  int num_slots, a_div, block_m;
  int safe;                     // entries of `sorted` that exist whatever num_post says
  float limit;
  // set by the launch.  rows16: the scales of 16 rows are alike; grid_log2: 1 << that is no more than the workgroups
  int k_shift, n_shift, rows16, grid_log2;
  double per_workgroup, per_block, per_unit;   // 1 / workgroups, 1 / row groups of a block, 1 / units of a row
};

// whether the streaming form can take this call (how many rows per expert it pays for depends on the caller's other form); runs: of row blocks with the
// same expert there are no more than this many (the experts, or what is known of them)
bool moe_stream_wants(const MoeStreamParams& p, int wfmt, int mode, int dtype, int64_t experts, int64_t runs);
int moe_stream_launch(const MoeStreamParams& p, int wfmt, int mode, int dtype, int64_t experts, hipStream_t stream);
