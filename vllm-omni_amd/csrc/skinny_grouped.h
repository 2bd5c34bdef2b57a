// Grouped (per-expert) form of the decode-batch linear kernel, shared between skinny_gemm.hip (the kernel) and
// fused_moe.hip (its caller): every workgroup row (grid.y) is one tile of <= 64 token rows that all use ONE expert's
// weight matrix; rows are gathered through the MoE alignment's maps.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mi {

struct GroupedGemmArgs {
  void* out;                    // [max_rows, n_out]
  const void* a_rows;           // MI_MOE_PLAIN: rows [max_rows, k]; else x [T, k] (row = sorted_pairs[r] / top_k)
  const void* weights;          // [E, (MI_MOE_GATED ? 2 : 1) * n_out, k]
  const int32_t* sorted_pairs;  // [max_rows]: pair index or -1 (padding)
  const int32_t* tile_expert;   // [max_tiles]
  const int32_t* num_tiles;     // [1], device
  const float* pair_weights;    // MI_MOE_RELU_SQUARED: what a pair's row is multiplied by, or nullptr
  int32_t max_tiles, form, n_out, k, top_k, rows_per_tile;
  int64_t a_row_stride, out_row_stride, weight_expert_stride;
  int dtype;
};

// MI_OK, or MI_ERR_UNSUPPORTED when the shape is outside the ring kernel's envelope (the caller then runs its
// direct-from-global kernel).
int launch_grouped_skinny(const GroupedGemmArgs& a, hipStream_t s);
// Tiles of 32 or 64 rows (expert_stream.hip); MI_ERR_UNSUPPORTED outside its envelope.
int launch_grouped_stream(const GroupedGemmArgs& a, hipStream_t s);
// Tiles of 128 or 256 rows (tall_gemm.hip); MI_ERR_UNSUPPORTED outside its envelope.
int launch_grouped_tall(const GroupedGemmArgs& a, hipStream_t s);

// Experts' weight rows a multiple of 4096 bytes apart: the k blocks of 256 weight rows (128 columns of a gated form) begin with that of their number
// among all experts' and go round.  One rule for every kernel of the grouped products: their sums keep one order.
inline bool grouped_turn(int64_t k) { return k % 2048 == 0; }
__device__ __forceinline__ int grouped_first_block(bool gated, int expert, int col, int n_out, int n_it) {
  const int unit = gated ? 128 : 256;
  return (int)((uint32_t)(expert * ((n_out + unit - 1) / unit) + col / unit) % (uint32_t)n_it);
}

}  // namespace mi
