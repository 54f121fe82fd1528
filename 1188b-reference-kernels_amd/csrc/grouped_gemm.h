// Arguments of the grouped GEMM forward kernels, shared by their sources.
#pragma once

#include "gemm_device.h"

namespace moe {

constexpr int kRowBytes = gemm::kBK * 2;  // 128: one tile row in LDS
constexpr int kChunks = gemm::kBK / 8;    // 8 chunks of 16 bytes per row

struct GemmArgs {
  const uint16_t *a;       // A rows, or the gather source x [a_src_rows, K]
  const int32_t *a_rows;   // gather: A row p = a[a_rows[p]] (nullptr: A row p = a[p])
  int64_t a_src_rows;      // gather: rows of x
  const uint16_t *w;
  const int32_t *offsets;
  uint16_t *out;
  int64_t M, K, N, G;
  int64_t ncols;   // output columns: N (NONE) or N / 2 (SWIGLU)
  int64_t ntiles;  // column tiles per expert
  int vec_out;     // output rows are 16-byte aligned (ncols % 8 == 0, aligned base)
  int *tails;      // ping-pong kernel: tail list (kTail* layout) or nullptr (tails in 256-row tiles)
  // Reduction split of the last tiles (ping-pong kernel, 0: none): the last split_tiles tiles of the
  // static order are left to grouped_gemm_split_kernel, which computes each as split_ways ranges of
  // split_steps K steps (the last range takes the rest) into fp32 planes of 256 x 256 (planes), and
  // split_sum_kernel adds each tile's planes in range order and rounds once.
  int split_tiles, split_ways, split_steps;
  float *planes;
};

__device__ __forceinline__ int swz(int row) { return (row >> 1) & (kChunks - 1); }

// The weight stream of short groups (expert_stream.hip). With p.tails it runs only if no group has more than
// 64 rows; otherwise it leaves all of them, and the tail list, to a ping-pong kernel launched after it.
void launch_expert_stream(const GemmArgs &p, bool swiglu, bool gather, hipStream_t s);

}  // namespace moe
