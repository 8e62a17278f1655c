// out = x W^T in tiles of 256 rows x 256 weight rows: the matrix products of prompts, of one matrix or grouped by expert,
// in bf16 or int8, with an activation over (gate, up) pairs of weight rows where one follows.
#pragma once

#include "common.h"

namespace hymeta {

struct TileGemmArgs {
  const char* x;                    // rows of k_bytes, x_stride bytes apart
  const char* w;                    // [experts,] N rows of k_bytes, next to each other
  uint16_t* out;                    // bf16 rows, out_stride elements apart
  const int32_t* expert_offsets;    // slots of expert e: [offsets[e], offsets[e + 1]); NULL: one matrix, rows 0 .. max_rows - 1
  const int32_t* a_rows;            // source row of slot s = a_rows[s] / a_rows_div, a_rows[s] < max_rows; or NULL: s
  const int32_t* scale_rows;        // index into row_scale per slot, or NULL: s
  const float* row_scale;           // factor of a row's sums, or NULL
  const float* x_scale;             // int8: per source row
  const float* w_scale;             // int8: per weight row, [experts,] N
  const uint16_t* bias;             // bf16 [N] of the one matrix, or NULL
  int64_t x_stride, w_stride_e, out_stride;
  int32_t a_rows_div, max_rows, N, k_bytes, expert_begin, expert_end;
  int32_t act;                      // HYMETA_GEMM_ACT_*: out has N / 2 columns, weight rows are gate rows, then up rows
  float act_limit, act_alpha;
  float* slabs;                     // slices > 1 (bf16): the sums of K's slices, [slices][max_rows][N], instead of out
  int32_t slices;
  uint32_t a_rows_inv;              // the launch's: 2^32 / a_rows_div, rounded up
};

// Whether the tiles take the problem: whole steps of 128 bytes, whole 16-byte stores, unsigned 32-bit offsets into x (whose rows do
// not run backwards) and 32-bit ones into an expert's weights, as many experts as a wave has lanes.  (Alignment of the pointers to 16 bytes is the caller's to check.)
bool tile_gemm_fits(const TileGemmArgs& a);
// Slices that K is cut into where one bf16 matrix has so few tiles that they leave the chip idle; 1: none.  At most 64 MiB of sums.
// reduced: a launch of its own adds the slices, else the consumer does while it reads them.
int tile_gemm_slices(const TileGemmArgs& a, bool reduced);
void tile_gemm_launch(const TileGemmArgs& a, bool int8, hipStream_t s);

}  // namespace hymeta
