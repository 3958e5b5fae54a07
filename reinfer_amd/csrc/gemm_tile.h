// gemm_tile.hip: products of up to 512 rows, reached through the entry points of gemm_wide.hip. epilogue: 0 plain, 1 gate over
// weight rows interleaved in runs of 8, 2 added to C, 3 a float plane for each K range.
#pragma once
#include "common.h"

struct RaTilePlan {
  int cols;                      // features of a tile
  int ranges, range_k;           // K ranges, and the k of each (the last may have fewer)
};
// What is done with the sums (all of it optional but alpha; none of it for planes)
struct RaTileEnd {
  const float* in_ss;            // [in_parts, M] partial sums of squares of the rows behind A, whose RMSNorm the product carries (64 rows)
  int in_parts;
  float in_eps, in_inv_width;
  const bf16_t* bias;            // [N], plain and added
  float alpha;                   // added: alpha times the product
  int half;                      // plain and gated: the result is bfloat16
  bool keep;                     // the weights by the caches' usual policy
};

extern "C" int ra_gemm_tile_takes(int epilogue, int M, int N, int K);
RaTilePlan ra_tile_plan(int M, int N, int K, bool cut);
// 128 rows; with planes 512; plain and added 64
int ra_tile_product(int epilogue, const RaTilePlan& plan, const void* A, int lda, const void* W, void* C, int ldc, int M, int N, int K,
                    RaTileEnd end, hipStream_t stream);
// planes[z][m][n] = A[m, range z] . W[n, range z]^T
int ra_tile_ranges(const RaTilePlan& plan, const void* A, int lda, const void* W, float* planes, int M, int N, int K, bool keep,
                   hipStream_t stream);
