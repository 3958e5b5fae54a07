// gemm_prompt.hip: products of many rows in bfloat16 on tiles of 128 to 256 rows and 128 or 256 weight rows.
#pragma once
#include "common.h"

struct RaPromptPlan {
  int rows, cols;                // of a tile
  int ranges, range_k;           // K ranges, and the k of each (the last may have fewer)
  float us;                      // what the product is expected to take
};

// Whether the kernel takes products of this shape: whole steps of 64 k, four or more, and weight rows in runs of 16.
static inline bool ra_prompt_shape(int N, int K) { return N >= 16 && N % 16 == 0 && K % 64 == 0 && K >= 256 && K <= (1 << 22); }
// The tile and ranges (from `least` to `most`) of the least expected time, plane_us for each range's float plane among it.
RaPromptPlan ra_prompt_plan(int M, int N, int K, int least, int most, float plane_us);
// C = A . W^T: epilogue 0 bfloat16, 1 bfloat16 silu(gate) * up over weight rows interleaved in runs of 8, 2 C += alpha * (float),
// 3 float, with more than one range a plane [M, N] for each
int ra_prompt_product(const RaPromptPlan& plan, int epilogue, const void* A, const void* W, void* C, int M, int N, int K, int lda,
                      int ldc, float alpha, hipStream_t stream);
