// gemm_prompt.hip: products of many rows in bfloat16 on tiles of 128 to 256 rows and 128 or 256 weight rows.
#pragma once
#include "common.h"

struct RaPromptPlan {
  int rows, cols;                // of a tile
  int ranges, range_k;           // K ranges, and the k of each (the last may have fewer)
  int rounds;                    // of workgroups
  float us;                      // what the product is expected to take
};

// Whether the kernel takes products of this shape: whole steps of 64 k, four or more, and weight rows in runs of 16.
static inline bool ra_prompt_shape(int N, int K) { return N >= 16 && N % 16 == 0 && K % 64 == 0 && K >= 256 && K <= (1 << 22); }
// The tile of the least expected time for a product in ranges of range_k (a multiple of 64) k; no ranges where the last one would
// have fewer steps than the kernel's least.
RaPromptPlan ra_prompt_plan(int M, int N, int K, int range_k);
// C = A . W^T: epilogue 0 bfloat16, 1 bfloat16 silu(gate) * up over weight rows interleaved in runs of 8, 2 C += alpha * (float),
// 3 float, with more than one range a plane [M, N] for each
int ra_prompt_product(const RaPromptPlan& plan, int epilogue, const void* A, const void* W, void* C, int M, int N, int K, int lda,
                      int ldc, float alpha, hipStream_t stream);

// Experts over pairs sorted by expert (moe_grouped.hip). plan: [0] tiles in all, from [4] on four ints a tile: expert | pairs << 16,
// the first pair, the expert's first tile, the expert's tiles. slots: pair (token * top + choice) by place in the sorted run.
struct RaExpertsPlan {
  int rows, up_cols, down_cols;  // of a tile: sorted pairs, and weight rows of the up (and gate) and the down product
  int past;                      // the weights are read once, past the caches' usual policy
};
// false: not a shape of this kernel (widths in steps of 64, operands within reach of a descriptor)
bool ra_prompt_experts_plan(int pairs, int experts, int ff, int width, int gated, long tokens, long ldx, long ld_down,
                            RaExpertsPlan* plan);
// kind 0: relu(a . w^T)^2, 1: silu(gate) * up of an expert's gate rows and its up rows behind them, both of tokens' rows and times
// the pair's weight, in bfloat16; 2: a . w^T of pairs' rows in float, an expert's K columns of w's rows side by side
int ra_prompt_experts(int rows, int cols, int kind, const void* a, long tokens, int lda, const void* w, int ldw, void* out, int N,
                      int K, const int* plan, const int* slots, const float* weights, int top, long most, int past, hipStream_t stream);
