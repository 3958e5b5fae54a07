// gemm_tile.hip: products of 65 to 512 rows, reached through the entry points of gemm_wide.hip. epilogue: 0 plain, 1 gate over
// weight rows interleaved in runs of 8, 2 added to C.
#pragma once
#include "common.h"

extern "C" int ra_gemm_tile_takes(int epilogue, int M, int N, int K);
void ra_tile_plan(int M, int N, int K, int* ranges, int* range_k);
// planes[z][m][n] = A[m, range z] . W[n, range z]^T
int ra_tile_ranges(const void* A, int lda, const void* W, float* planes, int M, int N, int K, int ranges, int range_k,
                   hipStream_t stream);
// C[M, N / 2] = silu(gate) * up in bfloat16
int ra_tile_gated(const void* A, int lda, const void* W, void* C, int ldc, int M, int N, int K, hipStream_t stream);
