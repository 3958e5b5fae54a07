// What the two forms of the prompt attention share: heads of any size but 256 elements (attention_prefill.hip) and of 256
// (attention_prefill_wide.hip).
#pragma once
#include "common.h"
#include "reinfer_hip.h"

#define FP_KT 64          // keys per round
#define FPW_D 256         // the wide form: head size,
#define FPW_WAVES 4       // waves of a workgroup
#define FPW_NC 2          // column tiles of a wave,
// and keys up to which the other form's eight waves are ahead (the same bits). There / here, us, 16 query heads on 1 and on 8 KV heads:
// one prompt of 5 tokens 7.9 / 10.6, 7.7 / 10.4; of 64 12.7 / 13.2, 11.5 / 13.1; of 112 15.9 / 16.1, 14.7 / 14.6; of 128 17.4 / 16.1,
// 15.8 / 15.9; of 192 21.6 / 18.6, 20.2 / 18.6; a hundred of 100 tokens 99.7 / 106.9, 102.5 / 104.7
#define FPW_FEW_KEYS 112

__device__ __forceinline__ float fp_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// A listed tile may be one of several parts of a query tile, each with a range of keys (split.ranges, three
// ints a listed tile: first key, one past the last, both multiples of the round; and the part's slot, or -1
// for a tile that is whole): a part leaves its float sums (the outputs before the division, the running
// maximum and the sum of each column) in its slot, and a second kernel adds a tile's parts up. A portion
// of few queries deep in a long prompt is a handful of tiles with thousands of keys each, and a 2048-token
// prompt is one tile a CU of which the last has 32 times the keys of the first: cut by keys, the heavy
// tiles spread over the CUs that would idle.
struct FpSplit {
  const int* ranges;       // [listed tiles][3], or null: every tile is whole
  float* part_o;           // [slots][workgroups a tile][columns][DMAX]
  float* part_ml;          // [slots][workgroups a tile][columns][2]
};

// FLAGS & FP_MOD: the scores are changed before the softmax (RaScoreMod: a tanh cap, a per-head distance term); the scaled
// and changed score then replaces the product in the registers, and scale_log2 is log2(e) alone
// FLAGS & FP_KEEP: a window that keeps the first `keep` keys; the rounds that hold them and lie below the window's
// first round are walked before it.
// FLAGS & FP_CHUNK: the window is the query's own chunk of `window` keys, counted from position 0.
enum { FP_MOD = 1, FP_KEEP = 2, FP_CHUNK = 4 };

// one launch of the wide form (operands as its checked caller has them)
void ra_prefill_wide(int grid, const bf16_t* q, int q_stride, bf16_t* out, int out_stride, const bf16_t* kcache, const bf16_t* vcache,
                     const int* block_tables, int max_blocks, const int* tile_info, int block_size, int Hq, int Hkv, int hg,
                     float scale_log2, int window, int aligned, int keep, const FpSplit& sp, float scale, const RaScoreMod& mod,
                     const RaHeadOut& ho, hipStream_t stream);
