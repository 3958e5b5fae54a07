// A mixture of experts over many tokens (bfloat16): a token's rows meet its chosen experts' matrices alone. The token-expert
// pairs are sorted by expert on the device, tiles of a sorted run of pairs go through that expert's up (and gate) projection
// with the activation and the routing weight in the epilogue, the results through its down projection into float rows, and
// a last kernel adds a token's rows in the order of its choices. Nothing of the routing reaches the host: grids are sized
// for the most tiles there can be, and workgroups without one leave.
//
// Running every expert over every token instead (two library products, experts laid side by side) executes experts / top
// times the flops at twice the rate: 1900 tokens of width 4096, 4 of 16 experts of 1536, 810 us in all against 274 here.
// The products of widths in steps of 64 run on gemm_prompt.hip's tiles (405 -> 274 us in all with weights from memory; 1859 tokens
// and gated experts of 1024 312 -> 228; 300 tokens of the first 143 -> 110), the others on the kernel below, which is bound by LDS
// (560 to 730 TFLOP/s): every product's operands are read from it by two waves each, and written from registers between two
// barriers.
#include "common.h"
#include "gemm_prompt.h"
#include "reinfer_hip.h"

namespace {

#define MOE_SORT_THREADS 1024

// plan: [0] tiles in all, then from [4] four ints a tile: expert | slots (1..tile_rows) << 16, first slot, the expert's first tile
// and its tiles.
// slots[slot] = pair (token * top + choice), place[pair] = slot, or -1 for an id past the experts (the token's row itself), or
// -2 for a pair that counts for nothing: an expert that the token names again further on weighs what it weighs there, as where
// all experts run over all tokens. distinct: no token names one twice, nobody looks (8192 tokens, 4 choices: 50 us less).
__global__ void __launch_bounds__(MOE_SORT_THREADS)
moe_sort_kernel(const int* __restrict__ ids, int pairs, int top, bool distinct, int experts, int tile_rows,
                int* __restrict__ plan, int* __restrict__ slots, int* __restrict__ place) {
  extern __shared__ int sorted[];           // [experts] counts, then cursors; [experts] first tiles
  int* count = sorted;
  int* tile0 = sorted + experts;
  for (int e = threadIdx.x; e < experts; e += MOE_SORT_THREADS) count[e] = 0;
  __syncthreads();
  for (int p = threadIdx.x; p < pairs; p += MOE_SORT_THREADS) {
    const int e = ids[p];
    bool counts = e >= 0 && e < experts;
    if (!distinct) {
      for (int x = p + 1, end = p - p % top + top; counts && x < end; ++x) counts = ids[x] != e;
      place[p] = counts ? 0 : -2;
    }
    if (counts) atomicAdd(&count[e], 1);
  }
  __syncthreads();
  if (threadIdx.x < RA_WAVE) {               // one wave: running sums over the experts, 64 at a time
    int slot = 0, tile = 0;
    for (int base = 0; base < experts; base += RA_WAVE) {
      const int e = base + (int)threadIdx.x;
      const int c = e < experts ? count[e] : 0, n = (c + tile_rows - 1) / tile_rows;
      int cs = c, ns = n;
      for (int d = 1; d < RA_WAVE; d <<= 1) {
        const int co = __shfl_up(cs, d, RA_WAVE), no = __shfl_up(ns, d, RA_WAVE);
        if ((int)threadIdx.x >= d) {
          cs += co;
          ns += no;
        }
      }
      if (e < experts) {
        const int first = slot + cs - c;
        tile0[e] = tile + ns - n;
        for (int i = 0; i < n; ++i) {
          int* t = plan + 4 + 4 * (tile0[e] + i);
          t[0] = e | (c - i * tile_rows < tile_rows ? c - i * tile_rows : tile_rows) << 16;
          t[1] = first + i * tile_rows;
          t[2] = tile0[e];
          t[3] = n;
        }
        count[e] = first;                    // from here on: the expert's next free slot
      }
      slot += __shfl(cs, RA_WAVE - 1, RA_WAVE);
      tile += __shfl(ns, RA_WAVE - 1, RA_WAVE);
    }
    if (threadIdx.x == 0) plan[0] = tile;
  }
  __syncthreads();
  // which slot of its expert's run a pair gets does not matter: its row is computed the same in each
  for (int p = threadIdx.x; p < pairs; p += MOE_SORT_THREADS) {
    const int e = ids[p];
    const bool counts = e >= 0 && e < experts && (distinct || place[p] == 0);      // place: this thread's own writes
    const int slot = counts ? atomicAdd(&count[e], 1) : e >= experts ? -1 : -2;
    place[p] = slot;
    if (slot >= 0) slots[slot] = p;
  }
}

enum { MOE_RELU2 = 0, MOE_GATED = 1, MOE_DOWN = 2 };
#define MOE_BK 64

struct GroupedArgs {
  const bf16_t* a;                           // rows: tokens (by pair / top) or, MOE_DOWN, slots
  int lda;
  const bf16_t* w;
  int ldw;                                   // elements from one weight row to the next
  int K, N;                                  // N: results a slot (features; with a gate the gated ones)
  const int *plan, *slots;
  const float* weights;                      // by pair
  int top;
  void* out;                                 // [slots, N]: bfloat16, or float for MOE_DOWN
};

// A workgroup of four waves: BM slots of one expert by BN weight rows, 64 k a step. Both tiles go through registers, asked
// for one step ahead, into one LDS buffer between two barriers; two or three workgroups a CU keep the matrix cores busy over
// each other's barriers. A row of a tile is 8 pieces of 16 bytes, piece p of row r at place p ^ (r % 8): eight rows' reads
// of one piece fall on different banks.
template <int BM, int BN, int MODE>
__global__ void __launch_bounds__(256, 2) moe_grouped_kernel(GroupedArgs g) {
  constexpr int TM = BM / 64, TN = BN / 64;  // 32 x 32 tiles of a wave: 2 x 2 waves
  constexpr int LA = BM / 32, LB = BN / 32;  // 16-byte pieces a thread stages
  constexpr int BF = MODE == MOE_GATED ? BN / 2 : BN;      // results a tile has a slot
  __shared__ __attribute__((aligned(16))) bf16_t as[BM * MOE_BK];
  __shared__ __attribute__((aligned(16))) bf16_t ws[BN * MOE_BK];
  // tiles run along the slots of a weight panel, then along panels, then experts; each XCD gets a run of them, so that what
  // neighbours share meets in its L2
  const int panels = (g.N + BF - 1) / BF;
  const int tiles = g.plan[0] * panels, each = (tiles + RA_XCDS - 1) / RA_XCDS;
  const int at = (int)blockIdx.x / RA_XCDS, tile_no = (int)blockIdx.x % RA_XCDS * each + at;
  if (at >= each || tile_no >= tiles) return;
  int expert, slot0, rows, panel;
  {
    // an expert's tiles stand side by side in the plan: its panels are walked tile by tile
    const int* t = g.plan + 4 + 4 * (tile_no / panels);
    const int first = t[2], n = t[3], within = tile_no - first * panels;
    panel = within / n;
    t = g.plan + 4 + 4 * (first + within % n);
    expert = t[0] & 0xFFFF;
    rows = t[0] >> 16;
    slot0 = t[1];
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int piece = tid & 7, srow = tid >> 3;              // staging: rows srow + 32 i
  const int n0 = panel * BF;
  const bf16_t *ap[LA], *wp[LB];
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int r = srow + 32 * i, slot = slot0 + (r < rows ? r : rows - 1);
    const int row = MODE == MOE_DOWN ? slot : g.slots[slot] / g.top;
    ap[i] = g.a + (size_t)row * g.lda + piece * 8;
  }
#pragma unroll
  for (int i = 0; i < LB; ++i) {
    const int r = srow + 32 * i;
    size_t row;
    int col = 0;
    if (MODE == MOE_GATED) {                 // runs of 32 rows: gate, up of the same features, gate, ...
      int f = n0 + (r >> 6) * 32 + (r & 31);
      f = f < g.N ? f : g.N - 1;
      row = (size_t)expert * 2 * g.N + (r >> 5 & 1) * g.N + f;
    } else {
      const int f = n0 + r < g.N ? n0 + r : g.N - 1;
      row = MODE == MOE_DOWN ? f : (size_t)expert * g.N + f;
      if (MODE == MOE_DOWN) col = expert * g.K;
    }
    wp[i] = g.w + row * g.ldw + col + piece * 8;
  }
  bf16x8_t ar[LA], wr[LB];
  auto fetch = [&](int k) {
    const bool ok = k + piece * 8 < g.K;     // K is a multiple of 8
    const int o = ok ? k : -piece * 8;
    const bf16x8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < LA; ++i) {
      ar[i] = *(const bf16x8_t*)(ap[i] + o);
      if (!ok) ar[i] = zero;
    }
#pragma unroll
    for (int i = 0; i < LB; ++i) {
      wr[i] = *(const bf16x8_t*)(wp[i] + o);
      if (!ok) wr[i] = zero;
    }
  };
  f32x16_t acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
  const int lrow = lane & 31, half = lane >> 5;
  fetch(0);
  for (int k = 0; k < g.K; k += MOE_BK) {
    const int place = (piece ^ (srow & 7)) * 8;
#pragma unroll
    for (int i = 0; i < LA; ++i) *(bf16x8_t*)(as + (srow + 32 * i) * MOE_BK + place) = ar[i];
#pragma unroll
    for (int i = 0; i < LB; ++i) *(bf16x8_t*)(ws + (srow + 32 * i) * MOE_BK + place) = wr[i];
    __syncthreads();
    if (k + MOE_BK < g.K) fetch(k + MOE_BK);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < MOE_BK / 16; ++s) {
      const int p = ((s * 2 + half) ^ (lrow & 7)) * 8;
      bf16x8_t x[TM], y[TN];
#pragma unroll
      for (int j = 0; j < TM; ++j) x[j] = *(const bf16x8_t*)(as + (wm + j * 32 + lrow) * MOE_BK + p);
#pragma unroll
      for (int i = 0; i < TN; ++i) y[i] = *(const bf16x8_t*)(ws + (wn + i * 32 + lrow) * MOE_BK + p);
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(y[i], x[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  // a lane holds slot lane % 32 of a tile, weight rows 8 (e / 4) + 4 (lane / 32) + e % 4
#pragma unroll
  for (int j = 0; j < TM; ++j) {
    const int r = wm + j * 32 + lrow;
    if (r >= rows) continue;
    const size_t slot = slot0 + r;
    const float p = MODE == MOE_DOWN ? 1.f : g.weights[g.slots[slot]];
#pragma unroll
    for (int i = 0; i < TN; i += MODE == MOE_GATED ? 2 : 1)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = n0 + (MODE == MOE_GATED ? wn / 2 + i * 16 : wn + i * 32) + q * 8 + half * 4;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float u = acc[i][j][q * 4 + e];
          if (MODE == MOE_RELU2) {
            const float z = fmaxf(u, 0.f);
            v[e] = p * (z * z);
          } else if (MODE == MOE_GATED) {
            v[e] = p * (u / (1.f + expf(-u))) * acc[(i + 1) % TN][j][q * 4 + e];
          } else {
            v[e] = u;
          }
        }
        if (MODE == MOE_DOWN) {
          float* o = (float*)g.out + slot * g.N + n;
          if (n + 3 < g.N && g.N % 4 == 0) *(f32x4_t*)o = (f32x4_t){v[0], v[1], v[2], v[3]};
          else
            for (int e = 0; e < 4; ++e)
              if (n + e < g.N) o[e] = v[e];
        } else {
          bf16_t* o = (bf16_t*)g.out + slot * g.N + n;
          if (n + 3 < g.N && g.N % 4 == 0) *(bf16x4_t*)o = (bf16x4_t){(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
          else
            for (int e = 0; e < 4; ++e)
              if (n + e < g.N) o[e] = (bf16_t)v[e];
        }
      }
  }
}

// y[t] = more[t] (times sigmoid(more_logit[t])) + the sum over choices of the pair's float row + the weights of choices that
// name no matrices, times x[t]: added times alpha into the float stream, or written in bfloat16. Four columns a thread.
// Bound by reading the pairs' rows: 7600 of 4096 in 28 us, 5.5 TB/s with the stream read and written.
__global__ void __launch_bounds__(256)
moe_sum_kernel(const float* __restrict__ rows, const int* __restrict__ place, const float* __restrict__ weights, int top,
               const bf16_t* __restrict__ x, int ldx, const float* __restrict__ more, const float* __restrict__ more_logit,
               int ld_logit, float* __restrict__ resid, bf16_t* __restrict__ out, float alpha, int width) {
  const size_t t = blockIdx.y;
  const int n = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (n >= width) return;
  f32x4_t y = {0.f, 0.f, 0.f, 0.f};
  if (more) {
    const float p = more_logit ? 1.f / (1.f + expf(-more_logit[t * ld_logit])) : 1.f;
    y = *(const f32x4_t*)(more + t * width + n);
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] *= p;
  }
  float same = 0.f;
  for (int j = 0; j < top; ++j) {
    const int s = place[t * top + j];
    if (s >= 0) y += *(const f32x4_t*)(rows + (size_t)s * width + n);
    else if (s == -1) same += weights[t * top + j];
  }
  if (same != 0.f) {
    const bf16x4_t v = *(const bf16x4_t*)(x + t * ldx + n);
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] += same * (float)v[i];
  }
  if (resid) {
    f32x4_t* r = (f32x4_t*)(resid + t * width + n);
    f32x4_t v = *r;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = fmaf(alpha, y[i], v[i]);
    *r = v;
  } else {
    *(bf16x4_t*)(out + t * width + n) = (bf16x4_t){(bf16_t)y[0], (bf16_t)y[1], (bf16_t)y[2], (bf16_t)y[3]};
  }
}

template <int BM, int BN, int MODE>
void launch(const GroupedArgs& g, long most_tiles, hipStream_t stream) {
  constexpr int BF = MODE == MOE_GATED ? BN / 2 : BN;
  const long blocks = (most_tiles * ((g.N + BF - 1) / BF) + RA_XCDS - 1) / RA_XCDS * RA_XCDS;
  moe_grouped_kernel<BM, BN, MODE><<<(unsigned)blocks, 256, 0, stream>>>(g);
}

}  // namespace

#define MOE_TILE 128

// Tiles of 128 slots that sorted pairs can make at most.
static long most_tiles(int pairs, int experts) { return pairs / MOE_TILE + (pairs < experts ? pairs : experts); }

struct GroupedScratch {
  size_t plan, slots, place, act, rows, all;
};
static GroupedScratch grouped_scratch(int n_tokens, int top, int experts, int ff, int width) {
  const size_t pairs = (size_t)n_tokens * top;
  const size_t bytes[5] = {(size_t)(4 + 4 * most_tiles((int)pairs, experts)) * 4, pairs * 4, pairs * 4, pairs * ff * 2,
                           pairs * width * 4};
  size_t at[6] = {0};
  for (int i = 0; i < 5; ++i) at[i + 1] = at[i] + (bytes[i] + 255) / 256 * 256;
  return {at[0], at[1], at[2], at[3], at[4], at[5]};
}

extern "C" long ra_moe_grouped_scratch(int n_tokens, int top, int experts, int ff, int width) {
  if (n_tokens <= 0 || top <= 0 || experts <= 0 || ff <= 0 || width <= 0) return 0;
  return (long)grouped_scratch(n_tokens, top, experts, ff, width).all;
}

extern "C" int ra_moe_grouped(const void* x, int ldx, const void* w_up, const void* w_down, int ld_down, const int* ids,
                              const float* weights, int top, int distinct, int experts, int ff, int gated, int n_tokens, int width,
                              const float* more, const float* more_logit, int ld_logit, float* resid, void* out, float alpha,
                              void* scratch, long scratch_bytes, int keep, hipStream_t stream) {
  RA_CHECK(n_tokens > 0 && top > 0 && experts > 0 && ff > 0 && width > 0, "moe_grouped: %d tokens, %d of %d experts of %d",
           n_tokens, top, experts, ff);
  RA_CHECK((long)n_tokens * top <= 1L << 24 && n_tokens <= 65535 && experts <= 4096, "moe_grouped: %d tokens, %d of %d experts",
           n_tokens, top, experts);
  RA_CHECK(width % 8 == 0 && ff % 8 == 0 && ldx >= width && ld_down >= experts * ff,
           "moe_grouped: width %d and experts of %d in steps of 8, rows of %d and %d", width, ff, ldx, ld_down);
  RA_CHECK(ra_rows_16b(x, ldx, 2) && ra_rows_16b(w_up, width, 2) && ra_rows_16b(w_down, ld_down, 2) &&
               ra_rows_16b(more, width, 4) && ra_rows_16b(resid, width, 4) && ra_rows_16b(out, width, 2),
           "moe_grouped: rows are whole 16-byte pieces");
  RA_CHECK((resid == nullptr) != (out == nullptr), "moe_grouped: the result goes into the stream or into out");
  const GroupedScratch at = grouped_scratch(n_tokens, top, experts, ff, width);
  RA_CHECK(scratch && (uintptr_t)scratch % 256 == 0 && scratch_bytes >= (long)at.all,
           "moe_grouped: scratch of %ld bytes, needs %zu", scratch_bytes, at.all);
  RaExpertsPlan tile;
  const bool tiled = ra_prompt_experts_plan(n_tokens * top, experts, ff, width, gated, n_tokens, ldx, ld_down, &tile);
  char* s = (char*)scratch;
  int *plan = (int*)(s + at.plan), *slots = (int*)(s + at.slots), *place = (int*)(s + at.place);
  const int pairs = n_tokens * top;
  moe_sort_kernel<<<1, MOE_SORT_THREADS, (size_t)experts * 8, stream>>>(ids, pairs, top, distinct != 0, experts,
                                                                        tiled ? tile.rows : MOE_TILE, plan, slots, place);
  RA_LAUNCH_CHECK("moe_grouped (sort)");
  const long most = most_tiles(pairs, experts);
  if (tiled) {
    if (int rc = ra_prompt_experts(tile.rows, tile.up_cols, gated ? 1 : 0, x, n_tokens, ldx, w_up, width, s + at.act, ff, width, plan,
                                   slots, weights, top, most, tile.past && !keep, stream))
      return rc;
    if (int rc = ra_prompt_experts(tile.rows, tile.down_cols, 2, s + at.act, pairs, ff, w_down, ld_down, s + at.rows, width, ff, plan,
                                   slots, weights, top, most, tile.past && !keep, stream))
      return rc;
  } else {
  // 256 weight rows a tile where that still leaves every CU two workgroups: half the reads of the slots' rows (gate and up
  // 1859 tokens, experts of 1024, width 4096: 171 us against 208; down 100 against 115; but up 7600 x 4096 x 1536, 384 tiles
  // of the larger kind, 157 against 144)
  const int fill = 2 * ra_cu_count();
  const GroupedArgs up = {(const bf16_t*)x, ldx, (const bf16_t*)w_up, width, width, ff, plan, slots, weights, top, s + at.act};
  if (!gated) {
    if (most * ((ff + 255) / 256) >= fill) launch<128, 256, MOE_RELU2>(up, most, stream);
    else launch<128, 128, MOE_RELU2>(up, most, stream);
  } else {
    if (most * ((ff + 127) / 128) >= fill) launch<128, 256, MOE_GATED>(up, most, stream);
    else launch<128, 128, MOE_GATED>(up, most, stream);
  }
  RA_LAUNCH_CHECK("moe_grouped (up)");
  const GroupedArgs down = {(const bf16_t*)(s + at.act), ff, (const bf16_t*)w_down, ld_down, ff, width, plan, slots, weights,
                            top, s + at.rows};
  if (most * ((width + 255) / 256) >= fill) launch<128, 256, MOE_DOWN>(down, most, stream);
  else launch<128, 128, MOE_DOWN>(down, most, stream);
  RA_LAUNCH_CHECK("moe_grouped (down)");
  }
  moe_sum_kernel<<<dim3((width / 4 + 255) / 256, n_tokens), 256, 0, stream>>>(
      (const float*)(s + at.rows), place, weights, top, (const bf16_t*)x, ldx, more, more_logit, ld_logit, resid,
      (bf16_t*)out, alpha, width);
  RA_LAUNCH_CHECK("moe_grouped (sum)");
  return 0;
}
