// Products of many rows in bfloat16, C[M,N] = A[M,K] . W[N,K]^T: the projections of prompts. They are bound by the matrix cores
// (and behind those by the chip's power: on operands of zeros the same instructions run a quarter faster), so what counts is that
// the matrix cores never wait and that every CU has work until the end.
//
// A workgroup of four waves, one a SIMD with all of its registers, takes tiles of 128 to 256 rows and 128 or 256 weight rows, 64 k a
// step; a wave holds a quarter of the tile's sums. Operands go straight to LDS by loads of whole 128-byte lines, two or three steps
// ahead (as LDS allows), and from there to registers half a step ahead, so that in the middle of a step there is one barrier, with
// products of the first half still to issue behind it, and nowhere else a wait. Reads and fetches stand between the products, one
// to two products apart: a wave issues in order, and a fetch holds the issue while the CU's other waves' fetches are taken (all of
// a step's fetches in one place: 1.14 PFLOP/s at 2048 x 24576 x 4096; spread out 1.26; with the barrier moved in among the
// products, no scalar work at the seam and the sums kept in their registers 1.39, and 1.45 at 8192 x 10240 x 5120; without any
// fetches 1.65 and 1.76). Weights through registers instead of straight to LDS: 5 to 15 % slower. Loads past the caches' usual
// policy (non-temporal): 2 to 50 % slower. The workgroups stay (one a CU) and ask for the next tile's first stages before they
// write a tile's sums.
//
// The tile is chosen for the fewest part-filled rounds of workgroups, which is what the library's own product loses on: with the gate
// 3000 x 24576 x 4096 459 us against 599 with the library and the gate's kernel, 2048 x 19456 x 2560 169 against 214, 512 x 51200 x
// 5120 226 against 285; 3000 x 6144 x 4096 115 against 136, but 8192 x 6144 x 4096, whose rounds are full in any tile, 282 against 267
// (ra_gemm_prompt_takes). Weight rows of a tile are permuted (gp_row) so that a lane's sums are stored 16 bytes at a time.
#include <type_traits>
#include <utility>
#include <math.h>

#include "common.h"
#include "gemm_prompt.h"
#include "reinfer_hip.h"

namespace {

#define GP_BK 64
#define GP_LDS (160 * 1024)
#define GP_STEPS 4                 // least steps of a tile

typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));

enum { GP_PLAIN = 0, GP_GATED = 1, GP_ADD = 2, GP_FLOAT = 3, GP_MOE_RELU2 = 4, GP_MOE_GATED = 5, GP_MOE_DOWN = 6 };
// what decides where a tile's weight rows lie and how its sums are stored
__host__ __device__ constexpr int gp_form(int epi) {
  return epi == GP_MOE_RELU2 ? GP_PLAIN : epi == GP_MOE_GATED ? GP_GATED : epi == GP_MOE_DOWN ? GP_FLOAT : epi;
}

struct PromptArgs {
  const bf16_t* a;
  const bf16_t* w;
  void* c;
  int M, N, K, lda, ldw, ldc;
  float alpha;
  int m_tiles, n_tiles, band;
  int ranges, range_steps;        // GP_FLOAT: c is [ranges][M][N], a range of range_steps * 64 k in each
  // experts (gemm_prompt.h): M is the tokens, a tile one of the plan's by a panel of columns
  const int *plan, *slots;
  const float* weights;
  int top;
};

template <class F, int... I>
__device__ __forceinline__ void gp_each(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
// f(0) ... f(N - 1) with the number as a constant
template <int N, class F>
__device__ __forceinline__ void gp_for(F&& f) {
  gp_each(f, std::make_integer_sequence<int, N>{});
}

// The instructions stay in the order that they are written in: operand reads and fetches between the products.
#define GP_ORDER __builtin_amdgcn_sched_barrier(0)

// Written by hand so that a sum stays in its registers: of 64 sums that fill the accumulation registers the compiler moves
// a few to and fro in every step.
__device__ __forceinline__ void gp_mfma(f32x4_t& c, const bf16x8_t& w, const bf16x8_t& a) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(w), "v"(a));
}
// The wait states between a product and an ordinary access to its sums, which the compiler does not see in the assembly.
template <int TN, int TM>
__device__ __forceinline__ void gp_settle(f32x4_t (&acc)[TN][TM]) {
  f32x4_t* p = &acc[0][0];
#pragma unroll
  for (int i = 0; i < TN * TM; i += 4)
    asm volatile("s_nop 15\n\ts_nop 3" : "+a"(p[i]), "+a"(p[i + 1]), "+a"(p[i + 2]), "+a"(p[i + 3]));
}

// The weight row (of a wave's columns) that row r of 16-wide tile i stands for, chosen so that a lane's sums of neighbouring
// tiles are eight features side by side, one 16-byte store: plain in pairs of tiles; gated in fours, the gate and up rows of
// four features and of the next four (weight rows alternate in runs of eight).
template <int EPI>
__device__ __forceinline__ constexpr int gp_row(int i, int r) {
  if (EPI == GP_PLAIN) return (i >> 1) * 32 + (r >> 2) * 8 + (i & 1) * 4 + (r & 3);
  if (EPI == GP_GATED) return (i >> 2) * 64 + (r >> 2) * 16 + (i & 1) * 8 + ((i >> 1) & 1) * 4 + (r & 3);
  return i * 16 + r;
}
// Piece p of 16 bytes of row r lies at place p ^ key(r): the 16 rows of a tile that are read together, two to 256 bytes, then
// fall on all banks.
template <int EPI>
__device__ __forceinline__ constexpr int gp_key(int r) {
  if (EPI == GP_PLAIN) return ((r >> 1) & 1) | ((r >> 3) & 3) << 1;
  if (EPI == GP_GATED) return ((r >> 1) & 1) | ((r >> 4) & 3) << 1;
  return (r >> 1) & 7;
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t gp_rsrc(const bf16_t* p, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p), 0,
                                           (int)(bytes > 0xFFFFFF00ull ? 0xFFFFFF00u : (unsigned)bytes), 0x00020000);
}

// Operation t of OPS between MF products, L of which (evenly spread) are fetches, the rest operand reads: whether it is a
// fetch, the number among its kind, and the product that it stands behind (all of them in the first 9/10, and before the last
// seven, behind which the slots move on).
template <int MF, int OPS, int L>
struct GpOps {
  static constexpr int SPAN = MF * 9 / 10 < MF - 7 ? MF * 9 / 10 : MF - 7;
  static constexpr int fetches(int t) { return t * L / OPS; }
  static constexpr bool fetch(int t) { return fetches(t) != fetches(t + 1); }
  static constexpr int place(int t) { return t * SPAN / OPS; }
  // operations that stand behind products before m
  static constexpr int before(int m) {
    int t = 0;
    while (t < OPS && place(t) < m) ++t;
    return t;
  }
};

// STREAM: the weights past the caches' usual policy (experts of a tile each; RA_STREAM_BYTES in common.h)
template <int TM, int TN, int KIND, bool STREAM = false>
__global__ void __launch_bounds__(256, 1) gemm_prompt_kernel(PromptArgs g) {
  constexpr bool MOE = KIND >= GP_MOE_RELU2;
  constexpr int EPI = gp_form(KIND);
  constexpr int BM = 32 * TM, BN = 32 * TN, PA = TM, PB = TN;      // a wave's fetches a step: 8 rows (1 KB) each
  constexpr int SA = BM * GP_BK, SW = BN * GP_BK;                  // elements of a slot
  // Stages that the fetches run ahead, and slots: three where LDS holds them (the weights first, which come from memory), else two.
  // The rows' slot of stage s + DA is written in the first half of step s, when that of stage s - 1 is the last one free; the
  // weights' of stage s + DW in the second half, when that of stage s is.
  constexpr int DW = (3 * SA + 3 * SW) * 2 <= GP_LDS ? 3 : 2, DA = DW == 3 && (4 * SA + 3 * SW) * 2 <= GP_LDS ? 3 : 2;
  constexpr int NA = DA + 1, NW = DW;
  // fetches that may be under way when stage s + 1 has to be there, in the middle of step s
  constexpr int ROWS_AHEAD = (DA - 1) * (PA + PB), WEIGHTS_AHEAD = (DW - 1) * PA + (DW - 2) * PB;
  constexpr int UNDER_WAY = ROWS_AHEAD < WEIGHTS_AHEAD ? ROWS_AHEAD : WEIGHTS_AHEAD;
  __shared__ __attribute__((aligned(1024))) bf16_t lds[NA * SA + NW * SW];
  const int total = (MOE ? g.plan[0] : g.m_tiles) * g.n_tiles * g.ranges, each = (total + RA_XCDS - 1) / RA_XCDS;
  const int xcd = (int)blockIdx.x % RA_XCDS, stride = (int)gridDim.x / RA_XCDS;
  const int end = min(each, total - xcd * each);
  int at = (int)blockIdx.x / RA_XCDS;
  if (at >= end) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // a tile of experts: whose, the sorted pairs from `first` on, and the panel of columns; an expert's tiles run along the pairs of
  // a panel, then along panels
  int expert = 0, pairs = 0;
  auto moe_place = [&](int at, int& m0, int& n0) {
    const int tile = xcd * each + at;
    const int* t = g.plan + 4 + 4 * (tile / g.n_tiles);
    const int first = t[2], n = t[3], in = tile - first * g.n_tiles;
    t = g.plan + 4 + 4 * (first + in % n);
    expert = t[0] & 0xFFFF;
    pairs = t[0] >> 16;
    m0 = t[1];
    n0 = in / n * BN;
  };
  int m0, n0, z = 0;
  if (MOE) moe_place(at, m0, n0);
  unsigned a_off[PA], w_off[PB];
#pragma unroll
  for (int i = 0; i < PA; ++i) {
    const int r = (wave * PA + i) * 8 + (lane >> 3), p = (lane & 7) ^ ((r >> 1) & 7);
    int row = r;
    if (MOE && KIND != GP_MOE_DOWN) row = g.slots[m0 + min(r, pairs - 1)] / g.top;         // the pair's token
    a_off[i] = ((unsigned)row * (unsigned)g.lda + p * 8) * 2u;
  }
#pragma unroll
  for (int i = 0; i < PB; ++i) {
    const int r = (wave * PB + i) * 8 + (lane >> 3), p = (lane & 7) ^ gp_key<EPI>(r);
    const int row = KIND == GP_MOE_GATED ? ((r >> 3) & 1) * g.N + (r >> 4) * 8 + (r & 7) : r;  // gate rows, then all up rows
    w_off[i] = ((unsigned)row * (unsigned)g.ldw + p * 8) * 2u;
  }
  float share[TM];                          // what the pairs of this lane's sums weigh
  if (KIND == GP_MOE_RELU2 || KIND == GP_MOE_GATED) {
#pragma unroll
    for (int j = 0; j < TM; ++j) share[j] = g.weights[g.slots[m0 + min((wave >> 1) * (BM / 2) + j * 16 + (lane & 15), pairs - 1)]];
  }
  bf16_t* const la = lds + wave * PA * 8 * GP_BK;
  bf16_t* const lw = lds + NA * SA + wave * PB * 8 * GP_BK;
  auto fetch_a = [&](int i, int slot, __amdgpu_buffer_rsrc_t rs, int k) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rs, (__attribute__((address_space(3))) void*)(la + slot + i * 8 * GP_BK), 16, (int)a_off[i], k, 0, 0);
  };
  auto fetch_w = [&](int i, int slot, __amdgpu_buffer_rsrc_t rs, int k) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rs, (__attribute__((address_space(3))) void*)(lw + slot + i * 8 * GP_BK), 16, (int)w_off[i], k, 0, STREAM ? RA_STREAM : 0);
  };
  // range by range, in a range bands of `band` row tiles, inside a band column by column
  auto place = [&](int at, int& m0, int& n0, int& z) {
    int tile = xcd * each + at;
    z = 0;
    if (g.ranges > 1) {
      z = tile / (g.m_tiles * g.n_tiles);
      tile -= z * (g.m_tiles * g.n_tiles);
    }
    const int per = g.band * g.n_tiles, b = tile / per, in = tile % per;
    const int rows = min(g.band, g.m_tiles - b * g.band);
    m0 = (b * g.band + in % rows) * BM;
    n0 = in / rows * BN;
  };
  auto steps_of = [&](int z) { return min(g.range_steps, g.K / GP_BK - z * g.range_steps); };
  // from a tile's first row to the end of the matrix: rows past the end become zeros and cost no fetch
  auto a_of = [&](int m0) {
    if (KIND == GP_MOE_DOWN) return gp_rsrc(g.a + (size_t)m0 * g.lda, ((size_t)(pairs - 1) * g.lda + g.K) * 2);
    if (MOE) return gp_rsrc(g.a, ((size_t)(g.M - 1) * g.lda + g.K) * 2);
    return gp_rsrc(g.a + (size_t)m0 * g.lda, ((size_t)(g.M - 1 - m0) * g.lda + g.K) * 2);
  };
  auto w_of = [&](int n0) {
    if (KIND == GP_MOE_DOWN) return gp_rsrc(g.w + (size_t)n0 * g.ldw + (size_t)expert * g.K, ((size_t)(g.N - 1 - n0) * g.ldw + g.K) * 2);
    if (KIND == GP_MOE_GATED) return gp_rsrc(g.w + ((size_t)expert * 2 * g.N + n0 / 2) * g.ldw, (size_t)(2 * g.N - n0 / 2) * g.ldw * 2);
    if (MOE) return gp_rsrc(g.w + ((size_t)expert * g.N + n0) * g.ldw, (size_t)(g.N - n0) * g.ldw * 2);
    return gp_rsrc(g.w + (size_t)n0 * g.ldw, (size_t)(g.N - n0) * g.ldw * 2);
  };
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
  const int lr = lane & 15, lc = lane >> 4;
  const int ax0 = (lc ^ (lr >> 1)) * 8, ax1 = ((4 + lc) ^ (lr >> 1)) * 8;
  const int key = gp_key<EPI>(gp_row<EPI>(0, lr));       // the same in every tile
  const int wx0 = (lc ^ key) * 8, wx1 = ((4 + lc) ^ key) * 8;
  const bf16_t* const ab = lds + (wm + lr) * GP_BK;
  const bf16_t* const wb = lds + NA * SA + (wn + gp_row<EPI>(0, lr)) * GP_BK;
  bf16x8_t x0[TM], y0[TN], x1[TM], y1[TN];
  if (!MOE) place(at, m0, n0, z);
  __amdgpu_buffer_rsrc_t ar = a_of(m0), wr = w_of(n0);
  // where along K (bytes) the next stage of rows and of weights lies
  int ka = z * g.range_steps * GP_BK * 2, kw = ka, a_step = GP_BK * 2, w_step = GP_BK * 2;
#pragma unroll
  for (int s = 0; s < DW; ++s) {            // in the order of their steps: rows first
    if (s < DA) {
#pragma unroll
      for (int i = 0; i < PA; ++i) fetch_a(i, s * SA, ar, ka);
      ka += a_step;
    }
#pragma unroll
    for (int i = 0; i < PB; ++i) fetch_w(i, s * SW, wr, kw);
    kw += w_step;
  }
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((DA - 1) * PA + (DW - 1) * PB) : "memory");
#pragma unroll
  for (int i = 0; i < TN; ++i) y0[i] = *(const bf16x8_t*)(wb + gp_row<EPI>(i, 0) * GP_BK + wx0);
#pragma unroll
  for (int j = 0; j < TM; ++j) x0[j] = *(const bf16x8_t*)(ab + j * 16 * GP_BK + ax0);
  // the slots (elements) of stage s and of those behind it, the last one the next to be written, and the next reads
  int as[NA], ws[NW];
#pragma unroll
  for (int i = 0; i < NA; ++i) as[i] = i * SA;
#pragma unroll
  for (int i = 0; i < NW; ++i) ws[i] = i * SW;
  const bf16_t *ra1 = ab + ax1, *rw1 = wb + wx1, *ra0 = ab + SA + ax0, *rw0 = wb + SW + wx0;
  while (true) {
    f32x4_t acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    gp_settle(acc);
    const int next = MOE ? end : at + stride;      // experts: a tile a workgroup
    int next_m = 0, next_n = 0, next_z = 0;
    if (next < end) place(next, next_m, next_n, next_z);
    const int steps = steps_of(z);       // GP_STEPS or more, so that fetches are one tile ahead at most
    for (int s = 0; s < steps; ++s) {
      // the first 32 k's products, the second 32 k's operand reads; the last row of products is left for behind the barrier
      {
        constexpr int MF = TM * (TN - 1);
        using Ops = GpOps<MF, TM + TN + PA, PA>;
        gp_for<MF>([&](auto mc) {
          constexpr int m = mc, t0 = Ops::before(m);
          gp_mfma(acc[m / TM][m % TM], y0[m / TM], x0[m % TM]);
          GP_ORDER;
          gp_for<Ops::before(m + 1) - t0>([&](auto tc) {
            constexpr int t = t0 + tc, f = Ops::fetches(t), r = t - f;
            if constexpr (Ops::fetch(t)) fetch_a(f, as[DA], ar, ka);
            else if constexpr (r < TN) y1[r] = *(const bf16x8_t*)(rw1 + gp_row<EPI>(r, 0) * GP_BK);
            else x1[r - TN] = *(const bf16x8_t*)(ra1 + (r - TN) * 16 * GP_BK);
            GP_ORDER;
          });
        });
      }
      // This wave's reads of stage s are done, and of its fetches all but those of the rows of stage s + 2; the barrier makes
      // that true of all waves: stage s + 1 is there, and the weights' slot of stage s may be written.
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(UNDER_WAY) : "memory");
      GP_ORDER;
      {
        constexpr int MF = TM * (TN + 1);
        using Ops = GpOps<MF, TM + TN + PB, PB>;
        // the last weights and all rows are in use until the first TM products are out: with reads at their places the last
        // row's operands are the TN-th read, and the first products behind the barrier come before it
        gp_for<MF>([&](auto mc) {
          constexpr int m = mc, t0 = Ops::before(m);
          if constexpr (m < TM) gp_mfma(acc[TN - 1][m], y0[TN - 1], x0[m]);
          else gp_mfma(acc[m / TM - 1][m % TM], y1[m / TM - 1], x1[m % TM]);
          GP_ORDER;
          gp_for<Ops::before(m + 1) - t0>([&](auto tc) {
            constexpr int t = t0 + tc, f = Ops::fetches(t), r = t - f;
            static_assert(Ops::fetch(t) || r < TN - 1 || m >= TM - 1, "a read of a register that a product behind it needs");
            if constexpr (Ops::fetch(t)) fetch_w(f, ws[0], wr, kw);
            else if constexpr (r < TN) y0[r] = *(const bf16x8_t*)(rw0 + gp_row<EPI>(r, 0) * GP_BK);
            else x0[r - TN] = *(const bf16x8_t*)(ra0 + (r - TN) * 16 * GP_BK);
            GP_ORDER;
          });
          if constexpr (m == MF - 6) {         // the slots move on by one stage
            const int ta = as[0], tw = ws[0];
#pragma unroll
            for (int i = 0; i + 1 < NA; ++i) as[i] = as[i + 1];
#pragma unroll
            for (int i = 0; i + 1 < NW; ++i) ws[i] = ws[i + 1];
            as[NA - 1] = ta;
            ws[NW - 1] = tw;
            ka += a_step;
            kw += w_step;
            GP_ORDER;
          }
          if constexpr (m == MF - 5) { ra1 = ab + as[0] + ax1; GP_ORDER; }
          if constexpr (m == MF - 4) { rw1 = wb + ws[0] + wx1; GP_ORDER; }
          if constexpr (m == MF - 3) { ra0 = ab + as[1] + ax0; GP_ORDER; }
          if constexpr (m == MF - 2) { rw0 = wb + ws[1] + wx0; GP_ORDER; }
        });
      }
      // from its last stage on the next tile's are asked for; behind the last tile nothing (and the place along K stays 0)
      if (s + 1 + DA == steps) {
        ar = next < end ? a_of(next_m) : gp_rsrc(g.a, 0);
        ka = next_z * g.range_steps * GP_BK * 2;
        if (next >= end) a_step = 0;
      }
      if (s + 1 + DW == steps) {
        wr = next < end ? w_of(next_n) : gp_rsrc(g.w, 0);
        kw = next_z * g.range_steps * GP_BK * 2;
        if (next >= end) w_step = 0;
      }
    }
    gp_settle(acc);
    GP_ORDER;
    // A lane holds row lane % 16 of a tile, weight rows gp_row(i, 4 (lane / 16) + e). What lies past the last row or column is past
    // the descriptor, which spans the result from the tile's first value on.
    constexpr int SIZE = EPI == GP_PLAIN || EPI == GP_GATED ? 2 : 4;
    const int cols = KIND == GP_GATED ? g.N / 2 : g.N, c0 = EPI == GP_GATED ? n0 / 2 : n0;
    const int left = MOE ? pairs : min(g.M - m0, BM);
    const __amdgpu_buffer_rsrc_t cr = __builtin_amdgcn_make_buffer_rsrc(
        (char*)g.c + (((size_t)(EPI == GP_FLOAT ? z : 0) * g.M + m0) * g.ldc + c0) * SIZE, 0,
        (int)(((unsigned)(left - 1) * (unsigned)g.ldc + (cols - c0)) * SIZE), 0x00020000);
    const unsigned row0 = (unsigned)(wm + lr) * (unsigned)g.ldc * SIZE, row_step = 16u * (unsigned)g.ldc * SIZE;
    // where the value in column n (from the tile's first) of row tile j lies
    auto spot = [&](int j, int n) { return (int)(c0 + n < cols ? row0 + j * row_step + n * SIZE : 0xFFFFFFF0u); };
    if constexpr (EPI == GP_ADD) {
      // half a row of tiles at a time; as many of the stream's old values as there are registers for are asked for ahead (the
      // next half alone: 1733 x 4096 x 4096 62.4 us, so 58.6)
      constexpr int H = TN / 2, AHEAD = (TM * TN <= 32 ? 32 : TM * TN < 64 ? 16 : 8) / H;
      f32x4_t old[AHEAD][H];
      auto ask = [&](int u) {
#pragma unroll
        for (int i = 0; i < H; ++i)
          old[u % AHEAD][i] = __builtin_bit_cast(
              f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(cr, spot(u >> 1, wn + ((u & 1) * H + i) * 16 + lc * 4), 0, 0));
      };
#pragma unroll
      for (int u = 0; u < AHEAD && u < 2 * TM; ++u) ask(u);
#pragma unroll
      for (int u = 0; u < 2 * TM; ++u) {
        GP_ORDER;
#pragma unroll
        for (int i = 0; i < H; ++i) {
          f32x4_t v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = fmaf(g.alpha, acc[(u & 1) * H + i][u >> 1][e], old[u % AHEAD][i][e]);
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), cr,
                                                 spot(u >> 1, wn + ((u & 1) * H + i) * 16 + lc * 4), 0, 0);
        }
        if (u + AHEAD < 2 * TM) ask(u + AHEAD);
      }
    } else {
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        if (EPI == GP_GATED) {
#pragma unroll
          for (int i = 0; i < TN; i += 4) {
            bf16x8_t o;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const float u = acc[i + (e >> 2) * 2][j][e & 3];
              const float gate = u / (1.f + expf(-u));
              o[e] = (bf16_t)((MOE ? share[j] * gate : gate) * acc[i + (e >> 2) * 2 + 1][j][e & 3]);
            }
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, o), cr,
                                                   spot(j, wn / 2 + (i >> 2) * 32 + lc * 8), 0, 0);
          }
        } else if (EPI == GP_PLAIN) {
#pragma unroll
          for (int i = 0; i < TN; i += 2) {
            bf16x8_t o;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const float u = acc[i + (e >> 2)][j][e & 3], r = fmaxf(u, 0.f);
              o[e] = (bf16_t)(MOE ? share[j] * (r * r) : u);
            }
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, o), cr,
                                                   spot(j, wn + (i >> 1) * 32 + lc * 8), 0, 0);
          }
        } else {
#pragma unroll
          for (int i = 0; i < TN; ++i)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, acc[i][j]), cr, spot(j, wn + i * 16 + lc * 4), 0, 0);
        }
        GP_ORDER;
      }
    }
    if (next >= end) break;
    at = next; m0 = next_m; n0 = next_n; z = next_z;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

template <int TM, int TN, int EPI>
int prompt_launch(PromptArgs g, hipStream_t stream) {
  g.m_tiles = (g.M + 32 * TM - 1) / (32 * TM);
  g.n_tiles = (g.N + 32 * TN - 1) / (32 * TN);
  const long total = (long)g.m_tiles * g.n_tiles * g.ranges, blocks = (total + RA_XCDS - 1) / RA_XCDS * RA_XCDS;
  const long room = ra_cu_count() / RA_XCDS * RA_XCDS;
  g.band = TM >= 2 * TN ? 4 : 8;
  gemm_prompt_kernel<TM, TN, EPI><<<(unsigned)(blocks < room ? blocks : room), 256, 0, stream>>>(g);
  RA_LAUNCH_CHECK("gemm_prompt");
  return 0;
}

template <int TM, int TN, bool STREAM>
int prompt_experts(PromptArgs g, int kind, long most, hipStream_t stream) {
  const int rows = kind == GP_MOE_GATED ? 2 * g.N : g.N;        // weight rows of an expert
  g.n_tiles = (rows + 32 * TN - 1) / (32 * TN);
  const unsigned blocks = (unsigned)((most * g.n_tiles + RA_XCDS - 1) / RA_XCDS * RA_XCDS);
  if (kind == GP_MOE_RELU2) gemm_prompt_kernel<TM, TN, GP_MOE_RELU2, STREAM><<<blocks, 256, 0, stream>>>(g);
  else if (kind == GP_MOE_GATED) gemm_prompt_kernel<TM, TN, GP_MOE_GATED, STREAM><<<blocks, 256, 0, stream>>>(g);
  else gemm_prompt_kernel<TM, TN, GP_MOE_DOWN, STREAM><<<blocks, 256, 0, stream>>>(g);
  RA_LAUNCH_CHECK("gemm_prompt (experts)");
  return 0;
}

template <int TM, int TN>
int prompt_epilogue(const PromptArgs& g, int epilogue, hipStream_t stream) {
  switch (epilogue) {
    case GP_PLAIN: return prompt_launch<TM, TN, GP_PLAIN>(g, stream);
    case GP_GATED: return prompt_launch<TM, TN, GP_GATED>(g, stream);
    case GP_ADD: return prompt_launch<TM, TN, GP_ADD>(g, stream);
    default: return prompt_launch<TM, TN, GP_FLOAT>(g, stream);
  }
}

}  // namespace

// What a tile of `rows` x `cols` costs, measured on MI355X over products of 128 to 3000 rows (4096 to 25600 k, one to eight
// ranges; the tile so chosen is within 4 % of the fastest at each of 23 shapes): a start, then for each round of workgroups an
// end that grows with the tile and the steps, each a part of its own (barrier, first operands) and one that grows with the tile,
// the more the fuller the chip is (power and fetches). It ranks tiles; beside the library's times it is corrected (below), as many
// full rounds take a tenth longer. Ten prices, 0.1 us of the host.
RaPromptPlan ra_prompt_plan(int M, int N, int K, int range_k) {
  static const int sides[10][2] = {{256, 256}, {224, 256}, {192, 256}, {160, 256}, {128, 256},
                                   {256, 128}, {224, 128}, {192, 128}, {160, 128}, {128, 128}};
  RaPromptPlan best = {0, 0, 0, 0, 0, 1e30f};
  const int slots = ra_cu_count() / RA_XCDS, steps = K / GP_BK, each = range_k / GP_BK, ranges = (steps + each - 1) / each;
  if (steps - (ranges - 1) * each < GP_STEPS) return best;
  for (const auto& side : sides) {
    const long tiles = (long)((M + side[0] - 1) / side[0]) * ((N + side[1] - 1) / side[1]) * ranges;
    const long rounds = ((tiles + RA_XCDS - 1) / RA_XCDS + slots - 1) / slots;
    const float fill = (float)tiles / (float)(rounds * slots * RA_XCDS), area = (float)side[0] * side[1] / 65536.f;
    const float us = 6.f + rounds * (11.2f * area + each * (0.227f + 0.623f * area + fill * (0.027f + 0.282f * area)));
    if (us < best.us) best = {side[0], side[1], ranges, range_k, (int)rounds, us};
  }
  return best;
}

int ra_prompt_product(const RaPromptPlan& plan, int epilogue, const void* A, const void* W, void* C, int M, int N, int K, int lda,
                      int ldc, float alpha, hipStream_t stream) {
  RA_CHECK(M > 0 && ra_prompt_shape(N, K) && lda % 8 == 0 && lda >= K && lda <= (1 << 22) && (uintptr_t)A % 16 == 0 &&
               (uintptr_t)W % 16 == 0 && (uintptr_t)C % 16 == 0 && ldc % 8 == 0 && ldc <= (1 << 21) &&
               ldc >= (epilogue == GP_GATED ? N / 2 : N),
           "gemm_prompt: [%d, %d, %d] with rows of strides %d and %d", M, N, K, lda, ldc);
  const int range_steps = plan.range_k / GP_BK;
  RA_CHECK(plan.ranges >= 1 && plan.range_k % GP_BK == 0 && (long)(plan.ranges - 1) * range_steps + GP_STEPS <= K / GP_BK &&
               (long)plan.ranges * plan.range_k >= K && (plan.ranges == 1 || (epilogue == GP_FLOAT && ldc == N)),
           "gemm_prompt: %d ranges of %d k for %d", plan.ranges, plan.range_k, K);
  PromptArgs g = {(const bf16_t*)A, (const bf16_t*)W, C, M, N, K, lda, K, ldc, alpha, 0, 0, 0, plan.ranges, range_steps};
  switch (plan.rows * 1000 + plan.cols) {
    case 256256: return prompt_epilogue<8, 8>(g, epilogue, stream);
    case 224256: return prompt_epilogue<7, 8>(g, epilogue, stream);
    case 192256: return prompt_epilogue<6, 8>(g, epilogue, stream);
    case 160256: return prompt_epilogue<5, 8>(g, epilogue, stream);
    case 128256: return prompt_epilogue<4, 8>(g, epilogue, stream);
    case 256128: return prompt_epilogue<8, 4>(g, epilogue, stream);
    case 224128: return prompt_epilogue<7, 4>(g, epilogue, stream);
    case 192128: return prompt_epilogue<6, 4>(g, epilogue, stream);
    case 160128: return prompt_epilogue<5, 4>(g, epilogue, stream);
    case 128128: return prompt_epilogue<4, 4>(g, epilogue, stream);
  }
  return ra_fail("gemm_prompt: no tiles of %d x %d", plan.rows, plan.cols);
}

// As ra_prompt_plan, of a product of `tiles` row tiles known beforehand
static float experts_cost(long tiles, int rows, int weight_rows, int K, int cols) {
  const int slots = ra_cu_count() / RA_XCDS;
  const long all = tiles * ((weight_rows + cols - 1) / cols), rounds = ((all + RA_XCDS - 1) / RA_XCDS + slots - 1) / slots;
  const float fill = (float)all / (float)(rounds * slots * RA_XCDS), area = (float)rows * cols / 65536.f;
  return 6.f + rounds * (11.2f * area + (K / GP_BK) * (0.227f + 0.623f * area + fill * (0.027f + 0.282f * area)));
}

bool ra_prompt_experts_plan(int pairs, int experts, int ff, int width, int gated, long tokens, long ldx, long ld_down,
                            RaExpertsPlan* plan) {
  if (ff % 64 || width % 64 || ff < 256 || width < 256 || experts > 0xFFFF || ((tokens - 1) * ldx + width) * 2 > 0xFFFFFF00l ||
      2l * ff * width * 2 > 0xFFFFFF00l || 256l * ld_down * 2 > 0xFFFFFF00l)
    return false;
  const float mean = (float)pairs / experts;
  float best = 1e30f;
  for (int rows = 128; rows <= 256; rows += 64) {
    // an expert's pairs, a deviation above the mean, in whole tiles
    const long tiles = (long)experts * (long)ceilf((mean + sqrtf(mean)) / rows);
    const int up = gated ? 2 * ff : ff;
    const float u[2] = {experts_cost(tiles, rows, up, width, 128), experts_cost(tiles, rows, up, width, 256)};
    const float d[2] = {experts_cost(tiles, rows, width, ff, 128), experts_cost(tiles, rows, width, ff, 256)};
    const float us = fminf(u[0], u[1]) + fminf(d[0], d[1]);
    if (us < best) {
      best = us;
      // An expert of one tile reads its weights once: they are asked for past the caches' usual policy. 16 experts of 1536 x 4096, four
      // a token, with their gate, 300 tokens 157 us, so 142, 600 185, 167; with two tiles an expert, 1000 tokens, the other way
      // round, 268 and 285. 128 experts of 768 x 2048, eight a token: 1000 tokens 333, 307, 3000 488, 449; 6000, two tiles, 858 and 891.
      const bool once = tiles <= experts && (size_t)experts * ff * width * sizeof(bf16_t) >= RA_STREAM_BYTES;
      *plan = {rows, u[0] < u[1] ? 128 : 256, d[0] < d[1] ? 128 : 256, once};
    }
  }
  return true;
}

int ra_prompt_experts(int rows, int cols, int kind, const void* a, long tokens, int lda, const void* w, int ldw, void* out, int N,
                      int K, const int* plan, const int* slots, const float* weights, int top, long most, int past, hipStream_t stream) {
  PromptArgs g = {(const bf16_t*)a, (const bf16_t*)w, out, (int)tokens, N, K, lda, ldw, N, 1.f, 0, 0, 1, 1, K / GP_BK,
                  plan, slots, weights, top};
  const int k = GP_MOE_RELU2 + kind;
#define RA_EXPERTS(TM, TN) return past ? prompt_experts<TM, TN, true>(g, k, most, stream) : prompt_experts<TM, TN, false>(g, k, most, stream);
  switch (rows * 1000 + cols) {
    case 256256: RA_EXPERTS(8, 8)
    case 192256: RA_EXPERTS(6, 8)
    case 128256: RA_EXPERTS(4, 8)
    case 256128: RA_EXPERTS(8, 4)
    case 192128: RA_EXPERTS(6, 4)
    case 128128: RA_EXPERTS(4, 4)
  }
#undef RA_EXPERTS
  return ra_fail("gemm_prompt: no tiles of %d x %d for experts", rows, cols);
}

// Whether a product is this kernel's: 0 no, 1 yes, 2 it could be, but few of its tiles are there and the library's product in float
// with the gate's kernel behind it is ahead. (us, here / library, weights from memory.)
// Up to 128 rows the weights' way from memory is the bound, and gemm_tile.hip's smaller stages are ahead. With a gate it is ahead of
// the library and the gate's kernel from there on (129 rows of 24576 x 4096 51 / 59, 512 of 19456 x 2560 57 / 62, 4096 of 24576 x 4096
// 577 / 593), a plain product from 513 rows on (513 rows of 6144 x 4096 31 / 36; below, wide ones would be, 300 rows of 12288 x 4096
// 45 / 52, most not, 512 rows of 6144 x 4096 38 / 36).
// A workgroup walks all of K at 0.35 to 0.45 us a step however few there are, and the library has smaller tiles: where tiles of
// 128 x 128 fill less than half of the chip, it is ahead with K above 2048 (gated 256 rows of 2048 x 4096 38 / 19, of 4096 x 2560
// 30 / 20, 512 of 4096 x 4096 38 / 33, but 513, 160 tiles, 31 / 38, and 256 rows of 8192 x 2048 23 / 29, of 6144 x 1024 14 / 19),
// a plain product, which has no gate's kernel to save, up to three quarters (513 rows of 1024 x 8192 52 / 29, of 2048 x 4096
// 29 / 24, 768 of 4096 x 4096 38 / 33; 1800 of 2048 x 4096, 240 tiles, 32 / 36), and with a shorter K up to half (1024 rows of 2048 x
// 2048 21 / 17; 1280, 160 tiles, 21 / 21, 513 of 4096 x 1024 11 / 15).
// Where tiles of 256 x 256 fill their rounds to 95 % and no column of them is padding, the library's product of that size is ahead of a
// plain one here: 8192 rows of 6144 x 4096 282 / 267, 4096 of 12288 x 4096 287 / 270, 4096 of 4096 x 4096 96 / 90; beside such
// numbers of rows it is behind, 6000 of 12288 x 4096 442 / 547, 3000 of 6144 x 4096 115 / 136. With a gate it is behind in both
// (4096 of 24576 x 4096 577 / 593). Left are a few plain products that nothing here tells from others, 4 to 8 % (8192 of 5376 x 4096
// 263 / 250, 513 of 16448 x 4096 77 / 71).
// One that adds into the stream, of more than half of the chip's tiles (1024 rows of 2048 x 2048 24 / 18), is priced beside the
// library's. What a product takes here by that price is 5 % less in a single round and 12 % more in many, and 12 % more in any where
// the rows fill every tile (all workgroups then walk K in step, where a row tile of few rows runs ahead and brings the weights into
// the caches); the library's time for weights from memory is its products at 1.45 PFLOP/s, 12 us and 3 ns a k. Over 300 products of
// 24 shapes the choice is 2.7 % ahead of the library alone and nowhere more than 8 % behind it (2048 rows of 5120 x 8192 148 / 137):
// 2048 rows of 2560 x 4096 47 / 48, 3000 of 5120 x 8192 192 / 187, 1733 of 5120 x 25600 382 / 682, but 768 of 4096 x 4096 42 / 36,
// 1536 of 2560 x 9728 94 / 89. Above 3072 rows the library multiplies without adding, which it does faster (4096 rows of 4096 x 4096
// 95 us; adding 117, here 121).
// K stays whole, though two to six ranges would be ahead up to 1500 rows (1024 rows of 2560 x 9728 64 us against 85 in the library):
// a row's sums then do not depend on how many rows share the call, so that a prompt gives the same bits alone and among others.
extern "C" int ra_gemm_prompt_takes(int epilogue, int M, int N, int K) {
  if (M <= 128 || !ra_prompt_shape(N, K) || (size_t)N * K < (4u << 20)) return 0;
  const long cus = ra_cu_count(), tiles = (long)((M + 127) / 128) * ((N + 127) / 128);
  if (epilogue == GP_GATED) return K > 2048 && tiles * 2 <= cus ? 2 : 1;
  if (epilogue == GP_PLAIN) {
    if (M <= 512 || (K > 2048 ? tiles * 4 <= cus * 3 : tiles * 2 <= cus)) return 0;
    const long large = (long)((M + 255) / 256) * (N / 256), rounds = (large + cus - 1) / cus;
    return N % 256 != 0 || large * 100 < rounds * cus * 95;
  }
  if (epilogue != GP_ADD || M <= 256 || M > 3072 || tiles * 2 <= cus) return 0;
  const RaPromptPlan p = ra_prompt_plan(M, N, K, K);
  const float adding = (float)M * N * 4.f / 4.5e6f;        // the stream read and written at the end
  return p.us * (M % p.rows == 0 ? 1.12f : 1.12f - 0.17f / p.rounds) + adding <=
         (float)((double)M * N * K * 2.0 / 1.45e9) + 12.f + 0.003f * K;
}

// bfloat16, many rows (ra_gemm_prompt_takes): epilogue 0 C = A . W^T in bfloat16; 1 bfloat16 silu(gate) * up; 2 float C += alpha *
// (A . W^T); 3 float C = A . W^T, or with more than one range C[ranges][M][N]. tile_rows 0: the plan's own choice.
extern "C" int ra_gemm_prompt(const void* A, const void* W, void* C, int epilogue, int M, int N, int K, int lda, int ldc,
                              float alpha, int tile_rows, int tile_cols, int ranges, hipStream_t stream) {
  RA_CHECK(epilogue >= 0 && epilogue <= 3, "gemm_prompt: epilogue %d", epilogue);
  RA_CHECK(M > 0 && ra_prompt_shape(N, K), "gemm_prompt: a product of [%d, %d, %d]", M, N, K);
  RA_CHECK(ranges >= 1, "gemm_prompt: %d ranges", ranges);
  RaPromptPlan plan = ra_prompt_plan(M, N, K, (K / GP_BK + ranges - 1) / ranges * GP_BK);
  RA_CHECK(plan.ranges == ranges, "gemm_prompt: K of %d does not cut into %d ranges", K, ranges);
  if (tile_rows) {
    plan.rows = tile_rows;
    plan.cols = tile_cols;
  }
  return ra_prompt_product(plan, epilogue, A, W, C, M, N, K, lda, ldc, alpha, stream);
}
