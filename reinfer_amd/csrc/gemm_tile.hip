// Products of up to 128 rows in bfloat16, C[M,N] = A[M,K] . W[N,K]^T: decode steps of 17 rows and more, short prompts (and up to 512
// rows where N or K does not fit gemm_prompt.hip's steps). Reached through the entry points of gemm_wide.hip.
//
// They are bound by reading the weights once, and beside that by the rows, which every workgroup reads again from the caches: a CU
// takes 24 KB/us of the chip's weight stream and some 96 KB/us of rows (40 bytes a clock; four waves alone take 30), and the two
// times add up, however many loads are under way. So all CUs get the same share of the weights (tiles of 64 to 160 features, and K
// ranges where those are few: tile_plan), a wide tile where rows are many, and nothing else may stand between the loads:
//  - the workgroups stay (one a CU, five to ten waves) and take tiles b, b + grid, ...; their loads go straight to LDS through a
//    ring of 128 KB (three to six stages of 64 k) that runs on across the ends of tiles;
//  - one barrier a stage, in the middle of its products: the first half's operands are read behind the barrier before it, so that
//    products are there to issue when it falls; loads and operand reads stand between the products (with a step's loads issued at
//    its head and its operands read at once 24576 x 4096 took 47 us at 97 rows, 44 with another stage; so 41 to 42);
//  - workgroups start their walk over K at different stages and wrap round: the rows that are read at one moment, a whole K apart,
//    would otherwise fall on few memory channels (K of 4096: 47 us without, 42 with; of 2560 the same).
// A row of a stage is 8 pieces of 16 bytes, piece p of row r at place p ^ (r / 2 % 8): the 16 rows of an operand, two to 256 bytes,
// then fall on all banks. Loads write LDS in the order of their lanes, so it is their addresses that are permuted, inside 128 bytes.
//
// In a chain of launches, weights from memory, with the adding kernel where there is one, us before (17 to 64 rows: weights through
// registers, a workgroup a tile; above: tiles of 128 rows with a step's loads at its head) / now: 151936 x 2560 in float at 48 rows 178 /
// 156, x 4096 254 / 227; 19456 x 2560 with its gate at 48 rows 24.5 / 23.4, 64 28.7 / 24.7, 97 30.3 / 28.8; 24576 x 4096 at 97 rows
// 47.5 / 40.5; 4096 x 12288 added at 48 rows 29.4 / 25.9, 97 31.1 / 29.8; 2560 x 4096 at 48 rows 15.7 / 13.7. A plain read of the
// weights of these takes 121, 195, 16.5, 31.6, 16.5 and 5.1.
#include <type_traits>
#include <utility>

#include "common.h"
#include "reinfer_hip.h"
#include "gemm_tile.h"
#include "gemm_prompt.h"

namespace {

#define GT_BK 64
#define GT_SIDE 128
#define GT_RING (128 * 1024)
#define GT_SPAN 0x7FFFFF00ull      // bytes that a descriptor covers, from a tile's first row on

typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));

enum { GT_PLAIN = 0, GT_GATED = 1, GT_ADD = 2, GT_PART = 3, GT_PLAIN_HALF = 4 };

struct TileArgs {
  const bf16_t* a;
  const bf16_t* w;
  void* c;                                   // GT_PART: float [ranges][M][N]
  int M, N, K, lda, ldc;
  int m_tiles, n_tiles, ranges, range_k;
  unsigned m_part, z_part;                   // 2^32 over m_tiles and over ranges, rounded up (0: over one)
  RaTileEnd end;
};

template <class F, int... I>
__device__ __forceinline__ void gt_each(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void gt_for(F&& f) {
  gt_each(f, std::make_integer_sequence<int, N>{});
}
// The instructions stay in the order that they are written in.
#define GT_ORDER __builtin_amdgcn_sched_barrier(0)

// e^x to an ulp or two in seven instructions: 2^(x log2 e), with what the product lost and the rest of log2 e put back to first order
__device__ __forceinline__ float gt_exp(float x) {
  const float c = fminf(fmaxf(x, -126.f), 126.f), hi = c * 0x1.715476p+0f;         // beyond, 1 + e^x is 1 or infinite
  const float lost = fmaf(c, 0x1.715476p+0f, -hi) + c * 0x1.4ae0c0p-26f;
  return __builtin_amdgcn_exp2f(hi) * fmaf(lost, 0x1.62e430p-1f, 1.f);
}

__device__ __forceinline__ int gt_key(int row) { return (row >> 1) & 7; }

// BMT x TN tiles of 16 rows x 16 features, shared out over WM x WN waves. QUICK: results whose rows start at whole pieces, a bias where
// they are plain only and, with the gate, in bfloat16, so that an end is a few stores; what is left takes any end, in four times the code
// (a launch runs each line of its code for the first time, from memory: with one end for all, 19456 x 2560 with its gate took 30.5 us at
// 97 rows, so 28.8; with a bias 51200 x 5120 at 17 rows 101.7, so 81.5, without one 82.3 and 81.1).
template <int BMT, int TN, int WM, int WN, int EPI, bool QUICK, bool STREAM>
__global__ void __launch_bounds__(64 * WM * WN) gemm_tile_kernel(TileArgs g) {
  constexpr int NW = WM * WN, MT = BMT / WM, NT = TN / WN;
  static_assert(BMT % WM == 0 && TN % WN == 0);
  constexpr int BM = 16 * BMT, BN = 16 * TN;
  constexpr int PA = (2 * BMT + NW - 1) / NW, PB = (2 * TN + NW - 1) / NW, P = PA + PB;   // a wave's loads a stage: 8 rows (1 KB) each
  constexpr int SLOT = (BM + BN) * GT_BK, ROOM = GT_RING / 2 / SLOT, STAGES = ROOM < 6 ? ROOM : 6;
  constexpr unsigned NOWHERE = 0x80000000u;
  constexpr bool SUMS = BM <= 64 && EPI != GT_PART;          // a carried norm's row factor may be applied here
  // The ring, where loads of no row go, and each wave's share of the rows' sums of squares: one array, since between several the
  // compiler tells the ring's loads and reads apart by itself and waits for every load in front of every read.
  __shared__ __attribute__((aligned(1024))) bf16_t lds[STAGES * SLOT + 512 + (SUMS ? NW * BM * 2 : 0)];
  float* const row_ss = (float*)(lds + STAGES * SLOT + 512);       // [NW][BM]
  const int total = g.m_tiles * g.n_tiles * g.ranges, stride = (int)gridDim.x;
  int at = (int)blockIdx.x;
  if (at >= total) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  // A tile: the row tiles of a panel and range of weights follow one another. Workgroups go round the XCDs, so that of eight ranges an
  // XCD has one, and its L2 that part of the rows. Of four it would have one too, in every other panel, and where panels lie whole
  // megabytes apart (128 rows of 4096) their loads come a quarter slower: there neighbouring pairs of panels start their ranges one on
  // (8192 x 4096 at 17 / 48 / 97 rows 19.7 / 21.1 / 25.8 us, so 16.0 / 18.6 / 22.7, 8192 x 8192 31.7 / 32.8 / 39.5, 26.2 / 28.8 / 34.7;
  // elsewhere 3 % either way, with eight ranges up to 17 % slower).
  const bool turned = g.ranges == 4 && ((unsigned)BN * (unsigned)g.K & ((1u << 19) - 1)) == 0;
  auto place = [&](int tile, int& m0, int& z, int& n) {
    const int in = g.m_part ? (int)__umulhi((unsigned)tile, g.m_part) : tile;
    m0 = (tile - in * g.m_tiles) * BM;
    n = g.z_part ? (int)__umulhi((unsigned)in, g.z_part) : in;
    z = in - n * g.ranges;
    if (turned) z = (z + n / 2) & 3;
  };

  // The carried norm's partial sums of squares. Up to eight a row (a product cut into ranges wrote them, one for 1024 columns): lane group
  // q asks for parts q and 4 + q of its rows here, ahead of the first stages, and looks at them when the tile is done. More (one for 16
  // columns, of up to 32 rows): the waves and their lane groups share the parts out, and their sums meet in LDS, both in a fixed order.
  const int wm = wave / WN, wn = wave % WN;
  const bool many = SUMS && g.end.in_parts > 8;
  float held[MT][2];
#pragma unroll
  for (int j = 0; j < MT; ++j) held[j][0] = held[j][1] = 0.f;
  if (SUMS && !many) {
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      const float* ss = g.end.in_ss + min((wm * MT + j) * 16 + r, g.M - 1);
      if (q < g.end.in_parts) held[j][0] = ss[(size_t)q * g.M];
      if (4 + q < g.end.in_parts) held[j][1] = ss[(size_t)(4 + q) * g.M];
    }
  }

  // Loads past a descriptor's end return zeros and touch no memory: rows past M or N, pieces past the K range and stages past the
  // workgroup's last tile are loads like any other, so that the waits count loads exactly.
  unsigned a_off[PA], w_off[PB];
  const int l8 = lane >> 3;
#pragma unroll
  for (int i = 0; i < PA; ++i) {
    const int row = (i * NW + wave) * 8 + l8;
    a_off[i] = row < min(BM, g.M) ? (unsigned)(((size_t)row * g.lda + ((lane & 7) ^ gt_key(row)) * 8) * 2) : NOWHERE;
  }
#pragma unroll
  for (int i = 0; i < PB; ++i) {
    const int row = (i * NW + wave) * 8 + l8;
    w_off[i] = row < BN ? (unsigned)(((size_t)row * g.K + ((lane & 7) ^ gt_key(row)) * 8) * 2) : NOWHERE;
  }
  // where in a stage this lane's pieces lie: the rows of a load and of the next are 8 NW apart, which an odd NW makes another key
  const int piece[2] = {((lane & 7) ^ gt_key(wave * 8 + l8)) * 8, ((lane & 7) ^ gt_key((NW + wave) * 8 + l8)) * 8};
  // where the loads are: stage f_s of tile f_at
  int f_at = at, f_s = 0, f_k0, f_k1, f_steps, f_rot, f_k = 0;
  unsigned f_past[2];                        // the top bit where a piece lies past the K range
  const bf16_t *f_a, *f_w;
  unsigned a_bytes, w_bytes;                 // from there to the end: 0 behind the last tile, where nothing is asked for
  auto enter = [&]() {
    int m0, z, n;
    place(f_at, m0, z, n);
    f_k0 = z * g.range_k;
    f_k1 = min(f_k0 + g.range_k, g.K);
    f_steps = (f_k1 - f_k0 + GT_BK - 1) / GT_BK;
    f_rot = (int)((unsigned)(n / 8 * 5) % (unsigned)f_steps);
    f_a = g.a + (size_t)m0 * g.lda;
    a_bytes = (unsigned)(((size_t)(g.M - 1 - m0) * g.lda + g.K) * 2);
    f_w = g.w + (size_t)n * BN * g.K;
    w_bytes = (unsigned)((size_t)min(g.N - n * BN, BN) * g.K * 2);
  };
  auto aim = [&]() {                         // at the stage that is asked for next
    const int k = f_k0 + (f_s + f_rot < f_steps ? f_s + f_rot : f_s + f_rot - f_steps) * GT_BK;
    f_k = k * 2;
    f_past[0] = k + piece[0] < f_k1 ? 0u : NOWHERE;
    f_past[1] = NW % 2 == 0 ? f_past[0] : k + piece[1] < f_k1 ? 0u : NOWHERE;
  };
  auto move = [&]() {
    if (++f_s == f_steps) {
      f_s = 0;
      f_at += stride;
      if (f_at < total) enter();
      else a_bytes = w_bytes = 0;
    }
  };
  auto fetch = [&](int i, int slot) {        // load i of the stage's P
    bf16_t* to = lds + slot * SLOT;
    const bool rows_of_w = i < PB;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(rows_of_w ? f_w : f_a), 0,
                                                                          (int)(rows_of_w ? w_bytes : a_bytes), 0x00020000);
    if (rows_of_w) {
      const int rows = i * NW + wave;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc, (__attribute__((address_space(3))) void*)(2 * TN % NW == 0 || rows < 2 * TN ? to + (BM + rows * 8) * GT_BK : lds + STAGES * SLOT),
          16, (int)(w_off[i < PB ? i : 0] | f_past[i & 1]), f_k, 0, STREAM ? RA_STREAM : 0);
    } else {
      const int j = i - PB, rows = j * NW + wave;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc, (__attribute__((address_space(3))) void*)(2 * BMT % NW == 0 || rows < 2 * BMT ? to + rows * 8 * GT_BK : lds + STAGES * SLOT),
          16, (int)(a_off[i < PB ? 0 : j] | f_past[j & 1]), f_k, 0, 0);
    }
  };
  enter();
#pragma unroll
  for (int s = 0; s < STAGES; ++s) {
    aim();
#pragma unroll
    for (int i = 0; i < P; ++i) fetch(i, s);
    move();
  }
  if (many) {
    constexpr int EACH = 8;                  // parts of a lane that are asked for at once
    for (int j = 0; j < BMT && j * 16 < g.M; ++j) {
      const float* ss = g.end.in_ss + min(j * 16 + r, g.M - 1);
      float t = 0.f;
      for (int p = 4 * wave + q; p < g.end.in_parts; p += 4 * NW * EACH) {
        float v[EACH];
#pragma unroll
        for (int i = 0; i < EACH; ++i) v[i] = ss[(size_t)min(p + 4 * NW * i, g.end.in_parts - 1) * g.M];
#pragma unroll
        for (int i = 0; i < EACH; ++i) t += p + 4 * NW * i < g.end.in_parts ? v[i] : 0.f;
      }
      t += __shfl_xor(t, 16, RA_WAVE);
      t += __shfl_xor(t, 32, RA_WAVE);
      if (q == 0) row_ss[wave * BM + j * 16 + r] = t;
    }
  }
  const int x0 = (q ^ gt_key(r)) * 8, x1 = ((4 + q) ^ gt_key(r)) * 8;
  const bf16_t* const ab = lds + (wm * 16 * MT + r) * GT_BK;
  const bf16_t* const wb = lds + (BM + wn * 16 * NT + r) * GT_BK;
  bf16x8_t xa[MT], ya[NT], xb[MT], yb[NT];   // operands of the first and of the second 32 k
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(P * (STAGES - 1)) : "memory");
#pragma unroll
  for (int i = 0; i < NT; ++i) ya[i] = *(const bf16x8_t*)(wb + i * 16 * GT_BK + x0);
#pragma unroll
  for (int j = 0; j < MT; ++j) xa[j] = *(const bf16x8_t*)(ab + j * 16 * GT_BK + x0);
  auto row_factor = [&](int j) {
    float t = held[j][0] + held[j][1];
    if (many) {
      t = 0.f;
      for (int w = 0; w < NW; ++w) t += row_ss[w * BM + (wm * MT + j) * 16 + r];
    } else {
      t += __shfl_xor(t, 16, RA_WAVE);
      t += __shfl_xor(t, 32, RA_WAVE);
    }
    return rsqrtf(t * g.end.in_inv_width + g.end.in_eps);
  };
  int slot = 0;
  for (; at < total; at += stride) {
    int m0, z, n_at;
    place(at, m0, z, n_at);
    const int n0 = n_at * BN;
    const int k0 = z * g.range_k, steps = (min(k0 + g.range_k, g.K) - k0 + GT_BK - 1) / GT_BK;
    f32x4_t acc[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < steps; ++s) {
      const int behind = slot + 1 == STAGES ? 0 : slot + 1;
      const bf16_t *a1 = ab + slot * SLOT + x1, *w1 = wb + slot * SLOT + x1;
      const bf16_t *a0 = ab + behind * SLOT + x0, *w0 = wb + behind * SLOT + x0;
      aim();
      GT_ORDER;
      gt_for<NT * MT>([&](auto c) {
        constexpr int i = c / MT, j = c % MT;
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ya[i], xa[j], acc[i][j], 0, 0, 0);
        GT_ORDER;
        if constexpr (c == 0) {
#pragma unroll
          for (int t = 0; t < MT; ++t) xb[t] = *(const bf16x8_t*)(a1 + t * 16 * GT_BK);
        }
        if constexpr (j == 0) yb[i] = *(const bf16x8_t*)(w1 + i * 16 * GT_BK);
        GT_ORDER;
      });
      // This wave's reads of this stage are done, and of its loads all but those of the STAGES - 2 behind the next one; the barrier
      // makes that true of all waves: the next stage is there, and this one's slot may be written.
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(P * (STAGES - 2)) : "memory");
      GT_ORDER;
      gt_for<NT * MT>([&](auto c) {
        constexpr int i = c / MT, j = c % MT, f0 = c * P / (NT * MT), f1 = (c + 1) * P / (NT * MT);
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(yb[i], xb[j], acc[i][j], 0, 0, 0);
        GT_ORDER;
        if constexpr (c == 0) {
#pragma unroll
          for (int t = 0; t < MT; ++t) xa[t] = *(const bf16x8_t*)(a0 + t * 16 * GT_BK);
        }
        if constexpr (j == 0) ya[i] = *(const bf16x8_t*)(w0 + i * 16 * GT_BK);
        gt_for<f1 - f0>([&](auto f) { fetch(f0 + f, slot); });
        GT_ORDER;
      });
      move();
      slot = behind;
    }
    // lane (r, q) holds rows r of a tile, features 4 q + e
    constexpr bool HALF = EPI == GT_GATED || EPI == GT_PLAIN_HALF;
    const int cols = EPI == GT_GATED ? g.N / 2 : g.N;
    if constexpr (QUICK) {
      // past the descriptor, which spans the result from the tile's first row on, lies what is past the last row or column
      const int SIZE = HALF ? 2 : 4, left = min(g.M - m0, BM);
      const __amdgpu_buffer_rsrc_t cr = __builtin_amdgcn_make_buffer_rsrc(
          (char*)g.c + ((size_t)(EPI == GT_PART ? z : 0) * g.M + m0) * g.ldc * SIZE, 0,
          (int)(((size_t)(left - 1) * g.ldc + cols) * SIZE), 0x00020000);
      constexpr bool PLAIN = EPI == GT_PLAIN || EPI == GT_PLAIN_HALF;
      f32x4_t bias[PLAIN ? NT : 1];
      if (PLAIN && g.end.bias) {
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) bias[PLAIN ? i : 0][e] = to_f32(g.end.bias[min(n0 + (wn * NT + i) * 16 + q * 4 + e, cols - 1)]);
      }
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        const int row = (wm * MT + j) * 16 + r;
        const float rstd = SUMS && g.end.in_parts > 0 ? row_factor(j) : 1.f;
#pragma unroll
        for (int i = 0; i < NT; ++i) {
          const int first = n0 + (wn * NT + i) * 16, n = EPI == GT_GATED ? first / 2 + (q & 1) * 4 : first + q * 4;
          const unsigned to = (row < left && n < cols && (EPI != GT_GATED || q < 2)) ? ((unsigned)row * (unsigned)g.ldc + n) * SIZE : 0xFFFFFFF0u;
          f32x4_t v = acc[i][j];
          if (SUMS) v *= rstd;
          if (PLAIN && g.end.bias) v += bias[PLAIN ? i : 0];
          if constexpr (EPI == GT_GATED) {   // rows 0-7 of a tile are gate, 8-15 up of the same features: those sit two groups on
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float up = __shfl_xor(v[e], 32, RA_WAVE);
              v[e] = v[e] * __builtin_amdgcn_rcpf(1.f + gt_exp(-v[e])) * up;
            }
          }
          if constexpr (HALF) {
            const bf16x4_t o = {(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2_t, o), cr, to, 0, 0);
          } else {
            if constexpr (EPI == GT_ADD)
              v = v * g.end.alpha + __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(cr, to, 0, 0));
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), cr, to, 0, 0);
          }
        }
      }
      continue;
    }
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      const int row = (wm * MT + j) * 16 + r, m = m0 + row;
      const float rstd = SUMS && g.end.in_parts > 0 ? row_factor(j) : 1.f;
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const int first = n0 + (wn * NT + i) * 16, n = first + q * 4;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = SUMS ? acc[i][j][e] * rstd : acc[i][j][e];
        if constexpr (EPI == GT_GATED) {     // rows 0-7 of a tile are gate, 8-15 up of the same features: those sit two groups on
          float up[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) up[e] = __shfl_xor(v[e], 32, RA_WAVE);
          if (m >= g.M || q >= 2 || first >= g.N) continue;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = v[e] * __builtin_amdgcn_rcpf(1.f + gt_exp(-v[e])) * up[e];
        } else {
          if (m >= g.M || n >= g.N) continue;
        }
        const int col = EPI == GT_GATED ? first / 2 + q * 4 : n;
        const size_t to = (EPI == GT_PART ? ((size_t)z * g.M + m) * g.N : (size_t)m * g.ldc) + col;
        if constexpr (EPI == GT_PLAIN || EPI == GT_ADD) {
          if (g.end.bias) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += col + e < cols ? to_f32(g.end.bias[col + e]) : 0.f;
          }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (col + e >= cols) continue;
          if (EPI != GT_PART && EPI != GT_ADD && g.end.half) {
            ((bf16_t*)g.c)[to + e] = (bf16_t)v[e];
          } else {
            float* c = (float*)g.c + to + e;
            *c = EPI == GT_ADD ? v[e] * g.end.alpha + *c : v[e];
          }
        }
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // loads that are still on their way to LDS
}

// With one row of tiles the weights are read once: past the caches' usual policy (RA_STREAM_BYTES in common.h; 48 rows of 24576 x 4096
// with its gate 37.1 us, so 34.8, of 6144 x 4096 12.7, 12.0, 97 rows 15.3, 14.3).
template <int BMT, int TN, int WM, int WN, int EPI, bool QUICK = true>
int tile_launch(TileArgs g, hipStream_t stream) {
  g.m_tiles = (g.M + 16 * BMT - 1) / (16 * BMT);
  g.n_tiles = (g.N + 16 * TN - 1) / (16 * TN);
  const long total = (long)g.m_tiles * g.n_tiles * g.ranges, cus = ra_cu_count();
  RA_CHECK(total < 1L << 27 && g.ranges <= 16, "gemm_tile: too many tiles");         // where 2^32 over 16 divides exactly
  g.m_part = g.m_tiles > 1 ? 0xFFFFFFFFu / (unsigned)g.m_tiles + 1u : 0u;
  g.z_part = g.ranges > 1 ? 0xFFFFFFFFu / (unsigned)g.ranges + 1u : 0u;
  const unsigned grid = (unsigned)(total < cus ? total : cus);
  if (QUICK && g.m_tiles == 1 && ra_streams((size_t)g.N * g.K * sizeof(bf16_t), g.end.keep))
    gemm_tile_kernel<BMT, TN, WM, WN, EPI, QUICK, QUICK><<<grid, 64 * WM * WN, 0, stream>>>(g);
  else
    gemm_tile_kernel<BMT, TN, WM, WN, EPI, QUICK, false><<<grid, 64 * WM * WN, 0, stream>>>(g);
  RA_LAUNCH_CHECK("gemm_tile");
  return 0;
}

// Five to ten waves, which fetch rows faster than four (36 against 30 bytes a clock). Above 64 rows a gated tile of 80 features has
// four, each with its two row tiles of all features. Of 16400 to 20480 features at 65 to 128 rows, four / ten waves, K of 1024 13.0 / 12.7
// us, 1536 to 2560 the same within 1 % (19456 x 2560 27.7 / 27.9 at 97 rows), 4096 34.0 / 34.6, 5120 45.0 / 47.2, 8192 63.4 / 66.6.
template <int EPI>
int tile_cols(const TileArgs& g, int cols, hipStream_t stream) {
#define RA_GT(BMT, TN, WM, WN) return tile_launch<BMT, TN, WM, WN, EPI>(g, stream)
  constexpr bool MANY = EPI == GT_GATED || EPI == GT_PART;       // the epilogues of more than 64 rows
  if (g.M <= 32) {
    switch (cols) {
      case 64: RA_GT(2, 4, 2, 4);
      case 80: RA_GT(2, 5, 2, 5);
      case 96: RA_GT(2, 6, 2, 3);
      case 112: RA_GT(2, 7, 1, 7);
      case 160: RA_GT(2, 10, 2, 5);
      default: RA_GT(2, 8, 2, 4);
    }
  }
  if (g.M <= 64) {
    switch (cols) {
      case 64: RA_GT(4, 4, 2, 4);
      case 80: RA_GT(4, 5, 2, 5);
      case 96: RA_GT(4, 6, 2, 3);
      case 112: RA_GT(4, 7, 1, 7);
      case 160: RA_GT(4, 10, 2, 5);
      default: RA_GT(4, 8, 2, 4);
    }
  }
  if constexpr (MANY) {
    switch (cols) {
      case 64: RA_GT(8, 4, 4, 2);
      case 80: if constexpr (EPI == GT_GATED) RA_GT(8, 5, 4, 1); else RA_GT(8, 5, 2, 5);
      case 96: RA_GT(8, 6, 4, 2);
      case 112: RA_GT(8, 7, 1, 7);
      default: RA_GT(8, 8, 2, 4);
    }
  }
#undef RA_GT
  return ra_fail("gemm_tile: %d rows", g.M);
}

// any end, in tiles of one width
template <int EPI>
int tile_any(const TileArgs& g, hipStream_t stream) {
  if (g.M <= 64) return tile_launch<4, 8, 2, 4, EPI, false>(g, stream);
  if constexpr (EPI == GT_GATED || EPI == GT_PART) return tile_launch<8, 8, 2, 4, EPI, false>(g, stream);
  return ra_fail("gemm_tile: %d rows", g.M);
}

}  // namespace

static long tile_count(int M, int N) { return (long)((M + GT_SIDE - 1) / GT_SIDE) * ((N + GT_SIDE - 1) / GT_SIDE); }

// K ranges of 129 rows and more: as many as fill the chip once, of at least 512 k (shorter ones are all start and end), at most 16 (each
// is a float plane to write and read again). They follow from N, K and the rows of tiles alone, so that a row has the same sums at any of 129
// to 256 rows (to 384, to 512). Ranges of the exact number of rows, which gemm_prompt.hip's tiles could have, would be faster (the two
// at 5120 x 25600 with 160 rows 92 / 70 us, with 384 139 / 114, 4096 x 12288 with 512 74 / 63, most shapes within 5 %), but then one
// more request in a step changes every row's last bits.
static void many_rows_ranges(int M, int N, int K, int* ranges, int* range_k) {
  long s = ra_cu_count() / tile_count(M, N);
  if (s > K / 512) s = K / 512;
  if (s > 16) s = 16;
  if (s < 1) s = 1;
  *range_k = ((K + (int)s - 1) / (int)s + GT_BK - 1) / GT_BK * GT_BK;
  *ranges = (K + *range_k - 1) / *range_k;
}

// The features of a tile and, where the product may be cut, its K ranges, by what a CU reads: a round of workgroups takes its share of
// the weights at 6.2 TB/s for the chip and at most 26 KB/us a CU, and the rows at 96 KB/us; ranges write and read a plane each at
// 8 TB/s. Of the shapes and rows measured (4096 to 24576 x 2560 to 12288, 24 to 128 rows) the plan is within 4 % of the fastest tile and
// ranges. It does not depend on the exact number of rows (up to 64 and up to 128 have one each), and so neither do a row's sums.
RaTilePlan ra_tile_plan(int M, int N, int K, bool cut) {
  RaTilePlan best = {GT_SIDE, 1, (K + GT_BK - 1) / GT_BK * GT_BK};
  if (M > GT_SIDE) {
    if (cut) many_rows_ranges(M, N, K, &best.ranges, &best.range_k);
    return best;
  }
  const int cus = ra_cu_count(), most = cut ? (K / 512 < 16 ? K / 512 : 16) : 1;
  const float rows = M <= 64 ? 48.f : 112.f;
  float least = 1e30f;
  for (int cols = M <= 64 ? 160 : 128; cols >= 64; cols -= cols > 128 ? 32 : 16) {
    if (cols > GT_SIDE && (size_t)cols * K * 2 >= GT_SPAN) continue;
    const int tiles = (N + cols - 1) / cols;
    const int fits = tiles < cus ? cus / tiles : 1, top = fits < most ? fits : most;
    for (int s = top > 1 ? top : 1; s >= 1 && s + 1 >= top; --s) {       // as many ranges as fill the chip once, or one less
      const int range_k = ((K + s - 1) / s + GT_BK - 1) / GT_BK * GT_BK, ranges = (K + range_k - 1) / range_k;
      const int all = tiles * ranges, full = all / cus, left = all % cus;
      const float w = cols * (float)range_k * 2e-3f, a = rows * (float)range_k * 2e-3f / 96.f;
      float us = full * (w * cus / 6200.f + a) + (left ? a + w / fminf(26.f, 6200.f / left) : 0.f);
      if (cut) us += ranges * rows * N * 1e-6f;
      if (us < least) {
        least = us;
        best = {cols, ranges, range_k};
      }
    }
  }
  return best;
}

// Of 65 to 512 rows. Products that are cut and whose ranges fill three quarters of the chip, or that are small (the library has too few
// tiles for those as well): 9216 x 4096 at 128 rows, 216 of 256 CUs, takes 27 us against the library's 30. 11264 x 4096, 176 CUs, is
// refused though it takes 29 against 32 now (this line was drawn with the tiles of before, which took 34); 22528 x 4096, whose tiles do
// not fill the chip and cannot be cut, takes 40 against 46 at 65 rows, 49 against 47 at 128. Above 256 rows only a long K,
// where the planes are few beside the weights, and more than that share of the chip (4096 x 12288 at 384 rows, 192 CUs,
// 70 us on gemm_prompt.hip's tiles against 69, though at 300 rows 57 against 69; at 512 rows, all of them, 74 against 80); the line
// is the same for all rows of a row of tiles, as the sums are. Beyond 512 the library's larger tiles read less. What adds into
// the stream with up to 128 rows also finishes the norm behind it, which outweighs a poor fill. A gated product, which is
// not cut, where one row of tiles fills half of the chip. Below 8 MB of weights (a router, gates) both take the few us of
// their launches, and the calls stay where they were. (Counted in tiles of 128 x 128, whatever the plan.)
extern "C" int ra_gemm_tile_takes(int epilogue, int M, int N, int K) {
  if (M <= 64 || M > 512 || N < 1 || K < 1024 || (size_t)N * K < (4u << 20) || (size_t)N * K * 2 > 0xFFFFFF00ull) return 0;
  const long cus = ra_cu_count(), tiles = tile_count(M, N);
  if (epilogue == 1) return M <= GT_SIDE && tiles <= cus && tiles * 2 > cus;
  int ranges, range_k;
  many_rows_ranges(M, N, K, &ranges, &range_k);
  if (ranges < 2) return 0;
  if (M > 256) return K >= 8192 && tiles * ranges * 4 > cus * 3;
  return (epilogue == 2 && M <= GT_SIDE) || tiles * 4 <= cus || tiles * ranges * 4 >= cus * 3;
}

int ra_tile_product(int epilogue, const RaTilePlan& plan, const void* A, int lda, const void* W, void* C, int ldc, int M, int N, int K,
                    RaTileEnd end, hipStream_t stream) {
  RA_CHECK(M > 0 && N > 0 && K > 0 && K % 8 == 0 && lda % 8 == 0 && lda >= K && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0,
           "gemm_tile: [%d, %d, %d] with rows of stride %d must be whole 16-byte pieces", M, N, K, lda);
  RA_CHECK((size_t)(plan.cols > GT_SIDE ? plan.cols : GT_SIDE) * K * 2 < GT_SPAN && ((size_t)(M - 1) * lda + K) * 2 < GT_SPAN,
           "gemm_tile: an operand of [%d, %d, %d] is larger than a descriptor covers", M, N, K);
  RA_CHECK(plan.ranges >= 1 && plan.range_k % GT_BK == 0 && (long)(plan.ranges - 1) * plan.range_k < K &&
               (long)plan.ranges * plan.range_k >= K && (plan.ranges == 1 || epilogue == GT_PART),
           "gemm_tile: %d ranges of %d k for %d", plan.ranges, plan.range_k, K);
  RA_CHECK(epilogue != GT_GATED || N % 16 == 0, "gemm_tile: the gate takes whole runs of 16 features");
  if (!end.in_ss) end.in_parts = 0;
  const int cols = epilogue == GT_GATED ? N / 2 : N;
  const bool half = end.half && (epilogue == GT_PLAIN || epilogue == GT_GATED);
  const bool quick = (!end.bias || epilogue == GT_PLAIN) && cols % 4 == 0 && ldc % 4 == 0 && ldc <= (1 << 22) && (uintptr_t)C % (half ? 8 : 16) == 0 &&
                     (half || epilogue != GT_GATED);
  TileArgs g = {(const bf16_t*)A, (const bf16_t*)W, C, M, N, K, lda, ldc, 0, 0, plan.ranges, plan.range_k, 0, 0, end};
  switch (epilogue) {
    case GT_PLAIN:
      if (!quick) return tile_any<GT_PLAIN>(g, stream);
      return half ? tile_cols<GT_PLAIN_HALF>(g, plan.cols, stream) : tile_cols<GT_PLAIN>(g, plan.cols, stream);
    case GT_GATED: return quick ? tile_cols<GT_GATED>(g, plan.cols, stream) : tile_any<GT_GATED>(g, stream);
    case GT_ADD: return quick ? tile_cols<GT_ADD>(g, plan.cols, stream) : tile_any<GT_ADD>(g, stream);
    default: return quick ? tile_cols<GT_PART>(g, plan.cols, stream) : tile_any<GT_PART>(g, stream);
  }
}

// planes[z][m][n] = A[m, range z] . W[n, range z]^T
int ra_tile_ranges(const RaTilePlan& plan, const void* A, int lda, const void* W, float* planes, int M, int N, int K, bool keep,
                   hipStream_t stream) {
  if (M > GT_SIDE && ra_prompt_shape(N, K)) {
    const RaPromptPlan p = ra_prompt_plan(M, N, K, plan.range_k);
    if (p.ranges == plan.ranges) return ra_prompt_product(p, 3, A, W, planes, M, N, K, lda, N, 1.f, stream);
  }
  RaTileEnd end = {};
  end.keep = keep;
  return ra_tile_product(GT_PART, plan, A, lda, W, planes, N, M, N, K, end, stream);
}
