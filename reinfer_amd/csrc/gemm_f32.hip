// Matrix products of the 32-bit path, C[M,N] = A[M,K] . W[N,K]^T (+ bias[N]), on the bfloat16 matrix cores, to float precision.
//
// A float is the sum of three bfloat16 numbers, exactly (but for bits below 2^-133): its value rounded, what that leaves rounded, and the
// rest. Of the nine products of the parts the six largest are summed, in float; what is left out is below 2^-25 of a product, a
// rounding of the sum 2^-24 of it. Measured against 64 bits over normal random numbers the sums are nearer than those of the
// float matrix cores: K 2560 3.43e-7 of the result's norm against 4.08e-7, K 4096 3.47 / 4.09, K 9728 5.59 / 6.27 (a product of
// 32 k is rounded into its sum once a term, where the float cores round for every four k).
//
// Up to 32 rows (gemm_f32_stream_kernel) the product is bound by reading the weights once. A workgroup has 16 features, its
// waves share K out and add their sums through LDS in a fixed order. The weights go by way of a piece of LDS of each wave's own:
// loaded in the products' order a load is 64 bytes of each of 16 rows, half a line each, and takes twice the time of whole lines.
// Splitting is issue time beside the loads' waits: with the next loads asked for behind it 15 % slower, with the rows split by every
// lane that multiplies them 10 %. Weights from memory, float matrix cores / here, us: 4 rows 6144 x 2560 19.7 / 17.0, 2560 x 4096
// 14.3 / 13.8, 19456 x 2560 41.4 / 39.1, 2560 x 9728 29.5 / 26.0, 151936 x 2560 265 / 271; 16 rows 23.5 / 21.7, 16.4 / 15.5, 51 / 48,
// 36.7 / 33.0; 32 rows 36.6 / 34.0, 25.8 / 23.4, 80.5 / 79, 57 / 54.5. Runs of 64 k, or three or four in flight, are slower.
//
// From 33 rows on (gemm_f32_tile_kernel) tiles of both operands go through LDS, split on the way. Six bfloat16 products take 96 cycles
// of a matrix core where the float ones take 256. What bounds them is issue: of a SIMD's time at 256 rows a tile 53 % are products, 27 %
// other vector instructions, which find little room beside them, and 18 % waits; and the chip's power, whose clock is 1.95 GHz
// (on zeros 2.35 and a sixth faster). In a loop over other weights, float matrix cores / here, us: 1119 x 19456 x 2560 880 / 620 (180
// TFLOP/s), 1119 x 2560 x 9728 500 / 330, 2048 x 19456 x 2560 1520 / 1030, 300 x 6144 x 2560 103 / 84, 64 x 19456 x 2560 71 / 62. Tiles
// split by every wave that multiplies them, the compiler's order, two waves a SIMD: 664 for the first. Dot products with (-1, 0) to take
// a part off gave 1 %.
#include <type_traits>

#include "common.h"
#include "reinfer_hip.h"

namespace {

// ------------------------------------------------------------------------------------------------ a float in three parts
struct F32Parts {
  bf16x8_t h, m, l;
};
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
// Two floats rounded, as the low and the high half of a word; what that leaves of them stays behind. (The empty statement has the
// compiler take the halves from the word: left to itself it converts each float once more for that.)
__device__ __forceinline__ unsigned f32_part(float& a, float& b) {
  unsigned u = __builtin_bit_cast(unsigned, (bf16x2_t){(bf16_t)a, (bf16_t)b});
  asm("" : "+v"(u));
  a -= __builtin_bit_cast(float, u << 16);
  b -= __builtin_bit_cast(float, u & 0xFFFF0000u);
  return u;
}
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ F32Parts f32_split(f32x4_t a, f32x4_t b) {
  float v[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  u32x4_t p[3];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) p[i][e] = f32_part(v[2 * e], v[2 * e + 1]);
  return {__builtin_bit_cast(bf16x8_t, p[0]), __builtin_bit_cast(bf16x8_t, p[1]), __builtin_bit_cast(bf16x8_t, p[2])};
}
// Term t of the product of two floats in parts, the smallest first: every kernel adds them in this order.
#define F32_TERMS 6
__device__ __forceinline__ f32x4_t f32_term(int t, const F32Parts& w, const F32Parts& a, f32x4_t c) {
  const bf16x8_t& x = t == 0 ? w.l : t == 2 || t == 3 ? w.m : w.h;
  const bf16x8_t& y = t == 1 ? a.l : t == 2 || t == 4 ? a.m : a.h;
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, c, 0, 0, 0);
}
// The parts of an infinity and of a float that rounds to one are no numbers, and a part that is zero times an infinity is none either: a
// sum that is not finite is worked out again from the floats.
__device__ __forceinline__ bool f32_off(float v) { return !(fabsf(v) <= 3.402823466e38f); }
__device__ __forceinline__ float f32_again(const float* __restrict__ a, const float* __restrict__ w, int K) {
  float s = 0.f;
  for (int k = 0; k < K; k += 4) {
    const f32x4_t x = *(const f32x4_t*)(a + k), y = *(const f32x4_t*)(w + k);
#pragma unroll
    for (int e = 0; e < 4; ++e) s = fmaf(x[e], y[e], s);
  }
  return s;
}

// ------------------------------------------------------------------------------------------------ the order of the sums
// K is summed in up to eight blocks of at least 512 k, whose number and length follow from K alone. A block is one chain of
// 16x16x32 products over its pieces of 32 k, six a piece. The blocks' sums are added in their order, then the bias. Both kernels
// keep this order, so a row's result does not depend on how many rows stand beside it: a request's 32-bit results are the same
// bits alone and in any step.
struct KBlocks {
  int n, k;                                // how many, and k of one (a multiple of 64)
};
KBlocks k_blocks(int K) {
  int n = K / 512;
  n = n < 1 ? 1 : n > 8 ? 8 : n;
  const int k = ((K + n - 1) / n + 63) / 64 * 64;
  return {(K + k - 1) / k, k};
}

// ------------------------------------------------------------------------------------------------ up to 32 rows
// Workgroups that stay: tile b, b + grid, ... of 16 features, all M rows, a wave a block of K. A wave's loads run two runs of 32 k
// ahead, on across the ends of tiles, and are unconditional: through a buffer descriptor a load past its end returns zeros and
// touches no memory, so rows past N or M, pieces past the block and runs past the last tile count like any other load and cost
// nothing.
//
// ROWS is the rows that there is room for. Up to 16 are split once, shared out over the lanes, and handed round in LDS like the
// weights; 32 would take too much of it, and there a lane splits what it loads in the products' order.
#define RA_WAVE_HANDOVER                                   \
  do {                                                     \
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); \
    __builtin_amdgcn_wave_barrier();                       \
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront"); \
  } while (0)
#define F32_BK 32
template <int ROWS>
struct F32Stream {
  static constexpr int MT = (ROWS + 15) / 16;
  static constexpr bool SHARED = ROWS <= 16;
  static constexpr int W_BYTES = 16 * F32_BK * 4, A_BYTES = SHARED ? 3 * ROWS * F32_BK * 2 : 0;   // of a wave's run in LDS
  static constexpr int SUM_BYTES = 2 * MT * RA_WAVE * 16;
  static constexpr int lds(int waves) { return waves * (W_BYTES + A_BYTES + SUM_BYTES); }
};
template <int ROWS>
__global__ void __launch_bounds__(8 * RA_WAVE, 4)
gemm_f32_stream_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                       float* __restrict__ C, int M, int N, int K, int lda, int ldc, int block_k) {
  using Form = F32Stream<ROWS>;
  constexpr int MT = Form::MT, DEPTH = 2;
  constexpr bool SHARED = Form::SHARED;
  constexpr unsigned NOWHERE = 0xFFFFFFF0u;
  constexpr int CH = F32_BK / 4;           // 16-byte pieces of a weight row in a run
  constexpr int LOADS = 2, LR = 8;         // loads of a run, rows of one: whole lines, lane after lane
  constexpr int A_LOADS = SHARED ? ROWS / LR : 2 * MT, A_PART = ROWS * F32_BK * 2;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int lane = threadIdx.x & 63, waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4, wr = lane / CH, wc = lane % CH;
  f32x4_t* const sums = (f32x4_t*)lds;     // [2][waves][MT][64]: of one tile while the next one's may already be written
  char* const own = lds + waves * Form::SUM_BYTES + wave * (Form::W_BYTES + Form::A_BYTES);
  // this wave's run of weights on its way into the products' order: piece c of row r at place c ^ r, from where the products' rows are
  // read without conflicts; and of rows, three parts of [ROWS][32], of which piece c (8 k) of row r lies at place c ^ r / 4
  f32x4_t* const laid = (f32x4_t*)own;
  char* const rows = own + Form::W_BYTES;
  auto spot = [&](int m, int c) { return rows + m * F32_BK * 2 + (c ^ (m >> 2 & 3)) * 16; };
  const int k0 = wave * block_k, k1 = min(k0 + block_k, K);
  const int n_steps = block_k / F32_BK;    // even, and the same for every wave: all meet at a tile's end
  const int n_tiles = (N + 15) / 16;
  const int n_mine = (n_tiles - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
  const int total = n_mine * n_steps;
  const __amdgpu_buffer_rsrc_t w_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(W), 0, (int)((size_t)N * K * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t a_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(A), 0, (int)(((size_t)(M - 1) * lda + K) * 4), 0x00020000);
  f32x4_t w[DEPTH][LOADS], a[DEPTH][A_LOADS];
  int l_q = 0, l_step = 0, l_n = (int)blockIdx.x * 16;             // where the loads are
  auto load_w = [&](int d) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int k = k0 + l_step * F32_BK + wc * 4, n = l_n + i * LR + wr;
      const unsigned off = l_q < total && k < k1 && n < N ? (unsigned)(((size_t)n * K + k) * 4) : NOWHERE;
      w[d][i] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, off, 0, 0));
    }
  };
  auto load_a = [&](int d) {                   // and on to the next run
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) {
      const int k = k0 + l_step * F32_BK + (SHARED ? wc * 4 : q * 8 + i % 2 * 4);          // a multiple of 4
      const int m = SHARED ? i * LR + wr : i / 2 * 16 + r;
      const unsigned off = l_q < total && k < k1 && m < M ? (unsigned)(((size_t)m * lda + k) * 4) : NOWHERE;
      a[d][i] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, off, 0, 0));
    }
    ++l_q;
    if (++l_step == n_steps) {
      l_step = 0;
      l_n += (int)gridDim.x * 16;
    }
  };
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) {
    load_w(d);
    load_a(d);
  }
  f32x4_t acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  int step = 0, n0 = (int)blockIdx.x * 16, buf = 0;                // where the products are
  for (int base = 0; base < total; base += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      // this wave's alone: LDS takes its accesses in their order, and the fences have the compiler keep that order where lanes
      // read what others wrote, and write what others have read
      RA_WAVE_HANDOVER;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) laid[(i * LR + wr) * CH + (wc ^ wr)] = w[d][i];
      if constexpr (SHARED) {
#pragma unroll
        for (int i = 0; i < A_LOADS; ++i) {
          float v[4] = {a[d][i][0], a[d][i][1], a[d][i][2], a[d][i][3]};
#pragma unroll
          for (int p = 0; p < 3; ++p) {
            const unsigned lo = f32_part(v[0], v[1]), hi = f32_part(v[2], v[3]);
            *(unsigned long long*)(spot(i * LR + wr, wc >> 1) + (wc & 1) * 8 + p * A_PART) = lo | (unsigned long long)hi << 32;
          }
        }
      }
      RA_WAVE_HANDOVER;
      // the run DEPTH ahead is asked for as soon as this one's registers are free
      __builtin_amdgcn_sched_barrier(0);
      load_w(d);
      if (SHARED) load_a(d);
      __builtin_amdgcn_sched_barrier(0);
      const F32Parts y = f32_split(laid[r * CH + ((q * 2) ^ (r & 7))], laid[r * CH + ((q * 2 + 1) ^ (r & 7))]);
      F32Parts x[MT];
      if constexpr (SHARED) {                  // columns of the product past ROWS are others again, and nobody's
        const char* from = spot(r & (ROWS - 1), q);
        x[0] = {*(const bf16x8_t*)from, *(const bf16x8_t*)(from + A_PART), *(const bf16x8_t*)(from + 2 * A_PART)};
      } else {
#pragma unroll
        for (int t = 0; t < MT; ++t) x[t] = f32_split(a[d][2 * t], a[d][2 * t + 1]);
      }
#pragma unroll
      for (int e = 0; e < F32_TERMS; ++e)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = f32_term(e, y, x[t], acc[t]);
      if (!SHARED) {
        __builtin_amdgcn_sched_barrier(0);
        load_a(d);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    step += DEPTH;
    if (step < n_steps) continue;
    // a tile is complete: lane has row lane % 16, features 4 (lane / 16) .. + 3. One barrier a tile: its sums are read
    // while the next tile's go to the other buffer, and a wave writes a buffer again only behind the next barrier.
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      sums[((buf * waves + wave) * MT + t) * RA_WAVE + lane] = acc[t];
      acc[t] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    for (int t = wave; t < MT; t += waves) {
      f32x4_t v = sums[(buf * waves * MT + t) * RA_WAVE + lane];
#pragma unroll
      for (int x = 1; x < 8; ++x)
        if (x < waves) v += sums[((buf * waves + x) * MT + t) * RA_WAVE + lane];
      const int m = t * 16 + r;
      if (m < M) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int f = n0 + q * 4 + i;
          if (f < N) C[(size_t)m * ldc + f] = bias ? v[i] + bias[f] : v[i];
        }
        if (f32_off(v[0]) || f32_off(v[1]) || f32_off(v[2]) || f32_off(v[3])) {
#pragma unroll 1
          for (int f = n0 + q * 4; f < min(n0 + q * 4 + 4, N); ++f)
            if (f32_off(C[(size_t)m * ldc + f])) {
              const float u = f32_again(A + (size_t)m * lda, W + (size_t)f * K, K);
              C[(size_t)m * ldc + f] = bias ? u + bias[f] : u;
            }
        }
      }
    }
    buf ^= 1;
    step = 0;
    n0 += (int)gridDim.x * 16;
  }
}

// ------------------------------------------------------------------------------------------------ from 33 rows on
#define F32_LDS __attribute__((address_space(3)))

struct F32Tile {
  const float* a;
  const float* w;
  const float* bias;
  float* c;                                // ranges > 1: the blocks' sums, [blocks][M][N]
  int M, N, K, lda, ldc, m_tiles, n_tiles, ranges;
  int block_k, range_blocks;               // k of a block (a multiple of 64), blocks of a range
};

// Large tiles' products are in assembly, so that a sum stays in its registers (of sums that fill the accumulation registers the
// compiler moves some to and fro, and spills others at the ends of blocks). It then does not see the wait states that belong between a
// product and an ordinary access to its sums, or between a copy of an operand, which it may make ahead of a block, and the product.
__device__ __forceinline__ void f32_term_kept(int t, const F32Parts& w, const F32Parts& a, f32x4_t& c) {
  const bf16x8_t& x = t == 0 ? w.l : t == 2 || t == 3 ? w.m : w.h;
  const bf16x8_t& y = t == 1 ? a.l : t == 2 || t == 4 ? a.m : a.h;
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(x), "v"(y));
}
template <int TN, int TM>
__device__ __forceinline__ void f32_settle(f32x4_t (&acc)[TN][TM]) {
  f32x4_t* p = &acc[0][0];
#pragma unroll
  for (int i = 0; i < TN * TM; i += 4)
    asm volatile("s_nop 15\n\ts_nop 3" : "+a"(p[i]), "+a"(p[i + 1]), "+a"(p[i + 2]), "+a"(p[i + 3]));
}
template <int TN>
__device__ __forceinline__ void f32_ready(const F32Parts (&y)[TN], const F32Parts& x) {
#pragma unroll
  for (int i = 0; i < TN; ++i) asm volatile("s_nop 3" ::"v"(y[i].h), "v"(y[i].m), "v"(y[i].l));
  asm volatile("s_nop 3" ::"v"(x.h), "v"(x.m), "v"(x.l));
}
// The instructions stay in the order that they are written in.
#define F32_ORDER __builtin_amdgcn_sched_barrier(0)

// A workgroup of four waves a tile of 32 TM rows and 128 features and range of k, in 2 x 2 quarters. A step is 32 k of both
// operands: read from memory as floats, in whole lines, two steps ahead, into registers; split, each once a workgroup, and written to
// LDS one step ahead, part by part in tiles of 16 rows in the products' order: the 16 bytes of row r, k 8 q .. + 7 lie at place
// 16 q + r, or r ^ 8 for q 2 and 3; the lanes that write side by side hold pieces of q 0 and 2 of four rows and of q 1 and 3 of the
// four behind them, which fall on all banks. A tile's operands have descriptors of their own, whose ends are those of the
// matrices: rows past them are zeros.
//
// A step's products go row tile by row tile, all four columns' operands in registers and a row tile's read one ahead. The barrier stands
// before the last row tile: there all of stage s has been read and all of stage s + 1 written, so that the next operands are
// read, and the first pieces of stage s + 2 written, behind products that are still to issue. Splitting stands between the
// products as well: a wave issues in order, and has the SIMD to itself but for tiles of 64 rows, of which a CU holds two.
template <int TM, bool CUT>
__global__ void __launch_bounds__(256, TM == 2 ? 2 : 1) gemm_f32_tile_kernel(F32Tile g) {
  constexpr int TN = 4, BM = 32 * TM, BN = 128;
  constexpr bool KEPT = TM >= 6;
  constexpr int PA = BM / 32, PB = BN / 32, P = PA + PB;          // a thread's pieces of a stage: one of every 32 rows
  constexpr int EARLY = P / TM;                                   // of them, written behind the barrier
  constexpr int TILE = 3 * 1024, STAGE = (BM + BN) / 16 * TILE;   // bytes
  constexpr unsigned NOWHERE = 0xFFFFFFF0u;
  __shared__ __attribute__((aligned(1024))) char lds[2 * STAGE];
  // the row tiles of a panel and range of weights follow one another, and each XCD gets a run of tiles
  const long total = (long)g.m_tiles * g.n_tiles * g.ranges, each = (total + RA_XCDS - 1) / RA_XCDS;
  const long at = blockIdx.x / RA_XCDS, tile = blockIdx.x % RA_XCDS * each + at;
  if (at >= each || tile >= total) return;
  const int m0 = (int)(tile % g.m_tiles) * BM;
  const int z = (int)(tile / g.m_tiles % g.ranges), n0 = (int)(tile / g.m_tiles / g.ranges) * BN;
  const int range_k = g.block_k * g.range_blocks, block_steps = g.block_k / F32_BK;
  const int k0 = z * range_k, k1 = min(k0 + range_k, g.K), steps = (k1 - k0 + 63) / 64 * 2;   // pairs, as a block's are
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int a_rows = min(BM, g.M - m0), w_rows = min(BN, g.N - n0);
  const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(g.a + (size_t)m0 * g.lda), 0, (int)(unsigned)(((size_t)(a_rows - 1) * g.lda + g.K) * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(g.w + (size_t)n0 * g.K), 0, (int)(unsigned)((size_t)w_rows * g.K * 4), 0x00020000);
  // piece c (16 bytes, 4 k) of row lr of each 32
  const int c = lane & 7, lr = wave * 8 + ((lane >> 3) & 3) + 4 * ((lane >> 5) ^ ((c >> 1) & 1));
  unsigned off[P];
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const int r = lr + (i < PA ? i : i - PA) * 32;
    off[i] = r < (i < PA ? a_rows : w_rows) ? ((unsigned)r * (unsigned)(i < PA ? g.lda : g.K) + c * 4) * 4u : 0x80000000u;
  }
  F32_LDS char* to[2];
  to[0] = (F32_LDS char*)lds + (lr >> 4) * TILE + (c >> 1) * 256 + (((lr & 15) ^ ((c >> 2) * 8)) * 16) + (c & 1) * 8;
  // stage s waits in held[s % 2] until it is split; behind that its registers are those of stage s + 2
  f32x4_t held[2][P];
  auto load = [&](int s, int i, int set) {
    const unsigned k = (unsigned)(k0 + s * F32_BK);
    const unsigned o = k + c * 4 < (unsigned)k1 ? off[i] + k * 4u : NOWHERE;         // past the range's end: zeros
    held[set][i] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(i < PA ? a_rsrc : w_rsrc, (int)o, 0, 0));
  };
  unsigned part[3][2];
  // a piece's way to LDS in operations of about five instructions: its first and second two floats, the writes, the next load
  constexpr int OPS = 6;
  auto piece = [&](int i, int op, int set, int buf, int next) {
    if (op < 4) {
      f32x4_t& v = held[set][i];
      float a = v[op >> 1 << 1], b = v[(op >> 1 << 1) + 1];
      if ((op & 1) == 0) {
        part[0][op >> 1] = f32_part(a, b);
      } else {
        part[1][op >> 1] = f32_part(a, b);
        part[2][op >> 1] = f32_part(a, b);
      }
      v[op >> 1 << 1] = a;
      v[(op >> 1 << 1) + 1] = b;
    } else if (op == 4) {
      F32_LDS char* d = to[buf] + i * 2 * TILE;
#pragma unroll
      for (int x = 0; x < 3; ++x) *(F32_LDS unsigned long long*)(d + x * 1024) = part[x][0] | (unsigned long long)part[x][1] << 32;
    } else {
      load(next, i, set);
    }
  };
  f32x4_t sum[TN][TM];                       // of the blocks before this one
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) sum[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  const int wm = (wave >> 1) * TM * 16, wn = (wave & 1) * 64;
  const int row = lane & 15, quarter = lane >> 4;
  const F32_LDS char* const from = (F32_LDS char*)lds + quarter * 256 + ((row ^ ((quarter >> 1) * 8)) * 16);
  const F32_LDS char *xs[2] = {from + wm / 16 * TILE}, *ys[2] = {from + (BM + wn) / 16 * TILE};
  // of both buffers, and not known to the compiler as one behind the other: an access holds 16 bits of offset, and it would add the
  // rest to the first one's address each time
  to[1] = to[0] + STAGE;
  xs[1] = xs[0] + STAGE;
  ys[1] = ys[0] + STAGE;
#pragma unroll
  for (int i = 0; i < 2; ++i) asm("" : "+v"(to[i]), "+v"(xs[i]), "+v"(ys[i]));
  auto read = [&](const F32_LDS char* s) {     // the operands of a 16-row tile
    typedef const F32_LDS bf16x8_t part_t;
    return F32Parts{*(part_t*)s, *(part_t*)(s + 1024), *(part_t*)(s + 2048)};
  };
  F32Parts x[2], y[TN];
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int i = 0; i < P; ++i) load(s, i, s);
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int i = 0; i < (s ? EARLY : P); ++i)
#pragma unroll
      for (int op = 0; op < OPS; ++op) piece(i, op, s, s, s + 2);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
  for (int i = 0; i < TN; ++i) y[i] = read(ys[0] + i * TILE);
  x[0] = read(xs[0]);
  const int ld = CUT ? g.N : g.ldc;
  const float* b = CUT ? nullptr : g.bias;
  const bool whole = g.N % 4 == 0 && ld % 4 == 0 && (uintptr_t)g.c % 16 == 0;
  auto step = [&](int s, f32x4_t (&acc)[TN][TM], auto odd) {
    constexpr int buf = odd, MF = TN * F32_TERMS;                 // products of a row tile
    constexpr int LATE = (P - EARLY) * OPS, FIRST = MF * (TM - 1);
    F32_ORDER;
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      if (j == TM - 1) {
        // this wave's pieces of stage s + 1 are written and its reads of stage s done; behind the barrier that is so of all waves
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        F32_ORDER;
      }
#pragma unroll
      for (int m = 0; m < MF; ++m) {
        // all four columns in turn; in the last row tile two, as their operands are then free for the next stage's in the middle and
        // at the end, and so in the first, where the other two are on their way
        const bool two = j == 0 || j == TM - 1;
        const int i = two ? m / (2 * F32_TERMS) * 2 + m % 2 : m % TN, t = two ? m % (2 * F32_TERMS) / 2 : m / TN;
        if constexpr (KEPT) f32_term_kept(t, y[i], x[j & 1], acc[i][j]);
        else acc[i][j] = f32_term(t, y[i], x[j & 1], acc[i][j]);
        F32_ORDER;
        if (j < TM - 1) {
          const int at = j * MF + m;
          if (m == 1) { x[(j + 1) & 1] = read(xs[buf] + (j + 1) * TILE); F32_ORDER; }
#pragma unroll
          for (int o = at * LATE / FIRST; o < (at + 1) * LATE / FIRST; ++o) {
            piece(EARLY + o / OPS, o % OPS, buf ^ 1, buf ^ 1, s + 3);
            F32_ORDER;
          }
        } else {
          if (m == 1) { x[0] = read(xs[buf ^ 1]); F32_ORDER; }
          if (m == MF / 2) {
            y[0] = read(ys[buf ^ 1]); F32_ORDER;
            y[1] = read(ys[buf ^ 1] + TILE); F32_ORDER;
          }
#pragma unroll
          for (int o = m * EARLY * OPS / MF; o < (m + 1) * EARLY * OPS / MF; ++o) {
            piece(o / OPS, o % OPS, buf, buf, s + 4);
            F32_ORDER;
          }
        }
      }
    }
    y[2] = read(ys[buf ^ 1] + 2 * TILE); F32_ORDER;
    y[3] = read(ys[buf ^ 1] + 3 * TILE); F32_ORDER;
  };
  for (int s = 0, block = z * g.range_blocks; s < steps; ++block) {
    f32x4_t acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    if constexpr (KEPT) {
      f32_settle(acc);
      f32_ready(y, x[0]);
    }
    for (const int end = min(s + block_steps, steps); s < end; s += 2) {
      step(s, acc, std::integral_constant<int, 0>{});
      step(s + 1, acc, std::integral_constant<int, 1>{});
    }
    if constexpr (KEPT) f32_settle(acc);
    if (!CUT) {                              // the blocks are added here, as the adding kernel does it
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) sum[i][j][e] += acc[i][j][e];
    }
    if (CUT || s == steps) {
      // a lane holds row lane % 16 of the tile, features 4 (lane / 16) .. + 3
      float* out = CUT ? g.c + (size_t)block * g.M * g.N : g.c;
      int m_at = m0 + wm + row;
      asm volatile("" : "+v"(m_at));         // addresses are worked out here and not kept in registers through the steps
      bool off = false;
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        const int m = m_at + j * 16;
        if (m >= g.M) continue;
#pragma unroll
        for (int i = 0; i < TN; ++i) {
          const int n = n0 + wn + i * 16 + quarter * 4;
          if (n >= g.N) continue;
          f32x4_t v;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[e] = CUT ? acc[i][j][e] : sum[i][j][e];
            off |= f32_off(v[e]);
            if (b && n + e < g.N) v[e] += b[n + e];
          }
          if (whole) {
            *(f32x4_t*)(out + (size_t)m * ld + n) = v;
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (n + e < g.N) out[(size_t)m * ld + n + e] = v[e];
          }
        }
      }
      if (!CUT && off) {
#pragma unroll 1
        for (int m = m_at; m < min(m_at + TM * 16, g.M); m += 16)
#pragma unroll 1
          for (int i = 0; i < TN * 4; ++i) {
            const int n = n0 + wn + (i >> 2) * 16 + quarter * 4 + (i & 3);
            if (n >= g.N || !f32_off(out[(size_t)m * ld + n])) continue;
            const float u = f32_again(g.a + (size_t)m * g.lda, g.w + (size_t)n * g.K, g.K);
            out[(size_t)m * ld + n] = b ? u + b[n] : u;
          }
      }
    }
  }
}

// C = the blocks' sums added in their order (+ bias): a workgroup takes 1024 features of a row, four a thread, read 16 bytes at
// a time where rows allow it. It is bound by reading the planes.
__global__ void __launch_bounds__(256)
gemm_f32_add_kernel(F32Tile g, int planes, float* __restrict__ C, const float* __restrict__ bias, bool whole) {
  const int n = (blockIdx.y * 256 + threadIdx.x) * 4;
  if (n >= g.N) return;
  const size_t m = blockIdx.x, size = (size_t)g.M * g.N;
  const float* p = g.c + m * g.N + n;
  float* c = C + m * g.ldc + n;
  f32x4_t v = {0.f, 0.f, 0.f, 0.f};
  if (whole) {
    v = *(const f32x4_t*)p;
    for (int r = 1; r < planes; ++r) v += *(const f32x4_t*)(p + r * size);
  } else {
    for (int e = 0; e < 4 && n + e < g.N; ++e) {
      v[e] = p[e];
      for (int r = 1; r < planes; ++r) v[e] += p[r * size + e];
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (n + e >= g.N) break;
    if (f32_off(v[e])) v[e] = f32_again(g.a + m * g.lda, g.w + (size_t)(n + e) * g.K, g.K);
    if (bias) v[e] += bias[n + e];
  }
  if (whole) *(f32x4_t*)c = v;
  else
    for (int e = 0; e < 4 && n + e < g.N; ++e) c[e] = v[e];
}

// The tile kernel's plan: rows of a tile, and how many of K's blocks a workgroup takes (it adds them in its registers; several ranges of
// blocks go to planes that the adding kernel adds). The price is a CU's share of the workgroups at what a step takes in tiles of so
// many rows (measured), and the planes written and read again.
struct TilePlan {
  int rows, blocks, block_k, range_blocks, ranges;
};
TilePlan tile_plan(int M, int N, int K) {
  const long cus = ra_cu_count();
  // us a step of 32 k: of one workgroup on a CU, and of two, side by side where there is room (tiles of 64 rows), else in turn
  const struct { int rows; double one, two; } forms[] = {{64, 1.05, 1.42}, {128, 1.48, 2.96}, {192, 1.93, 3.86}, {256, 2.53, 5.06}};
  const KBlocks kb = k_blocks(K);
  TilePlan best = {};
  double best_us = 0.0;
  for (const auto& f : forms) {
    const long tiles = (long)((M + f.rows - 1) / f.rows) * ((N + 127) / 128);
    for (int take = kb.n; take >= 1; --take) {
      const int ranges = (kb.n + take - 1) / take;
      const long load = (tiles * ranges + cus - 1) / cus;
      double us = (load / 2 * f.two + load % 2 * f.one) * take * kb.k / F32_BK + load;
      if (ranges > 1) us += 3.0 + (double)kb.n * M * N * 8.0 / 5e6;
      if (best.rows == 0 || us < best_us) {
        best = {f.rows, kb.n, kb.k, take, ranges};
        best_us = us;
      }
    }
  }
  return best;
}

template <int TM>
void tile_launch(const F32Tile& g, bool cut, unsigned blocks, hipStream_t stream) {
  if (cut) gemm_f32_tile_kernel<TM, true><<<blocks, 256, 0, stream>>>(g);
  else gemm_f32_tile_kernel<TM, false><<<blocks, 256, 0, stream>>>(g);
}

int tile_go(const TilePlan& p, const float* A, const float* W, const float* bias, float* C, int M, int N, int K, int lda,
            int ldc, float* scratch, hipStream_t stream) {
  const bool cut = p.ranges > 1;
  F32Tile g = {A, W, bias, cut ? scratch : C, M, N, K, lda, ldc, (M + p.rows - 1) / p.rows, (N + 127) / 128, p.ranges,
               p.block_k, p.range_blocks};
  const long total = (long)g.m_tiles * g.n_tiles * g.ranges, blocks = (total + RA_XCDS - 1) / RA_XCDS * RA_XCDS;
  RA_CHECK(blocks <= 0x7FFFFFFFL, "gemm_f32: [%d, %d] in one launch", M, N);
  if (p.rows == 64) tile_launch<2>(g, cut, (unsigned)blocks, stream);
  else if (p.rows == 128) tile_launch<4>(g, cut, (unsigned)blocks, stream);
  else if (p.rows == 192) tile_launch<6>(g, cut, (unsigned)blocks, stream);
  else tile_launch<8>(g, cut, (unsigned)blocks, stream);
  RA_LAUNCH_CHECK("gemm_f32");
  if (cut) {
    const bool whole = N % 4 == 0 && ldc % 4 == 0 && (uintptr_t)C % 16 == 0 && (uintptr_t)scratch % 16 == 0;
    gemm_f32_add_kernel<<<dim3(M, (N + 1023) / 1024), 256, 0, stream>>>(g, p.blocks, C, bias, whole);
    RA_LAUNCH_CHECK("gemm_f32 (ranges)");
  }
  return 0;
}

}  // namespace

#define F32_STREAM_ROWS 32

extern "C" int ra_gemm_f32_supports(const void* A, const void* W, int K, int lda) {
  // Sums of fewer than 512 k stay in the plain kernel's one chain: they belong to layers so small that a launch is most of
  // either's time, and a read-out that divides by a sum with cancellation shows the order of theirs a thousandfold. A tile's
  // rows are addressed from its first one in 31 bits.
  return K >= 512 && K % 4 == 0 && lda < (1 << 21) && K < (1 << 21) && ra_rows_16b(A, lda, 4) && ra_rows_16b(W, K, 4);
}

extern "C" long ra_gemm_f32_scratch(int M, int N, int K) {
  if (M <= F32_STREAM_ROWS) return 0;
  const TilePlan p = tile_plan(M, N, K);
  return p.ranges > 1 ? (long)p.blocks * M * N : 0;
}

extern "C" int ra_gemm_f32(const float* A, const float* W, const float* bias, float* C, int M, int N, int K, int lda,
                           int ldc, float* scratch, long scratch_floats, hipStream_t stream) {
  RA_CHECK(M > 0 && N > 0 && K > 0, "gemm_f32: empty product (%d, %d, %d)", M, N, K);
  RA_CHECK(lda >= K && ldc >= N, "gemm_f32: row strides (%d, %d) below the row lengths (%d, %d)", lda, ldc, K, N);
  RA_CHECK(ra_gemm_f32_supports(A, W, K, lda), "gemm_f32: rows of %d (stride %d) are not 16-byte pieces", K, lda);
  if (M <= F32_STREAM_ROWS) {
    // a descriptor covers less than 4 GiB of weights: a larger matrix goes in runs of features
    const KBlocks kb = k_blocks(K);
    const long most = 0xFFFFFF00L / ((long)K * 4) / 16 * 16;
    RA_CHECK(most > 0 && ((long)(M - 1) * lda + K) * 4 < 0xFFFFFF00L, "gemm_f32: rows of %d (stride %d) are too long", K, lda);
    for (long n0 = 0; n0 < N; n0 += most) {
      const int n = (int)(N - n0 < most ? N - n0 : most);
      const int tiles = (n + 15) / 16, cus = ra_cu_count();
      const float *w = W + (size_t)n0 * K, *b = bias ? bias + n0 : nullptr;
#define RA_GO(ROWS) \
  gemm_f32_stream_kernel<ROWS><<<grid < tiles ? grid : tiles, kb.n * RA_WAVE, F32Stream<ROWS>::lds(kb.n), stream>>>( \
      A, w, b, C + n0, M, n, K, lda, ldc, kb.k)
      // as many workgroups as the registers hold, 16 waves a CU
      const int grid = 16 / kb.n * cus;
      if (M > 16) RA_GO(32);
      else if (M > 8) RA_GO(16);
      else RA_GO(8);
#undef RA_GO
      RA_LAUNCH_CHECK("gemm_f32");
    }
    return 0;
  }
  const TilePlan p = tile_plan(M, N, K);
  RA_CHECK(p.ranges == 1 || (scratch && scratch_floats >= (long)p.blocks * M * N), "gemm_f32: scratch of %ld floats, needs %ld",
           scratch_floats, (long)p.blocks * M * N);
  return tile_go(p, A, W, bias, C, M, N, K, lda, ldc, scratch, stream);
}
