// Matrix products of the 32-bit path, C[M,N] = A[M,K] . W[N,K]^T (+ bias[N]), on the bfloat16 matrix cores, to float precision.
//
// A float is the sum of three bfloat16 numbers: its value rounded, what that leaves rounded, and the rest (Henry, Tang and Heinecke,
// "Leveraging the bfloat16 Artificial Intelligence Datatype for Higher-Precision Computations", 2019). Split 2^24 times as large it is so
// exactly down to the last subnormal bit. Of the nine products of the parts the six largest are summed, in float: the largest in a sum
// of its own, the five others in a second one, 2^8 times smaller. What this keeps, U being 2^-24:
//   one product   what is left out of it is below 1.001 U of it (2 2^-8 2^-17 and 2^-34; 0.99 for the mantissa 1 + 2^-8 - 2^-17), and one
//                 rounding, below U: measured up to 0.94 of a last place, a float product 0.50;
//   a sum         is rounded once for every eight k (a product of 32 k adds them eight at a time), where the float matrix cores round for every
//                 one. Over normal random numbers the error against 64 bits is 1.35e-7 of the result's norm at K 2560 (float matrix cores
//                 4.08e-7), 1.39e-7 at 4096 (4.09e-7) and 2.12e-7 at 9728 (6.27e-7). With all six products in one sum it was 3.43, 3.47
//                 and 5.59e-7 and had a mean of -0.6, -0.7 and -1.7e-7, for these cores cut what lies below 2^-31 of the largest
//                 that they add towards minus infinity, and did so six times for every eight k; now the mean is below 1e-9;
//   magnitudes    all floats; rows of 2^-140 are as near as others. Sums past 2^80 and what is not finite are worked out again from the floats.
//
// Up to 32 rows (gemm_f32_stream_kernel) the product is bound by reading the weights once. A workgroup has 16 features, its
// waves share K out and add their sums through LDS in a fixed order. The weights go by way of a piece of LDS of each wave's own:
// loaded in the products' order a load is 64 bytes of each of 16 rows, half a line each, and takes twice the time of whole lines.
// Splitting is issue time beside the loads' waits: with the next loads asked for behind it 15 % slower, with the rows split by every
// lane that multiplies them 10 %. Weights from memory, float matrix cores / here, us: 4 rows 6144 x 2560 19.7 / 17.4, 2560 x 4096
// 15.8 / 14.3, 19456 x 2560 41.5 / 39.2, 2560 x 9728 29.3 / 26.2; 12 rows 21.8 / 20.9, 17.5 / 16.1, 46.9 / 45.0, 33.4 / 31.3; 32 rows
// 37.5 / 33.0, 28.0 / 24.8, 80 / 73.5, 56.2 / 50.8. Where the stream is at memory rate splitting costs what it takes: 4 rows 151936 x 2560
// 264 / 270 (5.8 TB/s), 12 rows 324 / 329, 32 rows 554 / 507; 20 or 24 waves a CU in place of 16 are no faster there, and a tenth
// slower from 12 rows on. Runs of 64 k, or three or four in flight, are slower.
//
// From 33 rows on (gemm_f32_tile_kernel) tiles of both operands go through LDS, split on the way. Six bfloat16 products take 96 cycles
// of a matrix core where the float ones take 256. What bounds them is the chip's power (the clock is 1.93 GHz; on zeros 2.4 and a quarter
// faster) and issue: beside each product stand one and a half other vector instructions. In a loop over other weights, float matrix
// cores / here, us: 1119 x 19456 x 2560 875 / 606 (184 TFLOP/s), 1119 x 2560 x 9728 470 / 317, 2048 x 19456 x 2560 1510 / 1052, 300 x 6144 x 2560
// 96 / 68, 64 x 19456 x 2560 65 / 59. One wave a SIMD with tiles of 256 rows (one sum; with two they do not fit its registers) took 602, 303, 995,
// 85 and 61; all eight products but the smallest 774 for the first where six took 677. Dot products with (-1, 0) to take a part off: tiles
// 3 to 8 % slower, streams of 12 rows 1.5 % faster, of 4 rows no different.
#include <type_traits>

#include "common.h"
#include "reinfer_hip.h"

namespace {

// ------------------------------------------------------------------------------------------------ a float in three parts
struct F32Parts {
  bf16x8_t h, m, l;
};
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
// Two floats rounded, as the low and the high half of a word (the empty statement has the compiler take the halves from the word: left to
// itself it converts each float once more for that), and what that leaves of them.
__device__ __forceinline__ unsigned f32_pack(float a, float b) {
  unsigned u = __builtin_bit_cast(unsigned, (bf16x2_t){(bf16_t)a, (bf16_t)b});
  asm("" : "+v"(u));
  return u;
}
__device__ __forceinline__ void f32_rest(unsigned u, float& a, float& b) {
  a -= __builtin_bit_cast(float, u << 16);
  b -= __builtin_bit_cast(float, u & 0xFFFF0000u);
}
__device__ __forceinline__ unsigned f32_part(float& a, float& b) {
  const unsigned u = f32_pack(a, b);
  f32_rest(u, a, b);
  return u;
}
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
// Floats are split 2^24 times as large, so that the last bit of the smallest is no part's below what bfloat16 holds; a sum is 2^48 times as
// large, then.
#define F32_SCALE 0x1p24f
__device__ __forceinline__ F32Parts f32_split(f32x4_t a, f32x4_t b) {
  float v[8];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] = a[e] * F32_SCALE;
    v[4 + e] = b[e] * F32_SCALE;
  }
  u32x4_t p[3];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) p[i][e] = f32_part(v[2 * e], v[2 * e + 1]);
  return {__builtin_bit_cast(bf16x8_t, p[0]), __builtin_bit_cast(bf16x8_t, p[1]), __builtin_bit_cast(bf16x8_t, p[2])};
}
// Term t of the product of two floats in parts, the smallest first: every kernel adds them in this order. The largest has a sum of its own;
// the others' sum is some 2^8 times smaller, and so are its roundings.
#define F32_TERMS 6
__device__ __forceinline__ f32x4_t f32_term(int t, const F32Parts& w, const F32Parts& a, f32x4_t c) {
  const bf16x8_t& x = t == 0 ? w.l : t == 2 || t == 3 ? w.m : w.h;
  const bf16x8_t& y = t == 1 ? a.l : t == 2 || t == 4 ? a.m : a.h;
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, c, 0, 0, 0);
}
struct F32Sum {
  f32x4_t h, s;                            // of the largest term, of the others
};
__device__ __forceinline__ void f32_add_term(int t, const F32Parts& w, const F32Parts& a, F32Sum& c) {
  if (t == F32_TERMS - 1) c.h = f32_term(t, w, a, c.h);
  else c.s = f32_term(t, w, a, c.s);
}
// A block's sum; each operation is rounded by itself wherever it stands.
__device__ __forceinline__ f32x4_t f32_block(const F32Sum& c) {
#pragma clang fp contract(off)
  f32x4_t v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = (c.h[e] + c.s[e]) * (1.f / F32_SCALE / F32_SCALE);
  return v;
}
__device__ __forceinline__ f32x4_t f32_plus(f32x4_t a, f32x4_t b) {
#pragma clang fp contract(off)
#pragma unroll
  for (int e = 0; e < 4; ++e) a[e] += b[e];
  return a;
}

// The parts of an infinity and of a float that is one 2^24 times as large are no numbers: a block's sum that is not finite is worked out
// again from the floats, on the float matrix cores, by a wave for 16 rows and 16 features: four products for every 16 k, of k 0, 4, 8, 12,
// then 1, 5, 9, 13, .... a and w: the first row and feature, of `rows` and `features` that there are.
// With a NaN in one row a product takes, us (without): 8 rows 2560 x 9728 35 (24), 300 x 6144 x 2560 168 (68), 1119 x 6144 x 2560 361 (196); 300
// rows of NaN 391.
__device__ __forceinline__ bool f32_off(f32x4_t v) {
  return !(fabsf(v[0]) <= 3.402823466e38f && fabsf(v[1]) <= 3.402823466e38f && fabsf(v[2]) <= 3.402823466e38f && fabsf(v[3]) <= 3.402823466e38f);
}
__device__ __forceinline__ f32x4_t f32_again(const float* a, int lda, int rows, const float* w, int ldw, int features, int k0, int k1,
                                             f32x4_t v) {
  const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
  const float *x = a + (size_t)min(r, rows - 1) * lda, *y = w + (size_t)min(r, features - 1) * ldw;
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  f32x4_t c = zero;
  for (int k = k0; k < k1; k += 64) {
    f32x4_t f[4], g[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int at = k + i * 16 + q * 4;
      f[i] = at < k1 ? *(const f32x4_t*)(y + at) : zero;
      g[i] = at < k1 ? *(const f32x4_t*)(x + at) : zero;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(f[i / 4][i % 4], g[i / 4][i % 4], c, 0, 0, 0);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = fabsf(v[e]) <= 3.402823466e38f ? v[e] : c[e];
  return v;
}

// ------------------------------------------------------------------------------------------------ the order of the sums
// K is summed in up to eight blocks of at least 512 k, whose number and length follow from K alone. A block is two chains of
// 16x16x32 products over its pieces of 32 k, one and five a piece, that are added at its end; where that is not finite, its sum from the
// floats. The blocks' sums are added in their order, then the bias. Both kernels keep this order, so a row's result does not depend on
// how many rows stand beside it: a request's 32-bit results are the same bits alone and in any step.
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
template <int ROWS, bool STREAM>
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
      w[d][i] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, off, 0, STREAM ? RA_STREAM : 0));
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
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  F32Sum acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = {zero, zero};
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
          float v[4] = {a[d][i][0] * F32_SCALE, a[d][i][1] * F32_SCALE, a[d][i][2] * F32_SCALE, a[d][i][3] * F32_SCALE};
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
        for (int t = 0; t < MT; ++t) f32_add_term(e, y, x[t], acc[t]);
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
      f32x4_t v = f32_block(acc[t]);
      if (__any(f32_off(v))) v = f32_again(A + (size_t)t * 16 * lda, lda, M - t * 16, W + (size_t)n0 * K, K, N - n0, k0, k1, v);
      sums[((buf * waves + wave) * MT + t) * RA_WAVE + lane] = v;
      acc[t] = {zero, zero};
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    for (int t = wave; t < MT; t += waves) {
      f32x4_t v = zero;
#pragma unroll
      for (int x = 0; x < 8; ++x)
        if (x < waves) v = f32_plus(v, sums[((buf * waves + x) * MT + t) * RA_WAVE + lane]);
      const int m = t * 16 + r;
      if (m < M) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int f = n0 + q * 4 + i;
          if (f < N) C[(size_t)m * ldc + f] = bias ? v[i] + bias[f] : v[i];
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

// The instructions stay in the order that they are written in.
#define F32_ORDER __builtin_amdgcn_sched_barrier(0)

// Four neighbouring features of a row, n the first of N.
__device__ __forceinline__ void f32_store(float* to, f32x4_t v, const float* bias, int n, int N, bool whole) {
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (bias && n + e < N) v[e] += bias[n + e];
  if (whole) {
    *(f32x4_t*)to = v;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) to[e] = v[e];
  }
}
// 16 rows and features by a wave, straight from memory: blocks first to past, each as the tiles have it, or from the floats where that
// is not finite, added in their order. For tiles that hold a result that is not finite.
__device__ __forceinline__ void f32_write_again(const F32Tile& g, int m0, int n0, int first, int past, float* out, int ld,
                                                const float* bias, bool whole) {
  const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4, rows = g.M - m0, features = g.N - n0;
  const float *a = g.a + (size_t)m0 * g.lda, *w = g.w + (size_t)n0 * g.K;
  const float *x = a + (size_t)min(r, rows - 1) * g.lda, *y = w + (size_t)min(r, features - 1) * g.K;
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  f32x4_t sum = zero;
  for (int block = first; block < past; ++block) {
    const int k0 = block * g.block_k, k1 = min(k0 + g.block_k, g.K);
    F32Sum acc = {zero, zero};
    for (int k = k0; k < k1; k += 64) {
      f32x4_t f[4], h[4];                  // 8 k of each of two pieces
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int at = k + i / 2 * 32 + q * 8 + i % 2 * 4;
        f[i] = at < k1 ? *(const f32x4_t*)(y + at) : zero;
        h[i] = at < k1 ? *(const f32x4_t*)(x + at) : zero;
      }
#pragma unroll
      for (int i = 0; i < 4; i += 2) {
        const F32Parts wp = f32_split(f[i], f[i + 1]), ap = f32_split(h[i], h[i + 1]);
#pragma unroll
        for (int t = 0; t < F32_TERMS; ++t) f32_add_term(t, wp, ap, acc);
      }
    }
    f32x4_t v = f32_block(acc);
    if (__any(f32_off(v))) v = f32_again(a, g.lda, rows, w, g.K, features, k0, k1, v);
    sum = f32_plus(sum, v);
  }
  if (r < rows && q * 4 < features) f32_store(out + (size_t)(m0 + r) * ld + n0 + q * 4, sum, bias, n0 + q * 4, g.N, whole);
}

// A workgroup of WM x WN waves a tile of 32 WM rows and 128 features and range of k; a wave 32 rows and 16 TN features of it. A step is 32 k of
// both operands: read from memory as floats, in whole lines, two steps ahead, into registers; split, each once a workgroup, and written to
// LDS one step ahead, part by part in tiles of 16 rows in the products' order: the 16 bytes of row r, k 8 q .. + 7 lie at place
// 16 q + r, or r ^ 8 for q 2 and 3; the lanes that write side by side hold pieces of q 0 and 2 of four rows and of q 1 and 3 of the
// four behind them. A tile's operands have descriptors of their own, whose ends are those of the matrices: rows past them are zeros.
//
// A step's products go row tile by row tile, two columns in turn, with all columns' operands in registers. The barrier stands between the
// row tiles: there all of stage s has been read and all of stage s + 1 written (a few products before: 4 % of the time), so that the next
// operands are read, and the first pieces of stage s + 2 written, behind products that are still to issue. Splitting stands between the
// products as well, two or three instructions at a time. Two waves a SIMD fill each other's gaps: one, with tiles of 128 rows in quarters
// of 64 and four columns in turn, took 880 us where two take 774 (eight products, 1119 x 19456 x 2560).
template <int WM, int WN, int TN, bool CUT>
__global__ void __launch_bounds__(WM * WN * RA_WAVE, 2) gemm_f32_tile_kernel(F32Tile g) {
  constexpr int TM = 2, BM = WM * TM * 16, BN = WN * TN * 16;
  constexpr int ROWS = WM * WN * 8, PA = BM / ROWS, PB = BN / ROWS, P = PA + PB;     // a thread's pieces of a stage: one of every so many rows
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
  // piece c (16 bytes, 4 k) of row lr of each ROWS
  const int c = lane & 7, lr = wave * 8 + ((lane >> 3) & 3) + 4 * ((lane >> 5) ^ ((c >> 1) & 1));
  unsigned off[P];
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const int r = lr + (i < PA ? i : i - PA) * ROWS;
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
  // a piece's way to LDS in operations of about three instructions, which is what there is room for beside a product: its first and second
  // two floats, the writes, the next load
  constexpr int OPS = 10;
  auto piece = [&](int i, int op, int set, int buf, int next) {
    if (op < 8) {
      const int two = op >> 2;
      f32x4_t& v = held[set][i];
      float a = v[2 * two], b = v[2 * two + 1];
      if (op % 4 == 0) {
        a *= F32_SCALE;
        b *= F32_SCALE;
        part[0][two] = f32_pack(a, b);
      } else if (op % 4 == 1) {
        f32_rest(part[0][two], a, b);
      } else if (op % 4 == 2) {
        part[1][two] = f32_pack(a, b);
      } else {
        f32_rest(part[1][two], a, b);
        part[2][two] = f32_pack(a, b);
      }
      v[2 * two] = a;
      v[2 * two + 1] = b;
    } else if (op == 8) {
      F32_LDS char* d = to[buf] + i * (ROWS / 16) * TILE;
#pragma unroll
      for (int x = 0; x < 3; ++x) *(F32_LDS unsigned long long*)(d + x * 1024) = part[x][0] | (unsigned long long)part[x][1] << 32;
    } else {
      load(next, i, set);
    }
  };
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  f32x4_t sum[TN][TM];                       // of the blocks before this one
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) sum[i][j] = zero;
  const int wm = wave / WN * TM * 16, wn = wave % WN * TN * 16;
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
  auto step = [&](int s, F32Sum (&acc)[TN][TM], auto odd) {
    constexpr int buf = odd, MF = TN * F32_TERMS;                 // of a row tile
    // the last write of stage s + 1 some products before the barrier, which waits for it
    constexpr int LATE = (P - EARLY) * OPS, FIRST = MF * (TM - 1) - (TN == 4 ? 6 : 2);
    F32_ORDER;
#pragma unroll
    for (int u = 0; u < TM; ++u) {
      if (u == TM - 1) {
        // this wave's pieces of stage s + 1 are written and its reads of stage s done; behind the barrier that is so of all waves
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        F32_ORDER;
      }
#pragma unroll
      for (int m = 0; m < MF; ++m) {
        const int i = m / (2 * F32_TERMS) * 2 + m % 2;
        f32_add_term(m % (2 * F32_TERMS) / 2, y[i], x[u], acc[i][u]);
        F32_ORDER;
        if (u < TM - 1) {
          const int at = u * MF + m;
          if (m == 1) { x[1] = read(xs[buf] + TILE); F32_ORDER; }
#pragma unroll
          for (int o = at * LATE / FIRST; o < LATE && o < (at + 1) * LATE / FIRST; ++o) {
            piece(EARLY + o / OPS, o % OPS, buf ^ 1, buf ^ 1, s + 3);
            F32_ORDER;
          }
        } else {
          if (m == 1) { x[0] = read(xs[buf ^ 1]); F32_ORDER; }
          if (TN == 4 && m == MF / 2) {
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
#pragma unroll
    for (int i = TN - 2; i < TN; ++i) { y[i] = read(ys[buf ^ 1] + i * TILE); F32_ORDER; }
  };
  for (int s = 0, block = z * g.range_blocks; s < steps; ++block) {
    F32Sum acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) acc[i][j] = {zero, zero};
    for (const int end = min(s + block_steps, steps); s < end; s += 2) {
      step(s, acc, std::integral_constant<int, 0>{});
      step(s + 1, acc, std::integral_constant<int, 1>{});
    }
    if (!CUT) {                              // the blocks are added here, as the adding kernel does it
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) sum[i][j] = f32_plus(sum[i][j], f32_block(acc[i][j]));
    }
    if (CUT || s == steps) {
      // a lane holds row lane % 16 of the tile, features 4 (lane / 16) .. + 3
      float* out = CUT ? g.c + (size_t)block * g.M * g.N : g.c;
      int m_at = m0 + wm + row;
      asm volatile("" : "+v"(m_at));         // addresses are worked out here and not kept in registers through the steps
      unsigned off = 0;                      // a bit for 16 rows and features that hold a result that is not finite
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        const int m = m_at + j * 16;
        if (m >= g.M) continue;
#pragma unroll
        for (int i = 0; i < TN; ++i) {
          const int n = n0 + wn + i * 16 + quarter * 4;
          if (n >= g.N) continue;
          f32x4_t v = CUT ? f32_block(acc[i][j]) : sum[i][j];
          off |= (unsigned)f32_off(v) << (j * TN + i);
          f32_store(out + (size_t)m * ld + n, v, b, n, g.N, whole);
        }
      }
      if (__any(off != 0)) {
        const int first = CUT ? block : 0, past = CUT ? block + 1 : (g.K + g.block_k - 1) / g.block_k;
#pragma unroll 1
        for (int j = 0; j < TM * TN; ++j)
          if (__any(off >> j & 1))
            f32_write_again(g, m0 + wm + j / TN * 16, n0 + wn + j % TN * 16, first, past, out, ld, b, whole);
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
  f32x4_t v = {0.f, 0.f, 0.f, 0.f};
  for (int r = 0; r < planes; ++r) {
    f32x4_t x = {0.f, 0.f, 0.f, 0.f};
    if (whole) x = *(const f32x4_t*)(p + r * size);
    else
      for (int e = 0; e < 4 && n + e < g.N; ++e) x[e] = p[r * size + e];
    v = f32_plus(v, x);
  }
  f32_store(C + m * g.ldc + n, v, bias, n, g.N, whole);
}

// The tile kernel's plan: the form of a tile, and how many of K's blocks a workgroup takes (it adds them in its registers; several ranges of
// blocks go to planes that the adding kernel adds). The price is a CU's share of the workgroups at what a step of 32 k takes in
// tiles of that form and a start of some 4 us (measured), and the planes written and read again.
struct TilePlan {
  int form, blocks, block_k, range_blocks, ranges;
};
struct TileForm {
  int rows;
  double one, two;                         // us a step: of one workgroup on a CU, and of two, side by side or in turn
  bool beside;
};
// 64 rows by eight waves are ahead while each CU has one tile, by four, two of them on a CU, from two tiles on: 64 x 2560 x 9728 41.5 / 48.1 us,
// 160 x 6144 x 2560 55.1 / 52.9, 64 x 19456 x 2560 66.6 / 61; 128 rows from there on where they are there: 100 x 19456 x 2560 105 / 97.5
// and 91, 300 x 2560 x 9728 - / 125 and 112.
constexpr TileForm tile_forms[] = {{64, 0.85, 1.70, false}, {64, 1.03, 1.60, true}, {128, 1.38, 2.76, false}};
TilePlan tile_plan(int M, int N, int K) {
  const long cus = ra_cu_count();
  const KBlocks kb = k_blocks(K);
  TilePlan best = {};
  double best_us = -1.0;
  for (int form = 0; form < 3; ++form) {
    const TileForm& f = tile_forms[form];
    const long tiles = (long)((M + f.rows - 1) / f.rows) * ((N + 127) / 128);
    for (int take = kb.n; take >= 1; --take) {
      const int ranges = (kb.n + take - 1) / take;
      const long load = (tiles * ranges + cus - 1) / cus;
      double us = (load / 2 * f.two + load % 2 * f.one) * take * kb.k / F32_BK + 4.0 * (f.beside ? (load + 1) / 2 : load);
      if (ranges > 1) us += 3.0 + (double)kb.n * M * N * 8.0 / 1e7;
      if (best_us < 0.0 || us < best_us) {
        best = {form, kb.n, kb.k, take, ranges};
        best_us = us;
      }
    }
  }
  return best;
}

template <int WM, int WN, int TN>
void tile_launch(const F32Tile& g, bool cut, unsigned blocks, hipStream_t stream) {
  if (cut) gemm_f32_tile_kernel<WM, WN, TN, true><<<blocks, WM * WN * RA_WAVE, 0, stream>>>(g);
  else gemm_f32_tile_kernel<WM, WN, TN, false><<<blocks, WM * WN * RA_WAVE, 0, stream>>>(g);
}

int tile_go(const TilePlan& p, const float* A, const float* W, const float* bias, float* C, int M, int N, int K, int lda,
            int ldc, float* scratch, hipStream_t stream) {
  const bool cut = p.ranges > 1;
  const int rows = tile_forms[p.form].rows;
  F32Tile g = {A, W, bias, cut ? scratch : C, M, N, K, lda, ldc, (M + rows - 1) / rows, (N + 127) / 128, p.ranges,
               p.block_k, p.range_blocks};
  const long total = (long)g.m_tiles * g.n_tiles * g.ranges, blocks = (total + RA_XCDS - 1) / RA_XCDS * RA_XCDS;
  RA_CHECK(blocks <= 0x7FFFFFFFL, "gemm_f32: [%d, %d] in one launch", M, N);
  if (p.form == 0) tile_launch<2, 4, 2>(g, cut, (unsigned)blocks, stream);
  else if (p.form == 1) tile_launch<2, 2, 4>(g, cut, (unsigned)blocks, stream);
  else tile_launch<4, 2, 4>(g, cut, (unsigned)blocks, stream);
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
                           int ldc, float* scratch, long scratch_floats, int keep, hipStream_t stream) {
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
  do {                                                                                                                               \
    if (past) gemm_f32_stream_kernel<ROWS, true><<<grid < tiles ? grid : tiles, kb.n * RA_WAVE, F32Stream<ROWS>::lds(kb.n), stream>>>( \
        A, w, b, C + n0, M, n, K, lda, ldc, kb.k);                                                                                   \
    else gemm_f32_stream_kernel<ROWS, false><<<grid < tiles ? grid : tiles, kb.n * RA_WAVE, F32Stream<ROWS>::lds(kb.n), stream>>>(    \
        A, w, b, C + n0, M, n, K, lda, ldc, kb.k);                                                                                   \
  } while (0)
      const bool past = ra_streams((size_t)N * K * sizeof(float), keep);
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
