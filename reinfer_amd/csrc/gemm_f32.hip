// Matrix products of the 32-bit path, C[M,N] = A[M,K] . W[N,K]^T (+ bias[N]), on the float matrix cores: the products are
// full float ones and the sums are float, as in gemm_plain.hip, which keeps the rows that 16-byte accesses cannot read.
//
// An operand of the 16x16x4 and 32x32x2 products is one float a lane at (row, k slot). Which k a slot stands for is free as
// long as both operands agree, so a lane reads four neighbouring k with one 16-byte access and the four products that
// follow take one element of it each.
//
// Up to 32 rows (gemm_f32_stream_kernel) the product is bound by reading the weights once. A workgroup has 16 features, its
// waves share K out and add their sums through LDS in a fixed order; both operands go from memory to the matrix cores
// without LDS. At 4 rows 19456 x 2560 takes 41 us (4.8 TB/s) and 151936 x 2560 281 us (5.5 TB/s), where the plain kernel
// took 406 us for the first; with more rows the activations, which every workgroup reads again, cost as much as the weights
// (19456 x 2560 at 32 rows 96 us, as much as the other kernel at 33).
//
// From 33 rows on (gemm_f32_tile_kernel) tiles of both operands go through LDS, 32 k at a time: fetched into registers
// while the tile before is multiplied, written to the other of two buffers, one barrier a step. The float matrix cores do
// 256 flops a clock and CU, and a 128 x 128 tile wants 8 bytes a clock from L2, a 64 x 64 one 16, which is what L2 gives:
// 100 to 107 TFLOP/s of 157 (2048 x 19456 x 2560 1.92 ms; 300 rows 360 us against 561 of the plain kernel, 300 x 2560 x 9728
// 191 us against 1350).
#include "common.h"
#include "reinfer_hip.h"

namespace {

__device__ __forceinline__ f32x4_t load4(const float* p, bool ok) {
  f32x4_t v = *(const f32x4_t*)p;
  if (!ok) v = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  return v;
}

// ------------------------------------------------------------------------------------------------ up to 32 rows
// Workgroups that stay: tile b, b + grid, ... of 16 features, all M rows (MT tiles of 16), WAVES waves. A wave's loads run
// DEPTH runs of 32 U k ahead, on across the ends of tiles, and are unconditional: through a buffer descriptor a load past
// its end returns zeros and touches no memory, so rows past N or M, pieces past K and runs past the last tile count like any
// other load and cost nothing. A tile's runs are padded to a multiple of DEPTH, so that it ends where a round of the
// ring does.
template <int WAVES, int MT, int U, int DEPTH>
__global__ void __launch_bounds__(WAVES * RA_WAVE, 4)
gemm_f32_stream_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                       float* __restrict__ C, int M, int N, int K, int lda, int ldc) {
  constexpr int SPAN = WAVES * U * 32;     // k of one run of all waves
  constexpr unsigned NOWHERE = 0xFFFFFFF0u;
  __shared__ f32x4_t sums[2][WAVES][MT][RA_WAVE];        // of one tile while the next one's may already be written
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, q = lane >> 4;
  const int n_steps = (K + SPAN - 1) / SPAN;
  const int n_steps_p = (n_steps + DEPTH - 1) / DEPTH * DEPTH;
  const int n_tiles = (N + 15) / 16;
  const int n_mine = (n_tiles - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
  const int total = n_mine * n_steps_p;
  const __amdgpu_buffer_rsrc_t w_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(W), 0, (int)((size_t)N * K * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t a_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(A), 0, (int)(((size_t)(M - 1) * lda + K) * 4), 0x00020000);
  f32x4_t w[DEPTH][U][2], a[DEPTH][U][MT][2];
  int l_q = 0, l_step = 0, l_n = (int)blockIdx.x * 16 + r;         // where the loads are
#define RA_F32_LOAD(d)                                                                                        \
  do {                                                                                                        \
    const bool live_ = l_q < total && l_step < n_steps;                                                       \
    _Pragma("unroll") for (int u = 0; u < U; ++u)                                                             \
      _Pragma("unroll") for (int j = 0; j < 2; ++j) {                                                         \
        const int k_ = l_step * SPAN + (wave * U + u) * 32 + j * 16 + q * 4;                                  \
        const bool ok_ = live_ && k_ < K;            /* K is a multiple of 4 */                               \
        const unsigned off_ = ok_ && l_n < N ? (unsigned)(((size_t)l_n * K + k_) * 4) : NOWHERE;              \
        w[d][u][j] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, off_, 0, 0));  \
        _Pragma("unroll") for (int t = 0; t < MT; ++t) {                                                      \
          const int m_ = t * 16 + r;                                                                          \
          const unsigned at_ = ok_ && m_ < M ? (unsigned)(((size_t)m_ * lda + k_) * 4) : NOWHERE;             \
          a[d][u][t][j] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, at_, 0, 0)); \
        }                                                                                                     \
      }                                                                                                       \
    ++l_q;                                                                                                    \
    if (++l_step == n_steps_p) {                                                                              \
      l_step = 0;                                                                                             \
      l_n += (int)gridDim.x * 16;                                                                             \
    }                                                                                                         \
  } while (0)
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) RA_F32_LOAD(d);
  f32x4_t acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  int step = 0, n0 = (int)blockIdx.x * 16, buf = 0;                // where the products are
  for (int base = 0; base < total; base += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int t = 0; t < MT; ++t)
              acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[d][u][j][e], a[d][u][t][j][e], acc[t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);   // the run DEPTH ahead is asked for once this one's registers are free
      RA_F32_LOAD(d);
      __builtin_amdgcn_sched_barrier(0);
    }
    step += DEPTH;
    if (step < n_steps_p) continue;
    // a tile is complete: lane has row lane % 16, features 4 (lane / 16) .. + 3. One barrier a tile: its sums are read
    // while the next tile's go to the other buffer, and a wave writes a buffer again only behind the next barrier.
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      sums[buf][wave][t][lane] = acc[t];
      acc[t] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (wave < MT) {
      f32x4_t v = sums[buf][0][wave][lane];
#pragma unroll
      for (int x = 1; x < WAVES; ++x) v += sums[buf][x][wave][lane];
      const int m = wave * 16 + r;
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
#undef RA_F32_LOAD
}

// ------------------------------------------------------------------------------------------------ from 33 rows on
#define F32_BK 32
// A row of a tile in LDS is 8 pieces of 16 bytes, piece p of row r at place p ^ (r % 8): eight rows' reads of one piece fall
// on different banks.
__device__ __forceinline__ int piece_at(int row, int piece) { return row * F32_BK + ((piece ^ (row & 7)) << 2); }

// One workgroup of four waves: rows [B blockIdx.y, +B), features [B blockIdx.x, +B), k of range blockIdx.z.
// ranges == 1: C with the bias; else the range's float sums into part[blockIdx.z][M][N].
template <int B>
__global__ void __launch_bounds__(256)
gemm_f32_tile_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                     float* __restrict__ C, float* __restrict__ part, int M, int N, int K, int lda, int ldc,
                     int range_k) {
  constexpr int T = B / 64;                // 32 x 32 tiles a side of a wave's quarter
  constexpr int L = B * F32_BK / 4 / 256;  // 16-byte pieces a thread and operand
  __shared__ float lds[4 * B * F32_BK];    // two buffers of both operands: 64 KB at B = 128
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.y * B, n0 = blockIdx.x * B;
  const int k0 = blockIdx.z * range_k, k1 = k0 + range_k < K ? k0 + range_k : K;
  const int steps = (k1 - k0 + F32_BK - 1) / F32_BK;
  // staging: piece i of a thread is row (tid + 256 i) / 8, k 4 ((tid + 256 i) % 8)
  const float *ag[L], *wg[L];
  const int kp = (tid & 7) * 4;
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int row = (tid + 256 * i) >> 3;
    ag[i] = A + (size_t)(m0 + row < M ? m0 + row : M - 1) * lda;
    wg[i] = W + (size_t)(n0 + row < N ? n0 + row : N - 1) * K;
  }
  f32x4_t as[L], ws[L];
  auto fetch = [&](int k) {
    const bool ok = k + kp < k1;
    const int at = ok ? k + kp : 0;
#pragma unroll
    for (int i = 0; i < L; ++i) {
      as[i] = load4(ag[i] + at, ok);
      ws[i] = load4(wg[i] + at, ok);
    }
  };
  auto stage = [&](int buf) {
    float* a = lds + buf * 2 * B * F32_BK;
    float* w = a + B * F32_BK;
#pragma unroll
    for (int i = 0; i < L; ++i) {
      const int at = piece_at((tid + 256 * i) >> 3, tid & 7);
      *(f32x4_t*)(a + at) = as[i];
      *(f32x4_t*)(w + at) = ws[i];
    }
  };
  f32x16_t acc[T][T];
#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int j = 0; j < T; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  const int wm = (wave >> 1) * (B / 2), wn = (wave & 1) * (B / 2);
  const int row = lane & 31, half = lane >> 5;

  fetch(k0);
  stage(0);
  __syncthreads();
  for (int s = 0; s < steps; ++s) {
    if (s + 1 < steps) fetch(k0 + (s + 1) * F32_BK);
    __builtin_amdgcn_sched_barrier(0);
    const float* a = lds + (s & 1) * 2 * B * F32_BK + wm * F32_BK;
    const float* w = lds + ((s & 1) * 2 + 1) * B * F32_BK + wn * F32_BK;
#pragma unroll
    for (int kk = 0; kk < F32_BK; kk += 8) {
      f32x4_t x[T], y[T];
#pragma unroll
      for (int i = 0; i < T; ++i) {
        x[i] = *(const f32x4_t*)(a + piece_at(i * 32 + row, kk / 4 + half));
        y[i] = *(const f32x4_t*)(w + piece_at(i * 32 + row, kk / 4 + half));
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < T; ++i)
#pragma unroll
          for (int j = 0; j < T; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(y[j][e], x[i][e], acc[i][j], 0, 0, 0);
    }
    if (s + 1 < steps) stage((s + 1) & 1);
    __syncthreads();
  }
  // a lane holds row lane % 32 of the tile, features 8 (e / 4) + 4 (lane / 32) + e % 4
  float* out = part ? part + (size_t)blockIdx.z * M * N : C;
  const int ld = part ? N : ldc;
  const float* b = part ? nullptr : bias;
#pragma unroll
  for (int i = 0; i < T; ++i) {
    const int m = m0 + wm + i * 32 + row;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < T; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int n = n0 + wn + j * 32 + g * 8 + half * 4;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) out[(size_t)m * ld + n + e] = b ? acc[i][j][g * 4 + e] + b[n + e] : acc[i][j][g * 4 + e];
      }
  }
}

__global__ void __launch_bounds__(256)
gemm_f32_add_kernel(const float* __restrict__ part, int ranges, const float* __restrict__ bias, float* __restrict__ C,
                    int M, int N, int ldc) {
  const size_t size = (size_t)M * N, i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= size) return;
  const int m = i / N, n = i % N;
  float v = part[i];
  for (int r = 1; r < ranges; ++r) v += part[r * size + i];
  C[(size_t)m * ldc + n] = bias ? v + bias[n] : v;
}

// The tile kernel's plan: 128 x 128 tiles where there are four a CU and more (2048 x 19456 x 2560: 1.91 ms against 2.02 ms),
// else 64 x 64 ones with K cut into as many ranges of at least 256 k as price lowest: a CU's share of the workgroups at the
// share of the matrix cores' rate that so many side by side reach (measured: one workgroup waits for memory most of the
// time), and the ranges' sums written and read again. (300 x 2560 x 9728: uncut 459 us, in 12 ranges 190; 33 x 19456 x
// 2560: 157 us, in 3 ranges 92.)
struct TilePlan {
  int side, ranges, range_k;
};
TilePlan tile_plan(int M, int N, int K) {
  const int cus = ra_cu_count();
  const long big = (long)((M + 127) / 128) * ((N + 127) / 128);
  if (big >= 4L * cus) return {128, 1, K};
  const long tiles = (long)((M + 63) / 64) * ((N + 63) / 64);
  const double reached[5] = {0.28, 0.48, 0.62, 0.72, 0.76};
  const double tile_us = 64.0 * 64.0 * 2.0 * K / 600e3;                       // one tile at a CU's full rate
  int best = 1;
  double best_us = 0.0;
  for (int r = 1; r <= 16 && (r == 1 || K / r >= 256); ++r) {
    const long load = (tiles * r + cus - 1) / cus;
    double us = (double)load / r * tile_us / reached[load < 5 ? load - 1 : 4];
    if (r > 1) us += 3.0 + (double)r * M * N * 8.0 / 5e6;
    if (r == 1 || us < best_us) {
      best = r;
      best_us = us;
    }
  }
  const int range_k = ((K + best - 1) / best + F32_BK - 1) / F32_BK * F32_BK;
  return {64, (K + range_k - 1) / range_k, range_k};
}

}  // namespace

#define F32_STREAM_ROWS 32

extern "C" int ra_gemm_f32_supports(const void* A, const void* W, int K, int lda) {
  return K > 0 && K % 4 == 0 && ra_rows_16b(A, lda, 4) && ra_rows_16b(W, K, 4);
}

extern "C" long ra_gemm_f32_scratch(int M, int N, int K) {
  if (M <= F32_STREAM_ROWS) return 0;
  const TilePlan p = tile_plan(M, N, K);
  return p.ranges > 1 ? (long)p.ranges * M * N : 0;
}

extern "C" int ra_gemm_f32(const float* A, const float* W, const float* bias, float* C, int M, int N, int K, int lda,
                           int ldc, float* scratch, long scratch_floats, hipStream_t stream) {
  RA_CHECK(M > 0 && N > 0 && K > 0, "gemm_f32: empty product (%d, %d, %d)", M, N, K);
  RA_CHECK(lda >= K && ldc >= N, "gemm_f32: row strides (%d, %d) below the row lengths (%d, %d)", lda, ldc, K, N);
  RA_CHECK(ra_gemm_f32_supports(A, W, K, lda), "gemm_f32: rows of %d (stride %d) are not 16-byte pieces", K, lda);
  if (M <= F32_STREAM_ROWS) {
    // a descriptor covers less than 4 GiB of weights: a larger matrix goes in runs of features
    const long most = 0xFFFFFF00L / ((long)K * 4) / 16 * 16;
    RA_CHECK(most > 0 && ((long)(M - 1) * lda + K) * 4 < 0xFFFFFF00L, "gemm_f32: rows of %d (stride %d) are too long", K, lda);
    for (long n0 = 0; n0 < N; n0 += most) {
      const int n = (int)(N - n0 < most ? N - n0 : most);
      const int tiles = (n + 15) / 16, cus = ra_cu_count();
      const float *w = W + (size_t)n0 * K, *b = bias ? bias + n0 : nullptr;
#define RA_GO(WAVES, MT, U, DEPTH, GRID) \
  gemm_f32_stream_kernel<WAVES, MT, U, DEPTH><<<(GRID) < tiles ? (GRID) : tiles, WAVES * RA_WAVE, 0, stream>>>( \
      A, w, b, C + n0, M, n, K, lda, ldc)
      // four waves and four workgroups a CU share many tiles out most evenly (6144 x 2560 at 4 rows: 19.0 us against 21.1
      // with eight waves and two), eight waves keep more in flight where a CU has one tile (2560 x 9728: 30.5 against 32.9)
      if (M > 16) RA_GO(8, 2, 1, 3, 2 * cus);
      else if (tiles <= cus) RA_GO(8, 1, 2, 2, cus);
      else RA_GO(4, 1, 2, 2, 4 * cus);
#undef RA_GO
      RA_LAUNCH_CHECK("gemm_f32");
    }
    return 0;
  }
  const TilePlan p = tile_plan(M, N, K);
  const bool cut = p.ranges > 1;
  RA_CHECK(!cut || (scratch && scratch_floats >= (long)p.ranges * M * N), "gemm_f32: scratch of %ld floats, needs %ld",
           scratch_floats, (long)p.ranges * M * N);
  const dim3 grid((N + p.side - 1) / p.side, (M + p.side - 1) / p.side, p.ranges);
  RA_CHECK(grid.y <= 65535, "gemm_f32: %d rows in one launch", M);
  float* part = cut ? scratch : nullptr;
  if (p.side == 128) gemm_f32_tile_kernel<128><<<grid, 256, 0, stream>>>(A, W, bias, C, part, M, N, K, lda, ldc, p.range_k);
  else gemm_f32_tile_kernel<64><<<grid, 256, 0, stream>>>(A, W, bias, C, part, M, N, K, lda, ldc, p.range_k);
  RA_LAUNCH_CHECK("gemm_f32");
  if (cut) {
    const size_t blocks = ((size_t)M * N + 255) / 256;
    gemm_f32_add_kernel<<<blocks, 256, 0, stream>>>(scratch, p.ranges, bias, C, M, N, ldc);
    RA_LAUNCH_CHECK("gemm_f32 (ranges)");
  }
  return 0;
}
