// The entry points of products with few rows that are not gemm_skinny.hip's:  C[M,N] = A[M,K] . W[N,K]^T, bfloat16 in, float
// accumulation on the matrix cores; the faster of the two from 17 rows on, and for wide gated products below that. The products are
// gemm_tile.hip's; here stand the rule which of the two kernels is ahead, and the kernels that add K ranges.
//
// With more than one row tile the activations weigh as much as the weights: a workgroup that owns 16 features and splits K over its
// waves (gemm_skinny.hip) reads all of A, once a wave slice, and with its registers full of row tiles it keeps too few bytes in flight
// to cover the memory latency (measured at 64 rows: 3 TB/s).
//
// Where N gives too few tiles of features to fill the chip, K is cut into S ranges; each writes its float partial result and a second
// kernel adds them in range order and applies the epilogue: deterministic, no atomics. Epilogues as in gemm_skinny.hip: plain
// (+ bias), SiLU gate over interleaved gate/up rows (S = 1 only), C += (float).
//
// An RMSNorm can ride on these products as on gemm_skinny's (y = rstd[m] * ((x .* w) . W^T)): the
// row factor is applied in the epilogue of whichever kernel finishes the product; the scaled copy
// and the partial sums of squares for the norm that follows an accumulating product are written by
// the adding kernel, which such a product then always runs: one partial sum per row and 1024 columns.
#include "common.h"
#include "reinfer_hip.h"
#include "gemm_tile.h"

enum { WEPI_PLAIN = 0, WEPI_SILU_PAIRS = 1, WEPI_ACCUM = 2 };

// RMSNorm carried by the product (all pointers may be null): see gemm_skinny.hip
struct WideNorm {
  const float* in_ss;      // [in_parts, M] partial sums of squares of the rows behind A
  int in_parts;
  float in_eps, in_inv_width;
  const void* out_w;       // [N] weight of the norm that follows (adding kernel only)
  int out_w_f32;
  bf16_t* out_x;           // [M, out_ldx] bf16(C_new * out_w)
  int out_ldx;
  float* out_ss;           // [ceil(N / 1024), M] sums of squares of C_new over 1024 columns
  float out_eps;           // >= 0 with out_ss null: the adding kernel finishes the norm, out_x = bf16(norm(C_new) * out_w)
  float acc_scale;         // the accumulating epilogue adds acc_scale times the product (1: the product itself)
};

// The ranges' values in four columns, added in range order (v), for which those of up to eight ranges are asked for in one trip.
#define GW_AHEAD 8
__device__ __forceinline__ void gw_ask(f32x4_t (&t)[GW_AHEAD], const float* __restrict__ p, size_t plane, int s0, int S) {
#pragma unroll
  for (int j = 0; j < GW_AHEAD; ++j) t[j] = *(const f32x4_t*)(p + (size_t)min(s0 + j, S - 1) * plane);
}
__device__ __forceinline__ void gw_add(float (&v)[4], const f32x4_t (&t)[GW_AHEAD], int s0, int S) {
#pragma unroll
  for (int j = 0; j < GW_AHEAD; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += s0 + j < S ? t[j][i] : 0.f;
}

// C = epilogue(sum over s of P[s]) for the K ranges of a split product, in range order; a workgroup
// takes 1024 columns of one row. The carried norm's row factor and, for the norm that follows an
// accumulating product, the scaled copy and the workgroup's sum of squares are applied here. Bound by trips to memory: all that a
// thread reads (eight ranges, the old values, the next norm's weights) is asked for at once (ranges six at a time and the rest
// behind their sum: the two kernels of 48 rows of 2560 x 4096 14.2 us, so 13.7; of 4096 x 12288 26.9, 25.9).
template <int EPI, typename TO>
__global__ void __launch_bounds__(256)
gemm_wide_reduce_kernel(const float* __restrict__ P, int S, const bf16_t* __restrict__ bias,
                        TO* __restrict__ C, int ldc, int M, int N, WideNorm nf) {
  __shared__ float red[17];
  const int n = (blockIdx.x * 256 + threadIdx.x) * 4;
  const int m = blockIdx.y;
  float v[4] = {0.f, 0.f, 0.f, 0.f}, old[4] = {0.f, 0.f, 0.f, 0.f}, w[4] = {0.f, 0.f, 0.f, 0.f};
  if (n < N) {
    const float* p = P + (size_t)m * N + n;
    const size_t plane = (size_t)M * N;
    const bool whole = n + 3 < N && (N & 3) == 0;
    f32x4_t t[GW_AHEAD];
    if (whole) gw_ask(t, p, plane, 0, S);
    if (EPI == WEPI_ACCUM) {
#pragma unroll
      for (int i = 0; i < 4; ++i) old[i] = to_f32(C[(size_t)m * ldc + min(n + i, N - 1)]);
      if (nf.out_x) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int c = min(n + i, N - 1);
          w[i] = nf.out_w_f32 ? ((const float*)nf.out_w)[c] : to_f32(((const bf16_t*)nf.out_w)[c]);
        }
      }
    }
    if (whole) {
      gw_add(v, t, 0, S);
      for (int s0 = GW_AHEAD; s0 < S; s0 += GW_AHEAD) {
        gw_ask(t, p, plane, s0, S);
        gw_add(v, t, s0, S);
      }
    } else {
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n + i < N) v[i] += p[(size_t)s * plane + i];
    }
  }
  float rstd = 1.f;
  if (nf.in_ss) {                              // the same for every thread: the threads share the parts out
    float t = 0.f;
    for (int p = threadIdx.x; p < nf.in_parts; p += blockDim.x) t += nf.in_ss[(size_t)p * M + m];
    rstd = rsqrtf(block_sum(t, red) * nf.in_inv_width + nf.in_eps);
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (n + i >= N) continue;
    float x = v[i] * rstd;
    if (bias) x += to_f32(bias[n + i]);
    if (EPI == WEPI_ACCUM) x = x * nf.acc_scale + old[i];
    C[(size_t)m * ldc + n + i] = from_f32<TO>(x);
    if (EPI == WEPI_ACCUM && nf.out_x) {
      nf.out_x[(size_t)m * nf.out_ldx + n + i] = from_f32<bf16_t>(x * w[i]);
      ss += x * x;
    }
  }
  if (EPI == WEPI_ACCUM && nf.out_x) {        // the same for every thread of the workgroup
    ss = block_sum(ss, red);
    if (threadIdx.x == 0) nf.out_ss[(size_t)blockIdx.x * M + m] = ss;
  }
}

// The same with a whole row a workgroup, which then also finishes the RMSNorm that follows an accumulating
// product: out_x = bf16(C_new * rsqrt(mean(C_new^2) + out_eps) * out_w). For the rows above those that the
// weight-streaming products take (65 to 128 requests decoding), where the products behind the norm are the
// library's and cannot apply a row factor: the norm then costs no kernel of its own. 1024 threads a row, each
// with CH chunks of 4 columns (N <= 4096 CH, N a multiple of 4): with few workgroups it is the loads in flight
// that count (256 threads with four chunks each, one after the other: 11 us against 7).
template <int CH>
__global__ void __launch_bounds__(1024)
gemm_wide_reduce_rows_kernel(const float* __restrict__ P, int S, const bf16_t* __restrict__ bias,
                             float* __restrict__ C, int ldc, int M, int N, WideNorm nf) {
  __shared__ float red[17];
  const int m = blockIdx.x;
  float rstd = 1.f;
  if (nf.in_ss) {                              // the same for every thread: the threads share the parts out
    float t = 0.f;
    for (int p = threadIdx.x; p < nf.in_parts; p += blockDim.x) t += nf.in_ss[(size_t)p * M + m];
    rstd = rsqrtf(block_sum(t, red) * nf.in_inv_width + nf.in_eps);
  }
  float x[CH][4], w[CH][4];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int n = (c * 1024 + threadIdx.x) * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) x[c][i] = w[c][i] = 0.f;
    if (n >= N) continue;
    const float* p = P + (size_t)m * N + n;
    const size_t plane = (size_t)M * N;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    f32x4_t t[GW_AHEAD];
    gw_ask(t, p, plane, 0, S);
    const f32x4_t c0 = *(const f32x4_t*)(C + (size_t)m * ldc + n);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      w[c][i] = nf.out_w_f32 ? ((const float*)nf.out_w)[n + i] : to_f32(((const bf16_t*)nf.out_w)[n + i]);
    gw_add(v, t, 0, S);
    for (int s0 = GW_AHEAD; s0 < S; s0 += GW_AHEAD) {
      gw_ask(t, p, plane, s0, S);
      gw_add(v, t, s0, S);
    }
    f32x4_t o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float y = v[i] * rstd;
      if (bias) y += to_f32(bias[n + i]);
      y = y * nf.acc_scale + c0[i];
      o[i] = y;
      x[c][i] = y;
      ss += y * y;
    }
    *(f32x4_t*)(C + (size_t)m * ldc + n) = o;
  }
  const float rout = rsqrtf(block_sum(ss, red) / (float)N + nf.out_eps);
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int n = (c * 1024 + threadIdx.x) * 4;
    if (n >= N) continue;
    bf16x4_t o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = from_f32<bf16_t>(x[c][i] * rout * w[c][i]);
    *(bf16x4_t*)(nf.out_x + (size_t)m * nf.out_ldx + n) = o;
  }
}

// How [M, N, K] runs: its tiles and K ranges, and whether the adding kernel finishes it. Ranges where tiles of 128 features do not fill
// three quarters of the chip's CUs, and where the adding kernel runs anyhow to write what the next norm needs; a gated product is never cut.
struct WidePlan {
  RaTilePlan tile;
  bool partial;
};
static WidePlan gw_plan(int epilogue, int M, int N, int K, bool emits = false) {
  const int cus = ra_cu_count(), fill = cus - cus / 4;
  const bool cut = epilogue != WEPI_SILU_PAIRS && (M > 64 || emits || (N + 127) / 128 < fill);
  WidePlan p = {ra_tile_plan(M, N, K, cut), false};
  p.partial = cut && (M > 64 || emits || p.tile.ranges > 1);
  return p;
}

// 1 where this kernel beats ra_gemm_skinny (measured on MI355X at 4 to 64 rows): from 17 rows on,
// except a small product whose K has to be cut (4096 x 4096: the second launch costs more than the
// shared activations save); from 9 rows for the gated product of a wide feed-forward.
extern "C" int ra_gemm_wide_preferred(int epilogue, int M, int N, int K) {
  if (M < 1) return 0;
  // 65 to 128 rows: what adds into the residual stream, cut into ranges, because the norm that follows can ride on it
  // (the other products of these rows are offered by ra_gemm_tile_takes)
  if (M > 64) return M <= 128 && epilogue == WEPI_ACCUM ? ra_gemm_tile_takes(epilogue, M, N, K) : 0;
  const RaTilePlan tile = gw_plan(epilogue, M, N, K).tile;
  // sizes are priced a CU: a product is "large" where every CU has more than 128 KiB of weights to stream
  // (on 256 CUs: more than 4096 x 4096 bfloat16)
  const int cus = ra_cu_count(), fill = cus - cus / 4;
  const bool large = (long)N * K * 2 > 131072L * cus;
  const int cb = (N + tile.cols - 1) / tile.cols;
  if (M < 17) {
    if (epilogue == WEPI_SILU_PAIRS)
      return (M > 8 && cb >= fill && cb * 10 >= ((cb + cus - 1) / cus) * cus * 8) ? 1 : 0;
    return (epilogue == WEPI_PLAIN && M > 8 && tile.ranges == 1 && cb >= 3 * cus) ? 1 : 0;
  }
  return (tile.ranges == 1 || large) ? 1 : 0;
}

// Floats of scratch that ra_gemm_wide needs for this product (0: none).
extern "C" long ra_gemm_wide_scratch(int epilogue, int M, int N, int K, int emits) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const WidePlan p = gw_plan(epilogue, M, N, K, emits != 0);
  return p.partial ? (long)p.tile.ranges * M * N : 0;
}

// Partial sums a row that an emitting product writes for the norm that follows an [M, N] result.
extern "C" int ra_gemm_wide_row_parts(int N) { return (N + 1023) / 1024; }

// the second half of a product cut into K ranges: adds them in range order and applies the epilogue
static int launch_wide_reduce(const void* bias, void* C, int ldc, int out_dtype, int epilogue, int M, int N, int S,
                              const float* scratch, const WideNorm& nf, hipStream_t stream) {
  if (nf.out_x && !nf.out_ss) {                // a whole row a workgroup: the norm that follows is finished here
    if (N <= 4096) gemm_wide_reduce_rows_kernel<1><<<M, 1024, 0, stream>>>(scratch, S, (const bf16_t*)bias, (float*)C, ldc, M, N, nf);
    else if (N <= 8192) gemm_wide_reduce_rows_kernel<2><<<M, 1024, 0, stream>>>(scratch, S, (const bf16_t*)bias, (float*)C, ldc, M, N, nf);
    else gemm_wide_reduce_rows_kernel<4><<<M, 1024, 0, stream>>>(scratch, S, (const bf16_t*)bias, (float*)C, ldc, M, N, nf);
    RA_LAUNCH_CHECK("gemm_wide reduce rows");
    return 0;
  }
  const dim3 rg((N + 1023) / 1024, M);
#define RA_GR(EPI, TO) \
  gemm_wide_reduce_kernel<EPI, TO><<<rg, 256, 0, stream>>>(scratch, S, (const bf16_t*)bias, (TO*)C, ldc, M, N, nf)
  if (epilogue == WEPI_ACCUM) RA_GR(WEPI_ACCUM, float);
  else if (out_dtype == RA_BF16) RA_GR(WEPI_PLAIN, bf16_t);
  else RA_GR(WEPI_PLAIN, float);
#undef RA_GR
  RA_LAUNCH_CHECK("gemm_wide reduce");
  return 0;
}

static int gemm_wide_impl(const void* A, const void* W, const void* bias, void* C, int out_dtype,
                          int epilogue, int M, int N, int K, int lda, int ldc, float* scratch,
                          long scratch_floats, const float* in_ss, int in_parts, float in_eps,
                          int in_width, const void* out_w, int out_w_dtype, void* out_x, int out_ldx,
                          float* out_ss, float out_eps, float acc_scale, int keep, hipStream_t stream) {
  RA_CHECK(M > 0 && N > 0 && K > 0, "gemm_wide: empty product (%d, %d, %d)", M, N, K);
  RA_CHECK(M <= 128 || ra_gemm_tile_takes(epilogue, M, N, K),
           "gemm_wide: %d rows; at most 128, or 512 where the tiled product is ahead", M);
  RA_CHECK(K % 8 == 0 && lda % 8 == 0, "gemm_wide: K (%d) and the row stride (%d) must be multiples of 8", K, lda);
  RA_CHECK(epilogue == WEPI_PLAIN || epilogue == WEPI_SILU_PAIRS || epilogue == WEPI_ACCUM,
           "gemm_wide: unknown epilogue %d", epilogue);
  RA_CHECK(epilogue != WEPI_ACCUM || out_dtype == RA_F32, "gemm_wide: accumulation is into a float matrix");
  const int n_out = epilogue == WEPI_SILU_PAIRS ? N / 2 : N;
  RA_CHECK(epilogue != WEPI_SILU_PAIRS || (N % 16 == 0 && bias == nullptr),
           "gemm_wide: the gated epilogue needs N (%d) in whole tiles of 16 and no bias", N);
  RA_CHECK(lda >= K && ldc >= n_out, "gemm_wide: row strides (%d, %d) below the row lengths (%d, %d)", lda, ldc, K, n_out);
  RA_CHECK(((uintptr_t)A % 16) == 0 && ((uintptr_t)W % 16) == 0, "gemm_wide: operands must be 16-byte aligned");
  RA_CHECK(out_dtype == RA_BF16 || out_dtype == RA_F32, "gemm_wide: unknown output dtype tag %d", out_dtype);
  WideNorm nf = {};
  nf.acc_scale = acc_scale;
  if (in_ss) {
    RA_CHECK(in_parts > 0 && in_width > 0 && in_eps >= 0.f, "gemm_wide: row sums need parts (%d), width (%d) and eps", in_parts, in_width);
    nf.in_ss = in_ss;
    nf.in_parts = in_parts;
    nf.in_eps = in_eps;
    nf.in_inv_width = 1.f / (float)in_width;
  }
  const bool emits = out_x || out_ss || out_w;
  const bool finishes = emits && !out_ss;      // the adding kernel finishes the norm that follows
  if (emits) {
    RA_CHECK(epilogue == WEPI_ACCUM, "gemm_wide: only the accumulating epilogue emits for a norm");
    RA_CHECK(out_x && out_w && (out_ss || out_eps >= 0.f),
             "gemm_wide: emitting needs the norm weight, the scaled copy and the partial sums (or, to finish the norm, its eps)");
    RA_CHECK(!finishes || (N % 4 == 0 && N <= 16384 && ldc % 4 == 0 && out_ldx % 4 == 0 && ((uintptr_t)C % 16) == 0 &&
                           ((uintptr_t)out_x % 8) == 0),
             "gemm_wide: finishing the norm takes rows of up to 16384 columns in steps of 4 (%d, strides %d and %d)", N, ldc, out_ldx);
    RA_CHECK(out_w_dtype == RA_BF16 || out_w_dtype == RA_F32, "gemm_wide: unknown norm weight dtype tag %d", out_w_dtype);
    RA_CHECK(out_ldx >= N, "gemm_wide: the scaled copy's row stride (%d) is below %d", out_ldx, N);
    nf.out_w = out_w;
    nf.out_w_f32 = out_w_dtype == RA_F32;
    nf.out_x = (bf16_t*)out_x;
    nf.out_ldx = out_ldx;
    nf.out_ss = out_ss;
    nf.out_eps = out_eps;
  }
  const long need = ra_gemm_wide_scratch(epilogue, M, N, K, emits);
  RA_CHECK(need == 0 || (scratch && scratch_floats >= need && ((uintptr_t)scratch % 16) == 0),
           "gemm_wide: this product needs %ld floats of scratch, got %ld", need, scratch_floats);
  const WidePlan p = gw_plan(epilogue, M, N, K, emits);
  if (p.partial) {
    // Above 48 rows the weights by the caches' usual policy: with the adding kernel behind it, 64 rows of 4096 x 4096 14.8 us (past it
    // 15.5), 128 of 2560 x 9728 22.5 (24.0), of 4096 x 12288 32.9 (33.9); at 24 rows 13.6 (12.5), 16.5 (15.4), 25.0 (23.3).
    if (int rc = ra_tile_ranges(p.tile, A, lda, W, scratch, M, N, K, keep || M > 48, stream)) return rc;
    return launch_wide_reduce(bias, C, ldc, out_dtype, epilogue, M, N, p.tile.ranges, scratch, nf, stream);
  }
  RA_CHECK(M <= 64 || (!in_ss && out_dtype == RA_BF16 && ra_gemm_tile_takes(epilogue, M, N, K)),
           "gemm_wide: with %d rows a gated product only where its tiles fill the chip, with a bfloat16 result and no norm", M);
  const RaTileEnd end = {nf.in_ss, nf.in_parts, nf.in_eps, nf.in_inv_width, (const bf16_t*)bias, acc_scale, out_dtype == RA_BF16, keep != 0};
  return ra_tile_product(epilogue, p.tile, A, lda, W, C, ldc, M, N, K, end, stream);
}

// K ranges that ra_gemm_wide_partial cuts [M, N, K] into (its result has that many [M, N] float planes).
extern "C" int ra_gemm_wide_ranges(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  return gw_plan(WEPI_PLAIN, M, N, K, true).tile.ranges;
}

// Only the first half of a split product: P[s][m][n] = A[m, range s] . W[n, range s]^T, float, for a
// consumer that adds the ranges itself (in range order) instead of the adding kernel.
extern "C" int ra_gemm_wide_partial(const void* A, const void* W, float* P, long p_floats, int M, int N, int K,
                                    int lda, int keep, hipStream_t stream) {
  RA_CHECK(M > 0 && N > 0 && K > 0, "gemm_wide: empty product (%d, %d, %d)", M, N, K);
  RA_CHECK(M <= 64 || ra_gemm_tile_takes(WEPI_PLAIN, M, N, K),
           "gemm_wide: %d rows; at most 64, or 512 where the tiled product is ahead", M);
  RA_CHECK(K % 8 == 0 && lda % 8 == 0 && lda >= K, "gemm_wide: K (%d) and the row stride (%d) must be multiples of 8", K, lda);
  RA_CHECK(((uintptr_t)A % 16) == 0 && ((uintptr_t)W % 16) == 0 && ((uintptr_t)P % 16) == 0,
           "gemm_wide: operands must be 16-byte aligned");
  const RaTilePlan tile = gw_plan(WEPI_PLAIN, M, N, K, true).tile;
  RA_CHECK(P && p_floats >= (long)tile.ranges * M * N, "gemm_wide: %d ranges of [%d, %d] need %ld floats, got %ld", tile.ranges, M, N,
           (long)tile.ranges * M * N, p_floats);
  // past the caches at any number of rows: by the usual policy / past it, 64 rows 6144 x 2560 10.8 / 10.3 us, 4096 x 12288 21.8 / 20.2, 128
  // rows 13.6 / 13.2 and 26.5 / 25.5
  return ra_tile_ranges(tile, A, lda, W, P, M, N, K, keep != 0, stream);
}

extern "C" int ra_gemm_wide_normed(const void* A, const void* W, const void* bias, void* C, int out_dtype,
                                   int epilogue, int M, int N, int K, int lda, int ldc, float* scratch,
                                   long scratch_floats, const float* in_ss, int in_parts, float in_eps,
                                   int in_width, const void* out_w, int out_w_dtype, void* out_x, int out_ldx,
                                   float* out_ss, float out_eps, int keep, hipStream_t stream) {
  return gemm_wide_impl(A, W, bias, C, out_dtype, epilogue, M, N, K, lda, ldc, scratch, scratch_floats, in_ss,
                        in_parts, in_eps, in_width, out_w, out_w_dtype, out_x, out_ldx, out_ss, out_eps, 1.f, keep, stream);
}

extern "C" int ra_gemm_wide(const void* A, const void* W, const void* bias, void* C, int out_dtype, int epilogue,
                            int M, int N, int K, int lda, int ldc, float* scratch, long scratch_floats,
                            int keep, hipStream_t stream) {
  return gemm_wide_impl(A, W, bias, C, out_dtype, epilogue, M, N, K, lda, ldc, scratch, scratch_floats,
                        nullptr, 0, 0.f, 0, nullptr, 0, nullptr, 0, nullptr, -1.f, 1.f, keep, stream);
}

// C += acc_scale * (A . W^T): the accumulating epilogue with a factor on the product
extern "C" int ra_gemm_wide_scaled(const void* A, const void* W, float* C, int M, int N, int K, int lda, int ldc,
                                   float* scratch, long scratch_floats, float acc_scale, int keep, hipStream_t stream) {
  return gemm_wide_impl(A, W, nullptr, C, RA_F32, WEPI_ACCUM, M, N, K, lda, ldc, scratch, scratch_floats,
                        nullptr, 0, 0.f, 0, nullptr, 0, nullptr, 0, nullptr, -1.f, acc_scale, keep, stream);
}
