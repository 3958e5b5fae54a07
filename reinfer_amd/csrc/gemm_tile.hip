// Products of 65 to 128 rows in bfloat16, C[M,N] = A[M,K] . W[N,K]^T: short prompts and the largest decode steps (and of up to 512
// rows where N or K does not fit gemm_prompt.hip's steps). They are
// bound by reading the weights once, and by how many CUs a few tiles of 128 x 128 can be spread over: K is cut into ranges
// until the tiles fill the chip once, each range's float sums go to a plane of their own, and the adding kernels of
// gemm_wide.hip add the planes in order and do what stands behind the product (bias, the float stream, the norm that
// follows). A gate and up projection of up to 128 rows whose tiles fill the chip uncut is finished here.
//
// A workgroup of four waves takes 64 k a step through a ring of three stages in LDS, filled by loads that go straight to
// LDS two steps ahead, with one barrier a step: a wave waits for its own loads of a stage, the barrier makes that true of
// all, and behind it the stage of the step before, which every wave has left, is asked for anew. A row of a stage is 8
// pieces of 16 bytes, piece p of row r at place p ^ (r % 8), so that eight rows' reads of one piece fall on different
// banks; the loads write LDS in the order of their lanes, so it is their addresses that are permuted, inside a row's 128
// bytes. What bounds a step are the 24 to 32 KB that its CU fetches, at 17 to 20 bytes a clock however few CUs run: four or
// five stages, two workgroups a CU with two stages each, and tiles of 256 changed a product by less than a tenth. Hence the
// gated product's tiles, which stand in one row, are the narrowest that the chip holds at once (19456 x 2560 at 128 rows:
// 203 tiles of 96 features 31.2 us, 152 of 128 34.5).
//
// With the adding kernel, 6144 x 4096 / 4096 x 4096 / 4096 x 12288, the library's product in brackets: 97 rows
// 19 / 16 / 29 us (23 / 18 / 41), 128 rows 20 / 18 / 31 (26 / 24 / 66). 24576 x 4096 with its gate at 97 rows 48 (54 with the
// gate's kernel). Above 128 rows these ranges run on gemm_prompt.hip's tiles where its shapes allow: 160 rows 24 / 19 / 36 us
// (28 / 21 / 40 here; library 28 / 27 / 76), 193 rows 26 / 21 / 39 (28 / 22 / 41; 25 / 22 / 54), 256 rows 30 / 23 / 44
// (30 / 24 / 45; 40 / 23 / 58).
#include "common.h"
#include "reinfer_hip.h"
#include "gemm_tile.h"
#include "gemm_prompt.h"

namespace {

#define GT_BK 64
#define GT_SIDE 128

enum { GT_GATED = 1, GT_PART = 3 };

struct TileArgs {
  const bf16_t* a;
  const bf16_t* w;
  void* c;                                   // GT_PART: float [ranges][M][N]; GT_GATED: bfloat16 [M][N / 2]
  int M, N, K, lda, ldc;
  unsigned a_bytes, w_bytes;
  int m_tiles, n_tiles, ranges, range_k;
};

template <int BN, int EPI>
__global__ void __launch_bounds__(256) gemm_tile_kernel(TileArgs g) {
  constexpr int BM = GT_SIDE, STAGES = 3;
  constexpr int WAVES_N = BN == 96 ? 1 : 2, WAVES_M = 4 / WAVES_N;
  constexpr int TM = BM / 32 / WAVES_M, TN = BN / 32 / WAVES_N;   // 32 x 32 tiles of a wave
  constexpr int ROWS = BM + BN, PA = BM / 32, PB = BN / 32;       // a wave's loads a stage: 8 rows (1 KB) each
  constexpr unsigned NOWHERE = 0xFFFFFFF0u;
  __shared__ __attribute__((aligned(1024))) bf16_t lds[STAGES * ROWS * GT_BK];
  // the row tiles of a panel and range of weights follow one another, and each XCD gets a run of tiles
  const int total = g.m_tiles * g.n_tiles * g.ranges, each = (total + RA_XCDS - 1) / RA_XCDS;
  const int at = (int)blockIdx.x / RA_XCDS, tile = (int)blockIdx.x % RA_XCDS * each + at;
  if (at >= each || tile >= total) return;
  const int m0 = tile % g.m_tiles * BM, z = tile / g.m_tiles % g.ranges, n0 = tile / g.m_tiles / g.ranges * BN;
  const int k0 = z * g.range_k, k1 = min(k0 + g.range_k, g.K), steps = (k1 - k0 + GT_BK - 1) / GT_BK;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(g.a), 0, (int)g.a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(g.w), 0, (int)g.w_bytes, 0x00020000);
  const int piece = (lane & 7) ^ (lane >> 3);
  // nobody stores what becomes of rows past the end: those of A are zeros from past the descriptor, which cost no fetch
  // (97 rows: 8 %), those of W, whose descriptor may span 4 GiB, read the last row
  unsigned a_off[PA], w_off[PB];
#pragma unroll
  for (int i = 0; i < PA; ++i) {
    const int r = m0 + (wave * PA + i) * 8 + (lane >> 3);
    a_off[i] = r < g.M ? (unsigned)(((size_t)r * g.lda + piece * 8) * 2) : 0x80000000u;
  }
#pragma unroll
  for (int i = 0; i < PB; ++i) {
    const int r = n0 + (wave * PB + i) * 8 + (lane >> 3);
    w_off[i] = (unsigned)(((size_t)(r < g.N ? r : g.N - 1) * g.K + piece * 8) * 2);
  }
  auto fetch = [&](int s, int buf) {
    const int k = k0 + s * GT_BK;
    const unsigned past = k + piece * 8 < k1 ? 0u : NOWHERE;      // pieces past the range's end become zeros
    bf16_t* to = lds + buf * ROWS * GT_BK;
#pragma unroll
    for (int i = 0; i < PA; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          a_rsrc, (__attribute__((address_space(3))) void*)(to + (wave * PA + i) * 8 * GT_BK), 16,
          (int)((a_off[i] + (unsigned)k * 2u) | past), 0, 0, 0);
#pragma unroll
    for (int i = 0; i < PB; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          w_rsrc, (__attribute__((address_space(3))) void*)(to + (BM + (wave * PB + i) * 8) * GT_BK), 16,
          (int)((w_off[i] + (unsigned)k * 2u) | past), 0, 0, 0);
  };
  f32x16_t acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  const int wm = wave / WAVES_N * (BM / WAVES_M), wn = wave % WAVES_N * (BN / WAVES_N);
  const int lrow = lane & 31, half = lane >> 5;
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s) fetch(s, s);
  int buf = 0;
  for (int s = 0; s < steps; ++s) {
    // this wave's loads of stage s are done when only those of the STAGES - 2 stages behind it are left, its reads of the
    // stage that is asked for next when no LDS read is left
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((PA + PB) * (STAGES - 2)) : "memory");
    fetch(s + STAGES - 1, buf == 0 ? STAGES - 1 : buf - 1);
    const bf16_t* as = lds + buf * ROWS * GT_BK;
    const bf16_t* ws = as + BM * GT_BK;
    // all operands of the step are asked for before its first product: they arrive while the products before them run
    bf16x8_t x[GT_BK / 16][TM], y[GT_BK / 16][TN];
#pragma unroll
    for (int ks = 0; ks < GT_BK / 16; ++ks) {
      const int p = ((ks * 2 + half) ^ (lrow & 7)) * 8;
#pragma unroll
      for (int i = 0; i < TN; ++i) y[ks][i] = *(const bf16x8_t*)(ws + (wn + i * 32 + lrow) * GT_BK + p);
#pragma unroll
      for (int j = 0; j < TM; ++j) x[ks][j] = *(const bf16x8_t*)(as + (wm + j * 32 + lrow) * GT_BK + p);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < GT_BK / 16; ++ks)
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(y[ks][i], x[ks][j], acc[i][j], 0, 0, 0);
    buf = buf + 1 == STAGES ? 0 : buf + 1;
  }
  // a lane holds row lane % 32 of a tile, weight rows 8 (e / 4) + 4 (lane / 32) + e % 4
  const bool whole = g.N % 4 == 0;
#pragma unroll
  for (int j = 0; j < TM; ++j) {
    const int m = m0 + wm + j * 32 + lrow;
    if (m >= g.M) continue;
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int q = 0; q < 4; q += EPI == GT_GATED ? 2 : 1) {
        const int n = n0 + wn + i * 32 + q * 8 + half * 4;
        if (n >= g.N) continue;
        if (EPI == GT_GATED) {               // 8 gate rows, then the 8 up rows of the same features
          bf16x4_t o;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float u = acc[i][j][q * 4 + e];
            o[e] = (bf16_t)(u / (1.f + expf(-u)) * acc[i][j][(q + 1) % 4 * 4 + e]);
          }
          *(bf16x4_t*)((bf16_t*)g.c + (size_t)m * g.ldc + (n0 + wn + i * 32) / 2 + q * 4 + half * 4) = o;
        } else {
          float* c = (float*)g.c + ((size_t)z * g.M + m) * g.N + n;
          f32x4_t v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = acc[i][j][q * 4 + e];
          if (whole) {
            *(f32x4_t*)c = v;
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (n + e < g.N) c[e] = v[e];
          }
        }
      }
  }
}

TileArgs tile_args(const void* A, int lda, const void* W, int M, int N, int K, int ranges, int range_k) {
  TileArgs g = {};
  g.a = (const bf16_t*)A;
  g.w = (const bf16_t*)W;
  g.M = M; g.N = N; g.K = K; g.lda = lda;
  g.a_bytes = (unsigned)(((size_t)(M - 1) * lda + K) * 2);
  g.w_bytes = (unsigned)((size_t)N * K * 2);
  g.m_tiles = (M + GT_SIDE - 1) / GT_SIDE;
  g.ranges = ranges; g.range_k = range_k;
  return g;
}

template <int BN, int EPI>
int tile_launch(TileArgs g, hipStream_t stream) {
  g.n_tiles = (g.N + BN - 1) / BN;
  const long total = (long)g.m_tiles * g.n_tiles * g.ranges, blocks = (total + RA_XCDS - 1) / RA_XCDS * RA_XCDS;
  gemm_tile_kernel<BN, EPI><<<(unsigned)blocks, 256, 0, stream>>>(g);
  RA_LAUNCH_CHECK("gemm_tile");
  return 0;
}

}  // namespace

static long tile_count(int M, int N) { return (long)((M + GT_SIDE - 1) / GT_SIDE) * ((N + GT_SIDE - 1) / GT_SIDE); }

// As many K ranges as fill the chip once, of at least 512 k (shorter ones are all start and end), at most 16 (each is a float
// plane to write and read again). They follow from N, K and the rows of tiles alone, so that a row has the same sums at any of 129
// to 256 rows (to 384, to 512). Ranges of the exact number of rows, which gemm_prompt.hip's tiles could have, would be faster (the two
// at 5120 x 25600 with 160 rows 92 / 70 us, with 384 139 / 114, 4096 x 12288 with 512 74 / 63, most shapes within 5 %), but then one
// more request in a step changes every row's last bits.
void ra_tile_plan(int M, int N, int K, int* ranges, int* range_k) {
  long s = ra_cu_count() / tile_count(M, N);
  if (s > K / 512) s = K / 512;
  if (s > 16) s = 16;
  if (s < 1) s = 1;
  *range_k = ((K + (int)s - 1) / (int)s + GT_BK - 1) / GT_BK * GT_BK;
  *ranges = (K + *range_k - 1) / *range_k;
}

// Products that are cut and whose ranges fill three quarters of the chip, or that are small (the library has too few tiles for
// those as well): 11264 x 4096 at 128 rows, 176 of 256 CUs, takes 34 us against the library's 32, 9216 x 4096, 216 CUs, 26
// against 30; 22528 x 4096, whose tiles do not fill the chip and cannot be cut, 49 against 45. Above 256 rows only a long K,
// where the planes are few beside the weights, and more than that share of the chip (4096 x 12288 at 384 rows, 192 CUs,
// 70 us on gemm_prompt.hip's tiles against 69, though at 300 rows 57 against 69; at 512 rows, all of them, 74 against 80); the line
// is the same for all rows of a row of tiles, as the sums are. Beyond 512 the library's larger tiles read less. What adds into
// the stream with up to 128 rows also finishes the norm behind it, which outweighs a poor fill. A gated product, which is
// not cut, where one row of tiles fills half of the chip. Below 8 MB of weights (a router, gates) both take the few us of
// their launches, and the calls stay where they were.
extern "C" int ra_gemm_tile_takes(int epilogue, int M, int N, int K) {
  if (M <= 64 || M > 512 || N < 1 || K < 1024 || (size_t)N * K < (4u << 20) || (size_t)N * K * 2 > 0xFFFFFF00ull) return 0;
  const long cus = ra_cu_count(), tiles = tile_count(M, N);
  if (epilogue == 1) return M <= GT_SIDE && tiles <= cus && tiles * 2 > cus;
  int ranges, range_k;
  ra_tile_plan(M, N, K, &ranges, &range_k);
  if (ranges < 2) return 0;
  if (M > 256) return K >= 8192 && tiles * ranges * 4 > cus * 3;
  return (epilogue == 2 && M <= GT_SIDE) || tiles * 4 <= cus || tiles * ranges * 4 >= cus * 3;
}

static int tile_check(const void* A, int lda, const void* W, int M, int N, int K) {
  RA_CHECK(M > 0 && N > 0 && K > 0 && K % 8 == 0 && lda % 8 == 0 && lda >= K && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0,
           "gemm_tile: [%d, %d, %d] with rows of stride %d must be whole 16-byte pieces", M, N, K, lda);
  RA_CHECK((size_t)N * K * 2 <= 0xFFFFFF00ull && ((size_t)M * lda + K) * 2 <= 0x7FFFFF00ull,
           "gemm_tile: an operand of [%d, %d, %d] is larger than a descriptor covers", M, N, K);
  return 0;
}

int ra_tile_ranges(const void* A, int lda, const void* W, float* planes, int M, int N, int K, int ranges, int range_k,
                   hipStream_t stream) {
  if (int rc = tile_check(A, lda, W, M, N, K)) return rc;
  if (M > GT_SIDE && ra_prompt_shape(N, K)) {
    const RaPromptPlan p = ra_prompt_plan(M, N, K, range_k);
    if (p.ranges == ranges) return ra_prompt_product(p, 3, A, W, planes, M, N, K, lda, N, 1.f, stream);
  }
  TileArgs g = tile_args(A, lda, W, M, N, K, ranges, range_k);
  g.c = planes;
  return tile_launch<GT_SIDE, GT_PART>(g, stream);
}

int ra_tile_gated(const void* A, int lda, const void* W, void* C, int ldc, int M, int N, int K, hipStream_t stream) {
  if (int rc = tile_check(A, lda, W, M, N, K)) return rc;
  RA_CHECK(M <= GT_SIDE && N % 16 == 0 && ldc % 4 == 0 && (uintptr_t)C % 8 == 0,
           "gemm_tile: the gate takes up to %d rows, whole runs of 16 features and an aligned result", GT_SIDE);
  TileArgs g = tile_args(A, lda, W, M, N, K, 1, K);
  g.c = C; g.ldc = ldc;
  const int cus = ra_cu_count();
  if ((N + 63) / 64 <= cus) return tile_launch<64, GT_GATED>(g, stream);
  if ((N + 95) / 96 <= cus) return tile_launch<96, GT_GATED>(g, stream);
  return tile_launch<GT_SIDE, GT_GATED>(g, stream);
}
