// Matrix products of the 32-bit path, C[M,N] = A[M,K] . W[N,K]^T (+ bias[N]), on the float matrix cores: the products are
// full float ones and the sums are float, as in gemm_plain.hip, which keeps the rows that 16-byte accesses cannot read.
//
// An operand of a 16x16x4 product is one float a lane at (row, k slot). Which k a slot stands for is free as long as both
// operands agree, so a lane reads four neighbouring k with one 16-byte access and the four products that follow take one
// element of it each.
//
// Up to 32 rows (gemm_f32_stream_kernel) the product is bound by reading the weights once. A workgroup has 16 features, its
// waves share K out and add their sums through LDS in a fixed order. The activations go from memory to the matrix cores, the
// weights by way of a piece of LDS of each wave's own: loaded in the products' order a load is 64 bytes of each of 16 rows, half a
// line each, and takes twice the time of whole lines of 4 rows (weights from memory at 4 rows, straight / by way of LDS: 6144 x 2560
// 23.6 / 20.0 us, 2560 x 4096 17.7 / 14.3, 19456 x 2560 45.8 / 41.6, 2560 x 9728 33.2 / 29.4, 151936 x 2560 298 / 265; at 32 rows
// 19456 x 2560 100 / 82; a product of 1000 x 1028, all start and end, 10.2 / 11.0). Three or four runs in flight instead of two
// change nothing. With more rows the activations, which every workgroup reads again, cost as much as the weights.
//
// From 33 rows on (gemm_f32_tile_kernel) tiles of both operands go through LDS, 32 k at a time, by loads that go straight
// there; two stages and one barrier a step. The float matrix cores do 256 flops a clock and CU and bound it. Tiles of 64 x 128
// leave room in LDS for three workgroups whose waits fall at different times; 128 x 128 with two or four stages had the
// matrix cores 70 to 83 % busy, deeper rings changed nothing. In a loop over other weights 1119 x 19456 x 2560 takes 0.87 ms
// (128 TFLOP/s of 157), 1119 x 2560 x 9728 0.47, 300 x 2560 x 9728 0.144; with 32x32x2 products, whose order of sums is
// another one than the other kernel's, 0.89, 0.51 and 0.155.
#include "common.h"
#include "reinfer_hip.h"

namespace {

// ------------------------------------------------------------------------------------------------ the order of the sums
// K is summed in up to eight blocks of at least 512 k, whose number and length follow from K alone. A block is one chain of
// 16x16x4 products over its pieces of 16 k: the four products of a piece take k 0, 4, 8, 12, then 1, 5, 9, 13, ... The blocks'
// sums are added in their order, then the bias. Both kernels keep this order, so a row's result does not depend on how many
// rows stand beside it: a request's 32-bit results are the same bits alone and in any step.
struct KBlocks {
  int n, k;                                // how many, and k of one (a multiple of 32)
};
KBlocks k_blocks(int K) {
  int n = K / 512;
  n = n < 1 ? 1 : n > 8 ? 8 : n;
  const int k = ((K + n - 1) / n + 31) / 32 * 32;
  return {(K + k - 1) / k, k};
}

// ------------------------------------------------------------------------------------------------ up to 32 rows
// Workgroups that stay: tile b, b + grid, ... of 16 features, all M rows (MT tiles of 16), a wave a block of K. A wave's loads
// run DEPTH runs of 32 U k ahead, on across the ends of tiles, and are unconditional: through a buffer descriptor a load past
// its end returns zeros and touches no memory, so rows past N or M, pieces past the block and runs past the last tile count
// like any other load and cost nothing. A tile's runs are padded to a multiple of DEPTH, so that it ends where a round of the
// ring does.
#define RA_WAVE_HANDOVER                                   \
  do {                                                     \
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); \
    __builtin_amdgcn_wave_barrier();                       \
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront"); \
  } while (0)
template <int MT, int U, int DEPTH>
__global__ void __launch_bounds__(8 * RA_WAVE, 4)
gemm_f32_stream_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                       float* __restrict__ C, int M, int N, int K, int lda, int ldc, int block_k) {
  constexpr int SPAN = U * 32;             // k of one run of a wave
  constexpr unsigned NOWHERE = 0xFFFFFFF0u;
  constexpr int CH = SPAN / 4;             // 16-byte pieces of a weight row in a run
  __shared__ f32x4_t sums[2][8][MT][RA_WAVE];            // of one tile while the next one's may already be written
  __shared__ f32x4_t laid[8][16 * CH];                   // a wave's run of weights on its way into the products' order
  const int lane = threadIdx.x & 63, waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int k0 = wave * block_k, k1 = min(k0 + block_k, K);
  const int n_steps = (block_k + SPAN - 1) / SPAN;       // the same for every wave: all meet at a tile's end
  const int n_steps_p = (n_steps + DEPTH - 1) / DEPTH * DEPTH;
  const int n_tiles = (N + 15) / 16;
  const int n_mine = (n_tiles - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
  const int total = n_mine * n_steps_p;
  const __amdgpu_buffer_rsrc_t w_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(W), 0, (int)((size_t)N * K * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t a_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(A), 0, (int)(((size_t)(M - 1) * lda + K) * 4), 0x00020000);
  // A load of weights takes whole lines of a few rows, lane after lane; piece c of row r of a run lies at place c ^ r in LDS, from
  // where the products' rows are read without conflicts.
  constexpr int LOADS = U * 2, LR = 16 / LOADS;          // loads of a run, rows of one
  const int wr = lane / CH, wc = lane % CH;
  f32x4_t w[DEPTH][LOADS], a[DEPTH][U][MT][2];
  int l_q = 0, l_step = 0, l_n = (int)blockIdx.x * 16;             // where the loads are
#define RA_F32_LOAD(d)                                                                                        \
  do {                                                                                                        \
    const bool live_ = l_q < total && l_step < n_steps;                                                       \
    _Pragma("unroll") for (int i = 0; i < LOADS; ++i) {                                                       \
      const int k_ = k0 + l_step * SPAN + wc * 4, n_ = l_n + i * LR + wr;                                     \
      const unsigned off_ = live_ && k_ < k1 && n_ < N ? (unsigned)(((size_t)n_ * K + k_) * 4) : NOWHERE;     \
      w[d][i] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, off_, 0, 0));       \
    }                                                                                                         \
    _Pragma("unroll") for (int u = 0; u < U; ++u)                                                             \
      _Pragma("unroll") for (int j = 0; j < 2; ++j) {                                                         \
        const int k_ = k0 + l_step * SPAN + u * 32 + j * 16 + q * 4;                                          \
        const bool ok_ = live_ && k_ < k1;           /* a multiple of 4 */                                    \
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
      // this wave's alone: LDS takes its accesses in their order, and the fences have the compiler keep that order where lanes
      // read what others wrote, and write what others have read
      f32x4_t* const mine = laid[wave];
      RA_WAVE_HANDOVER;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) mine[(i * LR + wr) * CH + (wc ^ ((i * LR + wr) & (CH - 1)))] = w[d][i];
      RA_WAVE_HANDOVER;
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const f32x4_t y = mine[r * CH + (((u * 2 + j) * 4 + q) ^ (r & (CH - 1)))];
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int t = 0; t < MT; ++t)
              acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(y[e], a[d][u][t][j][e], acc[t], 0, 0, 0);
        }
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
    for (int t = wave; t < MT; t += waves) {
      f32x4_t v = sums[buf][0][t][lane];
#pragma unroll
      for (int x = 1; x < 8; ++x)
        if (x < waves) v += sums[buf][x][t][lane];
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
#undef RA_F32_LOAD
}

// ------------------------------------------------------------------------------------------------ from 33 rows on
#define F32_BK 32

struct F32Tile {
  const float* a;
  const float* w;
  const float* bias;
  float* c;                                // ranges > 1: the blocks' sums, [blocks][M][N]
  int M, N, K, lda, ldc, m_tiles, n_tiles, ranges;
  int block_k, range_blocks;               // k of a block (a multiple of 32), blocks of a range
};

// One workgroup of four waves a tile of BM rows and BN features and range of k, in 2 x 2 quarters. A stage is 32 k of both
// operands, rows of 8 pieces of 16 bytes, piece p of row r at place p ^ (r % 8), so that eight rows' reads of one piece fall
// on different banks; loads that go straight to LDS write it in the order of their lanes, so it is their addresses that are
// permuted. A tile's operands have descriptors of their own, whose ends are those of the matrices: rows past them are zeros.
template <int BM, int BN, int STAGES, bool CUT>
__global__ void __launch_bounds__(256) gemm_f32_tile_kernel(F32Tile g) {
  constexpr int TM = BM / 32, TN = BN / 32;                       // 16 x 16 tiles a side of a wave's quarter
  constexpr int ROWS = BM + BN, PA = BM / 32, PB = BN / 32;       // a wave's loads a stage: 8 rows (1 KB) each
  constexpr unsigned NOWHERE = 0xFFFFFFF0u;
  __shared__ __attribute__((aligned(1024))) float lds[STAGES * ROWS * F32_BK];
  // the row tiles of a panel and range of weights follow one another, and each XCD gets a run of tiles
  const long total = (long)g.m_tiles * g.n_tiles * g.ranges, each = (total + RA_XCDS - 1) / RA_XCDS;
  const long at = blockIdx.x / RA_XCDS, tile = blockIdx.x % RA_XCDS * each + at;
  if (at >= each || tile >= total) return;
  const int m0 = (int)(tile % g.m_tiles) * BM;
  const int z = (int)(tile / g.m_tiles % g.ranges), n0 = (int)(tile / g.m_tiles / g.ranges) * BN;
  const int range_k = g.block_k * g.range_blocks, block_steps = g.block_k / F32_BK;
  const int k0 = z * range_k, k1 = min(k0 + range_k, g.K), steps = (k1 - k0 + F32_BK - 1) / F32_BK;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int a_rows = min(BM, g.M - m0), w_rows = min(BN, g.N - n0);
  const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(g.a + (size_t)m0 * g.lda), 0, (int)(((size_t)(a_rows - 1) * g.lda + g.K) * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(g.w + (size_t)n0 * g.K), 0, (int)((size_t)w_rows * g.K * 4), 0x00020000);
  const int piece = (lane & 7) ^ (lane >> 3);
  unsigned a_off[PA], w_off[PB];
#pragma unroll
  for (int i = 0; i < PA; ++i) {
    const int r = (wave * PA + i) * 8 + (lane >> 3);
    a_off[i] = r < a_rows ? (unsigned)(((size_t)r * g.lda + piece * 4) * 4) : 0x80000000u;
  }
#pragma unroll
  for (int i = 0; i < PB; ++i) {
    const int r = (wave * PB + i) * 8 + (lane >> 3);
    w_off[i] = r < w_rows ? (unsigned)(((size_t)r * g.K + piece * 4) * 4) : 0x80000000u;
  }
  auto fetch = [&](int s, int buf) {
    const int k = k0 + s * F32_BK;
    const unsigned past = k + piece * 4 < k1 ? 0u : NOWHERE;      // pieces past the range's end become zeros
    float* to = lds + buf * ROWS * F32_BK;
#pragma unroll
    for (int i = 0; i < PA; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          a_rsrc, (__attribute__((address_space(3))) void*)(to + (wave * PA + i) * 8 * F32_BK), 16,
          (int)((a_off[i] + (unsigned)k * 4u) | past), 0, 0, 0);
#pragma unroll
    for (int i = 0; i < PB; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          w_rsrc, (__attribute__((address_space(3))) void*)(to + (BM + (wave * PB + i) * 8) * F32_BK), 16,
          (int)((w_off[i] + (unsigned)k * 4u) | past), 0, 0, 0);
  };
  f32x4_t sum[TN][TM];                       // of the blocks before this one
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) sum[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
  const int row = lane & 15, quarter = lane >> 4;
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s) fetch(s, s);
  const int ld = CUT ? g.N : g.ldc;
  const float* b = CUT ? nullptr : g.bias;
  const bool whole = g.N % 4 == 0 && ld % 4 == 0 && (uintptr_t)g.c % 16 == 0;
  int buf = 0;
  for (int s = 0, block = z * g.range_blocks; s < steps; ++block) {
    f32x4_t acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    const int end = min(s + block_steps, steps);
    for (; s < end; ++s) {
      // this wave's loads of stage s are done when only those of the stages behind it are left (and, behind a block's end, its
      // stores), its reads of the stage that is
      // asked for next when no LDS read is left
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((PA + PB) * (STAGES - 2)) : "memory");
      fetch(s + STAGES - 1, buf == 0 ? STAGES - 1 : buf - 1);
      const float* as = lds + buf * ROWS * F32_BK + (wm + row) * F32_BK;
      const float* ws = lds + buf * ROWS * F32_BK + (BM + wn + row) * F32_BK;
#pragma unroll
      for (int kk = 0; kk < F32_BK / 16; ++kk) {
        f32x4_t x[TM], y[TN];
        const int p = ((kk * 4 + quarter) ^ (row & 7)) * 4;
#pragma unroll
        for (int j = 0; j < TM; ++j) x[j] = *(const f32x4_t*)(as + j * 16 * F32_BK + p);
#pragma unroll
        for (int i = 0; i < TN; ++i) y[i] = *(const f32x4_t*)(ws + i * 16 * F32_BK + p);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < TN; ++i)
#pragma unroll
            for (int j = 0; j < TM; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(y[i][e], x[j][e], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);     // one piece's operands at a time: three workgroups a CU have registers for no more
      }
      buf = buf + 1 == STAGES ? 0 : buf + 1;
    }
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
    }
  }
}

// C = the blocks' sums added in their order (+ bias): a workgroup takes 1024 features of a row, four a thread, read 16 bytes at
// a time where rows allow it. It is bound by reading the planes.
__global__ void __launch_bounds__(256)
gemm_f32_add_kernel(const float* __restrict__ part, int ranges, const float* __restrict__ bias, float* __restrict__ C,
                    int M, int N, int ldc, bool whole) {
  const int n = (blockIdx.y * 256 + threadIdx.x) * 4;
  if (n >= N) return;
  const size_t m = blockIdx.x, size = (size_t)M * N;
  const float* p = part + m * N + n;
  float* c = C + m * ldc + n;
  if (whole) {
    f32x4_t v = *(const f32x4_t*)p;
    for (int r = 1; r < ranges; ++r) v += *(const f32x4_t*)(p + r * size);
    if (bias)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += bias[n + e];
    *(f32x4_t*)c = v;
    return;
  }
  for (int e = 0; e < 4 && n + e < N; ++e) {
    float v = p[e];
    for (int r = 1; r < ranges; ++r) v += p[r * size + e];
    c[e] = bias ? v + bias[n + e] : v;
  }
}

// The tile kernel's plan: tiles of 64 x 128 or 64 x 64, and how many of K's blocks a workgroup takes (it adds them in its
// registers; several ranges of blocks go to planes that the adding kernel adds). The price is a CU's share of the workgroups at
// the share of the matrix cores' rate that so many side by side reach (measured), and the planes written and read again.
struct TilePlan {
  int bn, blocks, block_k, range_blocks, ranges;
};
TilePlan tile_plan(int M, int N, int K) {
  const long cus = ra_cu_count();
  const double reached[2][3] = {{0.70, 0.78, 0.81}, {0.79, 0.85, 0.87}};
  const int blocks = k_blocks(K).n, block_k = k_blocks(K).k;
  TilePlan best = {};
  double best_us = 0.0;
  for (int wide = 0; wide < 2; ++wide) {
    const int bn = wide ? 128 : 64;
    const long tiles = (long)((M + 63) / 64) * ((N + bn - 1) / bn);
    const double block_us = 64.0 * bn * 2.0 * block_k / 614e3;                // one tile's block at a CU's full rate
    for (int take = blocks; take >= 1; --take) {
      const int ranges = (blocks + take - 1) / take;
      const long load = (tiles * ranges + cus - 1) / cus;
      double us = (double)load * take * block_us / reached[wide][load < 3 ? load - 1 : 2];
      if (ranges > 1) us += 3.0 + (double)blocks * M * N * 8.0 / 5e6;
      if (best.bn == 0 || us < best_us) {
        best = {bn, blocks, block_k, take, ranges};
        best_us = us;
      }
    }
  }
  return best;
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
#define RA_GO(MT, U, DEPTH, GRID) \
  gemm_f32_stream_kernel<MT, U, DEPTH><<<(GRID) < tiles ? (GRID) : tiles, kb.n * RA_WAVE, 0, stream>>>( \
      A, w, b, C + n0, M, n, K, lda, ldc, kb.k)
      // as many workgroups as the registers hold, 16 waves a CU
      const int grid = 16 / kb.n * cus;
      if (M > 16) RA_GO(2, 1, 3, grid);
      else RA_GO(1, 2, 2, grid);
#undef RA_GO
      RA_LAUNCH_CHECK("gemm_f32");
    }
    return 0;
  }
  const TilePlan p = tile_plan(M, N, K);
  const bool cut = p.ranges > 1;
  RA_CHECK(!cut || (scratch && scratch_floats >= (long)p.blocks * M * N), "gemm_f32: scratch of %ld floats, needs %ld",
           scratch_floats, (long)p.blocks * M * N);
  F32Tile g = {A, W, bias, cut ? scratch : C, M, N, K, lda, ldc, (M + 63) / 64, (N + p.bn - 1) / p.bn, p.ranges,
               p.block_k, p.range_blocks};
  const long total = (long)g.m_tiles * g.n_tiles * g.ranges, blocks = (total + RA_XCDS - 1) / RA_XCDS * RA_XCDS;
  RA_CHECK(blocks <= 0x7FFFFFFFL, "gemm_f32: [%d, %d] in one launch", M, N);
  if (p.bn == 128 && cut) gemm_f32_tile_kernel<64, 128, 2, true><<<(unsigned)blocks, 256, 0, stream>>>(g);
  else if (p.bn == 128) gemm_f32_tile_kernel<64, 128, 2, false><<<(unsigned)blocks, 256, 0, stream>>>(g);
  else if (cut) gemm_f32_tile_kernel<64, 64, 2, true><<<(unsigned)blocks, 256, 0, stream>>>(g);
  else gemm_f32_tile_kernel<64, 64, 2, false><<<(unsigned)blocks, 256, 0, stream>>>(g);
  RA_LAUNCH_CHECK("gemm_f32");
  if (cut) {
    const bool whole = N % 4 == 0 && ldc % 4 == 0 && (uintptr_t)C % 16 == 0 && (uintptr_t)scratch % 16 == 0;
    gemm_f32_add_kernel<<<dim3(M, (N + 1023) / 1024), 256, 0, stream>>>(scratch, p.blocks, bias, C, M, N, ldc, whole);
    RA_LAUNCH_CHECK("gemm_f32 (ranges)");
  }
  return 0;
}
