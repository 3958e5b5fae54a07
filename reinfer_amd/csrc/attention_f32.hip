// Paged attention of the 32-bit path for head sizes 64, 128 and 256; attention_plain.hip says what it computes and keeps
// the other sizes and the bfloat16 twin.
//
// Both products run on the float matrix cores, 16 rows a workgroup: the heads that share a KV head, times tokens of a request. A float product of
// 16x16x4 is a chain of four fused multiply-adds, in order and each rounded, so vector units can walk the same chains: few tokens, whose
// products would be mostly empty columns, go there (attention_f32_token_kernel), and have the same bits. The tiles of 16 keys are dealt
// out to eight shares by their number, each with a running maximum and sums of its own, that are added up through LDS at the end in
// their order; waves take the shares one after the other. So a token's bits follow from its own position, whatever the step holds.
// Both tiles are read in the order they are stored in, 16 bytes a lane, and once for all of a workgroup's rows:
//   keys    are the products' rows and the queries their columns. Lane (slot = lane % 16, hi = lane / 16) has the slot's pieces of 8
//           entries hi, hi + 4, ...; entry e of a half of piece hi + 4 c is step e of chain 2 c + half. (With half as many chains the
//           error against 64 bits is 1.51e-7 of the norm in place of 1.35e-7; it was 1.46e-7 with a query a wave on the vector units);
//   values  are the rows of the second product, lane (entry = lane % 16, four slots from 4 (lane / 16)). The first one's results lie as
//           the second wants its columns: four keys of a row a lane. It starts from zero in every tile and is added to the sums so far.
// What is read of a tile ahead of its turn goes into the registers of the one before: keys behind the first product, values behind the
// second, through descriptors, whose loads past the last tile count like others. (Behind a branch all loads are waited for.)
//
// A query a workgroup on the vector units was bound by reading every tile again for each: four prompts of 60 to 500 tokens, 32 heads of
// 128 on 8 KV heads, 335 us, now 85; one of 600 248 / 62; 300 tokens behind 1000 363 / 97; 500 and 400 of 16 heads of 256 on 4, 318 / 94. On
// the bfloat16 cores, in three parts a float, it was 90 (keys and values split by every wave: 2800 cycles of vector instructions a wave
// and 32 keys), and the decode step below 21.0. Bound now by the matrix cores, busy 30 % of the time, and by loads, which are a tile
// ahead: 31 % of a wave's time; the next tile's scores beside this one's weights took a fifth longer (a wave's last are wasted). Decode
// steps, a token a workgroup: 1 at 300 keys 12.2 / 8.9, 4 of 70 to 505 14.8 / 12.7, 1 at 4000 64.8 / 47.3: bound by trips to memory and
// exchanges; through LDS each costs some hundred cycles, so they are the vector unit's own.
#include "common.h"
#include "reinfer_hip.h"

namespace {

struct F32Attention {
  const float* q;
  int q_stride;
  float* out;
  int out_stride;
  const float *kcache, *vcache;
  const int* block_tables;
  int max_blocks;
  const int *token_list, *seq_of_token, *positions;
  int n_tokens, heads;                     // heads: of a workgroup, of one KV head
  const int* cu_tokens;                    // the requests' first tokens, and the number of tokens behind them
  int n_requests;
  int tiles;                               // of 16 slots, of a block
  unsigned long long share;                // i / tiles is i * share >> 32
  int Hq, Hkv;
  float scale;
  int window, aligned, keep;
  RaScoreMod mod;
  RaHeadOut ho;
};

// Over the four rows of 16 lanes, in the vector unit. (The builtins for the swaps give their first result twice. The waits are the two
// that lie between a write by the vector unit and a swap, and as many behind it.)
__device__ __forceinline__ float sum_rows(float v) {
  float w = v;
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(v), "+v"(w));
  w = v += w;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(v), "+v"(w));
  return v + w;
}
__device__ __forceinline__ float sum_rows_far(float v) {                // the far rows first: (first + third) + (second + fourth)
  float w = v;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(v), "+v"(w));
  w = v += w;
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(v), "+v"(w));
  return v + w;
}
__device__ __forceinline__ float max_rows(float v) {
  float w = v;
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(v), "+v"(w));
  w = v = fmaxf(v, w);
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(v), "+v"(w));
  return fmaxf(v, w);
}
__device__ __forceinline__ int max16(int v) {
#pragma unroll
  for (int m = 8; m > 0; m >>= 1) v = max(v, __shfl_xor(v, m, RA_WAVE));
  return __builtin_amdgcn_readfirstlane(v);
}

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
// of 16 neighbouring lanes: pairs, quads, the mirrored half row and row
__device__ __forceinline__ float max_row(float v) {
  v = fmaxf(v, dpp<0xB1>(v));
  v = fmaxf(v, dpp<0x4E>(v));
  v = fmaxf(v, dpp<0x141>(v));
  return fmaxf(v, dpp<0x140>(v));
}

#define SHARES 8
#define ROWS 16
// Where a chain of a tile's is cut in two, e 0 and 1, 2 and 3: where the error against 64 bits was not below that of the kernel before (64,
// 1e-7 of the norm: a prompt of 600 1.33, whole chains 1.38, 1.25 so), or it costs nothing (values of 128: 1.35 / 1.30; of 256 they
// are registers too many).
#define SPLIT_KEYS(D) ((D) == 64)
#define SPLIT_VALUES(D) ((D) <= 128)

// The tiles of 16 keys that positions see: those with keys that are kept, then those from the first window's first key on. Tile i is share
// i % SHARES's.
struct F32Walk {
  int early, first, last;
  __device__ __forceinline__ int skip(int i) const {
    return i >= early && i < first ? i + (first - i + SHARES - 1) / SHARES * SHARES : i;
  }
};
__device__ __forceinline__ int block_of(const F32Attention& g, int i) { return (int)((unsigned)i * g.share >> 32); }
__device__ __forceinline__ int id_of(const F32Attention& g, const int* table, int i) {
  return ((const __attribute__((address_space(4))) int*)table)[block_of(g, i)];
}
__device__ __forceinline__ size_t base_of(const F32Attention& g, int kvh, int i, int id, int d) {
  return (((size_t)id * g.Hkv + kvh) * g.tiles + (i - block_of(g, i) * g.tiles)) * 16 * d;
}
// The shares' sums of one entry or four, in their order.
template <typename T>
__device__ __forceinline__ T add_shares(const float* ends, int ends_step, const float* sums, int step, float sink, float gate) {
  float top = -INFINITY, den = 0.f;
  for (int w = 0; w < SHARES; ++w) top = fmaxf(top, ends[w * ends_step]);
  T sum = {};
  for (int w = 0; w < SHARES; ++w) {
    const float lw = ends[w * ends_step + 1];
    if (lw == 0.f) continue;               // nothing seen
    const float f = expf(ends[w * ends_step] - top);
    const T y = *(const T*)(sums + w * step);
    if constexpr (sizeof(T) == 4) {
      sum = fmaf(f, y, sum);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[e] = fmaf(f, y[e], sum[e]);
    }
    den = fmaf(f, lw, den);
  }
  den += expf(sink - top);                 // no sink: minus infinity
  return sum * (gate / den);
}

// One share of a token's walk for GH heads of one KV head, by a wave, in the order of the kernel below to the last bit. Its products' chains
// of 16 are a lane each: chain 2 c + half takes entries half * 4 + e of pieces 4 c to 4 c + 3, e by e; chains c and c + w are added for w =
// half of them, a quarter, ...; of the values' it is the keys 0, 4, 8, 12, 1, 5, .... sums [GH][D], ends [GH][2]: maximum and sum.
template <int D, int GH>
__device__ __forceinline__ void walk_share(const F32Attention& g, int t, int h0, const int* table, int share, float* sums, float* ends) {
  constexpr int N = D / 64;                // chains, and entries of the values, of a lane: number lane / 16 + 4 j of the chains and runs
  const int lane = threadIdx.x & 63, lo16 = lane & 15, hi = lane >> 4;
  const int kvh = h0 / (g.Hq / g.Hkv), p = g.positions[t];
  const int lo = ra_first_key(p, g.window, g.aligned), kept = g.keep < lo ? g.keep : lo;
  const F32Walk walk = {(kept + 15) >> 4, lo >> 4, p >> 4};
  int i = walk.skip(share);
  float m[GH], l[GH], acc[GH][N];
#pragma unroll
  for (int h = 0; h < GH; ++h) {
    m[h] = -INFINITY;
    l[h] = 0.f;
#pragma unroll
    for (int j = 0; j < N; ++j) acc[h][j] = 0.f;
  }
  if (i <= walk.last) {
    f32x4_t q[GH][N][4];
    const int piece = (hi >> 1) * 4, half = hi & 1;      // chain hi + 4 j: pieces piece + 8 j + 0 .. 3
#pragma unroll
    for (int h = 0; h < GH; ++h) {
      const float* qv = g.q + (size_t)t * g.q_stride + (size_t)(h0 + h) * D + piece * 8 + half * 4;
#pragma unroll
      for (int j = 0; j < N; ++j)
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
          for (int e = 0; e < 4; ++e) q[h][j][x][e] = qv[j * 64 + x * 8 + e];
    }
    int id = id_of(g, table, i);
    while (true) {
      const int next = walk.skip(i + SHARES);
      const size_t at = base_of(g, kvh, i, id, D);
      f32x4_t k[N][4], v[N][4];
#pragma unroll
      for (int j = 0; j < N; ++j)
#pragma unroll
        for (int x = 0; x < 4; ++x) k[j][x] = *(const f32x4_t*)(g.kcache + at + ((piece + j * 8 + x) * 16 + lo16) * 8 + half * 4);
#pragma unroll
      for (int j = 0; j < N; ++j)
#pragma unroll
        for (int x = 0; x < 4; ++x) v[j][x] = *(const f32x4_t*)(g.vcache + at + (((hi + 4 * j) * 4 + x) * 16 + lo16) * 4);
      id = id_of(g, table, min(next, walk.last));        // the next one's, beside this one's keys
      const int key0 = i * 16, key = key0 + lo16;
      const bool seen = key <= p && (key >= lo || key < kept);
      // slots that nobody has written yet may hold anything: a probability of zero does not make a NaN harmless
      if (key0 + 15 > p || key0 < lo) {
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int at_key = key0 + x * 4 + e;
            const bool any = at_key <= p && (at_key >= lo || at_key < kept);
#pragma unroll
            for (int j = 0; j < N; ++j) v[j][x][e] = any ? v[j][x][e] : 0.f;
          }
      }
#pragma unroll
      for (int h = 0; h < GH; ++h) {
        float z[N];
#pragma unroll
        for (int j = 0; j < N; ++j) {
          float zz = z[j] = 0.f;
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int x = 0; x < 4; ++x) {
              float& to = SPLIT_KEYS(D) && e > 1 ? zz : z[j];
              to = fmaf(k[j][x][e], q[h][j][x][e], to);
            }
          if (SPLIT_KEYS(D)) z[j] += zz;
        }
#pragma unroll
        for (int w = N / 2; w > 0; w >>= 1)
#pragma unroll
          for (int j = 0; j < w; ++j) z[j] += z[j + w];
        const int a = h0 + h;
        float s = sum_rows_far(z[0]) * g.scale;
        if (g.mod.softcap > 0.f || g.mod.r1)
          s = ra_mod_score(s, g.mod.softcap, g.mod.r1 != nullptr, g.mod.r1 ? g.mod.r1[a] : 0.f, g.mod.r1 ? g.mod.r2[a] : 0.f, p - key);
        s = seen ? s : -INFINITY;
        const float top = fmaxf(m[h], max_row(s));
        const float corr = m[h] == -INFINITY ? 0.f : expf(m[h] - top), less = top == -INFINITY ? 0.f : top;      // all may be -inf
        m[h] = top;
        s = expf(s - less);
        l[h] = fmaf(l[h], corr, dpp<0x00>(s)) + dpp<0x55>(s);
        l[h] += dpp<0xAA>(s);
        l[h] += dpp<0xFF>(s);
        float y[2][N];
#pragma unroll
        for (int j = 0; j < N; ++j) y[0][j] = y[1][j] = 0.f;
#define KEY(x, e)                      \
  {                                    \
    const float w = dpp<0x150 + x * 4 + e>(s); \
    for (int j = 0; j < N; ++j) {      \
      float& to = y[SPLIT_VALUES(D) ? e / 2 : 0][j]; \
      to = fmaf(v[j][x][e], w, to);    \
    }                                  \
  }
#define KEYS(e) KEY(0, e) KEY(1, e) KEY(2, e) KEY(3, e)
        KEYS(0) KEYS(1) KEYS(2) KEYS(3)
#undef KEYS
#undef KEY
#pragma unroll
        for (int j = 0; j < N; ++j) acc[h][j] = fmaf(acc[h][j], corr, SPLIT_VALUES(D) ? y[0][j] + y[1][j] : y[0][j]);
      }
      if (next > walk.last) break;
      i = next;
    }
#pragma unroll
    for (int h = 0; h < GH; ++h) {
      l[h] += __shfl_xor(l[h], 4, RA_WAVE);
      l[h] += __shfl_xor(l[h], 8, RA_WAVE);
#pragma unroll
      for (int j = 0; j < N; ++j) sums[h * D + (hi + 4 * j) * 16 + lo16] = acc[h][j];
    }
  }
  if (lane == 0) {
#pragma unroll
    for (int h = 0; h < GH; ++h) {
      ends[h * 2] = m[h];
      ends[h * 2 + 1] = l[h];
    }
  }
}

// The first token of tile y when each request's tokens lie in tiles of nt of their own, and how many it has: none behind the last tile.
__device__ __forceinline__ int tile_of(const F32Attention& g, int nt, int y, int& tokens) {
  const int lane = threadIdx.x & 63;
  if (g.n_requests == 1) {                 // no trip to memory: a prompt of 700 73.7 us, with it 76.6
    tokens = max(0, min(nt, g.n_tokens - y * nt));
    return y * nt;
  }
  tokens = 0;
  for (int s0 = 0; s0 < g.n_requests; s0 += RA_WAVE) {
    const int s = s0 + lane, first = g.cu_tokens[min(s, g.n_requests)], past = g.cu_tokens[min(s + 1, g.n_requests)];
    const int mine = (past - first + nt - 1) / nt;
    int upto = mine;                       // of the requests up to the lane's
#pragma unroll
    for (int m = 1; m < RA_WAVE; m <<= 1) {
      const int other = __shfl_up(upto, m, RA_WAVE);
      upto += lane >= m ? other : 0;
    }
    const unsigned long long here = __ballot(y < upto);
    if (here) {
      const int l = __builtin_amdgcn_readfirstlane(__ffsll(here) - 1);
      const int at = __builtin_amdgcn_readlane(first, l) + (y - __builtin_amdgcn_readlane(upto - mine, l)) * nt;
      tokens = min(nt, __builtin_amdgcn_readlane(past, l) - at);
      return at;
    }
    y -= __builtin_amdgcn_readlane(upto, RA_WAVE - 1);
  }
  return 0;
}

// 16 rows: tokens of a request times the heads of a KV head.
template <int D, int WAVES>
__global__ void __launch_bounds__(WAVES * RA_WAVE) attention_f32_kernel(F32Attention g) {
  constexpr int KP = D / 32;               // pieces of 8 entries of a key a lane
  constexpr int VP = D / 16;               // runs of 16 entries of the values
  constexpr int LD = D + 4;
  // of a fixed size: one that is told at the launch and is above 64 KB is a host call more at each
  __shared__ __attribute__((aligned(16))) float part[SHARES * ROWS * LD], ends[SHARES * ROWS * 2];       // maximum and sum
  __shared__ int off[ROWS];                // rows with a result that is no finite number
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  const int lo16 = lane & 15, hi = lane >> 4;
  const int gh = g.heads;
  const int h0 = blockIdx.x * gh, kvh = h0 / (g.Hq / g.Hkv), a = h0 + lo16 % gh;
  int tokens;                              // the last ones first: theirs are the longest walks of a prompt
  const int i0 = tile_of(g, ROWS / gh, gridDim.y - 1 - blockIdx.y, tokens), rows = tokens * gh;
  if (rows == 0) return;
  const int t = i0 + min(lo16, rows - 1) / gh, pos = g.positions[t];
  float q[KP][8];                          // the products' columns
  {
    const float* qv = g.q + (size_t)t * g.q_stride + (size_t)a * D + hi * 8;
#pragma unroll
    for (int c = 0; c < KP; ++c)
#pragma unroll
      for (int e = 0; e < 8; ++e) q[c][e] = qv[c * 32 + e];
  }
  const float d1 = g.mod.r1 ? g.mod.r1[a] : 0.f, d2 = g.mod.r1 ? g.mod.r2[a] : 0.f;

  const bool mine = lo16 < rows;
  const int* table = g.block_tables + (size_t)__builtin_amdgcn_readfirstlane(g.seq_of_token[i0]) * g.max_blocks;
  const int p = mine ? pos : -1;         // a row that is not there sees nothing
  const int lo = mine ? ra_first_key(p, g.window, g.aligned) : 0;
  const int kept = mine ? (g.keep < lo ? g.keep : lo) : 0;
  const int end = max16(p), from = -max16(mine ? -lo : -0x7fffffff), keeps = max16(kept);      // over the rows
  const F32Walk walk = {(keeps + 15) >> 4, from >> 4, end >> 4};
  const int last = walk.last;
  for (int share = wave; share < SHARES; share += waves) {
    int i = walk.skip(share);
    if (i > last) {                      // a share without a tile
      if (lane < ROWS) {
        ends[(share * ROWS + lane) * 2] = -INFINITY;
        ends[(share * ROWS + lane) * 2 + 1] = 0.f;
      }
      continue;
    }
    float m = -INFINITY, l = 0.f;
    f32x4_t acc[VP], k[KP][2], v[VP];
#pragma unroll
    for (int b = 0; b < VP; ++b) acc[b] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    // behind the last tile a load counts like any other, and neither reads memory nor makes the others' wait a longer one
    auto load_keys = [&](int i, int id) {
      const auto tile = __builtin_amdgcn_make_buffer_rsrc((void*)(g.kcache + base_of(g, kvh, i, id, D)), 0, i <= last ? 16 * D * 4 : 0, 0x00020000);
#pragma unroll
      for (int c = 0; c < KP; ++c)
#pragma unroll
        for (int e = 0; e < 2; ++e)
          k[c][e] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(tile, (hi * 16 + lo16) * 32, c * 2048 + e * 16, 0));
    };
    auto load_values = [&](int i, int id) {
      const auto tile = __builtin_amdgcn_make_buffer_rsrc((void*)(g.vcache + base_of(g, kvh, i, id, D)), 0, i <= last ? 16 * D * 4 : 0, 0x00020000);
#pragma unroll
      for (int b = 0; b < VP; ++b)
        v[b] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(tile, (hi * 16 + lo16) * 16, b * 1024, 0));
    };
    int id = id_of(g, table, i), next = walk.skip(i + SHARES);
    load_keys(i, id);
    load_values(i, id);
    id = id_of(g, table, min(next, last));
    for (; i <= last;) {
      const int then = walk.skip(next + SHARES), id2 = id_of(g, table, min(then, last));
      f32x4_t z[2 * KP], zz[2 * KP];
#pragma unroll
      for (int c = 0; c < 2 * KP; ++c) z[c] = zz[c] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int c = 0; c < 2 * KP; ++c) {
          f32x4_t& to = SPLIT_KEYS(D) && e > 1 ? zz[c] : z[c];
          to = __builtin_amdgcn_mfma_f32_16x16x4f32(k[c >> 1][c & 1][e], q[c >> 1][(c & 1) * 4 + e], to, 0, 0, 0);
        }
      load_keys(next, id);
      if (SPLIT_KEYS(D)) {
#pragma unroll
        for (int c = 0; c < 2 * KP; ++c) z[c] += zz[c];
      }
#pragma unroll
      for (int w = KP; w > 0; w >>= 1)
#pragma unroll
        for (int c = 0; c < w; ++c) z[c] += z[c + w];
      const int key0 = i * 16 + hi * 4;
      float s[4], top = m;
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = z[0][e] * g.scale;
      if (g.mod.softcap > 0.f || g.mod.r1) {
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] = ra_mod_score(s[e], g.mod.softcap, g.mod.r1 != nullptr, d1, d2, p - key0 - e);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int key = key0 + e;
        s[e] = key <= p && (key >= lo || key < kept) ? s[e] : -INFINITY;
        top = fmaxf(top, s[e]);
      }
      top = max_rows(top);
      const float corr = m == -INFINITY ? 0.f : expf(m - top), less = top == -INFINITY ? 0.f : top;      // all may be -inf
      m = top;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[e] = expf(s[e] - less);
        l = e == 0 ? fmaf(l, corr, s[0]) : l + s[e];
      }
      // slots that nobody has written yet may hold anything: a probability of zero does not make a NaN harmless
      if (i * 16 + 15 > end || i * 16 < from) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int key = key0 + e;
          const bool any = key <= end && (key >= from || key < keeps);
#pragma unroll
          for (int b = 0; b < VP; ++b) v[b][e] = any ? v[b][e] : 0.f;
        }
      }
      f32x4_t y[2][VP];
#pragma unroll
      for (int b = 0; b < VP; ++b) y[0][b] = y[1][b] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int b = 0; b < VP; ++b) {
          f32x4_t& to = y[SPLIT_VALUES(D) ? e / 2 : 0][b];
          to = __builtin_amdgcn_mfma_f32_16x16x4f32(v[b][e], s[e], to, 0, 0, 0);
        }
      load_values(next, id);
#pragma unroll
      for (int b = 0; b < VP; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[b][e] = fmaf(acc[b][e], corr, SPLIT_VALUES(D) ? y[0][b][e] + y[1][b][e] : y[0][b][e]);
      i = next;
      next = then;
      id = id2;
    }
    l = sum_rows(l);
    float* row = part + (share * ROWS + lo16) * LD;
#pragma unroll
    for (int b = 0; b < VP; ++b) *(f32x4_t*)(row + b * 16 + hi * 4) = acc[b];
    if (hi == 0) {
      ends[(share * ROWS + lo16) * 2] = m;
      ends[(share * ROWS + lo16) * 2 + 1] = l;
    }
  }
  if (threadIdx.x < ROWS) off[threadIdx.x] = 0;
  __syncthreads();
  for (int x = threadIdx.x; x < rows * (D / 4); x += blockDim.x) {
    const int r = x / (D / 4), e0 = x % (D / 4) * 4, head = h0 + r % gh, token = i0 + r / gh;
    const f32x4_t y = add_shares<f32x4_t>(ends + r * 2, ROWS * 2, part + r * LD + e0, ROWS * LD,
                                          g.ho.sink ? g.ho.sink[head] : -INFINITY, ra_head_gate<float>(g.ho, token, head));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (!(fabsf(y[e]) <= 3.402823466e38f)) off[r] = 1;
      g.out[(size_t)token * g.out_stride + (size_t)head * D + e0 + e] = y[e];
    }
  }
  __syncthreads();
  // A key that a row does not see weighs zero there, and zero times a value that is no finite number is none: a row with such a result
  // is worked out again, from the keys it sees alone.
  for (int r = 0; r < rows; ++r) {
    if (!off[r]) continue;
    const int head = h0 + r % gh, token = i0 + r / gh;
    __syncthreads();
    for (int share = wave; share < SHARES; share += waves)
      walk_share<D, 1>(g, token, head, table, share, part + share * D, ends + share * 2);
    __syncthreads();
    for (int e = threadIdx.x; e < D; e += blockDim.x)
      g.out[(size_t)token * g.out_stride + (size_t)head * D + e] = add_shares<float>(
          ends, 2, part + e, D, g.ho.sink ? g.ho.sink[head] : -INFINITY, ra_head_gate<float>(g.ho, token, head));
  }
}

// A token on its own, a share a wave.
template <int D, int GH>
__global__ void __launch_bounds__(SHARES * RA_WAVE) attention_f32_token_kernel(F32Attention g) {
  __shared__ float part[SHARES][GH][D], ends[SHARES][GH][2];
  const int share = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h0 = blockIdx.x * GH;
  const int t = g.token_list ? g.token_list[blockIdx.y] : blockIdx.y;
  walk_share<D, GH>(g, t, h0, g.block_tables + (size_t)g.seq_of_token[t] * g.max_blocks, share, part[share][0], ends[share][0]);
  __syncthreads();
  for (int x = threadIdx.x; x < GH * D; x += blockDim.x) {
    const int h = x / D, e = x % D, a = h0 + h;
    g.out[(size_t)t * g.out_stride + (size_t)a * D + e] = add_shares<float>(
        &ends[0][h][0], GH * 2, &part[0][h][e], GH * D, g.ho.sink ? g.ho.sink[a] : -INFINITY, ra_head_gate<float>(g.ho, t, a));
  }
}

template <int D, int GH>
int go_tokens(const F32Attention& g, hipStream_t stream) {
  attention_f32_token_kernel<D, GH><<<dim3(g.Hq / GH, g.n_tokens), SHARES * RA_WAVE, 0, stream>>>(g);
  RA_LAUNCH_CHECK("attention_f32");
  return 0;
}

template <int D>
int go(F32Attention g, hipStream_t stream) {
  const int group = g.Hq / g.Hkv;
  const long cus = ra_cu_count();
  // all heads of a group, or as many of them as tokens fill 12 of the 16 rows with at least: keys and values are read once for them
  g.heads = 1;
  for (int h = 2; h <= ROWS; ++h)
    if (group % h == 0 && ROWS / h * h >= 12) g.heads = h;
  const int nt = ROWS / g.heads;
  // Tokens on their own until their workgroups wait for one another, and where the products' 16 columns would stay all but empty; a request's
  // tokens share what is read of its keys in the caches either way and go further so. Two heads of single tokens share what is read
  // of a key they both read, but for so few that the chip has room for each. us, a head each / two / 16 rows: 32 heads of 128 on 8 KV
  // heads at 300 keys, 4 tokens of 4 requests 12.4 / 10.5 / 16.0, 8 of 8 17.4 / 12.5 / 16.0, 16 of 16 29.5 / 17.9 / 17.6, 64 of 64 95 / 54 / 33; a
  // prompt of 24 9.3 / 9.7 / 11.2, 33 11.5 / 12.6 / 11.2, 64 15.6 / 16.5 / 11.6, 250 69 / 76 / 21, 24 tokens behind 1000 36 / 34 / 32; 8 single
  // ones beside a portion of 100 37 / 32 / 21 (of 40 heads 41 / - / 21). 32 on 32: 64 of 64 at 300 112 / - / 122, a prompt of 64 15.6 / -
  // / 11.8. 16 of 64 on 16: prompts of 64 7.6 / - / 9.4, 128 11.5 / - / 10.6, 250 22 / - / 12.5. 16 of 256 on 2: 8 of 8 at 300 17.7 / - / 26,
  // 16 of 16 27.8 / - / 26.3, 64 of 64 92 / - / 29. Over 29 steps of 13 shapes what is taken is nowhere more than 28 % behind the best (24 tokens
  // behind 1000, two heads would be ahead), in 17 of 377 more than 10 %.
  const bool two = D <= 128 && group % 2 == 0;
  const int each = g.n_requests > 0 ? g.n_tokens / g.n_requests : 1;        // tokens of a request, or so
  const double alone = (double)g.Hq * g.n_tokens / cus;                    // workgroups of a head and token, a CU's share
  const bool pair = two && each < 4 && alone > (D == 64 ? 0.75 : 0.35);
  const double least = each < 2 ? (D == 64 ? 1.25 : 1.0) : each < 4 ? 2.0 : D == 64 ? 6.0 : D == 128 ? 3.5 : 2.8;
  if (g.n_requests == 0 || g.heads * (each < nt ? each : nt) < 3 || alone < least * (pair ? 2 : 1)) {
    if constexpr (D <= 128)
      if (pair) return go_tokens<D, 2>(g, stream);
    return go_tokens<D, 1>(g, stream);
  }
  // eight waves, a share each, while that leaves CUs without a workgroup: 33 tokens behind 300 18.4 us, of four waves 20.2; 250 from their start 24.5
  // and 20.9
  const long pairs = g.Hq / g.heads, tiles = (g.n_tokens - g.n_requests) / nt + g.n_requests;        // at most
  const int waves = D > 128 || pairs * tiles > cus ? 4 : 8;
  constexpr int W = D <= 128 ? 8 : 4;
  attention_f32_kernel<D, W><<<dim3(pairs, tiles), waves * RA_WAVE, 0, stream>>>(g);
  RA_LAUNCH_CHECK("attention_f32");
  return 0;
}

}  // namespace

// Whether the kernel takes these sizes (16-byte reads of the cache besides; the queries are read element by element).
bool ra_attention_f32_takes(const void* kcache, const void* vcache, int d, int block_size, int max_blocks) {
  const long tiles = block_size / 16;      // a block's, and the range in which a product stands for a division by them
  return (d == 64 || d == 128 || d == 256) && (uintptr_t)kcache % 16 == 0 && (uintptr_t)vcache % 16 == 0
         && max_blocks * tiles * tiles < (1l << 32);
}

int ra_attention_f32(const float* q, int q_stride, float* out, int out_stride, const float* kcache, const float* vcache,
                     const int* block_tables, int max_blocks, const int* token_list, const int* seq_of_token,
                     const int* positions, int n_tokens, const int* cu_tokens, int n_requests, int block_size, int Hq, int Hkv, int d, float scale,
                     int window, int aligned, int keep, RaScoreMod mod, RaHeadOut ho, hipStream_t stream) {
  const F32Attention g = {q, q_stride, out, out_stride, kcache, vcache, block_tables, max_blocks, token_list, seq_of_token,
                          positions, n_tokens, 1, cu_tokens, n_requests, block_size / 16, (1ull << 32) / (block_size / 16) + 1, Hq, Hkv, scale, window, aligned, keep, mod, ho};
  if (d == 64) return go<64>(g, stream);
  if (d == 128) return go<128>(g, stream);
  if (d == 256) return go<256>(g, stream);
  return ra_fail("attention_f32: head size %d", d);
}
