// Paged attention of the 32-bit path for head sizes 64, 128 and 256; attention_plain.hip says what it computes and keeps
// the other sizes and the bfloat16 twin.
//
// A workgroup has one token and GH query heads of one KV head. The tiles of 16 keys are dealt out to eight shares, each with a
// running maximum and sums of its own, that are added up through LDS at the end in their order; its waves, two or eight, take
// the shares one after the other. So the order of a token's sums follows from its own position, whatever the step holds. Both
// tiles are read in the order they are stored in, 16 bytes a lane, and once for all GH heads:
//   keys    lane (slot = lane % 16, part = lane / 16) has the slot's pieces of 8 entries number part, part + 4, ...: its
//           share of the scores is a product with queries that stay in registers, two exchanges add the four shares;
//   values  lane (entry = lane % 16, four slots from 4 (lane / 16)) has four keys' values of one entry of every run of 16.
// The plain kernel reads an element a lane and access and walks the values key by key: bound by the latency of those reads.
// Four requests with prompts of 60 to 500 tokens and 12 further ones each, 32 heads of 128 on 8 KV heads: its calls take
// 339 us on average there, 33 us here. (Eight shares whatever the step holds cost prompts the sums' ends: 497 tokens from their
// start 169 us, 139 where each of two waves had one set of sums.) What bounds it now is the vector unit in prompts (every query reads the tiles from
// the caches again) and the trips to memory of a short walk in decode steps.
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
  int block_size, Hq, Hkv;
  float scale;
  int window, aligned, keep;
  RaScoreMod mod;
  RaHeadOut ho;
};

__device__ __forceinline__ float max16(float v) {
#pragma unroll
  for (int m = 8; m > 0; m >>= 1) v = fmaxf(v, __shfl_xor(v, m, RA_WAVE));
  return v;
}

#define SHARES 8

template <int D, int GH>
__global__ void __launch_bounds__(SHARES * RA_WAVE) attention_f32_kernel(F32Attention g) {
  constexpr int KP = D / 32;               // pieces of 8 entries of a key a lane
  constexpr int VP = D / 16;               // runs of 16 entries of the values
  __shared__ float part[SHARES][GH][D + 2];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int lo16 = lane & 15, hi = lane >> 4;
  const int h0 = blockIdx.x * GH, group = g.Hq / g.Hkv, kvh = h0 / group;
  const int t = g.token_list ? g.token_list[blockIdx.y] : blockIdx.y;
  const int p = g.positions[t];
  const int* table = g.block_tables + (size_t)g.seq_of_token[t] * g.max_blocks;
  float q[GH][KP][8];
#pragma unroll
  for (int h = 0; h < GH; ++h) {
    const float* qv = g.q + (size_t)t * g.q_stride + (size_t)(h0 + h) * D;
#pragma unroll
    for (int c = 0; c < KP; ++c)
#pragma unroll
      for (int e = 0; e < 8; ++e) q[h][c][e] = qv[(hi + 4 * c) * 8 + e];
  }
  // tiles of the kept first keys, then those from the window's first key on; a tile that holds the end of the one and the
  // start of the other comes twice, each time with its own keys alone
  const int lo = ra_first_key(p, g.window, g.aligned);
  const int kept = g.keep < lo ? g.keep : lo;
  const int kept_tiles = (kept + 15) >> 4, first = lo >> 4;
  const int tiles = kept_tiles + (p >> 4) - first + 1;
  for (int share = wave; share < SHARES; share += waves) {
    if (share >= tiles) {                    // a share without a tile
      if (lane < GH) {
        part[share][lane][D] = -INFINITY;
        part[share][lane][D + 1] = 0.f;
      }
      continue;
    }
    float acc[GH][VP], m[GH], l[GH];
#pragma unroll
    for (int h = 0; h < GH; ++h) {
#pragma unroll
      for (int b = 0; b < VP; ++b) acc[h][b] = 0.f;
      m[h] = -INFINITY;
      l[h] = 0.f;
    }
    for (int i = share; i < tiles; i += SHARES) {
      const bool early = i < kept_tiles;
      const int tile = early ? i : first + i - kept_tiles;
      const int from = early ? 0 : lo, to = early ? kept : p + 1;      // the keys of this tile that are seen
      const size_t at = ((size_t)table[tile * 16 / g.block_size] * g.Hkv + kvh) * g.block_size * D
                        + (size_t)(tile * 16 % g.block_size) * D;
      f32x4_t k[KP][2], v[VP];
#pragma unroll
      for (int c = 0; c < KP; ++c) {
        const float* kr = g.kcache + at + ((hi + 4 * c) * 16 + lo16) * 8;
        k[c][0] = *(const f32x4_t*)kr;
        k[c][1] = *(const f32x4_t*)(kr + 4);
      }
#pragma unroll
      for (int b = 0; b < VP; ++b) v[b] = *(const f32x4_t*)(g.vcache + at + ((b * 4 + hi) * 16 + lo16) * 4);
      const int key = tile * 16 + lo16;
      const bool seen = key >= from && key < to;
      // slots that nobody has written yet may hold anything: a probability of zero does not make a NaN harmless
      const int slot0 = tile * 16 + hi * 4;
#pragma unroll
      for (int b = 0; b < VP; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (slot0 + e < from || slot0 + e >= to) v[b][e] = 0.f;
#pragma unroll
      for (int h = 0; h < GH; ++h) {
        float s = 0.f;
#pragma unroll
        for (int c = 0; c < KP; ++c)
#pragma unroll
          for (int e = 0; e < 8; ++e) s = fmaf(q[h][c][e], k[c][e >> 2][e & 3], s);
        s += __shfl_xor(s, 16, RA_WAVE);
        s += __shfl_xor(s, 32, RA_WAVE);
        const int a = h0 + h;
        s = ra_mod_score(s * g.scale, g.mod.softcap, g.mod.r1 != nullptr, g.mod.r1 ? g.mod.r1[a] : 0.f,
                         g.mod.r1 ? g.mod.r2[a] : 0.f, p - key);
        if (!seen) s = -INFINITY;
        const float top = fmaxf(m[h], max16(s));
        const float corr = m[h] == -INFINITY ? 0.f : expf(m[h] - top);
        const float pr = seen ? expf(s - (top == -INFINITY ? 0.f : top)) : 0.f;      // all of a tile's scores may be -inf
        m[h] = top;
        l[h] = l[h] * corr + pr;
        float ps[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) ps[e] = __shfl(pr, hi * 4 + e, RA_WAVE);
#pragma unroll
        for (int b = 0; b < VP; ++b) {
          float sum = acc[h][b] * corr;
#pragma unroll
          for (int e = 0; e < 4; ++e) sum = fmaf(ps[e], v[b][e], sum);
          acc[h][b] = sum;
        }
      }
    }
    // a share's sums: l over its 16 slots, each entry over the four runs of slots
#pragma unroll
    for (int h = 0; h < GH; ++h) {
#pragma unroll
      for (int x = 8; x > 0; x >>= 1) l[h] += __shfl_xor(l[h], x, RA_WAVE);
#pragma unroll
      for (int b = 0; b < VP; ++b) {
        acc[h][b] += __shfl_xor(acc[h][b], 16, RA_WAVE);
        acc[h][b] += __shfl_xor(acc[h][b], 32, RA_WAVE);
        if (hi == 0) part[share][h][b * 16 + lo16] = acc[h][b];
      }
      if (lane == 0) {
        part[share][h][D] = m[h];
        part[share][h][D + 1] = l[h];
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < GH * D; i += blockDim.x) {
    const int h = i / D, e = i % D, a = h0 + h;
    float top = -INFINITY;
    for (int w = 0; w < SHARES; ++w) top = fmaxf(top, part[w][h][D]);
    float sum = 0.f, den = 0.f;
    for (int w = 0; w < SHARES; ++w) {
      if (part[w][h][D + 1] == 0.f) continue;      // nothing seen
      const float f = expf(part[w][h][D] - top);
      sum = fmaf(f, part[w][h][e], sum);
      den = fmaf(f, part[w][h][D + 1], den);
    }
    if (g.ho.sink) den += expf(g.ho.sink[a] - top);
    g.out[(size_t)t * g.out_stride + (size_t)a * D + e] = sum * (ra_head_gate<float>(g.ho, t, a) / den);
  }
}

template <int D, int GH>
int go(const F32Attention& g, int n_tokens, hipStream_t stream) {
  const int pairs = g.Hq / GH;
  // a wave a share where that fills the chip; with many tokens two, so that a short context still gives every wave a tile
  // or two
  const int waves = (long)pairs * n_tokens > 16L * ra_cu_count() ? 2 : 8;
  attention_f32_kernel<D, GH><<<dim3(pairs, n_tokens), waves * RA_WAVE, 0, stream>>>(g);
  RA_LAUNCH_CHECK("attention_f32");
  return 0;
}

}  // namespace

// Whether the kernel takes these sizes (16-byte reads of the cache besides; the queries are read element by element).
bool ra_attention_f32_takes(const void* kcache, const void* vcache, int d) {
  return (d == 64 || d == 128 || d == 256) && (uintptr_t)kcache % 16 == 0 && (uintptr_t)vcache % 16 == 0;
}

int ra_attention_f32(const float* q, int q_stride, float* out, int out_stride, const float* kcache, const float* vcache,
                     const int* block_tables, int max_blocks, const int* token_list, const int* seq_of_token,
                     const int* positions, int n_tokens, int block_size, int Hq, int Hkv, int d, float scale, int window,
                     int aligned, int keep, RaScoreMod mod, RaHeadOut ho, hipStream_t stream) {
  const F32Attention g = {q, q_stride, out, out_stride, kcache, vcache, block_tables, max_blocks, token_list, seq_of_token,
                          positions, block_size, Hq, Hkv, scale, window, aligned, keep, mod, ho};
  const bool even = Hq / Hkv % 2 == 0;     // two heads share what is read of a key where they read the same one
  if (d == 64) return even ? go<64, 2>(g, n_tokens, stream) : go<64, 1>(g, n_tokens, stream);
  if (d == 128) return even ? go<128, 2>(g, n_tokens, stream) : go<128, 1>(g, n_tokens, stream);
  if (d == 256) return go<256, 1>(g, n_tokens, stream);
  return ra_fail("attention_f32: head size %d", d);
}
