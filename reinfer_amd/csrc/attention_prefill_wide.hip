// Prompt attention for heads of 256 elements: the form of attention_prefill.hip (which says what a tile, a
// round and a part are) for a workgroup of four waves of two column tiles, one a SIMD, with all of its 512 registers.
//
// A column tile's outputs and queries alone are 96 registers here. In the other form's shape (eight waves of one column tile) a key or
// value read from LDS feeds one product, so that LDS bounds the kernel at twice the products' time, and nothing is left to read
// ahead with. Here it feeds two, the operands of half a round (128 registers) are read ahead of its products, and keys and values
// go straight to LDS. What a SIMD's only wave has to overlap is alternated in its stream: a column tile's exponentials with the
// scores of the next half and the outputs of the tile before. It is bound by LDS reads and products about evenly, in turns with
// what does not overlap (the first scores of a round, masks, the ends of the operands' reads).
// Against the other shape (16 query heads, 1 KV head, 1900 tokens in a window of 1024) 87 -> 65 us; 500 tokens 45 -> 35; 16 and 8
// heads, 2000 tokens 140 -> 93; 16 and 4, 7000 tokens 896 -> 562. At 128 elements the same scheme is slower than eight waves (64 and 8 heads, 7901 tokens 1035 ->
// 1483 us), and so are eight waves that take turns at products and exponentials between barriers (1100). Sizes of
// 129 to 255 stay with the other form too: padded to 256 this one reads and loads more than they need (192 elements, 16 and 8 heads,
// 2000 tokens 119 there, 127 here; 144 elements, 300 tokens 22 and 28). So do steps of few keys (FPW_FEW_KEYS).
#include <type_traits>
#include <utility>
#include "attention_prefill.h"

template <class F, int... I>
__device__ __forceinline__ void fpw_each(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void fpw_for(F&& f) {
  fpw_each(f, std::make_integer_sequence<int, N>{});
}
// The instructions stay in the order that they are written in.
#define FPW_ORDER __builtin_amdgcn_sched_barrier(0)

// Products written by hand, so that scores are made in the registers that the softmax reads (the compiler, told that a wave has
// 512, makes every result in the accumulation registers and moves each value over and back) while outputs and queries
// stay in the others.
__device__ __forceinline__ void fpw_first(f32x4_t& s, const bf16x8_t& k, const bf16x8_t& q) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(s) : "v"(k), "a"(q));
}
__device__ __forceinline__ void fpw_score(f32x4_t& s, const bf16x8_t& k, const bf16x8_t& q) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(s) : "v"(k), "a"(q));
}
__device__ __forceinline__ void fpw_output(f32x4_t& o, const bf16x8_t& v, const bf16x8_t& p) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(o) : "v"(v), "v"(p));
}
// The wait states that the compiler does not see in the assembly: between a product and an ordinary access to its result (and
// back), and between an ordinary write of an operand and the product that reads it.
template <int N>
__device__ __forceinline__ void fpw_rest_scores(f32x4_t (&x)[N]) {
#pragma unroll
  for (int i = 0; i < N; i += 2) asm volatile("s_nop 15\n\ts_nop 3" : "+v"(x[i]), "+v"(x[i + 1]));
}
template <int N>
__device__ __forceinline__ void fpw_rest_outputs(f32x4_t (&x)[N]) {
#pragma unroll
  for (int i = 0; i < N; i += 4) asm volatile("s_nop 15\n\ts_nop 3" : "+a"(x[i]), "+a"(x[i + 1]), "+a"(x[i + 2]), "+a"(x[i + 3]));
}
__device__ __forceinline__ void fpw_ready(bf16x8_t& x) { asm volatile("s_nop 3" : "+v"(x)); }

template <int FLAGS>
__global__ void __launch_bounds__(FPW_WAVES * RA_WAVE, 1)
flash_prefill_wide_kernel(const bf16_t* __restrict__ q, int q_stride, bf16_t* __restrict__ out, int out_stride,
                          const bf16_t* __restrict__ kcache, const bf16_t* __restrict__ vcache,
                          const int* __restrict__ block_tables, int max_blocks,
                          const int* __restrict__ tile_info,      // per tile: seq, first token row, n queries, first position
                          int block_size, int Hq, int Hkv, int HG, float scale_log2, int window,
                          int keep, FpSplit sp, float mod_scale, RaScoreMod mod, RaHeadOut ho) {
  constexpr int d = FPW_D, WAVES = FPW_WAVES, NC = FPW_NC;
  constexpr bool MOD = (FLAGS & FP_MOD) != 0, KEEP = (FLAGS & FP_KEEP) != 0, CHUNK = (FLAGS & FP_CHUNK) != 0;
  constexpr int NDT = d / 32;       // 32-wide d tiles of the score product
  constexpr int NOT = d / 16;       // 16-row d tiles of the output
  constexpr int TILE = 16 * d;      // elements of a tile of 16 slots in LDS
  __shared__ __attribute__((aligned(1024))) bf16_t ring[2 * 8 * TILE];        // two rounds of 4 tiles of K, 4 of V

  const int tid = threadIdx.x;
  const int lane = tid & (RA_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / RA_WAVE);      // scalar: tests on it are branches
  const int r = lane & 15, g = lane >> 4;
  const int G = Hq / Hkv;
  const int n_hgrp = G / HG;
  // Workgroups go round the chip's XCDs, each with an L2 of its own, in the order of their numbers: the
  // (KV head, head group) is the fast index, so that with 8 of them all query tiles of one KV head run on
  // one XCD and its keys and values fill one L2 instead of all of them. Later tiles see more keys: they
  // start first.
  const int gy = Hkv * n_hgrp;
  const int by = blockIdx.x % gy;
  const int tile = gridDim.x / gy - 1 - blockIdx.x / gy;
  const int kvh = by / n_hgrp, hgrp = by % n_hgrp;
  const int seq = tile_info[tile * 4 + 0];
  const int row0 = tile_info[tile * 4 + 1];
  const int nq = tile_info[tile * 4 + 2] & 0xffff;      // above it, which column tiles are computed: at 256 elements all are
  const int pos0 = tile_info[tile * 4 + 3];
  const int* table = block_tables + (size_t)seq * max_blocks;

  // column tile c = wave * NC + j: queries (c / HG) * 16 + r, head hgrp * HG + c % HG
  int qi[NC];
  bool q_live[NC];
  bf16x8_t qreg[NC][NDT];
  const bool biased = MOD && mod.r1 != nullptr;
  const float inv_cap = (MOD && mod.softcap > 0.f) ? 1.f / mod.softcap : 0.f;
  float r1h[NC], r2h[NC];               // the distance term's two numbers of each column tile's head
  int chunk_lo[NC];                     // CHUNK: the first key each column's query sees
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const int c = wave * NC + j;
    qi[j] = (c / HG) * 16 + r;
    q_live[j] = qi[j] < nq;
    chunk_lo[j] = CHUNK ? ra_first_key(pos0 + qi[j], window, 1) : 0;
    const int head = kvh * G + hgrp * HG + c % HG;
    r1h[j] = biased ? mod.r1[head] : 0.f;
    r2h[j] = biased ? mod.r2[head] : 0.f;
  }
  f32x4_t acc[NC][NOT];
  float m[NC], l[NC];
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    m[j] = q_live[j] ? -INFINITY : 0.f;      // a column without a query adds zeros and never asks for a new maximum
    l[j] = 0.f;
#pragma unroll
    for (int i = 0; i < NOT; ++i) acc[j][i] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  }

  // keys this tile of queries can see, and this wave's share of them
  const int last_pos = pos0 + nq - 1;
  const int first_key = ra_first_key(pos0, window, CHUNK ? 1 : 0);
  const int win_round = first_key / FP_KT * FP_KT;       // the round that holds the window's first key
  int kt_begin = win_round;
  int k_stop = last_pos;                      // the last key of this workgroup's rounds
  int slot = -1;
  if (sp.ranges) {
    kt_begin = max(kt_begin, sp.ranges[tile * 3 + 0]);
    k_stop = min(k_stop, sp.ranges[tile * 3 + 1] - 1);
    slot = sp.ranges[tile * 3 + 2];
  }
  // Kept first keys below the window's first round: rounds [kept_from, kept_from + kept) of this workgroup's share
  // take the places right below kt_begin; from there on a place is the key's own number.
  int kept = 0, kept_from = 0;
  if (KEEP) {
    int kept_end = min((keep + FP_KT - 1) / FP_KT * FP_KT, win_round);
    if (sp.ranges) {
      kept_from = sp.ranges[tile * 3 + 0];
      kept_end = min(kept_end, sp.ranges[tile * 3 + 1]);
    }
    kept = max(kept_end - kept_from, 0);
    if (k_stop < kt_begin) k_stop = kt_begin - 1;        // nothing of the window in this share: the kept rounds alone
  }
  const int place_begin = kt_begin - kept;
  auto key_of = [&](int place) -> int { return (KEEP && place < kt_begin) ? place - place_begin + kept_from : place; };
  const int w_q0 = (wave * NC / HG) * 16;                       // first query of the wave
  const int w_qend = ((wave * NC + NC - 1) / HG + 1) * 16;      // one past its last
  const int w_first_pos = pos0 + w_q0;
  const int w_last_pos = pos0 + min(w_qend, nq) - 1;            // < w_first_pos if the wave has no query
  // CHUNK: the first keys that the wave's first and last query see
  const int w_first_lo = CHUNK ? ra_first_key(w_first_pos, window, 1) : 0;
  const int w_last_lo = CHUNK ? ra_first_key(max(w_last_pos, w_first_pos), window, 1) : 0;

  // A round is four tiles of 16 slots of K and of V. Each wave asks for one of either, straight to LDS and in the cache's own order,
  // a round ahead. A tile outside the visible keys, and a round past the last, are loads like any other from a descriptor of no
  // bytes: zeros.
  const int bs_shift = __builtin_ctz(block_size);      // block sizes are powers of two here
  auto tile_live = [&](int kt) -> bool { return kt <= k_stop && (kt + 15 >= first_key || (KEEP && kt < keep)); };
  auto block_of = [&](int place) -> int {              // the block of this wave's tile of a round
    const int kt = key_of(place) + wave * 16;
    return place <= k_stop && tile_live(kt) ? table[kt >> bs_shift] : 0;
  };
  auto fetch = [&](int place, int slot, int blk) {
    const int kt = key_of(place) + wave * 16;
    const bool live = place <= k_stop && tile_live(kt);
    const size_t tile_at = live ? (((size_t)blk * Hkv + kvh) << bs_shift) * d + (size_t)((kt & (block_size - 1)) >> 4) * 16 * d : 0;
    auto ask_tile = [&](const bf16_t* cache, bf16_t* to) {
      const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(cache) + tile_at, 0, live ? 32 * d : 0, 0x00020000);
#pragma unroll
      for (int u = 0; u < TILE * 2 / 1024; ++u)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(to + u * 512), 16, lane * 16, u * 1024, 0, 0);
    };
    bf16_t* to = ring + slot * 8 * TILE;
    ask_tile(kcache, to + wave * TILE);
    ask_tile(vcache, to + (4 + wave) * TILE);
  };
  // Slots of this wave's tile outside the visible range may hold anything (a freed block's bits): their values are zeroed once the
  // tile is there. (Their keys need not be: the scores are replaced.)
  auto clean = [&](int place, int slot) {
    const int kt = key_of(place) + wave * 16;
    if (!tile_live(kt) || (kt + 15 <= last_pos && kt >= first_key)) return;
    bf16_t* v = ring + slot * 8 * TILE + (4 + wave) * TILE;
    for (int u = lane; u < d * 4; u += RA_WAVE) {         // 4 slots of one value row: slots 4 ((u / 16) % 4) + e
      bf16x4_t x = *(const bf16x4_t*)(v + u * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int key = kt + ((u >> 4) & 3) * 4 + e;
        if (key > last_pos || (key < first_key && !(KEEP && key < keep))) x[e] = (bf16_t)0.f;
      }
      *(bf16x4_t*)(v + u * 4) = x;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };

  const bf16x8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  // operands of one half (32 keys) of the round in `slot`
  auto k_operand = [&](int slot, int kp, int ks, int dt) -> bf16x8_t {
    return *(const bf16x8_t*)(ring + slot * 8 * TILE + (kp * 2 + ks) * TILE + ((dt * 4 + g) * 16 + r) * 8);
  };
  auto v_operand = [&](int slot, int kp, int ot) -> bf16x8_t {
    const bf16_t* v = ring + slot * 8 * TILE + (4 + kp * 2) * TILE + ((ot * 4 + g) * 16 + r) * 4;
    const bf16x4_t a = *(const bf16x4_t*)v, b = *(const bf16x4_t*)(v + TILE);
    return (bf16x8_t){a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  };
  using Scores = f32x4_t[2][NC];
  auto read_k = [&](bf16x8_t (&ka)[2][NDT], int slot, int kp) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) ka[ks][dt] = k_operand(slot, kp, ks, dt);
  };
  auto read_v = [&](bf16x8_t (&va)[NOT], int slot, int kp) {
#pragma unroll
    for (int ot = 0; ot < NOT; ++ot) va[ot] = v_operand(slot, kp, ot);
  };
  // product m of column tile j's scores: S^T[key][column] for 2 sub-tiles of 16 keys
  auto score = [&](Scores& S, const bf16x8_t (&ka)[2][NDT], auto jc, auto mc) {
    constexpr int j = jc, ks = mc % 2, dt = mc / 2;
    if (dt == 0) fpw_first(S[ks][j], ka[ks][dt], qreg[j][dt]);
    else fpw_score(S[ks][j], ka[ks][dt], qreg[j][dt]);
  };
  // changed and masked scores of the half from key kh on
  auto dress = [&](Scores& S, int kh) {
    if constexpr (MOD) {
      // a key past the query (masked below) counts as distance 0: its changed score is never used
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        const int q_pos = pos0 + qi[j];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int key = kh + ks * 16 + 4 * g + i;
            S[ks][j][i] = ra_mod_score_fast(S[ks][j][i] * mod_scale, mod.softcap, inv_cap, biased, r1h[j], r2h[j],
                                            max(q_pos - key, 0));
          }
      }
    }
    // keys strictly inside every query's view need no mask
    const bool inner = kh + 31 <= w_first_pos && w_qend <= nq &&
                       (CHUNK ? kh >= w_last_lo
                              : window <= 0 || kh >= w_last_pos - window + 1 || (KEEP && kh + 31 < keep));
    if (!inner) {
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        const int q_pos = pos0 + qi[j];
        const int q_lo = CHUNK ? chunk_lo[j] : (window > 0 && q_pos - window + 1 > 0) ? q_pos - window + 1 : 0;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int key = kh + ks * 16 + 4 * g + i;
            if (!(q_live[j] && key <= q_pos && (key >= q_lo || (KEEP && key < keep)))) S[ks][j][i] = -INFINITY;
          }
      }
    }
  };
  // Probabilities against the running maximum m first; m follows the true maximum only when
  // some probability comes out above 2^8 (the true maximum has grown by more than 8 in the
  // exponent): until then float sums and bfloat16 operands hold the larger values as well, and
  // the accumulators need no rescaling. A lane tests the 8 values it holds itself; the exchange
  // between lanes that finds a column's maximum is left to the rare branch, which the wave
  // takes as a whole, for every column: it rescales and computes the probabilities again. A
  // column that has seen no key yet (m = -inf) always takes it, so m never stays unset while
  // keys are visible. The lane's sum stands for its largest value: no probability is above 2^8 unless the sum is (it is
  // needed anyway; a sum above 2^8 of smaller values only rescales a round early).
  float p[8];
  // the rest of column tile j's softmax: its operand of the output product
  auto settle = [&](const Scores& S, auto jc, float big) -> bf16x8_t {
    constexpr int j = jc;
    if (__any(!(big <= 256.f) || m[j] == -INFINITY)) {           // an overflowed or undefined value counts as large
      float tmax = fmaxf(fmaxf(fmaxf(S[0][j][0], S[0][j][1]), fmaxf(S[0][j][2], S[0][j][3])),
                         fmaxf(fmaxf(S[1][j][0], S[1][j][1]), fmaxf(S[1][j][2], S[1][j][3])));
      tmax = fmaxf(tmax, __shfl_xor(tmax, 16, RA_WAVE));
      tmax = fmaxf(tmax, __shfl_xor(tmax, 32, RA_WAVE)) * scale_log2;    // the scale is positive
      const float mn = fmaxf(m[j], tmax);
      // a column with nothing visible so far keeps m = -inf and adds zeros
      const float corr = (mn == -INFINITY) ? 1.f : fp_exp2(m[j] - mn);
      l[j] *= corr;
      m[j] = mn;
      fpw_rest_outputs(acc[j]);
#pragma unroll
      for (int ot = 0; ot < NOT; ++ot) {
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[j][ot][i] *= corr;
        FPW_ORDER;
      }
      fpw_rest_outputs(acc[j]);
      const float base = (mn == -INFINITY) ? 0.f : mn;
      big = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        p[e] = fp_exp2(fmaf(S[e >> 2][j][e & 3], scale_log2, -base));
        big += p[e];
      }
    }
    bf16x8_t pb;
#pragma unroll
    for (int e = 0; e < 8; ++e) pb[e] = from_f32<bf16_t>(p[e]);
    l[j] += big;                                     // the lane's sum, of the second set where one was computed
    return pb;
  };
  // product ot of O^T[d][column] += V^T[d][key] P[key][column], 32 keys per instruction:
  // k-slots (g, e): e < 4 -> key 4g + e of the first 16-key tile, e >= 4 -> of the second
  auto output = [&](const bf16x8_t (&va)[NOT], bf16x8_t& pb, auto jc, auto mc) {
    constexpr int j = jc, ot = mc;
    if (ot == 0) fpw_ready(pb);
    fpw_output(acc[j][ot], va[ot], pb);
  };
  // Column tile j of a half: its probabilities, one value behind every few products, which are the scores of the half behind it (AHEAD)
  // and the outputs of the column tile before. A wave issues in order, so only what its own stream alternates overlaps.
  auto step = [&](const Scores& S, const bf16x8_t (&va)[NOT], bf16x8_t& pb, auto jc, auto ahead, Scores& next, const bf16x8_t (&ka)[2][NDT]) {
    constexpr int j = jc, SC = decltype(ahead)::value ? 2 * NDT : 0, OU = j > 0 ? NOT : 0, MF = SC + OU;
    static_assert(2 * NDT == NOT);         // in turn, where there are both
    const float base = (m[j] == -INFINITY) ? 0.f : m[j];
    float big = 0.f;
    auto value = [&](auto ec) {
      constexpr int e = ec;
      p[e] = fp_exp2(fmaf(S[e >> 2][j][e & 3], scale_log2, -base));      // masked: exp2(-inf) = 0
      big += p[e];
    };
    FPW_ORDER;
    fpw_for<MF>([&](auto mc) {
      constexpr int i = mc, e0 = i * 8 / MF, e1 = (i + 1) * 8 / MF;
      constexpr bool out = OU > 0 && (SC == 0 || i % 2 == 0);
      using Nth = std::integral_constant<int, (SC > 0 && OU > 0 ? i / 2 : i)>;
      if constexpr (out) output(va, pb, std::integral_constant<int, (j > 0 ? j - 1 : 0)>{}, Nth{});
      else score(next, ka, jc, Nth{});
      FPW_ORDER;
      fpw_for<e1 - e0>([&](auto ec) { value(std::integral_constant<int, e0 + decltype(ec)::value>{}); });
      FPW_ORDER;
    });
    if constexpr (MF == 0) fpw_for<8>([&](auto ec) { value(ec); });
    pb = settle(S, jc, big);
  };
  auto half = [&](const Scores& S, const bf16x8_t (&va)[NOT], auto ahead, Scores& next, const bf16x8_t (&ka)[2][NDT]) {
    bf16x8_t pb = zero8;
    fpw_for<NC>([&](auto jc) { step(S, va, pb, jc, ahead, next, ka); });
    FPW_ORDER;
    fpw_for<NOT>([&](auto mc) { output(va, pb, std::integral_constant<int, NC - 1>{}, mc); });
  };

  // one round of 64 keys
  auto compute = [&](int k0, int slot) {
    // a wave whose queries all lie before this round, or that has none, has nothing to add
    if (w_last_pos < w_first_pos || w_last_pos < k0) return;
    if (CHUNK ? k0 + FP_KT - 1 < w_first_lo
              : window > 0 && k0 + FP_KT - 1 < w_first_pos - window + 1 && !(KEEP && k0 < keep)) return;
    bf16x8_t ka[2][NDT], va[NOT];
    Scores s0, s1;
    read_k(ka, slot, 0);
    read_v(va, slot, 0);
    FPW_ORDER;                              // the reads stay ahead of the products
    fpw_for<2 * NDT>([&](auto mc) { fpw_for<NC>([&](auto jc) { score(s0, ka, jc, mc); }); });
    fpw_rest_scores(s0[0]);
    fpw_rest_scores(s0[1]);
    read_k(ka, slot, 1);
    dress(s0, k0);
    half(s0, va, std::true_type{}, s1, ka);
    read_v(va, slot, 1);
    fpw_rest_scores(s1[0]);
    fpw_rest_scores(s1[1]);
    dress(s1, k0 + 32);
    half(s1, va, std::false_type{}, s0, ka);
  };

  fetch(place_begin, 0, block_of(place_begin));
  int ask = place_begin + FP_KT;
  int blk = block_of(ask);
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const int head = kvh * G + hgrp * HG + (wave * NC + j) % HG;
    const bf16_t* qp = q + (size_t)(row0 + (q_live[j] ? qi[j] : 0)) * q_stride + (size_t)head * d;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) {
      const int e = dt * 32 + g * 8;
      qreg[j][dt] = q_live[j] ? *(const bf16x8_t*)(qp + e) : zero8;
    }
  }
  // the queries are waited for here: a wait left to the loop would be for all of a round's loads
#pragma unroll
  for (int j = 0; j < NC; ++j)
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) asm volatile("" : "+a"(qreg[j][dt]));
  // One barrier a round: behind it this round is there (each wave has waited for its own tiles), and the round before is done with,
  // whose slot the next one takes.
  int round = 0;
  for (int place = place_begin; place <= k_stop; place += FP_KT, ask += FP_KT) {       // the bounds are the same in every thread
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    clean(place, round);
    asm volatile("s_barrier" ::: "memory");
    const int now = blk;
    blk = block_of(ask + FP_KT);
    fetch(ask, round ^ 1, now);
    compute(key_of(place), round);
    round ^= 1;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // loads that are still on their way to LDS
#pragma unroll
  for (int j = 0; j < NC; ++j) fpw_rest_outputs(acc[j]);
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    // the lane groups hold partial sums of l over their own keys
    float lt = l[j];
    lt += __shfl_xor(lt, 16, RA_WAVE);
    lt += __shfl_xor(lt, 32, RA_WAVE);
    if (slot >= 0) {
      // a part: the sums as they are, for the kernel that adds the parts (a column without a query, or one
      // that saw none of this part's keys, leaves zeros and -inf or 0 as its maximum: both weigh nothing)
      const size_t col = ((size_t)slot * gy + by) * (WAVES * NC * 16) + (wave * NC + j) * 16 + r;
#pragma unroll
      for (int ot = 0; ot < NOT; ++ot)
        *(f32x4_t*)(sp.part_o + col * d + ot * 16 + 4 * g) = acc[j][ot];
      if (g == 0) {
        sp.part_ml[col * 2] = q_live[j] ? m[j] : -INFINITY;
        sp.part_ml[col * 2 + 1] = lt;
      }
      continue;
    }
    if (!q_live[j]) continue;
    const int head = kvh * G + hgrp * HG + (wave * NC + j) % HG;
    const float inv = ra_head_gate<bf16_t>(ho, row0 + qi[j], head) / (lt + ra_sink_term(ho, head, m[j]));
    bf16_t* op = out + (size_t)(row0 + qi[j]) * out_stride + (size_t)head * d;
#pragma unroll
    for (int ot = 0; ot < NOT; ++ot) {
      const int e = ot * 16 + 4 * g;
      bf16x4_t o4 = {from_f32<bf16_t>(acc[j][ot][0] * inv), from_f32<bf16_t>(acc[j][ot][1] * inv),
                     from_f32<bf16_t>(acc[j][ot][2] * inv), from_f32<bf16_t>(acc[j][ot][3] * inv)};
      *(bf16x4_t*)(op + e) = o4;
    }
  }
}

void ra_prefill_wide(int grid, const bf16_t* q, int q_stride, bf16_t* out, int out_stride, const bf16_t* kcache, const bf16_t* vcache,
                     const int* block_tables, int max_blocks, const int* tile_info, int block_size, int Hq, int Hkv, int hg,
                     float scale_log2, int window, int aligned, int keep, const FpSplit& sp, float scale, const RaScoreMod& mod,
                     const RaHeadOut& ho, hipStream_t stream) {
  const bool changed = mod.softcap > 0.f || mod.r1 != nullptr;
  const int flags = (changed ? FP_MOD : 0) | (aligned ? FP_CHUNK : keep > 0 ? FP_KEEP : 0);
#define RA_FPW(FL)                                                                                                \
  case FL:                                                                                                        \
    flash_prefill_wide_kernel<FL><<<grid, FPW_WAVES * RA_WAVE, 0, stream>>>(                                      \
        q, q_stride, out, out_stride, kcache, vcache, block_tables, max_blocks, tile_info, block_size, Hq, Hkv, hg, \
        scale_log2, window, keep, sp, scale, mod, ho);                                                            \
    break;
  switch (flags) {
    RA_FPW(0) RA_FPW(FP_MOD) RA_FPW(FP_KEEP) RA_FPW(FP_MOD | FP_KEEP) RA_FPW(FP_CHUNK) RA_FPW(FP_MOD | FP_CHUNK)
  }
#undef RA_FPW
}
