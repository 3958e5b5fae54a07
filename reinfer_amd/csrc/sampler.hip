// On-GPU sampling over [rows, vocab] float logits, many workgroups per row.
//   temperature <= 0: the first maximum (lowest id among equal maxima;
//     crates/cuda/src/engine.rs:6512-6520)
//   temperature  > 0: Gumbel-max, argmax_v( logit_v / T + g_v ),
//     g_v = -ln(-ln u_v), u_v = top 24 bits of mix(base ^ mix(v)) / 2^24
//     (crates/cuda/kernels/sampler_kernel.cu:61-77, 364-397), with
//     base = splitmix64(seed ^ position * golden): a pure function of the
//     request's seed, the position and the token id
//     (crates/scheduler/src/rng.rs:52-58), so a token does not depend on
//     what else is in the batch.
// Non-finite logits never win; a row without a finite logit yields -1.
// The reference's sampler is one 256-thread workgroup
// (sampler_kernel.cu:157); here stage 1 scans slices of the row in parallel
// and stage 2 merges the slice winners in a fixed order.
#include <mutex>
#include "common.h"
#include "reinfer_hip.h"

#define SAMPLE_THREADS 256
#define SAMPLE_SLICE 2048

__device__ __forceinline__ unsigned long long mix64(unsigned long long z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
__device__ __forceinline__ unsigned long long splitmix64(unsigned long long x) {
  return mix64(x + 0x9E3779B97F4A7C15ull);
}

struct Best {
  float val;
  int idx;
};
__device__ __forceinline__ Best better(Best a, Best b) {
  if (b.idx < 0) return a;
  if (a.idx < 0) return b;
  if (b.val > a.val || (b.val == a.val && b.idx < a.idx)) return b;
  return a;
}

__device__ __forceinline__ Best block_best(Best b, Best* red) {
#pragma unroll
  for (int m = RA_WAVE / 2; m > 0; m >>= 1) {
    Best o;
    o.val = __shfl_xor(b.val, m, RA_WAVE);
    o.idx = __shfl_xor(b.idx, m, RA_WAVE);
    b = better(b, o);
  }
  const int lane = threadIdx.x & (RA_WAVE - 1), wave = threadIdx.x / RA_WAVE;
  if (lane == 0) red[wave] = b;
  __syncthreads();
  Best r = red[0];
  for (int i = 1; i < SAMPLE_THREADS / RA_WAVE; ++i) r = better(r, red[i]);
  return r;
}

// A finite logit of token v as the draw compares it: itself at T <= 0, else over T and with its noise. False: it never wins.
__device__ __forceinline__ bool sample_value(float& x, int v, float T, unsigned long long base) {
  if (!(T > 0.f)) return true;
  const float u = (float)(mix64(base ^ mix64((unsigned long long)v)) >> 40) * (1.0f / 16777216.0f);
  if (u <= 0.f) return false;            // -ln(-ln 0) = -inf
  x = x / T - logf(-logf(u));
  return true;
}

__global__ void sample_stage1(const float* __restrict__ logits, int vocab, int row_stride,
                              const float* __restrict__ temperature,
                              const long long* __restrict__ seeds, const int* __restrict__ positions,
                              float* __restrict__ part_val, int* __restrict__ part_idx, int n_slices) {
  __shared__ Best red[SAMPLE_THREADS / RA_WAVE];
  const int row = blockIdx.y, slice = blockIdx.x;
  const float* lg = logits + (size_t)row * row_stride;
  const float T = temperature[row];
  const unsigned long long base =
      splitmix64((unsigned long long)seeds[row] ^ ((unsigned long long)positions[row] * 0x9E3779B97F4A7C15ull));
  Best b;
  b.val = -INFINITY;
  b.idx = -1;
  // a thread's logits are asked for in one trip to memory (one after the other, both stages: 1 row of
  // 151936 6.8 us, so 5.9; 48 rows 14.1, 11.4)
  constexpr int EACH = SAMPLE_SLICE / SAMPLE_THREADS;
  const int first = slice * SAMPLE_SLICE + threadIdx.x;
  float held[EACH];
#pragma unroll
  for (int j = 0; j < EACH; ++j) held[j] = first + j * SAMPLE_THREADS < vocab ? lg[first + j * SAMPLE_THREADS] : INFINITY;
#pragma unroll
  for (int j = 0; j < EACH; ++j) {
    const int v = first + j * SAMPLE_THREADS;
    float x = held[j];
    if (!isfinite(x)) continue;
    if (!sample_value(x, v, T, base)) continue;
    Best c;
    c.val = x;
    c.idx = v;
    b = better(b, c);
  }
  b = block_best(b, red);
  if (threadIdx.x == 0) {
    part_val[(size_t)row * n_slices + slice] = b.val;
    part_idx[(size_t)row * n_slices + slice] = b.idx;
  }
}

__global__ void sample_stage2(const float* __restrict__ part_val, const int* __restrict__ part_idx,
                              int n_slices, int* __restrict__ tokens) {
  __shared__ Best red[SAMPLE_THREADS / RA_WAVE];
  const int row = blockIdx.x;
  Best b;
  b.val = -INFINITY;
  b.idx = -1;
  for (int s = threadIdx.x; s < n_slices; s += SAMPLE_THREADS) {
    Best c;
    c.val = part_val[(size_t)row * n_slices + s];
    c.idx = part_idx[(size_t)row * n_slices + s];
    b = better(b, c);
  }
  b = block_best(b, red);
  if (threadIdx.x == 0) tokens[row] = b.idx;
}

extern "C" int ra_sample_slices(int vocab) { return (vocab + SAMPLE_SLICE - 1) / SAMPLE_SLICE; }

extern "C" int ra_sample(const float* logits, int n_rows, int vocab, int row_stride,
                         const float* temperature, const long long* seeds, const int* positions,
                         float* scratch_val, int* scratch_idx, int* tokens, hipStream_t stream) {
  RA_CHECK(n_rows > 0 && vocab > 0, "sample: empty input (%d rows, vocabulary %d)", n_rows, vocab);
  RA_CHECK(row_stride >= vocab, "sample: row stride %d below the vocabulary %d", row_stride, vocab);
  RA_CHECK(n_rows <= 65535, "sample: %d rows in one launch (max 65535)", n_rows);
  const int n_slices = ra_sample_slices(vocab);
  dim3 grid(n_slices, n_rows);
  sample_stage1<<<grid, SAMPLE_THREADS, 0, stream>>>(logits, vocab, row_stride, temperature, seeds,
                                                     positions, scratch_val, scratch_idx, n_slices);
  RA_LAUNCH_CHECK("sample stage 1");
  sample_stage2<<<n_rows, SAMPLE_THREADS, 0, stream>>>(scratch_val, scratch_idx, n_slices, tokens);
  RA_LAUNCH_CHECK("sample stage 2");
  return 0;
}

// ---------------------------------------------------------------------------
// The same two stages for callers that cannot allocate: the slice winners go
// to a file-scope array of device memory instead of buffers the caller brings.
// Each GPU holds its own copy of the array, at its own address, until the
// process ends (SAMPLE_STATIC_PAIRS * 8 bytes = 512 KiB). In host code the
// array's name is only a handle for hipGetSymbolAddress: the address it
// yields, looked up once per device with that device current, is what the
// kernels get. Stage 1 writes every pair that stage 2 reads, so nothing has to
// be cleared between calls; what an earlier call left beyond that is never read.
// ---------------------------------------------------------------------------
#define SAMPLE_STATIC_PAIRS 65536            // (row, slice) pairs a call may need
#define SAMPLE_STATIC_DEVICES 64

static __device__ __align__(256) unsigned char scratch[SAMPLE_STATIC_PAIRS * (sizeof(float) + sizeof(int))];

static void* scratch_of_device[SAMPLE_STATIC_DEVICES];     // device address of `scratch`, per GPU
static std::mutex scratch_lock;

static int static_scratch(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  RA_CHECK(e == hipSuccess, "sample_static: no current device: %s", hipGetErrorString(e));
  RA_CHECK(dev >= 0 && dev < SAMPLE_STATIC_DEVICES, "sample_static: device %d (at most %d are known)", dev,
           SAMPLE_STATIC_DEVICES);
  std::lock_guard<std::mutex> hold(scratch_lock);
  if (scratch_of_device[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    RA_CHECK(e == hipSuccess && p != nullptr, "sample_static: the scratch array has no address on device %d: %s", dev,
             hipGetErrorString(e));
    scratch_of_device[dev] = p;
  }
  *out = scratch_of_device[dev];
  return 0;
}

extern "C" long ra_sample_static_max_pairs(void) { return SAMPLE_STATIC_PAIRS; }

// Looks the array's address up for the current device, so that no later call has to: a caller that will
// run ra_sample_static under stream capture calls this once per device beforehand (a first call inside a
// capture would make the lookup inside it).
extern "C" int ra_sample_static_prepare(void) {
  void* base = nullptr;
  return static_scratch(&base);
}

extern "C" int ra_sample_static(const float* logits, int n_rows, int vocab, int row_stride,
                                const float* temperature, const long long* seeds, const int* positions,
                                int* tokens, hipStream_t stream) {
  RA_CHECK(n_rows > 0 && vocab > 0, "sample_static: empty input (%d rows, vocabulary %d)", n_rows, vocab);
  RA_CHECK(row_stride >= vocab, "sample_static: row stride %d below the vocabulary %d", row_stride, vocab);
  RA_CHECK(n_rows <= 65535, "sample_static: %d rows in one launch (max 65535)", n_rows);
  const int n_slices = ra_sample_slices(vocab);
  RA_CHECK((long)n_rows * n_slices <= SAMPLE_STATIC_PAIRS,
           "sample_static: %d rows of %d slices need %ld pairs of scratch, the array holds %d "
           "(use ra_sample with buffers of your own)",
           n_rows, n_slices, (long)n_rows * n_slices, SAMPLE_STATIC_PAIRS);
  void* base = nullptr;
  if (static_scratch(&base) != 0) return 1;
  float* part_val = (float*)base;
  int* part_idx = (int*)((unsigned char*)base + SAMPLE_STATIC_PAIRS * sizeof(float));
  dim3 grid(n_slices, n_rows);
  sample_stage1<<<grid, SAMPLE_THREADS, 0, stream>>>(logits, vocab, row_stride, temperature, seeds,
                                                     positions, part_val, part_idx, n_slices);
  RA_LAUNCH_CHECK("sample_static stage 1");
  sample_stage2<<<n_rows, SAMPLE_THREADS, 0, stream>>>(part_val, part_idx, n_slices, tokens);
  RA_LAUNCH_CHECK("sample_static stage 2");
  return 0;
}

// ---------------------------------------------------------------------------
// Filters and penalties, applied to a row of logits in place before ra_sample:
//   frequency/presence: logit -= count * freq + pres for tokens among the last
//     n of the request; repetition: logit > 0 divided, else multiplied by the
//     penalty (crates/cuda/kernels/sampler_kernel.cu:207-221);
//   then, on p = softmax(logit / T) and only if T > 0 (at T <= 0 the maximum
//     survives every filter, sampler_kernel.cu:236-252):
//   min_p: keep p >= min_p * max p; top_k: the k largest (value, then lower id);
//   top_p: keep p >= theta, theta the largest value with
//     sum_{kept, p >= theta} p >= top_p * (mass kept so far)
//   (order and boundary rules: sampler_kernel.cu:20-43, 287-372). Removed
//   tokens get -inf; ra_sample then applies the temperature and draws.
//
// A row is cut into slices, a workgroup each, and passes over it follow one another as launches:
//   1  bias and penalties of the slice's tokens, the slice's maximum of x = logit / T;
//   2  how many of its tokens, and how much of their mass e = exp(x - max x), fall into each of 512 bins a sixteenth wide
//      below the maximum (mass as whole numbers, so that sums do not depend on their order);
//   3  one workgroup a row adds the slices' bins: the bin in which the k-th largest lies, and the few in which the mass
//      reaches top_p's share, are then known;
//   4  the tokens of those bins, some dozens to hundreds, are listed;
//   5  one workgroup a row finds the exact boundaries among them;
//   6  every slice removes what lies below.
// One workgroup a row that bisected over the whole row, up to 94 passes, took 3.15 ms for 24 rows of 151936 however many
// rows there were; the six launches take 49 us for them (in a trace), each bound by its own start and one trip over the row.
// Where a token is drawn from the row at once (ra_sample_filtered) nothing is removed: the draw passes over what a filter would have
// taken, and only rows that penalties or a bias change are copied, in the first pass. For those 24 rows, half of them changed, that
// saves the copy of all rows, the last pass and a trip over memory each: in a trace 66 us of kernels, 85 with copies, so 56 and 63.
// Windows of 64 are counted eight tokens at a time: the first pass 14.1 -> 8.9 us.
// ---------------------------------------------------------------------------
#define FILTER_THREADS 256
#define FILTER_SLICE 4096        // 16 tokens a thread
#define FILTER_WINDOW 1024       // tokens of a window that are counted in LDS
#define FILTER_BINS 512
#define FILTER_BINS_A_UNIT 16.f
#define FILTER_ROW_THREADS 1024
#define FILTER_SHORT 2048        // listed tokens up to which every one is ranked against all others

__device__ __forceinline__ unsigned sortable(float v) {      // ascending order of floats as unsigned
  const unsigned b = __float_as_uint(v);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
// (value, lower id first) as one number
__device__ __forceinline__ unsigned long long filter_key(int v, float x) {
  return ((unsigned long long)sortable(x) << 32) | (unsigned)(~v);
}
__device__ __forceinline__ int filter_bin(float x, float mx) {
  return (int)fminf((mx - x) * FILTER_BINS_A_UNIT, (float)(FILTER_BINS - 1));
}

// Sum over FILTER_ROW_THREADS threads; `red` is LDS for a number a wave.
__device__ __forceinline__ unsigned long long filter_row_sum(unsigned long long v, unsigned long long* red) {
#pragma unroll
  for (int m = RA_WAVE / 2; m > 0; m >>= 1) v += __shfl_xor(v, m, RA_WAVE);
  const int lane = threadIdx.x & (RA_WAVE - 1), wave = threadIdx.x / RA_WAVE;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  unsigned long long t = 0;
  for (int i = 0; i < FILTER_ROW_THREADS / RA_WAVE; ++i) t += red[i];
  return t;
}

struct FilterRow {           // one per row, in device memory
  float temperature, top_p, min_p, repeat_penalty, frequency_penalty, presence_penalty;
  int top_k, window_off, window_len;
  int bias_off, bias_len;      // logit bias: bias_len pairs (token id, float bits) at window[bias_off]
  int pad;
};

// What the passes know of a row. A token is kept if e >= e_min, e >= theta and key >= key_min.
struct FilterPlan {
  unsigned long long key_min, mass, mass_before_k, mass_before_p;
  float mx, e_min, theta;
  int bin_k, rank_k;           // the k-th largest is number rank_k (from 1) of bin_k; bin_k -1: no such filter
  int bin_p0, bin_p1;          // top_p's boundary lies in one of these bins; bin_p0 -1: no such filter
  unsigned listed;
};

__device__ __forceinline__ bool filter_uses(const FilterRow& fr, int vocab) {
  return fr.temperature > 0.f && ((fr.top_k > 0 && fr.top_k < vocab) || (fr.top_p > 0.f && fr.top_p < 1.f) || fr.min_p > 0.f);
}

__device__ __forceinline__ bool filter_penalises(const FilterRow& fr) {
  return (fr.repeat_penalty > 1.f || fr.frequency_penalty > 0.f || fr.presence_penalty > 0.f) && fr.window_len > 0;
}
// The rows as they came, and those that the first pass changes, in a buffer of their own (null: changed where they are).
struct FilterLogits {
  const float* given;
  float* changed;
  int given_stride, changed_stride;
};
__device__ __forceinline__ const float* filter_row(const FilterLogits& l, const FilterRow& fr, int row) {
  return l.changed && (filter_penalises(fr) || fr.bias_len > 0) ? l.changed + (size_t)row * l.changed_stride
                                                                : l.given + (size_t)row * l.given_stride;
}

// A thread's 16 values of a slice, all asked for at once: value 4 q + e is token filter_at(from, q) + e. Past the row's end they
// are no numbers, which every pass leaves alone. Rows on a 16-byte boundary are read 16 bytes at a time.
__device__ __forceinline__ int filter_at(int from, int q) { return from + (q * FILTER_THREADS + (int)threadIdx.x) * 4; }
__device__ __forceinline__ void filter_read(const float* lg, int from, int to, float (&l)[16]) {
  const bool whole = (uintptr_t)lg % 16 == 0;            // `from` is a multiple of FILTER_SLICE
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int v = filter_at(from, q);
    if (whole && v + 3 < to) {
      const f32x4_t x = *(const f32x4_t*)(lg + v);
#pragma unroll
      for (int e = 0; e < 4; ++e) l[4 * q + e] = x[e];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) l[4 * q + e] = v + e < to ? lg[v + e] : NAN;
    }
  }
}

// Whether any of the window's tokens before `w` is `tok`, and how many are. Read eight at a time: with a loop that ends at the first
// one every read waits for the one before it.
__device__ __forceinline__ int filter_count(const int* win, int n, int w, int tok, bool* before) {
  int cnt = 0, early = 0;
#pragma unroll 8
  for (int x = 0; x < n; ++x) {
    const int same = win[x] == tok;
    cnt += same;
    early += same && x < w;
  }
  *before = early != 0;
  return cnt;
}

__global__ void __launch_bounds__(FILTER_THREADS)
filter_max_kernel(FilterLogits logits, int vocab, const FilterRow* __restrict__ rows, const int* __restrict__ window,
                  float* __restrict__ slice_max) {
  __shared__ float red[FILTER_THREADS / RA_WAVE];
  __shared__ int near_window[FILTER_WINDOW];
  __shared__ float slice[FILTER_SLICE];
  const FilterRow fr = rows[blockIdx.y];
  const float* lg = logits.given + (size_t)blockIdx.y * logits.given_stride;
  float* to_row = logits.changed ? logits.changed + (size_t)blockIdx.y * logits.changed_stride : const_cast<float*>(lg);
  const int tid = threadIdx.x, from = blockIdx.x * FILTER_SLICE, to = min(vocab, from + FILTER_SLICE);
  float l[16];
  filter_read(lg, from, to, l);              // asked for beside the row's options and its window
  const bool pen = filter_penalises(fr);
  if (pen || fr.bias_len > 0) {
    // the slice's logits change in LDS and, where they do, in the row
#pragma unroll
    for (int i = 0; i < 16; ++i) slice[filter_at(0, i >> 2) + (i & 3)] = l[i];
    // a window of usual length is read once and counted in LDS
    const int* win = window + fr.window_off;
    if (pen && fr.window_len <= FILTER_WINDOW) {
      for (int w = tid; w < fr.window_len; w += FILTER_THREADS) near_window[w] = win[w];
      win = near_window;
    }
    __syncthreads();
    // additive bias per token id, before everything else (crates/cuda/kernels/sampler_kernel.cu:189-203);
    // the caller lists every id once
    if (fr.bias_len > 0) {
      const int* bp = window + fr.bias_off;
      for (int b = tid; b < fr.bias_len; b += FILTER_THREADS) {
        const int tok = bp[2 * b];
        if (tok < from || tok >= to) continue;
        const float x = slice[tok - from];
        if (isfinite(x)) {
          slice[tok - from] = x + __int_as_float(bp[2 * b + 1]);
          if (!logits.changed) to_row[tok] = slice[tok - from];
        }
      }
      __syncthreads();
    }
    // penalties: the first occurrence of a token in the window carries its count
    if (pen) {
      for (int w = tid; w < fr.window_len; w += FILTER_THREADS) {
        const int tok = win[w];
        if (tok < from || tok >= to) continue;
        bool before;
        const int cnt = filter_count(win, fr.window_len, w, tok, &before);
        if (before) continue;
        float x = slice[tok - from];
        if (!isfinite(x)) continue;
        x -= fr.frequency_penalty * (float)cnt + fr.presence_penalty;
        if (fr.repeat_penalty > 1.f) x = x > 0.f ? x / fr.repeat_penalty : x * fr.repeat_penalty;
        slice[tok - from] = x;
        if (!logits.changed) to_row[tok] = x;
      }
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) l[i] = slice[filter_at(0, i >> 2) + (i & 3)];
    if (logits.changed) {
      const bool whole = (uintptr_t)to_row % 16 == 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int v = filter_at(from, q);
        if (whole && v + 3 < to) *(f32x4_t*)(to_row + v) = (f32x4_t){l[4 * q], l[4 * q + 1], l[4 * q + 2], l[4 * q + 3]};
        else
          for (int e = 0; e < 4 && v + e < to; ++e) to_row[v + e] = l[4 * q + e];
      }
    }
  }
  if (!filter_uses(fr, vocab)) return;
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < 16; ++i)
    if (isfinite(l[i])) mx = fmaxf(mx, l[i] / fr.temperature);
  mx = wave_max(mx);
  if ((tid & (RA_WAVE - 1)) == 0) red[tid / RA_WAVE] = mx;
  __syncthreads();
  if (tid == 0) {
    for (int i = 1; i < FILTER_THREADS / RA_WAVE; ++i) mx = fmaxf(mx, red[i]);
    slice_max[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = mx;
  }
}

// every thread gets the row's maximum
__device__ __forceinline__ float filter_row_max(const float* slice_max, int slices) {
  float mx = -INFINITY;
  for (int i = threadIdx.x & (RA_WAVE - 1); i < slices; i += RA_WAVE) mx = fmaxf(mx, slice_max[i]);
  return wave_max(mx);
}

__global__ void __launch_bounds__(FILTER_THREADS)
filter_bins_kernel(FilterLogits logits, int vocab, const FilterRow* __restrict__ rows,
                   const float* __restrict__ slice_max, unsigned long long* __restrict__ mass,
                   unsigned* __restrict__ count, float unit) {
  __shared__ unsigned long long m[FILTER_BINS];
  __shared__ unsigned c[FILTER_BINS];
  const FilterRow fr = rows[blockIdx.y];
  if (!filter_uses(fr, vocab)) return;
  const float* lg = filter_row(logits, fr, blockIdx.y);
  const int tid = threadIdx.x, from = blockIdx.x * FILTER_SLICE, to = min(vocab, from + FILTER_SLICE);
  const float mx = filter_row_max(slice_max + (size_t)blockIdx.y * gridDim.x, gridDim.x);
  if (mx == -INFINITY) return;               // no finite logit: ra_sample reports it
  const float e_min = fr.min_p > 0.f ? fr.min_p : 0.f;
  for (int b = tid; b < FILTER_BINS; b += FILTER_THREADS) {
    m[b] = 0ull;
    c[b] = 0u;
  }
  __syncthreads();
  float l[16];
  filter_read(lg, from, to, l);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    if (!isfinite(l[i])) continue;
    const float x = l[i] / fr.temperature, e = __expf(x - mx);
    const int b = filter_bin(x, mx);
    atomicAdd(&c[b], 1u);
    if (e >= e_min) atomicAdd(&m[b], (unsigned long long)(e * unit));
  }
  __syncthreads();
  const size_t at = ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * FILTER_BINS;
  for (int b = tid; b < FILTER_BINS; b += FILTER_THREADS) {
    mass[at + b] = m[b];
    count[at + b] = c[b];
  }
}

// One workgroup of FILTER_BINS threads a row.
__global__ void __launch_bounds__(FILTER_BINS)
filter_plan_kernel(int vocab, const FilterRow* __restrict__ rows, const float* __restrict__ slice_max, int slices,
                   const unsigned long long* __restrict__ mass, const unsigned* __restrict__ count,
                   FilterPlan* __restrict__ plans) {
  __shared__ unsigned long long m[FILTER_BINS];
  __shared__ unsigned c[FILTER_BINS];
  __shared__ FilterPlan plan;
  const FilterRow fr = rows[blockIdx.x];
  const int b = threadIdx.x;
  const float mx = filter_uses(fr, vocab) ? filter_row_max(slice_max + (size_t)blockIdx.x * slices, slices) : -INFINITY;
  if (mx == -INFINITY) {                     // nothing to remove
    if (b == 0) plans[blockIdx.x].mx = mx;
    return;
  }
  unsigned long long ms = 0ull;
  unsigned cs = 0u;
  const size_t at = (size_t)blockIdx.x * slices * FILTER_BINS + b;
#pragma unroll 8
  for (int i = 0; i < slices; ++i) {
    ms += mass[at + (size_t)i * FILTER_BINS];
    cs += count[at + (size_t)i * FILTER_BINS];
  }
  m[b] = ms;
  c[b] = cs;
  if (b == 0) plan = {0ull, 0ull, 0ull, 0ull, mx, fr.min_p > 0.f ? fr.min_p : 0.f, 0.f, -1, 0, -1, -1, 0u};
  __syncthreads();
  for (int d = 1; d < FILTER_BINS; d <<= 1) {            // m, c: of this bin and all above it
    const unsigned long long mo = b >= d ? m[b - d] : 0ull;
    const unsigned co = b >= d ? c[b - d] : 0u;
    __syncthreads();
    m[b] += mo;
    c[b] += co;
    __syncthreads();
  }
  const unsigned k = (unsigned)fr.top_k;
  const unsigned long long mb = b ? m[b - 1] : 0ull;
  const unsigned cb = b ? c[b - 1] : 0u;
  if (fr.top_k > 0 && k < c[FILTER_BINS - 1] && cb < k && k <= c[b]) {
    plan.bin_k = b;
    plan.rank_k = (int)(k - cb);
    plan.mass_before_k = mb;
  }
  __syncthreads();
  if (fr.top_p > 0.f && fr.top_p < 1.f) {
    // the mass left by top_k lies between these two, and with it what the boundary's bin must reach
    const int bk = plan.bin_k;
    const double p = (double)fr.top_p;
    const double least = p * (double)(bk >= 0 ? plan.mass_before_k : m[FILTER_BINS - 1]);
    const double most = p * (double)(bk >= 0 ? m[bk] : m[FILTER_BINS - 1]);
    if ((b == 0 || (double)mb < least) && (double)m[b] >= least) {
      plan.bin_p0 = b;
      plan.mass_before_p = mb;
    }
    if ((b == 0 || (double)mb < most) && (double)m[b] >= most) plan.bin_p1 = b;
    if (b == 0) plan.mass = m[FILTER_BINS - 1];
  }
  __syncthreads();
  if (b == 0) plans[blockIdx.x] = plan;
}

__global__ void __launch_bounds__(FILTER_THREADS)
filter_list_kernel(FilterLogits logits, int vocab, const FilterRow* __restrict__ rows,
                   FilterPlan* __restrict__ plans, int* __restrict__ list) {
  __shared__ unsigned found, base;
  __shared__ int mine[FILTER_SLICE];
  const FilterPlan p = plans[blockIdx.y];
  if (p.mx == -INFINITY || (p.bin_k < 0 && p.bin_p0 < 0)) return;
  const FilterRow fr = rows[blockIdx.y];
  const float* lg = filter_row(logits, fr, blockIdx.y);
  const float T = fr.temperature;
  const int tid = threadIdx.x, from = blockIdx.x * FILTER_SLICE, to = min(vocab, from + FILTER_SLICE);
  if (tid == 0) found = 0u;
  __syncthreads();
  float l[16];
  filter_read(lg, from, to, l);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    if (!isfinite(l[i])) continue;
    const int b = filter_bin(l[i] / T, p.mx);
    if (b == p.bin_k || (p.bin_p0 >= 0 && b >= p.bin_p0 && b <= p.bin_p1))
      mine[atomicAdd(&found, 1u)] = filter_at(from, i >> 2) + (i & 3);
  }
  __syncthreads();
  if (found == 0u) return;
  if (tid == 0) base = atomicAdd(&plans[blockIdx.y].listed, found);
  __syncthreads();
  for (unsigned i = tid; i < found; i += FILTER_THREADS) list[(size_t)blockIdx.y * vocab + base + i] = mine[i];
}

// Sum over eight neighbouring threads, all of which are there; whole numbers, so in any order.
template <typename T> __device__ __forceinline__ T eight_sum(T v) {
#pragma unroll
  for (int m = 4; m > 0; m >>= 1) v += __shfl_xor(v, m, RA_WAVE);
  return v;
}

// One workgroup a row: the boundaries among the listed tokens, whose order on the list means nothing.
__global__ void __launch_bounds__(FILTER_ROW_THREADS)
filter_select_kernel(FilterLogits logits, int vocab, const FilterRow* __restrict__ rows,
                     FilterPlan* __restrict__ plans, const int* __restrict__ list, float unit) {
  __shared__ unsigned long long red[FILTER_ROW_THREADS / RA_WAVE];
  __shared__ unsigned long long keys[FILTER_SHORT], masses[FILTER_SHORT];
  __shared__ float es[FILTER_SHORT];
  __shared__ short bins[FILTER_SHORT];
  __shared__ unsigned long long key_min;
  __shared__ unsigned theta_bits;
  const FilterPlan p = plans[blockIdx.x];
  if (p.mx == -INFINITY || (p.bin_k < 0 && p.bin_p0 < 0)) return;
  const FilterRow fr = rows[blockIdx.x];
  const float* lg = filter_row(logits, fr, blockIdx.x);
  const int* mine = list + (size_t)blockIdx.x * vocab;
  const int tid = threadIdx.x, n = (int)p.listed;
  const bool is_short = n <= FILTER_SHORT;
  struct Item {
    unsigned long long key, mass;
    float e;
    int bin;
  };
  auto read = [&](int i) {                   // listed token i, from memory
    const int v = mine[i];
    const float x = lg[v] / fr.temperature, e = __expf(x - p.mx);
    return Item{filter_key(v, x), e >= p.e_min ? (unsigned long long)(e * unit) : 0ull, e, filter_bin(x, p.mx)};
  };
  if (tid == 0) {
    key_min = 0ull;
    theta_bits = 0u;
  }
  if (is_short)
    for (int i = tid; i < n; i += FILTER_ROW_THREADS) {
      const Item it = read(i);
      keys[i] = it.key;
      masses[i] = it.mass;
      es[i] = it.e;
      bins[i] = (short)it.bin;
    }
  __syncthreads();
  if (p.bin_k >= 0) {
    if (is_short) {
      for (int i = tid >> 3; i < n; i += FILTER_ROW_THREADS >> 3) {      // eight threads a token
        if (bins[i] != p.bin_k) continue;
        const unsigned long long key = keys[i];
        int above = 0;
        for (int j = tid & 7; j < n; j += 8) above += bins[j] == p.bin_k && keys[j] > key;
        above = eight_sum(above);
        if (above == p.rank_k - 1) key_min = key;            // keys differ: the threads of one token
      }
    } else {
      unsigned long long lo = 0ull, hi = ~0ull;            // count(key >= lo) >= rank > count(key >= hi)
      while (hi - lo > 1ull) {
        const unsigned long long mid = lo + (hi - lo) / 2ull;
        unsigned long long c = 0ull;
        for (int i = tid; i < n; i += FILTER_ROW_THREADS) {
          const Item it = read(i);
          c += it.bin == p.bin_k && it.key >= mid;
        }
        if (filter_row_sum(c, red) >= (unsigned long long)p.rank_k) lo = mid; else hi = mid;
      }
      if (tid == 0) key_min = lo;
    }
    __syncthreads();
  }
  if (p.bin_p0 >= 0) {
    const unsigned long long kmin = key_min;
    unsigned long long left = p.mass;                      // the mass that top_k and min_p leave
    if (p.bin_k >= 0) {
      unsigned long long s = 0ull;
      for (int i = tid; i < n; i += FILTER_ROW_THREADS) {
        const Item it = is_short ? Item{keys[i], masses[i], es[i], bins[i]} : read(i);
        if (it.bin == p.bin_k && it.key >= kmin) s += it.mass;
      }
      left = p.mass_before_k + filter_row_sum(s, red);
    }
    const double need = (double)fr.top_p * (double)left;
    auto counts = [&](int bin, unsigned long long key) { return bin >= p.bin_p0 && bin <= p.bin_p1 && key >= kmin; };
    if (is_short) {
      for (int i = tid >> 3; i < n; i += FILTER_ROW_THREADS >> 3) {
        if (!counts(bins[i], keys[i]) || es[i] < p.e_min) continue;
        const float e = es[i];
        unsigned long long s = 0ull;
        for (int j = tid & 7; j < n; j += 8) s += es[j] >= e && counts(bins[j], keys[j]) ? masses[j] : 0ull;
        s = eight_sum(s) + p.mass_before_p;
        if ((tid & 7) == 0 && (double)s >= need) atomicMax(&theta_bits, __float_as_uint(e));
      }
    } else {
      unsigned lo = 0u, hi = 0x3F800001u;                  // mass(e >= lo) >= need > mass(e >= hi); e is at most 1
      while (hi - lo > 1u) {
        const unsigned mid = lo + (hi - lo) / 2u;
        unsigned long long s = 0ull;
        for (int i = tid; i < n; i += FILTER_ROW_THREADS) {
          const Item it = read(i);
          if (counts(it.bin, it.key) && __float_as_uint(it.e) >= mid) s += it.mass;
        }
        if ((double)(p.mass_before_p + filter_row_sum(s, red)) >= need) lo = mid; else hi = mid;
      }
      if (tid == 0) theta_bits = lo;
    }
    __syncthreads();
  }
  if (tid == 0) {
    plans[blockIdx.x].key_min = key_min;
    plans[blockIdx.x].theta = __uint_as_float(theta_bits);
  }
}

// Whether the filters leave token v, whose logit is finite (x: over the temperature).
__device__ __forceinline__ bool filter_keeps(const FilterPlan& p, int v, float x) {
  const float e = __expf(x - p.mx);
  return e >= p.e_min && e >= p.theta && filter_key(v, x) >= p.key_min;
}

// sample_stage1 over the tokens that the filters leave.
__global__ void __launch_bounds__(FILTER_THREADS)
filter_draw_kernel(FilterLogits logits, int vocab, const FilterRow* __restrict__ rows, const FilterPlan* __restrict__ plans,
                   const long long* __restrict__ seeds, const int* __restrict__ positions, float* __restrict__ part_val,
                   int* __restrict__ part_idx) {
  __shared__ Best red[FILTER_THREADS / RA_WAVE];
  const int row = blockIdx.y;
  const FilterRow fr = rows[row];
  const FilterPlan p = plans[row];
  const unsigned long long base =
      splitmix64((unsigned long long)seeds[row] ^ ((unsigned long long)positions[row] * 0x9E3779B97F4A7C15ull));
  const int from = blockIdx.x * FILTER_SLICE, to = min(vocab, from + FILTER_SLICE);
  const float T = fr.temperature;
  float l[16];
  filter_read(filter_row(logits, fr, row), from, to, l);
  Best b = {-INFINITY, -1};
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    if (!isfinite(l[i])) continue;
    const int v = filter_at(from, i >> 2) + (i & 3);
    if (p.mx != -INFINITY && !filter_keeps(p, v, l[i] / T)) continue;
    if (sample_value(l[i], v, T, base)) b = better(b, Best{l[i], v});
  }
  b = block_best(b, red);
  if (threadIdx.x == 0) {
    part_val[(size_t)row * gridDim.x + blockIdx.x] = b.val;
    part_idx[(size_t)row * gridDim.x + blockIdx.x] = b.idx;
  }
}

__global__ void __launch_bounds__(FILTER_THREADS)
filter_remove_kernel(float* __restrict__ logits, int vocab, int row_stride, const FilterRow* __restrict__ rows,
                     const FilterPlan* __restrict__ plans) {
  const FilterPlan p = plans[blockIdx.y];
  if (p.mx == -INFINITY) return;
  float* lg = logits + (size_t)blockIdx.y * row_stride;
  const float T = rows[blockIdx.y].temperature;
  const int from = blockIdx.x * FILTER_SLICE, to = min(vocab, from + FILTER_SLICE);
  const bool whole = (uintptr_t)lg % 16 == 0;
  float l[16];
  filter_read(lg, from, to, l);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int v = filter_at(from, q);
    f32x4_t o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool keep = !isfinite(l[4 * q + i]) || filter_keeps(p, v + i, l[4 * q + i] / T);
      o[i] = keep ? l[4 * q + i] : -INFINITY;
      if (!keep && !(whole && v + 3 < to)) lg[v + i] = -INFINITY;
    }
    if (whole && v + 3 < to) *(f32x4_t*)(lg + v) = o;
  }
}

// Scratch of a call, in the order of its parts: plans, the slices' bins (mass, count), their maxima, the lists.
static size_t filter_parts(int n_rows, int vocab, size_t (&off)[5]) {
  const size_t slices = (vocab + FILTER_SLICE - 1) / FILTER_SLICE, n = (size_t)n_rows;
  const size_t bytes[5] = {n * sizeof(FilterPlan), n * slices * FILTER_BINS * 8, n * slices * FILTER_BINS * 4,
                           n * slices * 4, n * (size_t)vocab * 4};
  size_t at = 0;
  for (int i = 0; i < 5; ++i) {
    off[i] = at;
    at += (bytes[i] + 15) / 16 * 16;
  }
  return at;
}

extern "C" long ra_filter_scratch(int n_rows, int vocab) {
  size_t off[5];
  return n_rows > 0 && vocab > 0 ? (long)filter_parts(n_rows, vocab, off) : 0;
}

static float filter_unit(int vocab) {
  // e = 1 in whole numbers: a whole row of ones stays below 2^63
  float unit = 1.f;
  for (int bits = 62, v = vocab; bits > 0; --bits, v >>= 1)
    if (v <= 1) {
      unit = (float)(1ull << bits);
      break;
    }
  return unit * 0.5f;
}

// Passes 1 to 5: the rows' plans.
static int filter_plans(const FilterLogits& l, int n_rows, int vocab, const FilterRow* fr, const int* window, char* s,
                        const size_t (&off)[5], hipStream_t stream) {
  FilterPlan* plans = (FilterPlan*)(s + off[0]);
  unsigned long long* mass = (unsigned long long*)(s + off[1]);
  unsigned* count = (unsigned*)(s + off[2]);
  float* slice_max = (float*)(s + off[3]);
  int* list = (int*)(s + off[4]);
  const int slices = (vocab + FILTER_SLICE - 1) / FILTER_SLICE;
  const float unit = filter_unit(vocab);
  const dim3 grid(slices, n_rows);
  filter_max_kernel<<<grid, FILTER_THREADS, 0, stream>>>(l, vocab, fr, window, slice_max);
  RA_LAUNCH_CHECK("filter_logits (maximum)");
  filter_bins_kernel<<<grid, FILTER_THREADS, 0, stream>>>(l, vocab, fr, slice_max, mass, count, unit);
  RA_LAUNCH_CHECK("filter_logits (bins)");
  filter_plan_kernel<<<n_rows, FILTER_BINS, 0, stream>>>(vocab, fr, slice_max, slices, mass, count, plans);
  RA_LAUNCH_CHECK("filter_logits (plan)");
  filter_list_kernel<<<grid, FILTER_THREADS, 0, stream>>>(l, vocab, fr, plans, list);
  RA_LAUNCH_CHECK("filter_logits (list)");
  filter_select_kernel<<<n_rows, FILTER_ROW_THREADS, 0, stream>>>(l, vocab, fr, plans, list, unit);
  RA_LAUNCH_CHECK("filter_logits (boundaries)");
  return 0;
}

extern "C" int ra_filter_logits(float* logits, int n_rows, int vocab, int row_stride, const void* rows,
                                const int* window, void* scratch, long scratch_bytes, hipStream_t stream) {
  RA_CHECK(n_rows > 0 && vocab > 0, "filter_logits: empty input (%d rows, vocabulary %d)", n_rows, vocab);
  RA_CHECK(row_stride >= vocab, "filter_logits: row stride %d below the vocabulary %d", row_stride, vocab);
  RA_CHECK(n_rows <= 65535, "filter_logits: %d rows in one launch (max 65535)", n_rows);
  RA_CHECK(rows != nullptr, "filter_logits: no row parameters");
  size_t off[5];
  const size_t need = filter_parts(n_rows, vocab, off);
  RA_CHECK(scratch != nullptr && scratch_bytes >= (long)need && (uintptr_t)scratch % 16 == 0,
           "filter_logits: scratch of %ld bytes, needs %zu on a 16-byte boundary", scratch_bytes, need);
  const FilterLogits l = {logits, nullptr, row_stride, 0};
  const FilterRow* fr = (const FilterRow*)rows;
  if (filter_plans(l, n_rows, vocab, fr, window, (char*)scratch, off, stream) != 0) return 1;
  filter_remove_kernel<<<dim3((vocab + FILTER_SLICE - 1) / FILTER_SLICE, n_rows), FILTER_THREADS, 0, stream>>>(
      logits, vocab, row_stride, fr, (const FilterPlan*)((char*)scratch + off[0]));
  RA_LAUNCH_CHECK("filter_logits (removal)");
  return 0;
}

// A token a row of what ra_filter_logits would leave, drawn as ra_sample draws it, the logits left as they are. changed: rows of
// changed_stride floats for those that penalties and biases change; the slices' best go to scratch_val and scratch_idx,
// ra_filter_slices a row. temperatures are the rows' own.
extern "C" int ra_filter_slices(int vocab) { return (vocab + FILTER_SLICE - 1) / FILTER_SLICE; }

extern "C" int ra_sample_filtered(const float* logits, int n_rows, int vocab, int row_stride, const void* rows, const int* window,
                                  float* changed, int changed_stride, void* scratch, long scratch_bytes, const long long* seeds,
                                  const int* positions, float* scratch_val, int* scratch_idx, int* tokens, hipStream_t stream) {
  RA_CHECK(n_rows > 0 && vocab > 0, "sample_filtered: empty input (%d rows, vocabulary %d)", n_rows, vocab);
  RA_CHECK(row_stride >= vocab && changed_stride >= vocab, "sample_filtered: row strides %d and %d below the vocabulary %d", row_stride,
           changed_stride, vocab);
  RA_CHECK(n_rows <= 65535, "sample_filtered: %d rows in one launch (max 65535)", n_rows);
  RA_CHECK(rows != nullptr && changed != nullptr && changed != logits, "sample_filtered: no row parameters, or no rows of its own");
  size_t off[5];
  const size_t need = filter_parts(n_rows, vocab, off);
  RA_CHECK(scratch != nullptr && scratch_bytes >= (long)need && (uintptr_t)scratch % 16 == 0,
           "sample_filtered: scratch of %ld bytes, needs %zu on a 16-byte boundary", scratch_bytes, need);
  const FilterLogits l = {logits, changed, row_stride, changed_stride};
  const FilterRow* fr = (const FilterRow*)rows;
  if (filter_plans(l, n_rows, vocab, fr, window, (char*)scratch, off, stream) != 0) return 1;
  const int slices = ra_filter_slices(vocab);
  filter_draw_kernel<<<dim3(slices, n_rows), FILTER_THREADS, 0, stream>>>(
      l, vocab, fr, (const FilterPlan*)((char*)scratch + off[0]), seeds, positions, scratch_val, scratch_idx);
  RA_LAUNCH_CHECK("sample_filtered (draw)");
  sample_stage2<<<n_rows, SAMPLE_THREADS, 0, stream>>>(scratch_val, scratch_idx, slices, tokens);
  RA_LAUNCH_CHECK("sample_filtered stage 2");
  return 0;
}
