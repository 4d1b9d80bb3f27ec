// Token selection on the device from float32 logits [rows, vocab]: first-index argmax for greedy
// rows; for sampled rows argmax(logits / T + g) with Gumbel noise g = -log(-log u), u hashed from
// (seed, counter, vocabulary index), and an optional nucleus (top-p) mask applied first. No
// [rows, vocab] temporaries: noise and probabilities are computed in registers. Every pass over a row is
// shared by SPARTS blocks; rows without a nucleus (greedy, or plain temperature) take one pass, whose best
// candidates the last kernel compares.
//
// Rows with a nucleus: the smallest probability that stays (the cut) is found by its bit pattern, ten bits
// a pass from the top. A pass adds the probabilities of what is left of the row into 1,024 bins, as whole
// numbers of 2^-46: whole sums do not depend on the order in which blocks add, so a row's token is the same
// in every batch and run, and nothing but the rounding of each probability down to a multiple of 2^-46 is lost.
// Six rows of 151,936 logits: 58 us in seven launches; one block per row that bisected on the bit pattern
// (31 passes) took 940. Up to 24,576 logits one block does all of it (sample_small_kernel).
#include "common.h"
#include "sampling.h"
#include <mutex>

__device__ __forceinline__ uint32_t mix32(uint32_t x) {
  x = ((x >> 16) ^ x) * 0x45D9F3Bu;
  x = ((x >> 16) ^ x) * 0x45D9F3Bu;
  return (x >> 16) ^ x;
}

// u in (0, 1): ((h >> 8) + 0.5) * 2^-24 evaluated in float32, kept below 1 (the float32 sum rounds
// the one input 2^24 - 1 up to 2^24, which would make the noise infinite).
__device__ __forceinline__ float hashed_uniform(uint32_t key, uint32_t v) {
  const uint32_t h = mix32(key + v * 0x9E3779B9u);
  const float u = ((float)(h >> 8) + 0.5f) * (1.0f / 16777216.0f);
  return fminf(u, 0.99999994f);
}

// A token's logit / T + Gumbel noise, the same bits in every kernel.
__device__ __forceinline__ float noisy(float z, float inv_t, uint32_t key, int i) {
  return fmaf(z, inv_t, -logf(-logf(hashed_uniform(key, (uint32_t)i))));
}

struct Best {
  float v;
  int i;
};

__device__ __forceinline__ Best better(Best a, Best b) {  // larger value, then smaller index
  return (b.v > a.v || (b.v == a.v && b.i < a.i)) ? b : a;
}

template <int NT> __device__ __forceinline__ Best block_best(Best b, Best* red) {
#pragma unroll
  for (int off = WAVE / 2; off > 0; off >>= 1) {
    Best o;
    o.v = __shfl_xor(b.v, off, WAVE);
    o.i = __shfl_xor(b.i, off, WAVE);
    b = better(b, o);
  }
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  __syncthreads();
  if (lane == 0) red[wave] = b;
  __syncthreads();
  Best t = red[0];
#pragma unroll
  for (int i = 1; i < NT / WAVE; ++i) t = better(t, red[i]);
  return t;
}

#define SPARTS 64  // blocks per row in the first kernel
#define SPT 256    // threads of such a block
#define NBINS 1024
#define NLEVELS 3   // ten bits each: probabilities lie in [0, 2), their bit patterns below 2^30
#define MASS_ONE 70368744177664.0f  // 2^46
#define NO_INDEX 0x7fffffff

typedef unsigned long long u64;

struct RowScratch {
  Best best[SPARTS];   // each part's best candidate (of the tokens above the cut, in rows with a nucleus)
  Best tie[SPARTS];    // ... and the best of those whose probability equals the cut
  int ties[SPARTS];    // how many of them the part holds
  float top[SPARTS];   // each part's largest logit / T
  float sum[SPARTS];   // each part's sum of exponentials
  u64 mass[NLEVELS][NBINS];
};
static_assert(sizeof(RowScratch) == 26368, "25.75 KiB, as sampling.h says");

// What a row with a nucleus needs to know of itself, the same bits in every kernel and block.
struct Nucleus {
  float inv_t, zmax, inv_sum;
  __device__ __forceinline__ float exponential(float z) const { return expf(fmaf(z, inv_t, -zmax)); }
  __device__ __forceinline__ float probability(float z) const { return exponential(z) * inv_sum; }
};

__device__ __forceinline__ u64 mass_of(float p) { return (u64)(p * MASS_ONE); }

// The mass the tokens that stay must reach: m < nucleus for a float mass m is mass < target here. At least 1: the narrowest
// nucleus holds the first most likely token, also where the caller's top_p is zero or less.
__device__ __forceinline__ u64 mass_target(float nucleus) { return nucleus > 0.f ? (u64)ceil((double)nucleus * (double)MASS_ONE) : 1ull; }

__device__ __forceinline__ float row_top(const RowScratch& s) {  // every thread of the block reads all parts
  float m = -INFINITY;
  for (int i = 0; i < SPARTS; ++i) m = fmaxf(m, s.top[i]);
  return m;
}

// Where the cut lies once `levels` histograms are complete: its leading 10 * levels bits, and the mass above all tokens that
// share them. found = 0: the row's whole mass is below the nucleus, everything stays.
struct Cut {
  uint32_t bits;
  u64 above;
  int found;
};

// One level further: which of the 1,024 bins holds the token that takes the mass to the target, from the largest down.
// 256 threads, four bins each; every thread returns the result.
__device__ __forceinline__ Cut next_level(Cut c, const u64* __restrict__ mass, u64 target, u64* scan, Cut* shared) {
  const int tid = threadIdx.x;
  u64 m[4], own = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) own += m[k] = mass[NBINS - 1 - (tid * 4 + k)];  // thread 0: the largest bins
  __syncthreads();
  scan[tid] = own;
  if (tid == 0) *shared = Cut{0u, 0ull, 0};
  __syncthreads();
  for (int off = 1; off < SPT; off <<= 1) {
    const u64 v = tid >= off ? scan[tid - off] : 0;
    __syncthreads();
    scan[tid] += v;
    __syncthreads();
  }
  u64 before = c.above + scan[tid] - own;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (before < target && before + m[k] >= target) *shared = Cut{(c.bits << 10) | (uint32_t)(NBINS - 1 - (tid * 4 + k)), before, 1};
    before += m[k];
  }
  __syncthreads();
  return *shared;
}

// The blocks of grid (rows, SPARTS) own a contiguous part of the vocabulary each.
__device__ __forceinline__ void part_of(int vocab, int part, int& begin, int& end) {
  const int per = (vocab + SPARTS - 1) / SPARTS;
  begin = min(vocab, part * per);
  end = min(vocab, begin + per);
}

// First kernel, grid (rows, SPARTS): the best candidate of a part of the vocabulary for rows without a nucleus: the largest
// logit (greedy), or the largest logit / T + noise. Rows with a nucleus: the part's largest logit / T; the row's bins are cleared.
__global__ __launch_bounds__(SPT) void sample_parts_kernel(const float* __restrict__ logits, int vocab, long long row_stride,
                                                           const float* __restrict__ temperature,
                                                           const float* __restrict__ top_p,
                                                           const unsigned* __restrict__ seed,
                                                           const int* __restrict__ counter, RowScratch* __restrict__ scratch) {
  __shared__ Best red[SPT / WAVE];
  const int row = blockIdx.x, part = blockIdx.y, tid = threadIdx.x;
  const float temp = temperature ? temperature[row] : 0.f;
  const bool sampled = temp > 0.f;
  const float* z = logits + (size_t)row * row_stride;
  int begin, end;
  part_of(vocab, part, begin, end);
  const float inv_t = sampled ? 1.f / temp : 1.f;
  RowScratch& s = scratch[row];
  Best b{-INFINITY, NO_INDEX};
  if (sampled && top_p && top_p[row] < 1.f) {
    for (int i = begin + tid; i < end; i += SPT) b.v = fmaxf(b.v, z[i] * inv_t);
    b = block_best<SPT>(b, red);
    if (tid == 0) s.top[part] = b.v;
    u64* bins = &s.mass[0][0];
    for (int i = part * SPT + tid; i < NLEVELS * NBINS; i += SPARTS * SPT) bins[i] = 0;
    return;
  }
  const uint32_t key = sampled ? mix32(seed[row] ^ mix32((uint32_t)counter[row])) : 0u;
  for (int i = begin + tid; i < end; i += SPT) {
    float v = z[i];
    if (sampled) v = noisy(v, inv_t, key, i);
    if (v > b.v) b = Best{v, i};
  }
  b = block_best<SPT>(b, red);
  if (tid == 0) s.best[part] = b;
}

// The passes of rows with a nucleus, grid (rows, SPARTS); other rows' blocks end at once. STEP 0: the part's sum of
// exponentials; 1 .. NLEVELS: the histogram of that level, over the probabilities that share the leading bits found so far;
// NLEVELS + 1: the part's best candidates above and at the cut.
template <int STEP>
__global__ __launch_bounds__(SPT) void sample_nucleus_kernel(const float* __restrict__ logits, int vocab, long long row_stride,
                                                             const float* __restrict__ temperature, const float* __restrict__ top_p,
                                                             const unsigned* __restrict__ seed, const int* __restrict__ counter,
                                                             RowScratch* __restrict__ scratch) {
  __shared__ Best red[SPT / WAVE];
  __shared__ float red_f[SPT / WAVE];
  __shared__ u64 scan[SPT];
  __shared__ Cut shared;
  __shared__ int tied;
  __shared__ u64 bins[STEP >= 1 && STEP <= NLEVELS ? NBINS : 1];
  const int row = blockIdx.x, part = blockIdx.y, tid = threadIdx.x;
  const float temp = temperature[row], nucleus = top_p[row];
  if (!(temp > 0.f && nucleus < 1.f)) return;
  const float* z = logits + (size_t)row * row_stride;
  RowScratch& s = scratch[row];
  int begin, end;
  part_of(vocab, part, begin, end);
  Nucleus n{1.f / temp, row_top(s), 0.f};
  if constexpr (STEP == 0) {
    float sum = 0.f;
    for (int i = begin + tid; i < end; i += SPT) sum += n.exponential(z[i]);
    sum = block_sum<SPT>(sum, red_f);
    if (tid == 0) s.sum[part] = sum;
  } else {
    float sum = 0.f;
    for (int i = 0; i < SPARTS; ++i) sum += s.sum[i];
    n.inv_sum = 1.f / sum;
    const u64 target = mass_target(nucleus);
    Cut c{0u, 0ull, 1};
#pragma unroll
    for (int l = 0; l + 1 < STEP; ++l)
      if (c.found) c = next_level(c, s.mass[l], target, scan, &shared);
    if constexpr (STEP <= NLEVELS) {
      if (!c.found) return;  // everything stays
      constexpr int SHIFT = 10 * (NLEVELS - STEP);
      for (int i = tid; i < NBINS; i += SPT) bins[i] = 0;
      __syncthreads();
      for (int i = begin + tid; i < end; i += SPT) {
        const float p = n.probability(z[i]);
        const uint32_t bits = __float_as_uint(p) >> SHIFT;
        if (p > 0.f && (STEP == 1 ? bits < NBINS : (bits >> 10) == c.bits)) atomicAdd(&bins[bits & (NBINS - 1)], mass_of(p));
      }
      __syncthreads();
      for (int i = tid; i < NBINS; i += SPT)
        if (bins[i]) atomicAdd(&s.mass[STEP - 1][i], bins[i]);
    } else {
      const float cut = c.found ? __uint_as_float(c.bits) : 0.f;
      const uint32_t key = mix32(seed[row] ^ mix32((uint32_t)counter[row]));
      Best b{-INFINITY, NO_INDEX}, t{-INFINITY, NO_INDEX};
      int ties = 0;
      if (tid == 0) tied = 0;
      for (int i = begin + tid; i < end; i += SPT) {
        const float p = n.probability(z[i]);
        if (p < cut) continue;
        const float v = noisy(z[i], n.inv_t, key, i);
        if (p == cut) {
          ++ties;
          if (v > t.v) t = Best{v, i};
        } else if (v > b.v) {
          b = Best{v, i};
        }
      }
      b = block_best<SPT>(b, red);  // (its barriers also stand between the clearing of `tied`, the sums and the reading)
      if (ties) atomicAdd(&tied, ties);
      t = block_best<SPT>(t, red);
      if (tid == 0) {
        s.best[part] = b;
        s.tie[part] = t;
        s.ties[part] = tied;
      }
    }
  }
}

// Last kernel, one block per row. temperature / top_p / seed / counter may be null: then every row is greedy. In a row with a
// nucleus the tokens at the cut stay in index order while the mass before them is below the nucleus: whole parts of them,
// then, in the part where that ends, one by one.
__global__ __launch_bounds__(SPT) void sample_rows_kernel(const float* __restrict__ logits, int vocab, long long row_stride,
                                                          const float* __restrict__ temperature, const float* __restrict__ top_p,
                                                          const unsigned* __restrict__ seed, const int* __restrict__ counter,
                                                          const RowScratch* __restrict__ scratch, int* __restrict__ tokens) {
  __shared__ Best red[SPT / WAVE];
  __shared__ u64 scan[SPT];
  __shared__ Cut shared;
  const int row = blockIdx.x, tid = threadIdx.x;
  const RowScratch& s = scratch[row];
  const float temp = temperature ? temperature[row] : 0.f;
  const float nucleus = (temp > 0.f && top_p) ? top_p[row] : 1.f;
  Best b = tid < SPARTS ? s.best[tid] : Best{-INFINITY, NO_INDEX};
  if (nucleus < 1.f) {
    const u64 target = mass_target(nucleus);
    Cut c{0u, 0ull, 1};
    for (int l = 0; l < NLEVELS; ++l)
      if (c.found) c = next_level(c, s.mass[l], target, scan, &shared);
    const float cut = c.found ? __uint_as_float(c.bits) : 0.f;
    long long keep = 0x7fffffffffffffffll;  // tokens at the cut that stay
    if (c.found) {
      const u64 each = mass_of(cut);
      keep = (long long)((target - c.above + each - 1) / each);
    }
    long long before = 0;  // tokens at the cut in the parts before this thread's
    if (tid < SPARTS) {
      for (int i = 0; i < tid; ++i) before += s.ties[i];
      if (before + s.ties[tid] <= keep) b = better(b, s.tie[tid]);
    }
    long long at = 0;
    int split = 0;
    while (split < SPARTS && at + s.ties[split] <= keep) at += s.ties[split++];
    if (split < SPARTS && at < keep) {
      Nucleus n{1.f / temp, row_top(s), 0.f};
      float sum = 0.f;
      for (int i = 0; i < SPARTS; ++i) sum += s.sum[i];
      n.inv_sum = 1.f / sum;
      const float* z = logits + (size_t)row * row_stride;
      const uint32_t key = mix32(seed[row] ^ mix32((uint32_t)counter[row]));
      int begin, end;
      part_of(vocab, split, begin, end);
      const int chunk = (end - begin + SPT - 1) / SPT;  // index order across threads: contiguous runs
      const int lo = min(end, begin + tid * chunk), hi = min(end, lo + chunk);
      int mine = 0;
      for (int i = lo; i < hi; ++i) mine += n.probability(z[i]) == cut;
      __syncthreads();
      scan[tid] = (u64)mine;
      __syncthreads();
      for (int off = 1; off < SPT; off <<= 1) {  // inclusive
        const u64 v = tid >= off ? scan[tid - off] : 0;
        __syncthreads();
        scan[tid] += v;
        __syncthreads();
      }
      long long rank = at + (long long)scan[tid] - mine;
      for (int i = lo; i < hi; ++i) {
        if (n.probability(z[i]) != cut || rank++ >= keep) continue;
        const float v = noisy(z[i], n.inv_t, key, i);
        b = better(b, Best{v, i});
      }
    }
  }
  b = block_best<SPT>(b, red);
  if (tid == 0) tokens[row] = b.i == NO_INDEX ? 0 : b.i;
}

// Few tokens in the vocabulary: one block does all of the above for a row, with the bins in LDS. Its passes over the row are short,
// and what the kernels above cost is seven launches of 64 blocks a row, most of them with next to nothing to do. Logits / T + noise
// and the masses are formed as above; the sum of exponentials is added in another order, which the vocabulary's size decides.
// Microseconds, the kernels above, this one (and one block that bisects, 31 passes), rows with a nucleus: 517 logits, one row 41,
// 13 (29), 300 rows 242, 19 (46); 8,000, 41, 23 (73) and 260, 33 (110); 24,000, 42, 42 (163) and 287, 67 (301); 32,000, 43, 51.
#define SMALL_VOCAB 24576
#define SMALL_NT 1024

// This thread's entry of the inclusive sum of `v` over the block's threads in order.
__device__ __forceinline__ u64 block_scan(u64 v, u64* waves) {
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
#pragma unroll
  for (int off = 1; off < WAVE; off <<= 1) {
    const u64 o = __shfl_up(v, off, WAVE);
    if (lane >= off) v += o;
  }
  __syncthreads();
  if (lane == WAVE - 1) waves[wave] = v;
  __syncthreads();
  for (int w = 0; w < wave; ++w) v += waves[w];
  return v;
}

__global__ __launch_bounds__(SMALL_NT) void sample_small_kernel(const float* __restrict__ logits, int vocab, long long row_stride,
                                                                const float* __restrict__ temperature, const float* __restrict__ top_p,
                                                                const unsigned* __restrict__ seed, const int* __restrict__ counter,
                                                                int* __restrict__ tokens) {
  constexpr int NT = SMALL_NT;
  static_assert(NT == NBINS, "a thread per bin");
  __shared__ Best red[NT / WAVE];
  __shared__ float red_f[NT / WAVE];
  __shared__ u64 waves[NT / WAVE], bins[NBINS];
  __shared__ Cut shared;
  const int row = blockIdx.x, tid = threadIdx.x;
  const float* z = logits + (size_t)row * row_stride;
  const float temp = temperature[row], nucleus = temp > 0.f ? top_p[row] : 1.f;
  const uint32_t key = temp > 0.f ? mix32(seed[row] ^ mix32((uint32_t)counter[row])) : 0u;
  Best b{-INFINITY, NO_INDEX};
  if (!(nucleus < 1.f)) {
    for (int i = tid; i < vocab; i += NT) {
      const float v = temp > 0.f ? noisy(z[i], 1.f / temp, key, i) : z[i];
      if (v > b.v) b = Best{v, i};
    }
    b = block_best<NT>(b, red);
    if (tid == 0) tokens[row] = b.i == NO_INDEX ? 0 : b.i;
    return;
  }
  Nucleus n{1.f / temp, 0.f, 0.f};
  for (int i = tid; i < vocab; i += NT) b.v = fmaxf(b.v, z[i] * n.inv_t);
  n.zmax = block_best<NT>(b, red).v;
  float sum = 0.f;
  for (int i = tid; i < vocab; i += NT) sum += n.exponential(z[i]);
  n.inv_sum = 1.f / block_sum<NT>(sum, red_f);
  const u64 target = mass_target(nucleus);
  Cut c{0u, 0ull, 1};
  for (int level = 0; level < NLEVELS && c.found; ++level) {
    const int shift = 10 * (NLEVELS - 1 - level);
    bins[tid] = 0;
    if (tid == 0) shared = Cut{0u, 0ull, 0};
    __syncthreads();
    for (int i = tid; i < vocab; i += NT) {
      const float p = n.probability(z[i]);
      const uint32_t bits = __float_as_uint(p) >> shift;
      if (p > 0.f && (level == 0 ? bits < NBINS : (bits >> 10) == c.bits)) atomicAdd(&bins[bits & (NBINS - 1)], mass_of(p));
    }
    __syncthreads();
    const u64 own = bins[NBINS - 1 - tid];  // the largest bins first
    const u64 before = c.above + block_scan(own, waves) - own;
    if (before < target && before + own >= target) shared = Cut{(c.bits << 10) | (uint32_t)(NBINS - 1 - tid), before, 1};
    __syncthreads();
    c = shared;
    __syncthreads();
  }
  const float cut = c.found ? __uint_as_float(c.bits) : 0.f;
  long long keep = 0x7fffffffffffffffll;  // tokens at the cut that stay, in index order
  if (c.found) {
    const u64 each = mass_of(cut);
    keep = (long long)((target - c.above + each - 1) / each);
  }
  b = Best{-INFINITY, NO_INDEX};
  Best t = b;
  u64 ties = 0;
  for (int i = tid; i < vocab; i += NT) {
    const float p = n.probability(z[i]);
    if (p < cut) continue;
    const float v = noisy(z[i], n.inv_t, key, i);
    if (p == cut) {
      ++ties;
      if (v > t.v) t = Best{v, i};
    } else if (v > b.v) {
      b = Best{v, i};
    }
  }
  const u64 upto = block_scan(ties, waves);
  if (tid == NT - 1) shared.above = upto;
  __syncthreads();
  if ((long long)shared.above <= keep) {
    b = better(b, t);
  } else {
    const int chunk = (vocab + NT - 1) / NT;  // index order across threads: contiguous runs
    const int lo = min(vocab, tid * chunk), hi = min(vocab, lo + chunk);
    u64 mine = 0;
    for (int i = lo; i < hi; ++i) mine += n.probability(z[i]) == cut;
    long long rank = (long long)(block_scan(mine, waves) - mine);
    for (int i = lo; i < hi; ++i) {
      if (n.probability(z[i]) != cut || rank++ >= keep) continue;
      b = better(b, Best{noisy(z[i], n.inv_t, key, i), i});
    }
  }
  b = block_best<NT>(b, red);
  if (tid == 0) tokens[row] = b.i == NO_INDEX ? 0 : b.i;
}

#define SAMPLE_BATCH 4096  // rows whose scratch one batch of launches uses; more rows come batch after batch

static int sample_launch(const float* logits, int rows, int vocab, long long row_stride, const float* temperature, const float* top_p,
                         const unsigned* seed, const int* counter, RowScratch* scratch, int* tokens, hipStream_t st) {
  if (temperature && top_p && vocab <= SMALL_VOCAB) {
    sample_small_kernel<<<rows, SMALL_NT, 0, st>>>(logits, vocab, row_stride, temperature, top_p, seed, counter, tokens);
    return launch_status();
  }
  for (int r0 = 0; r0 < rows; r0 += SAMPLE_BATCH) {
    const int n = rows - r0 < SAMPLE_BATCH ? rows - r0 : SAMPLE_BATCH;
    const float* z = logits + (size_t)r0 * row_stride;
    const float* t = temperature ? temperature + r0 : nullptr;
    const float* p = temperature && top_p ? top_p + r0 : nullptr;
    const unsigned* sd = seed ? seed + r0 : nullptr;
    const int* ct = counter ? counter + r0 : nullptr;
    const dim3 grid(n, SPARTS);
    sample_parts_kernel<<<grid, SPT, 0, st>>>(z, vocab, row_stride, t, p, sd, ct, scratch);
    if (p != nullptr) {
      sample_nucleus_kernel<0><<<grid, SPT, 0, st>>>(z, vocab, row_stride, t, p, sd, ct, scratch);
      sample_nucleus_kernel<1><<<grid, SPT, 0, st>>>(z, vocab, row_stride, t, p, sd, ct, scratch);
      sample_nucleus_kernel<2><<<grid, SPT, 0, st>>>(z, vocab, row_stride, t, p, sd, ct, scratch);
      sample_nucleus_kernel<3><<<grid, SPT, 0, st>>>(z, vocab, row_stride, t, p, sd, ct, scratch);
      sample_nucleus_kernel<4><<<grid, SPT, 0, st>>>(z, vocab, row_stride, t, p, sd, ct, scratch);
    }
    sample_rows_kernel<<<n, SPT, 0, st>>>(z, vocab, row_stride, t, p, sd, ct, scratch, tokens + r0);
  }
  return launch_status();
}

// Bytes of the scratch buffer ms_sample_rows needs for `rows` rows (-1: too many rows). The buffer may lie anywhere: what it
// holds starts at its first multiple of eight bytes.
extern "C" int ms_sample_scratch_bytes(int rows) {
  if ((long long)(rows > 0 ? rows : 0) * SPARTS * (long long)sizeof(Best) > 0x7fffffffLL) return -1;
  return rows <= 0 ? 0 : (rows < SAMPLE_BATCH ? rows : SAMPLE_BATCH) * (int)sizeof(RowScratch) + 8;
}

extern "C" int ms_sample_rows(const float* logits, int rows, int vocab, long long row_stride, const float* temperature,
                              const float* top_p, const unsigned* seed, const int* counter, void* scratch, int* tokens,
                              hipStream_t st) {
  if (rows <= 0) return MS_OK;
  if (vocab <= 0 || row_stride < vocab || scratch == nullptr) return MS_BAD_ARG;
  if (temperature != nullptr && (seed == nullptr || counter == nullptr)) return MS_BAD_ARG;
  scratch = (void*)(((size_t)scratch + 7) / 8 * 8);
  return sample_launch(logits, rows, vocab, row_stride, temperature, top_p, seed, counter, (RowScratch*)scratch, tokens, st);
}

// ---------------------------------------------------------------------------------------------
// The same kernels over a scratch buffer that lives in the library instead of in the caller's
// allocation, for callers that cannot allocate (declared in sampling.h).

static __device__ __align__(256) unsigned char sample_static_scratch[MS_SAMPLE_STATIC_MAX_ROWS * sizeof(RowScratch)];

#define MS_MAX_DEVICES 64
static void* sample_static_ptr[MS_MAX_DEVICES];  // per device: where that device's copy of the array lies
static std::mutex sample_static_mutex;

// The device address of the current device's copy of the array, looked up once per device. In host
// code the array's name is only a handle for this lookup; kernels are given the address it returns.
static void* sample_static_scratch_ptr() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MS_MAX_DEVICES) return nullptr;
  std::lock_guard<std::mutex> lock(sample_static_mutex);
  if (sample_static_ptr[dev] == nullptr) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(sample_static_scratch)) != hipSuccess) return nullptr;
    sample_static_ptr[dev] = p;
  }
  return sample_static_ptr[dev];
}

extern "C" int ms_sample_rows_static_max_rows() { return MS_SAMPLE_STATIC_MAX_ROWS; }

extern "C" int ms_sample_rows_static(const float* logits, int rows, int vocab, long long row_stride,
                                     const float* temperature, const float* top_p, const unsigned* seed,
                                     const int* counter, int* tokens, hipStream_t st) {
  if (rows <= 0) return MS_OK;
  if (rows > MS_SAMPLE_STATIC_MAX_ROWS) return MS_UNSUPPORTED;
  if (vocab <= 0 || row_stride < vocab || logits == nullptr || tokens == nullptr) return MS_BAD_ARG;
  if (temperature != nullptr && (seed == nullptr || counter == nullptr)) return MS_BAD_ARG;
  RowScratch* scratch = (RowScratch*)sample_static_scratch_ptr();
  if (scratch == nullptr) return MS_LAUNCH_FAILED;
  // Nothing in the array has to start at zero: the kernels write all they read of it, whatever an earlier call left.
  return sample_launch(logits, rows, vocab, row_stride, temperature, top_p, seed, counter, scratch, tokens, st);
}
