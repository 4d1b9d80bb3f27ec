// A mixture of feed-forward experts (gated, act(gate x) * up x, or plain, act(up x)): routing, a plan that sorts the step's
// (token, chosen expert) pairs by expert, the two products per expert over the sorted pairs, and the weighted sum back
// into the stream. Router outputs from `real` on are identity experts: they have no weights, their pairs are left out of
// the plan, and the weighted sum adds the token's own input for them.
//
// A step of T tokens that each choose `top` of E experts has P = T top pairs; pair p = t * top + j is token t's j-th
// choice (largest logit first). The plan cuts every expert's run of pairs into tiles of `tile_rows` pairs; the product
// kernels are launched over the most tiles a step can have (ceil(P / tile_rows) + min(E, P)) and a block whose tile
// holds no pair leaves at once: nothing is read back to the host, and a captured step replays.
//
// A pair's result depends on its own row and its expert's weights alone (every output element is one dot product, summed
// in an order that its place in a tile does not change), so neither the order of the pairs inside an expert's run nor
// which other pairs the step holds changes a token's result; how many pairs it holds picks the size of the tiles, and
// the kernels of different tile sizes add in different orders (rounding of float32 sums). The sum over a token's choices
// runs in the order of the choices.
#include "common.h"

#define MOE_MAX_EXPERTS 512
#define MOE_MAX_TOP WAVE

// ---------------------------------------------------------------------------------------------
// An expert's pairs are shared out evenly over its tiles, by 32 where tiles hold that many: two tiles of 128 and 122 pairs are
// done before one of 192 and one of 58. No tile holds more than tile_rows, and none is empty.
__device__ __forceinline__ int moe_pairs_per_tile(int pairs, int tiles, int tile_rows) {
  const int unit = min(tile_rows, 32);
  return ((pairs + max(tiles, 1) - 1) / max(tiles, 1) + unit - 1) / unit * unit;
}

// Where a plan goes, and for what: experts that have weights, pairs a tile, and the most tiles there can be.
struct MoePlan {
  int *order, *tile_expert, *tile_start, *tile_count;
  int4* tile_run;
  int experts, tile_rows, max_tiles;
};

static bool moe_plan_ok(const MoePlan& p, int pairs) {
  return p.order != nullptr && p.tile_expert != nullptr && p.tile_start != nullptr && p.tile_count != nullptr && p.tile_run != nullptr &&
         p.experts >= 1 && p.tile_rows >= 1 && p.max_tiles >= (pairs + p.tile_rows - 1) / p.tile_rows + (p.experts < pairs ? p.experts : pairs);
}

// The plan, one block of THREADS (ids in memory or in LDS): counts per expert, every expert's run of `order` (order[i] = the pair at
// sorted place i), and the tiles: tile n covers places tile_start[n] .. tile_start[n] + tile_count[n] - 1 of expert tile_expert[n]. Tiles past the
// last get a count of zero. Pairs whose id is E or more (identity experts) are in no run and no tile. tile_run: of every tile, its
// expert's first tile, tiles, first place and pairs; behind the counts stands how many tiles there are.
template <int THREADS>
__device__ __forceinline__ void moe_plan_block(const int* ids, int P, const MoePlan& plan) {
  const int E = plan.experts, tile_rows = plan.tile_rows, max_tiles = plan.max_tiles;
  __shared__ int counts[MOE_MAX_EXPERTS], offsets[MOE_MAX_EXPERTS], cursor[MOE_MAX_EXPERTS], tile_base[MOE_MAX_EXPERTS];
  __shared__ int total_tiles;
  const int tid = threadIdx.x;
  for (int e = tid; e < E; e += THREADS) { counts[e] = 0; cursor[e] = 0; }
  __syncthreads();
  for (int p = tid; p < P; p += THREADS)
    if (ids[p] < E) atomicAdd(&counts[max(ids[p], 0)], 1);
  __syncthreads();
  if (tid < WAVE) {  // running sums of the counts and of the tiles, 64 experts at a time
    int off = 0, nt = 0;
    for (int e0 = 0; e0 < E; e0 += WAVE) {
      const int e = e0 + tid, n = e < E ? counts[e] : 0, t = (n + tile_rows - 1) / tile_rows;
      int no = n, to = t;
#pragma unroll
      for (int d = 1; d < WAVE; d <<= 1) {
        const int a = __shfl_up(no, d, WAVE), b = __shfl_up(to, d, WAVE);
        if (tid >= d) no += a, to += b;
      }
      if (e < E) {
        offsets[e] = off + no - n;
        tile_base[e] = nt + to - t;
      }
      off += __shfl(no, WAVE - 1, WAVE);
      nt += __shfl(to, WAVE - 1, WAVE);
    }
    if (tid == 0) total_tiles = nt;
  }
  __syncthreads();
  for (int e = tid; e < E; e += THREADS) {
    const int n = (counts[e] + tile_rows - 1) / tile_rows;
    const int per = moe_pairs_per_tile(counts[e], n, tile_rows);
    for (int i = 0; i < n; ++i) {
      const int at = tile_base[e] + i;
      if (at >= max_tiles) break;
      plan.tile_expert[at] = e;
      plan.tile_start[at] = offsets[e] + i * per;
      plan.tile_count[at] = min(per, counts[e] - i * per);
      plan.tile_run[at] = make_int4(tile_base[e], n, offsets[e], counts[e]);
    }
  }
  if (tid == 0) plan.tile_count[max_tiles] = total_tiles;
  for (int n = total_tiles + tid; n < max_tiles; n += THREADS) {
    plan.tile_expert[n] = 0;
    plan.tile_start[n] = 0;
    plan.tile_count[n] = 0;
  }
  for (int p = tid; p < P; p += THREADS) {
    if (ids[p] >= E) continue;
    const int e = max(ids[p], 0);
    plan.order[offsets[e] + atomicAdd(&cursor[e], 1)] = p;
  }
}

// A step of up to MOE_PLANNED_TOKENS tokens is routed by one block of as many waves, which goes on to the plan with the ids still in LDS: that
// spares the plan's launch and its way to memory and back. One wave a token, and no more than two of them on a SIMD: with four, choosing costs
// more than the launch does. Microseconds of both in two launches and in one, 8 tokens: 4 of 32 experts 6.9, 5.9; 8 of 256 12.6, 12.0; 10 of 512
// 17.1, 16.2 (64 of 512, the most there are, 50.4, 51.3); 16 tokens by 16 waves: 8 of 32 9.2, 9.5; 8 of 256 12.8, 14.2; 10 of 512 17.2, 18.9.
#define MOE_PLANNED_TOKENS 8
#define MOE_ROUTE_WAVES(PLAN) ((PLAN) ? MOE_PLANNED_TOKENS : 4)

// ---------------------------------------------------------------------------------------------
// Routing: z = logits[t] + bias; the `top` largest z (ties: the lower index), largest first; weights = softmax over
// those alone. One wave per token. The logits may come as `splits` partial sums `stride` floats apart (the router's
// product over few rows leaves them so), added here in ascending order.
template <typename TB, bool PLAN>
__global__ __launch_bounds__(MOE_ROUTE_WAVES(PLAN) * WAVE) void moe_route_kernel(const float* __restrict__ logits, int ld, int splits, size_t stride,
                                                        const TB* __restrict__ bias, int T, int E, int top,
                                                        int* __restrict__ ids, float* __restrict__ weights, MoePlan plan) {
  __shared__ int all_ids[PLAN ? MOE_PLANNED_TOKENS * MOE_MAX_TOP : 1];
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int t = blockIdx.x * MOE_ROUTE_WAVES(PLAN) + wave;
  if (t < T) {
    float z[MOE_MAX_EXPERTS / WAVE];
#pragma unroll
    for (int i = 0; i < MOE_MAX_EXPERTS / WAVE; ++i) {
      const int e = lane + i * WAVE;
      z[i] = e < E ? sum_splits(logits + (size_t)t * ld + e, splits, stride) + (bias ? to_f32(bias[e]) : 0.f) : -INFINITY;
    }
    float chosen = 0.f;  // lane j keeps the j-th chosen logit and its expert
    int chosen_id = 0;
    for (int j = 0; j < top; ++j) {
      float best = -INFINITY;
      int at = 0x7fffffff;
#pragma unroll
      for (int i = 0; i < MOE_MAX_EXPERTS / WAVE; ++i)
        if (z[i] > best) { best = z[i]; at = lane + i * WAVE; }  // taken and absent experts hold -inf
#pragma unroll
      for (int off = WAVE / 2; off > 0; off >>= 1) {
        const float ob = __shfl_xor(best, off, WAVE);
        const int oa = __shfl_xor(at, off, WAVE);
        if (ob > best || (ob == best && oa < at)) { best = ob; at = oa; }
      }
      if (at >= E) at = j;  // logits that are no numbers: nothing to choose by, but the plan needs an expert that exists
#pragma unroll
      for (int i = 0; i < MOE_MAX_EXPERTS / WAVE; ++i)
        if (lane + i * WAVE == at) z[i] = -INFINITY;
      if (lane == j) chosen = best, chosen_id = at;
    }
    // every chosen logit is at most the first; the sum runs in the order of the choices
    const float m = __shfl(chosen, 0, WAVE);
    float sum = 0.f;
    for (int j = 0; j < top; ++j) sum += expf(__shfl(chosen, j, WAVE) - m);
    if (lane < top) {
      weights[(size_t)t * top + lane] = expf(chosen - m) / sum;
      ids[(size_t)t * top + lane] = chosen_id;
      if (PLAN) all_ids[t * top + lane] = chosen_id;
    }
  }
  if constexpr (PLAN) {
    __syncthreads();
    moe_plan_block<MOE_ROUTE_WAVES(true) * WAVE>(all_ids, T * top, plan);
  }
}

// experts > 0 (the router's outputs that have weights): the plan is made too, in what follows, for steps of up to ms_moe_planned_tokens().
extern "C" int ms_moe_planned_tokens() { return MOE_PLANNED_TOKENS; }
extern "C" int ms_moe_route(const float* logits, int ld, int splits, long long stride, const void* bias, int bias_is_bf16, int T,
                            int E, int top, int* ids, float* weights, int experts, int tile_rows, int max_tiles, int* order,
                            int* tile_expert, int* tile_start, int* tile_count, void* tile_run, hipStream_t st) {
  if (T <= 0) return MS_OK;
  if (logits == nullptr || ids == nullptr || weights == nullptr || E < 1 || top < 1 || top > E || ld < E || splits < 1 ||
      (splits > 1 && stride < (long long)T * ld))
    return MS_BAD_ARG;
  if (E > MOE_MAX_EXPERTS || top > MOE_MAX_TOP) return MS_UNSUPPORTED;
  const MoePlan plan{order, tile_expert, tile_start, tile_count, (int4*)tile_run, experts, tile_rows, max_tiles};
  if (experts > 0 && !moe_plan_ok(plan, T * top)) return MS_BAD_ARG;
  if (experts > 0 && (T > MOE_PLANNED_TOKENS || experts > MOE_MAX_EXPERTS)) return MS_UNSUPPORTED;
#define ROUTE(TB, PLAN) moe_route_kernel<TB, PLAN><<<(T - 1) / MOE_ROUTE_WAVES(PLAN) + 1, MOE_ROUTE_WAVES(PLAN) * WAVE, 0, st>>>(logits, ld, splits, (size_t)stride, (const TB*)bias, T, E, top, ids, weights, plan)
  if (experts > 0) { if (bias_is_bf16) ROUTE(bf16, true); else ROUTE(float, true); }
  else if (bias_is_bf16) ROUTE(bf16, false);
  else ROUTE(float, false);
#undef ROUTE
  return launch_status();
}

// ---------------------------------------------------------------------------------------------
// Routing by scores: s = softmax(logits[t]) over all E outputs, or, `sigmoid`, s = 1 / (1 + exp(-logits[t])) each on its own;
// the choice is made by c = s + correction (correction may be absent; sigmoid scores without one are chosen by their logits,
// which are in the same order and do not saturate), the weights are the chosen outputs' s, as they stand or, `renorm`, divided by their sum
// (+ 1e-20), times `factor`. With groups > 1 the E outputs form
// `groups` equal groups of neighbours, a group's score is its largest c, and only outputs of the `keep` best groups
// (ties: the lower group) can be chosen: the others' c counts as minus infinity. The `top` largest c are chosen, largest
// first (ties: the lower index). One wave per token; s and c of a token pass through the wave's own rows of LDS.
// PER: outputs a lane holds (64 PER cover them all).
template <typename TB, int PER, bool PLAN>
__global__ __launch_bounds__(MOE_ROUTE_WAVES(PLAN) * WAVE) void moe_route_scored_kernel(const float* __restrict__ logits, int ld, int splits, size_t stride,
                                                               const TB* __restrict__ correction, int T, int E, int top,
                                                               int groups, int keep, int sigmoid, int renorm, float factor,
                                                               int* __restrict__ ids, float* __restrict__ weights, MoePlan plan) {
  __shared__ float ss[MOE_ROUTE_WAVES(PLAN)][PER * WAVE], cs[MOE_ROUTE_WAVES(PLAN)][PER * WAVE];
  __shared__ int all_ids[PLAN ? MOE_PLANNED_TOKENS * MOE_MAX_TOP : 1];
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int t = blockIdx.x * MOE_ROUTE_WAVES(PLAN) + wave;
  const bool live = t < T;  // every wave stays for the block's barriers
  float c[PER];
  float m = -INFINITY;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = lane + i * WAVE;
    c[i] = (live && e < E) ? sum_splits(logits + (size_t)t * ld + e, splits, stride) : -INFINITY;
    m = fmaxf(m, c[i]);
  }
  m = wave_max(m);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    if (!sigmoid) c[i] = lane + i * WAVE < E ? expf(c[i] - m) : 0.f;
    sum += c[i];
  }
  sum = wave_sum(sum);
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = lane + i * WAVE;
    if (e < E) {
      const float sc = sigmoid ? 1.f / (1.f + expf(-c[i])) : c[i] / sum;
      ss[wave][e] = sc;
      if (correction || !sigmoid) c[i] = sc + (correction ? to_f32(correction[e]) : 0.f);
      cs[wave][e] = c[i];
    } else {
      c[i] = -INFINITY;
    }
  }
  if (groups > 1) {
    const int n = E / groups;
    __syncthreads();
    float gm[PER];  // lane l holds the scores of groups l, l + 64, ...
    bool taken[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int g = lane + i * WAVE;
      gm[i] = -INFINITY;
      taken[i] = false;
      if (g < groups)
        for (int k = 0; k < n; ++k) gm[i] = fmaxf(gm[i], cs[wave][g * n + k]);
    }
    __syncthreads();  // cs is read; from here on it says which groups stay (1) and which do not (0)
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (lane + i * WAVE < groups) cs[wave][lane + i * WAVE] = 0.f;
    for (int j = 0; j < keep; ++j) {
      float best = -INFINITY;
      int at = 0x7fffffff;
#pragma unroll
      for (int i = 0; i < PER; ++i)
        if (lane + i * WAVE < groups && !taken[i] && (at == 0x7fffffff || gm[i] > best)) { best = gm[i]; at = lane + i * WAVE; }
#pragma unroll
      for (int off = WAVE / 2; off > 0; off >>= 1) {
        const float ob = __shfl_xor(best, off, WAVE);
        const int oa = __shfl_xor(at, off, WAVE);
        if (oa != 0x7fffffff && (at == 0x7fffffff || ob > best || (ob == best && oa < at))) { best = ob; at = oa; }
      }
#pragma unroll
      for (int i = 0; i < PER; ++i)
        if (lane + i * WAVE == at) { taken[i] = true; cs[wave][at] = 1.f; }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = lane + i * WAVE;
      if (e < E && cs[wave][e / n] == 0.f) c[i] = -INFINITY;
    }
  } else {
    __syncthreads();
  }
  if (live) {
    float chosen = 0.f, total = 0.f;  // lane j keeps the j-th chosen score and its output; the scores' sum in the order of the choices
    int chosen_id = 0;
    for (int j = 0; j < top; ++j) {
      float best = -INFINITY;
      int at = 0x7fffffff;
#pragma unroll
      for (int i = 0; i < PER; ++i)
        if (c[i] > best) { best = c[i]; at = lane + i * WAVE; }
#pragma unroll
      for (int off = WAVE / 2; off > 0; off >>= 1) {
        const float ob = __shfl_xor(best, off, WAVE);
        const int oa = __shfl_xor(at, off, WAVE);
        if (ob > best || (ob == best && oa < at)) { best = ob; at = oa; }
      }
      if (at >= E) at = j;  // nothing left to choose by (no numbers, or fewer outputs in the kept groups than choices)
#pragma unroll
      for (int i = 0; i < PER; ++i)
        if (lane + i * WAVE == at) c[i] = -INFINITY;
      const float sc = ss[wave][at];
      total += sc;
      if (lane == j) chosen = sc, chosen_id = at;
    }
    if (lane < top) {
      weights[(size_t)t * top + lane] = (renorm ? chosen / (total + 1e-20f) : chosen) * factor;
      ids[(size_t)t * top + lane] = chosen_id;
      if (PLAN) all_ids[t * top + lane] = chosen_id;
    }
  }
  if constexpr (PLAN) {
    __syncthreads();
    moe_plan_block<MOE_ROUTE_WAVES(true) * WAVE>(all_ids, T * top, plan);
  }
}

extern "C" int ms_moe_route_scored(const float* logits, int ld, int splits, long long stride, const void* correction,
                                   int correction_is_bf16, int T, int E, int top, int groups, int keep, int sigmoid, int renorm,
                                   float factor, int* ids, float* weights, int experts, int tile_rows, int max_tiles, int* order,
                                   int* tile_expert, int* tile_start, int* tile_count, void* tile_run, hipStream_t st) {
  if (T <= 0) return MS_OK;
  if (logits == nullptr || ids == nullptr || weights == nullptr || E < 1 || top < 1 || top > E || ld < E || splits < 1 ||
      (splits > 1 && stride < (long long)T * ld) || groups < 1 || E % groups || keep < 1 || keep > groups)
    return MS_BAD_ARG;
  if (E > MOE_MAX_EXPERTS || top > MOE_MAX_TOP) return MS_UNSUPPORTED;
  const MoePlan plan{order, tile_expert, tile_start, tile_count, (int4*)tile_run, experts, tile_rows, max_tiles};
  if (experts > 0 && !moe_plan_ok(plan, T * top)) return MS_BAD_ARG;
  if (experts > 0 && (T > MOE_PLANNED_TOKENS || experts > MOE_MAX_EXPERTS)) return MS_UNSUPPORTED;
#define ROUTE_PLAN(TB, PER, PLAN) moe_route_scored_kernel<TB, PER, PLAN><<<(T - 1) / MOE_ROUTE_WAVES(PLAN) + 1, MOE_ROUTE_WAVES(PLAN) * WAVE, 0, st>>>(logits, ld, splits, (size_t)stride, (const TB*)correction, T, E, top, groups, keep, sigmoid, renorm, factor, ids, weights, plan)
#define ROUTE(TB, PER) do { if (experts > 0) ROUTE_PLAN(TB, PER, true); else ROUTE_PLAN(TB, PER, false); } while (0)
#define ROUTE_PER(TB) do { if (E <= WAVE) ROUTE(TB, 1); else if (E <= 2 * WAVE) ROUTE(TB, 2); else ROUTE(TB, MOE_MAX_EXPERTS / WAVE); } while (0)
  if (correction_is_bf16) ROUTE_PER(bf16); else ROUTE_PER(float);
#undef ROUTE_PER
#undef ROUTE
#undef ROUTE_PLAN
  return launch_status();
}

// ---------------------------------------------------------------------------------------------
// The plan by itself, for steps of more than MOE_PLANNED_TOKENS tokens.
__global__ __launch_bounds__(1024) void moe_plan_kernel(const int* __restrict__ ids, int P, MoePlan plan) { moe_plan_block<1024>(ids, P, plan); }

extern "C" int ms_moe_plan(const int* ids, int P, int E, int tile_rows, int max_tiles, int* order, int* tile_expert,
                           int* tile_start, int* tile_count, void* tile_run, hipStream_t st) {
  if (P <= 0) return MS_OK;
  const MoePlan plan{order, tile_expert, tile_start, tile_count, (int4*)tile_run, E, tile_rows, max_tiles};
  if (ids == nullptr || !moe_plan_ok(plan, P)) return MS_BAD_ARG;
  if (E > MOE_MAX_EXPERTS) return MS_UNSUPPORTED;
  moe_plan_kernel<<<1, 1024, 0, st>>>(ids, P, plan);
  return launch_status();
}

// ---------------------------------------------------------------------------------------------
// The experts' products on the matrix cores (bfloat16 operands, float32 sums, v_mfma_f32_16x16x32_bf16), operands
// straight from memory, 16 bytes a lane. A wave owns 16 pairs x 16 NT columns; a block's four waves split a tile of 64
// pairs by rows (NT = 4: 64 columns a block), a tile of 16 pairs by columns (64 NT columns a block: steps of few tokens,
// where every chosen expert has a tile of its own and its weights are streamed once; the fewer tiles the step can have,
// the narrower the waves' runs of columns, so that the chip still gets waves enough to stream with).
//   MODE 1 (gated): rows are x[token of the pair] (K = the model's width), two weights per expert, gate and up [E, N, K];
//          the result act(gate) * up (or what an activation with a limit makes of the two) goes to h[sorted place][N] in the compute type.
//   MODE 2 (plain first product): the same rows, one weight per expert; act(up) goes to h[sorted place][N].
//   MODE 0: rows are h[sorted place] (K = the experts' width), one weight per expert [E, N, K]; the result times the pair's
//          routing weight goes to y[pair][N] in float32.
// The routing weights may belong in front of the expert instead: given to a first product they multiply its float32
// results, W (w x) = w (W x), before the activation; the second product is then given none.
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 moe_bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float moe_floatx4;

// Eight consecutive elements from p + k, those at or past K zero. ALIGNED: one 16-byte load (K, the row strides and the
// bases are multiples of 8 elements, so a lane's eight are all inside or all outside).
template <bool ALIGNED> __device__ __forceinline__ moe_bf16x8 moe_load(const bf16* p, int k, int K, bool ok) {
  union { uint4 u; moe_bf16x8 v; bf16 e[8]; } x;
  x.u = make_uint4(0, 0, 0, 0);
  if (ALIGNED) {
    if (ok && k < K) x.u = *reinterpret_cast<const uint4*>(p + k);
  } else if (ok) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (k + i < K) x.e[i] = p[k + i];
  }
  return x.v;
}

template <int MODE, bool ALIGNED, int NT, bool KSPLIT = false>
__global__ __launch_bounds__(256) void moe_gemm_bf16_kernel(
    const bf16* __restrict__ a, int lda, const bf16* __restrict__ w1, const bf16* __restrict__ w2, void* __restrict__ out,
    const int* __restrict__ order, const int* __restrict__ tile_expert, const int* __restrict__ tile_start,
    const int* __restrict__ tile_count, const float* __restrict__ pair_weight, int top, int N, int K, int tile_rows, int act, float limit) {
  constexpr bool GATED = MODE == 1, FIRST = MODE != 0;
  const int count = tile_count[blockIdx.x];
  if (count == 0) return;
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE, l16 = lane % 16, grp = lane / 16;
  const bool by_rows = tile_rows == 64;
  const int m0 = by_rows ? wave * 16 : 0;
  // KSPLIT (16-pair tiles): the block's four waves share its 16 NT columns and take a quarter of K each (a multiple of 64),
  // so that four times the waves stream a step's weights; their sums meet in LDS and are added in wave order.
  const int n0 = (by_rows || KSPLIT) ? blockIdx.y * (16 * NT) : (blockIdx.y * 4 + wave) * (16 * NT);
  if (m0 >= count || n0 >= N) return;
  const int k_quarter = ((K + 3) / 4 + 63) / 64 * 64;
  const int k_lo = KSPLIT ? min(K, wave * k_quarter) : 0;
  const int k_hi = KSPLIT ? min(K, k_lo + k_quarter) : K;
  const int e = tile_expert[blockIdx.x], start = tile_start[blockIdx.x];
  const bool row_ok = m0 + l16 < count;
  const int place = start + m0 + (row_ok ? l16 : 0);
  const bf16* ap = a + (size_t)(FIRST ? order[place] / top : place) * lda;
  const bf16* wp1[NT];
  const bf16* wp2[NT];
  bool col_ok[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    col_ok[nt] = n0 + nt * 16 + l16 < N;
    const size_t at = ((size_t)e * N + (col_ok[nt] ? n0 + nt * 16 + l16 : 0)) * K;
    wp1[nt] = w1 + at;
    wp2[nt] = GATED ? w2 + at : nullptr;
  }
  moe_floatx4 acc1[NT], acc2[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) acc1[nt] = acc2[nt] = moe_floatx4{0.f, 0.f, 0.f, 0.f};
  // 64 k a step: a lane takes 16 consecutive k of its rows (two loads of 16 bytes: a wave reads a whole 128-byte line
  // of every row) and multiplies them in two products. Both operands are cut the same way, so the sum is over
  // every k once; within a step the order of k is that of the lanes' runs.
#pragma unroll(4 / NT)
  for (int k0 = k_lo; k0 < k_hi; k0 += 64) {
    const int kk = k0 + grp * 16;  // the lane's sixteen elements of this step
    moe_bf16x8 av[2], b1[NT][2], b2[NT][2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      av[u] = moe_load<ALIGNED>(ap, kk + 8 * u, k_hi, row_ok);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        b1[nt][u] = moe_load<ALIGNED>(wp1[nt], kk + 8 * u, k_hi, col_ok[nt]);
        if (GATED) b2[nt][u] = moe_load<ALIGNED>(wp2[nt], kk + 8 * u, k_hi, col_ok[nt]);
      }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        acc1[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[u], b1[nt][u], acc1[nt], 0, 0, 0);
        if (GATED) acc2[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[u], b2[nt][u], acc2[nt], 0, 0, 0);
      }
  }
  if constexpr (KSPLIT) {
    __shared__ float meet[3][GATED ? 2 * NT : NT][4][WAVE];
    if (wave > 0) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          meet[wave - 1][nt][r][lane] = acc1[nt][r];
          if (GATED) meet[wave - 1][NT + nt][r][lane] = acc2[nt][r];
        }
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 0; w < 3; ++w)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          acc1[nt][r] += meet[w][nt][r][lane];
          if (GATED) acc2[nt][r] += meet[w][NT + nt][r][lane];
        }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int m = m0 + grp * 4 + r;
    if (m >= count) continue;
    const int pair = order[start + m];
    const float pw = pair_weight ? pair_weight[pair] : 1.f;
    if (GATED) {
      bf16* o = (bf16*)out + (size_t)(start + m) * N + n0 + l16;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        if (col_ok[nt]) o[nt * 16] = static_cast<bf16>(gated_value(acc1[nt][r] * pw, acc2[nt][r] * pw, act, limit));
    } else if (FIRST) {
      bf16* o = (bf16*)out + (size_t)(start + m) * N + n0 + l16;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        if (col_ok[nt]) o[nt * 16] = static_cast<bf16>(activate(acc1[nt][r] * pw, act));
    } else {
      float* o = (float*)out + (size_t)pair * N + n0 + l16;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        if (col_ok[nt]) o[nt * 16] = acc1[nt][r] * pw;
    }
  }
}

// Tiles of 16 pairs x 16 columns whose four waves take a quarter of K each (as KSPLIT above, with the same sums in the same order), operands
// through LDS: what bounds a step of few tokens is the stream of its experts' weights, and a lane that reads 16 bytes of 16 rows
// each gets 5.0 TB/s of it. Here a load takes whole lines of 128 bytes, marked as read once, straight into a ring of STAGES steps of 64 k
// that belongs to the wave alone (no barrier in the loop), in the swizzle of the tiles below. K a multiple of 64, rows 16-byte aligned.
// Two steps and three or four blocks a CU: 72 to 96 KB of weights and rows under way; more steps leave fewer blocks (gated, 21 experts of
// 2,048 x 2,048: 56 us with two or three steps, 78 with four). Microseconds, the kernel above and this one, weights from memory, gated and
// second product: 8 tokens of 4 of 32 experts (2,048 -> 2,048) 72, 56 and 35, 31; 32 (2,048 -> 1,024) 60, 44 and 33, 26; 12 (4,096 ->
// 3,072) 254, 204 and 130, 102 (6.7 TB/s); 20 (1,024 -> 384) 17, 11 and 11, 8; 90 (4,096 -> 1,536) 184, 126 and 112, 86; 40 tokens of
// 6 of 160 (4,096 -> 1,536) 591, 449 and 317, 245; 1 token (2,048 -> 1,024) 11.8, 9.8 and 6.6, 5.4.
template <int MODE, int STAGES, int BLOCKS_PER_CU>
__global__ __launch_bounds__(256, BLOCKS_PER_CU) void moe_gemm_bf16_stream_kernel(
    const bf16* __restrict__ a, int lda, const bf16* __restrict__ w1, const bf16* __restrict__ w2, void* __restrict__ out,
    const int* __restrict__ order, const int* __restrict__ tile_expert, const int* __restrict__ tile_start,
    const int* __restrict__ tile_count, const float* __restrict__ pair_weight, int top, int N, int K, int act, float limit) {
  constexpr bool GATED = MODE == 1, FIRST = MODE != 0;
  constexpr int MATS = GATED ? 3 : 2;                 // rows of x, then the weights
  constexpr int STEP_BYTES = MATS * 2048, LOADS = MATS * 2;  // 16 rows of 128 bytes each, two load instructions
  extern __shared__ __attribute__((aligned(1024))) unsigned char moe_ring[];  // 4 * STAGES * STEP_BYTES
  const int count = tile_count[blockIdx.x];
  if (count == 0) return;
  const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), l16 = lane % 16, grp = lane / 16;
  const int n0 = blockIdx.y * 16;
  const int e = tile_expert[blockIdx.x], start = tile_start[blockIdx.x];
  const int k_quarter = ((K + 3) / 4 + 63) / 64 * 64;
  const int k_lo = min(K, wave * k_quarter), steps = (min(K, k_lo + k_quarter) - k_lo) / 64;
  unsigned char* ring = moe_ring + wave * STAGES * STEP_BYTES;
  const bf16* src[LOADS];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int R = j * 8 + lane / 8, chunk = (lane % 8) ^ ((R >> 1) & 7), k = k_lo + chunk * 8;
    const int place = start + min(R, count - 1);  // pairs that are not there: another's row, whose results are not stored
    src[j] = a + (size_t)(FIRST ? order[place] / top : place) * lda + k;
    const size_t at = ((size_t)e * N + min(n0 + R, N - 1)) * K + k;
    src[2 + j] = w1 + at;
    if (GATED) src[LOADS - 2 + j] = w2 + at;
  }
  auto issue = [&](int s) __attribute__((always_inline)) {
    unsigned char* to = ring + (s % STAGES) * STEP_BYTES;
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      const auto from = (const void __attribute__((address_space(1)))*)(src[j] + (size_t)s * 64);
      const auto at = (void __attribute__((address_space(3)))*)(to + j * 1024);
      if (j < 2) __builtin_amdgcn_global_load_lds(from, at, 16, 0, 0);
      else __builtin_amdgcn_global_load_lds(from, at, 16, 0, LOAD_ONCE);
    }
  };
  moe_floatx4 acc1 = moe_floatx4{0.f, 0.f, 0.f, 0.f}, acc2 = acc1;
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < steps) issue(s);
  for (int s = 0; s < steps; ++s) {
    // A step's place is free again: its fragments went into products a step ago. Loads come back in order, so the newest
    // STAGES - 1 steps may still be under way (near the end, where there are fewer, all are waited for).
    if (s + STAGES - 1 < steps) {
      issue(s + STAGES - 1);
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 1) * LOADS) : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    const unsigned char* at = ring + (s % STAGES) * STEP_BYTES + l16 * 128;
    moe_bf16x8 av[2], b1[2], b2[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int slot = ((2 * grp + u) ^ (l16 >> 1)) * 16;  // a lane's sixteen k of the step, as in the kernel above
      av[u] = *reinterpret_cast<const moe_bf16x8*>(at + slot);
      b1[u] = *reinterpret_cast<const moe_bf16x8*>(at + 2048 + slot);
      if (GATED) b2[u] = *reinterpret_cast<const moe_bf16x8*>(at + 4096 + slot);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[u], b1[u], acc1, 0, 0, 0);
      if (GATED) acc2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[u], b2[u], acc2, 0, 0, 0);
    }
    // the next loads overwrite what was read a step ago: the reads are done before any is issued
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  // The waves' sums meet in LDS, each in its own ring (nothing is under way any more), and are added in wave order.
  if (wave > 0) {
    float* meet = reinterpret_cast<float*>(ring);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      meet[r * WAVE + lane] = acc1[r];
      if (GATED) meet[(4 + r) * WAVE + lane] = acc2[r];
    }
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int w = 1; w < 4; ++w) {
    const float* meet = reinterpret_cast<const float*>(moe_ring + w * STAGES * STEP_BYTES);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      acc1[r] += meet[r * WAVE + lane];
      if (GATED) acc2[r] += meet[(4 + r) * WAVE + lane];
    }
  }
  if (n0 + l16 >= N) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int m = grp * 4 + r;
    if (m >= count) continue;
    const int pair = order[start + m];
    const float pw = pair_weight ? pair_weight[pair] : 1.f;
    if (FIRST) {
      const float v = GATED ? gated_value(acc1[r] * pw, acc2[r] * pw, act, limit) : activate(acc1[r] * pw, act);
      ((bf16*)out)[(size_t)(start + m) * N + n0 + l16] = static_cast<bf16>(v);
    } else {
      ((float*)out)[(size_t)pair * N + n0 + l16] = acc1[r] * pw;
    }
  }
}

// The same two products for steps with many pairs per expert (K a multiple of 64, rows 16-byte aligned): tiles of up to 32 MAX_FM pairs
// x 128 weight rows, K in slabs of 64 that go straight into LDS (global_load_lds, 16 bytes a lane) in a ring, one barrier per slab.
// Four waves a block in two by two, two blocks a CU: a wave owns every other run of 16 of the tile's pairs and 64 weight rows, so
// that a slab of 128 pairs takes 64 KB of fragment reads (eight waves of 32 x 64 read 96). The loop runs in half slabs: between the
// products of one set of fragments (32 k) the other set is read and, in a slab's second half, the loads of a later slab go out. A tile
// runs the loop made for its own number of runs (FM = pairs / 32, rounded up), so that an expert's last tile neither loads, reads nor
// multiplies rows that are not there; the plan cuts an expert's pairs evenly.
// What bounds it: with few pairs per expert the stream of the weights (537 MB of gate and up in 85 us, 6.3 TB/s); with many the loads
// (filling LDS and reading fragments from it take longer than the products) and,
// where K is short, what a block does before and after its loop. So:
//   * an XCD takes an eighth of the blocks, those of neighbouring tiles, the tiles of one expert and column run fastest: an expert's weights and rows
//     then come into one L2 once, where blocks in turn bring them into all eight (32 experts, 2,400 tokens 580 -> 565 us, 2,300 34.1 -> 33.0).
//     Where there are no more experts than XCDs and they have one or two tiles of 128 or 192 on average, the XCD of the expert with most pairs
//     would end last: there blocks go in turn, the columns of a tile fastest (8 experts, both products: 4,096 -> 4,608 of 96 pairs each 179 -> 162
//     us, 4,096 -> 3,072 of 378 313 -> 293, of 220 234 -> 227; 37 such steps 2.5 % less on average, one of them 5 % more). Eighths of the work, by the tiles' heights, measured slower: an
//     XCD with a block too many for its rounds of 64 takes a round more (2,000 tokens 92 -> 113);
//   * weights of an expert with one tile are marked as read once (200 tokens 95 -> 85 us; with two tiles it costs: 92 -> 103);
//   * the first slab's weights are asked for while the plan's indices are under way, the pairs' weights ahead of the loop, and an
//     activation is told apart once (the hardware's exp2 and reciprocal would save 4 of 102 us at 2,000 tokens, at four times the
//     activation's error).
// Microseconds, weights from memory, gated and second product, 32 experts of which a token runs 4 (before: eight waves, a slab's fragments
// read ahead of its products, tiles filled to the top, blocks in turn):
//   2000 tokens, 2048 -> 1024   110, 71  -> 102, 64       800 tokens, 4096 -> 1536   200, 98 -> 189, 100
//   2400 tokens, 4096 -> 3072   602, 317 -> 563, 308      600 tokens, 2048 -> 1024   72, 35  -> 67, 32
//   2300 tokens, 1024 -> 384    36, 27   -> 33, 23        200 tokens, 2048 -> 2048   95, 71  -> 84, 60
// In whole models prompts of 200 and 600 tokens take 5 to 12 % less, of 2,000 tokens level to 3 % (there the first row is 111, 65 -> 111, 67).
// Over 386 steps of 8 to 128 experts and 17 to 700 pairs each the two products take 6.5 % less on average. 21 of them take 1 to 7 % longer, one 10,
// half of these with 8 experts: their last round of blocks is often nearly empty, and a block alone on its CU has four waves now, not eight. The
// others have 16 to 64.
// A load instruction of a wave fills 1 KB of LDS in lane order, that is
// 8 tile rows of 128 bytes; the 16-byte chunk c of tile row R lands in slot c ^ ((R >> 1) & 7) of its row, so that a
// fragment read (16 rows, one chunk column) touches every bank once. The weight rows are the matrix instruction's first
// operand and the pairs its second: a lane ends up with four consecutive columns of one pair.
//   GATED: the tile's weight rows are blocks of 16 gate rows and 16 up rows in turn (64 columns of h a block), so that a
//          lane's fragments 2 i and 2 i + 1 are gate and up of the same four outputs.
// Pairs past the tile's count read the tile's last pair, weight rows past N the last row: their results are not stored.
// Every output element is one chain of products over k in ascending slabs, whatever the tile, the column and the pair's place in it. (Blocks that
// walk through k in step meet in the same memory channels, rows being a power of two apart. Sums that begin with a slab of the block's own avoid
// that, 600 tokens 67 -> 53 us, but a result then depends on its column and on the expert's number, and two models' logits came out 3 and 5 %
// further from 64 bits.)

// Block barrier after which at most N_ of this wave's loads are in flight (__syncthreads() would wait for all of them).
template <int N_> __device__ __forceinline__ void moe_wait_loads_and_block() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N_) : "memory");
}
// The same with at most n slabs of LOADS loads each in flight, n up to MOST.
template <int MOST, int LOADS> __device__ __forceinline__ void moe_wait_slabs_and_block(int n) {
  if constexpr (MOST > 0) {
    if (n < MOST) return moe_wait_slabs_and_block<MOST - 1, LOADS>(n);
  }
  moe_wait_loads_and_block<MOST * LOADS>();
}

constexpr int MOE_XCDS = 8;                                      // blocks are handed to the XCDs in turn
constexpr int MOE_BN = 128;                                      // weight rows of a tile
constexpr int moe_stage_bytes(int fm) { return (fm * 32 + MOE_BN) * 128; }
constexpr int moe_stages(int fm) { return fm == 1 ? 4 : fm == 2 ? 3 : 2; }  // what 80 KB hold
constexpr int moe_lds_bytes(int max_fm) {
  int most = 0;
  for (int fm = 1; fm <= max_fm; ++fm) most = moe_stages(fm) * moe_stage_bytes(fm) > most ? moe_stages(fm) * moe_stage_bytes(fm) : most;
  return most;
}

struct MoeTile {
  const bf16 *a, *w1, *w2;
  void* out;
  const int* order;
  const float* pair_weight;
  int lda, top, N, K, act;
  float limit;
  int n0, expert, start, count;  // first output column, and the tile's pairs
  bool once;                     // the expert has no other tile: its weights are read once
};

template <int MODE, int FM>
__device__ __forceinline__ void moe_tile(const MoeTile& t, unsigned char* lds) {
  constexpr bool GATED = MODE == 1, FIRST = MODE != 0;
  constexpr int FN = 4, KS = 64, ROW_BYTES = KS * 2, CPR = 8, RPI = 8, STAGES = moe_stages(FM);
  constexpr int XI = FM, WI = MOE_BN / (4 * RPI), LOADS = XI + WI, STAGE_BYTES = moe_stage_bytes(FM);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
  const int r = lane % 16, g = lane / 16;
  const int wr = wave / 2, wn = (wave % 2) * 64;
  const int slabs = t.K / KS;

  const int lrow = lane / CPR, lslot = lane % CPR;
  // What depends on the plan is asked for first, the weights of the first slab while it is under way. A slab's loads: weights (0 to
  // WI - 1; GATED: the first half of a wave's fill gate rows, the others up rows), then rows.
  int token[XI], pair[FM];
#pragma unroll
  for (int j = 0; j < XI; ++j) {
    const int place = t.start + min((wave * XI + j) * RPI + lrow, t.count - 1);
    token[j] = FIRST ? t.order[place] : place;
  }
  if (!FIRST || t.pair_weight) {
#pragma unroll
    for (int j = 0; j < FM; ++j) pair[j] = t.order[t.start + min((2 * j + wr) * 16 + r, t.count - 1)];
  }
  const bf16* src[LOADS];
#pragma unroll
  for (int j = 0; j < WI; ++j) {
    const int R = (wave * WI + j) * RPI + lrow;
    const int n = min(t.n0 + (GATED ? (R / 32) * 16 + R % 16 : R), t.N - 1);
    src[j] = (GATED && j >= WI / 2 ? t.w2 : t.w1) + ((size_t)t.expert * t.N + n) * t.K + ((lslot ^ ((R >> 1) & (CPR - 1))) * 8);
  }
  auto issue_one = [&](int slab, int j) __attribute__((always_inline)) {
    unsigned char* to = lds + (slab % STAGES) * STAGE_BYTES + (j < WI ? FM * 32 * ROW_BYTES + (wave * WI + j) * 1024 : (wave * XI + j - WI) * 1024);
    const auto from = (const void __attribute__((address_space(1)))*)(src[j] + (size_t)slab * KS);
    const auto at = (void __attribute__((address_space(3)))*)to;
    if (j < WI && t.once) __builtin_amdgcn_global_load_lds(from, at, 16, 0, LOAD_ONCE);
    else __builtin_amdgcn_global_load_lds(from, at, 16, 0, 0);
  };
#pragma unroll
  for (int j = 0; j < WI; ++j) issue_one(0, j);
#pragma unroll
  for (int j = 0; j < XI; ++j) {
    const int R = (wave * XI + j) * RPI + lrow;
    src[WI + j] = t.a + (size_t)(FIRST ? token[j] / t.top : token[j]) * t.lda + ((lslot ^ ((R >> 1) & (CPR - 1))) * 8);
  }
#pragma unroll
  for (int j = WI; j < LOADS; ++j) issue_one(0, j);
#pragma unroll
  for (int s = 1; s < STAGES; ++s)
    if (s < slabs) {
#pragma unroll
      for (int j = 0; j < LOADS; ++j) issue_one(s, j);
    }
  float pw[FM];
#pragma unroll
  for (int j = 0; j < FM; ++j) pw[j] = t.pair_weight ? t.pair_weight[pair[j]] : 1.f;

  moe_floatx4 acc[FN][FM];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) acc[i][j] = moe_floatx4{0.f, 0.f, 0.f, 0.f};
  const int sw = (r >> 1) & (CPR - 1);
  const int x_off = (wr * 16 + r) * ROW_BYTES, w_off = (FM * 32 + wn + r) * ROW_BYTES;

  moe_bf16x8 wf[2][FN], xf[2][FM];
  constexpr int PRODUCTS = FN * FM, READS = FN + FM;
  auto read_one = [&](int set, int slab, int q) __attribute__((always_inline)) {
    const unsigned char* stage = lds + (slab % STAGES) * STAGE_BYTES;
    const int slot = ((set * 4 + g) ^ sw) * 16;
    if (q < FN) wf[set][q < FN ? q : 0] = *reinterpret_cast<const moe_bf16x8*>(stage + w_off + q * 16 * ROW_BYTES + slot);
    else xf[set][q < FN ? 0 : q - FN] = *reinterpret_cast<const moe_bf16x8*>(stage + x_off + (q - FN) * 32 * ROW_BYTES + slot);
  };
  auto step = [&](int set, int read_slab, int load_slab, bool loads) __attribute__((always_inline)) {
    constexpr int SPAN = PRODUCTS > 6 ? PRODUCTS * 2 / 3 : PRODUCTS;  // the reads are out after two thirds of the products
#pragma unroll
    for (int p = 0; p < PRODUCTS; ++p) {
      acc[p / FM][p % FM] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[set][p / FM], xf[set][p % FM], acc[p / FM][p % FM], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < READS; ++q)
        if (q * SPAN / READS == p) read_one(1 - set, read_slab, q);
      if (loads) {
#pragma unroll
        for (int q = 0; q < LOADS; ++q)
          if (q * PRODUCTS / LOADS == p) issue_one(load_slab, q);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  moe_wait_slabs_and_block<STAGES - 1, LOADS>(slabs - 1);
#pragma unroll
  for (int q = 0; q < READS; ++q) read_one(0, 0, q);
  int k = 0;
  for (; k + STAGES < slabs; ++k) {
    step(0, k, 0, false);
    // Slab k + 1 is there for every wave, and every wave has read all of slab k.
    moe_wait_loads_and_block<LOADS * (STAGES - 2)>();
    step(1, k + 1, k + STAGES, true);
  }
  for (; k < slabs; ++k) {
    step(0, k, 0, false);
    moe_wait_slabs_and_block<STAGES - 2, LOADS>(slabs - 2 - k);
    step(1, k + 1, 0, false);  // behind the last slab: what is read lies in the ring and is not used
  }

  const int N = t.N;
  const bool vec = N % 4 == 0;
  // One straight run of code for each activation: told apart for each value, it cost more than the value.
  auto first = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int m = (2 * j + wr) * 16 + r;
      if (m >= t.count) continue;
      bf16* o = (bf16*)t.out + (size_t)(t.start + m) * N;
#pragma unroll
      for (int i = 0; i < FN; i += GATED ? 2 : 1) {
        const int col = t.n0 + (GATED ? wn / 2 + i / 2 * 16 : wn + i * 16) + g * 4;
        union { uint2 u; bf16 v[4]; } q;
#pragma unroll
        for (int c = 0; c < 4; ++c) q.v[c] = static_cast<bf16>(f(acc[i][j][c] * pw[j], acc[GATED ? i + 1 : i][j][c] * pw[j]));
        if (vec && col + 3 < N) *reinterpret_cast<uint2*>(o + col) = q.u;
        else
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (col + c < N) o[col + c] = q.v[c];
      }
    }
  };
  if constexpr (GATED) {
    static_assert(MS_GATED_COUNT == 3, "one case per activation below");
    if (t.act == MS_ACT_SILU) first([&](float a, float b) { return gated_value(a, b, MS_ACT_SILU, t.limit); });
    else if (t.act == MS_ACT_GELU_TANH) first([&](float a, float b) { return gated_value(a, b, MS_ACT_GELU_TANH, t.limit); });
    else first([&](float a, float b) { return gated_value(a, b, MS_ACT_SWIGLU_CLAMPED, t.limit); });
  } else if constexpr (FIRST) {
    if (t.act == MS_ACT_RELU_SQUARED) first([&](float a, float) { return activate(a, MS_ACT_RELU_SQUARED); });
    else if (t.act == MS_ACT_SILU) first([&](float a, float) { return activate(a, MS_ACT_SILU); });
    else first([&](float a, float) { return activate(a, t.act); });
  } else {
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      if ((2 * j + wr) * 16 + r >= t.count) continue;
      float* o = (float*)t.out + (size_t)pair[j] * N;
#pragma unroll
      for (int i = 0; i < FN; ++i) {
        const int col = t.n0 + wn + i * 16 + g * 4;
        const float4 v = make_float4(acc[i][j][0] * pw[j], acc[i][j][1] * pw[j], acc[i][j][2] * pw[j], acc[i][j][3] * pw[j]);
        if (vec && col + 3 < N) *reinterpret_cast<float4*>(o + col) = v;
        else
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (col + c < N) o[col + c] = c == 0 ? v.x : c == 1 ? v.y : c == 2 ? v.z : v.w;
      }
    }
  }
}

template <int MODE, int MAX_FM>
__global__ __launch_bounds__(256, 2) void moe_gemm_bf16_lds_kernel(
    const bf16* __restrict__ a, int lda, const bf16* __restrict__ w1, const bf16* __restrict__ w2, void* __restrict__ out,
    const int* __restrict__ order, const int* __restrict__ tile_expert, const int* __restrict__ tile_count, const int4* __restrict__ tile_run,
    const float* __restrict__ pair_weight, int max_tiles, unsigned cols, bool by_xcd, int top, int N, int K, int act, float limit) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char moe_lds[];
  const unsigned blocks = (unsigned)tile_count[max_tiles] * cols;  // at most as many as are launched: 31 bits
  unsigned at = blockIdx.x, end = blocks;
  if (by_xcd) {
    const unsigned xcd = blockIdx.x % MOE_XCDS;
    at = (unsigned)((unsigned long)xcd * blocks / MOE_XCDS) + blockIdx.x / MOE_XCDS;
    end = (unsigned)((xcd + 1ul) * blocks / MOE_XCDS);
  }
  if (at >= end) return;
  const unsigned any = at / cols;
  const int expert = tile_expert[any];
  const int4 run = tile_run[any];  // the expert's first tile, its tiles, its first place and its pairs
  unsigned tile = any - run.x, column = at % cols;
  if (by_xcd) {
    const unsigned local = at - (unsigned)run.x * cols;
    tile = local % run.y, column = local / run.y;
  }
  const int per = moe_pairs_per_tile(run.w, run.y, MAX_FM * 32), lo = (int)tile * per;
  const int start = run.z + lo, count = min(per, run.w - lo);
  const MoeTile t{a, w1, w2, out, order, pair_weight, lda, top, N, K, act, limit,
                  (int)column * (MODE == 1 ? MOE_BN / 2 : MOE_BN), expert, start, count, run.y == 1};
  const int fm = (count + 31) / 32;
  if (fm <= 1) moe_tile<MODE, 1>(t, moe_lds);
  else if (fm == 2) moe_tile<MODE, 2>(t, moe_lds);
  else if constexpr (MAX_FM > 2) {
    if (fm == 3) moe_tile<MODE, 3>(t, moe_lds);
    else if (fm == 4) moe_tile<MODE, 4>(t, moe_lds);
    else if constexpr (MAX_FM > 4) {
      if (fm == 5) moe_tile<MODE, 5>(t, moe_lds);
      else moe_tile<MODE, 6>(t, moe_lds);
    }
  }
}

template <int MODE, int MAX_FM>
static int moe_launch_lds(const void* a, int lda, const void* w1, const void* w2, void* out, const int* order, const int* tile_expert,
                          const int* tile_count, const void* tile_run, const float* pair_weight, int max_tiles, int experts, int top,
                          int N, int K, int act, float limit, hipStream_t st) {
  constexpr int lds_bytes = moe_lds_bytes(MAX_FM);
  static bool ready = false;  // more than 48 KB of LDS is asked for once per kernel
  if (!ready) {
    if (hipFuncSetAttribute((const void*)moe_gemm_bf16_lds_kernel<MODE, MAX_FM>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            lds_bytes) != hipSuccess)
      return MS_LAUNCH_FAILED;
    ready = true;
  }
  const int width = MODE == 1 ? MOE_BN / 2 : MOE_BN, cols = (N + width - 1) / width;
  const long blocks = ((long)cols * max_tiles + MOE_XCDS - 1) / MOE_XCDS * MOE_XCDS;
  if (blocks > 0x7fffffffl) return MS_BAD_ARG;
  const bool by_xcd = experts > MOE_XCDS || MAX_FM == 2 || max_tiles > 3 * experts;  // max_tiles: one an expert, and the pairs over a tile's
  moe_gemm_bf16_lds_kernel<MODE, MAX_FM><<<(unsigned)blocks, 256, lds_bytes, st>>>((const bf16*)a, lda, (const bf16*)w1, (const bf16*)w2, out, order,
                                                                                   tile_expert, tile_count, (const int4*)tile_run, pair_weight,
                                                                                   max_tiles, cols, by_xcd, top, N, K, act, limit);
  return launch_status();
}

// The same two products in true float32 on the vector units: 64 x 64 tiles through LDS, every output element one chain of
// fused multiply-adds over k in ascending order.
template <int MODE>
__global__ __launch_bounds__(256) void moe_gemm_f32_kernel(
    const float* __restrict__ a, int lda, const float* __restrict__ w1, const float* __restrict__ w2, float* __restrict__ out,
    const int* __restrict__ order, const int* __restrict__ tile_expert, const int* __restrict__ tile_start,
    const int* __restrict__ tile_count, const float* __restrict__ pair_weight, int top, int N, int K, int act, float limit) {
  constexpr bool GATED = MODE == 1, FIRST = MODE != 0;
  const int count = tile_count[blockIdx.x];
  if (count == 0) return;
  __shared__ float As[16][64 + 4];
  __shared__ float W1s[16][64 + 4];
  __shared__ float W2s[GATED ? 16 : 1][64 + 4];
  const int tid = threadIdx.x;
  const int e = tile_expert[blockIdx.x], start = tile_start[blockIdx.x];
  const int n0 = blockIdx.y * 64;
  const int tx = tid % 16, ty = tid / 16;      // 16 x 16 threads, 4 x 4 outputs each
  const int lr = tid / 4, lk = (tid % 4) * 4;  // loader: row within the tile, k offset
  const bool a_ok = lr < count;
  const float* arow = a + (size_t)(a_ok ? (FIRST ? order[start + lr] / top : start + lr) : 0) * lda;
  const bool w_ok = n0 + lr < N;
  const size_t wat = ((size_t)e * N + (w_ok ? n0 + lr : 0)) * K;
  float acc1[4][4], acc2[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc1[i][j] = acc2[i][j] = 0.f;
  for (int k0 = 0; k0 < K; k0 += 16) {
    float av[4], wv1[4], wv2[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = k0 + lk + i;
      av[i] = (a_ok && k < K) ? arow[k] : 0.f;
      wv1[i] = (w_ok && k < K) ? w1[wat + k] : 0.f;
      wv2[i] = (GATED && w_ok && k < K) ? w2[wat + k] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      As[lk + i][lr] = av[i];
      W1s[lk + i][lr] = wv1[i];
      if (GATED) W2s[lk + i][lr] = wv2[i];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      float x[4], u[4], v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = As[k][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        u[j] = W1s[k][tx * 4 + j];
        v[j] = GATED ? W2s[k][tx * 4 + j] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          acc1[i][j] = fmaf(x[i], u[j], acc1[i][j]);
          if (GATED) acc2[i][j] = fmaf(x[i], v[j], acc2[i][j]);
        }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = ty * 4 + i;
    if (m >= count) continue;
    const int pair = order[start + m];
    const float pw = pair_weight ? pair_weight[pair] : 1.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n >= N) continue;
      if (GATED) out[(size_t)(start + m) * N + n] = gated_value(acc1[i][j] * pw, acc2[i][j] * pw, act, limit);
      else if (FIRST) out[(size_t)(start + m) * N + n] = activate(acc1[i][j] * pw, act);
      else out[(size_t)pair * N + n] = acc1[i][j] * pw;
    }
  }
}

// a: the rows ([tokens, lda] for a first product, [P, lda] sorted places for the second); w1 (and w2, gated): [E, N, K];
// out: h [P, N] (a first product, the compute type) or y [P, N] float32. mode: 0 the second product, 1 the gated first
// product, 2 the plain first product. tile_rows: 16, 64, 128 or 192 in bfloat16 (from 128 on: K a multiple of 64 and 16-byte aligned
// rows), 64 in float32.
extern "C" int ms_moe_gemm(const void* a, int lda, const void* w1, const void* w2, void* out, int is_bf16, int mode,
                           const int* order, const int* tile_expert, const int* tile_start, const int* tile_count, const void* tile_run,
                           const float* pair_weight, int max_tiles, int experts, int top, int N, int K, int tile_rows, int act,
                           float limit, hipStream_t st) {
  if (max_tiles <= 0 || N <= 0) return MS_OK;
  const bool gated = mode == 1;
  if (mode < 0 || mode > 2 || a == nullptr || w1 == nullptr || (gated && w2 == nullptr) || out == nullptr || order == nullptr ||
      tile_expert == nullptr || tile_start == nullptr || tile_count == nullptr || tile_run == nullptr || experts < 1 || top < 1 ||
      K <= 0 || lda < K || (gated && (act < 0 || act >= MS_GATED_COUNT || (act == MS_ACT_SWIGLU_CLAMPED && !(limit > 0.f)))) || (mode == 2 && !ms_act_ungated_ok(act)))
    return MS_BAD_ARG;
  if (is_bf16) {
    if (tile_rows != 16 && tile_rows != 64 && tile_rows != 128 && tile_rows != 192) return MS_BAD_ARG;
    const bool rows16 = (size_t)a % 16 == 0 && (size_t)w1 % 16 == 0 && (!gated || (size_t)w2 % 16 == 0) && lda % 8 == 0;
    if (tile_rows >= 64 && K % 64 == 0 && rows16 && (mode != 0 || (size_t)out % 16 == 0)) {
#define MOE_LDS_MODE(G, ...) moe_launch_lds<G, __VA_ARGS__>(a, lda, w1, w2, out, order, tile_expert, tile_count, tile_run, pair_weight, max_tiles, experts, top, N, K, act, limit, st)
#define MOE_LDS(...) (mode == 1 ? MOE_LDS_MODE(1, __VA_ARGS__) : mode == 2 ? MOE_LDS_MODE(2, __VA_ARGS__) : MOE_LDS_MODE(0, __VA_ARGS__))
      return tile_rows == 192 ? MOE_LDS(6) : tile_rows == 128 ? MOE_LDS(4) : MOE_LDS(2);
#undef MOE_LDS
#undef MOE_LDS_MODE
    }
    if (tile_rows >= 128) return MS_UNSUPPORTED;  // the caller plans these tiles only where the kernel above takes them
    // 16-pair tiles whose K is no multiple of 64: min(E, pairs) of them at most are in use, each times the column blocks; the narrowest run of columns
    // with which that is under four blocks a CU.
    int nt = 4;
    if (tile_rows == 16) {
      const long busy = max_tiles / 2 + 1;  // about half of the launched tiles hold pairs
      while (nt > 1 && busy * ((N + 64 * nt - 1) / (64 * nt)) < 1024) nt /= 2;
    }
    const bool aligned = K % 8 == 0 && lda % 8 == 0 && (size_t)a % 16 == 0 && (size_t)w1 % 16 == 0 && (!gated || (size_t)w2 % 16 == 0);
    if (tile_rows == 16 && aligned && K % 64 == 0 && (N + 15) / 16 <= 65535) {
      const dim3 grid(max_tiles, (N + 15) / 16);
#define MOE_STREAM(G, BLOCKS) moe_gemm_bf16_stream_kernel<G, 2, BLOCKS><<<grid, 256, 4 * 2 * (G == 1 ? 3 : 2) * 2048, st>>>((const bf16*)a, lda, (const bf16*)w1, (const bf16*)w2, out, order, tile_expert, tile_start, tile_count, pair_weight, top, N, K, act, limit)
      if (mode == 1) MOE_STREAM(1, 3);
      else if (mode == 2) MOE_STREAM(2, 4);
      else MOE_STREAM(0, 4);
#undef MOE_STREAM
      return launch_status();
    }
#define MOE_ARGS (const bf16*)a, lda, (const bf16*)w1, (const bf16*)w2, out, order, tile_expert, tile_start, tile_count, pair_weight, top, N, K, tile_rows, act, limit
    // still few blocks at the narrowest columns: the waves of a block share 16 columns and split K
    if (tile_rows == 16 && nt == 1 && aligned && K >= 512 && (max_tiles / 2 + 1) * ((N + 63) / 64) < 2048 && (N + 15) / 16 <= 65535) {
      const dim3 grid(max_tiles, (N + 15) / 16);
      if (mode == 1) moe_gemm_bf16_kernel<1, true, 1, true><<<grid, 256, 0, st>>>(MOE_ARGS);
      else if (mode == 2) moe_gemm_bf16_kernel<2, true, 1, true><<<grid, 256, 0, st>>>(MOE_ARGS);
      else moe_gemm_bf16_kernel<0, true, 1, true><<<grid, 256, 0, st>>>(MOE_ARGS);
      return launch_status();
    }
    const int cols = tile_rows == 64 ? 64 : 64 * nt;
    const dim3 grid(max_tiles, (N + cols - 1) / cols);
    if (grid.y > 65535) return MS_BAD_ARG;
#define MOE(G, A, T) moe_gemm_bf16_kernel<G, A, T><<<grid, 256, 0, st>>>(MOE_ARGS)
#define MOE_NT(G, A) do { if (nt == 4) MOE(G, A, 4); else if (nt == 2) MOE(G, A, 2); else MOE(G, A, 1); } while (0)
#define MOE_AL(G) do { if (aligned) MOE_NT(G, true); else MOE_NT(G, false); } while (0)
    if (mode == 1) MOE_AL(1);
    else if (mode == 2) MOE_AL(2);
    else MOE_AL(0);
#undef MOE_AL
#undef MOE_NT
#undef MOE
#undef MOE_ARGS
  } else {
    if (tile_rows != 64) return MS_BAD_ARG;
    const dim3 grid(max_tiles, (N + 63) / 64);
    if (grid.y > 65535) return MS_BAD_ARG;
#define MOE_F32(G) moe_gemm_f32_kernel<G><<<grid, 256, 0, st>>>((const float*)a, lda, (const float*)w1, (const float*)w2, (float*)out, order, tile_expert, tile_start, tile_count, pair_weight, top, N, K, act, limit)
    if (mode == 1) MOE_F32(1);
    else if (mode == 2) MOE_F32(2);
    else MOE_F32(0);
#undef MOE_F32
  }
  return launch_status();
}

// ---------------------------------------------------------------------------------------------
// stream[t][n] += scale[n] (where it is given) times (the sum over j < top of y[t * top + j][n], in ascending j, plus the extra
// term). With ids: a choice whose id is `real` or more is an identity expert, and its term is weights[t * top + j] * x[t][n] (y
// holds nothing for it). The extra term (extra not nullptr) is what a feed-forward that every token runs put out, as
// `extra_splits` partial sums extra_stride floats apart, [T, N] each, times sigmoid(z[t]) where z is given: one number per token,
// the first column of rows z_ld apart that come as z_splits partial sums z_stride floats apart.
// A thread owns VEC consecutive columns of a token.
struct MoeExtra {
  const float* sum;
  int splits;
  size_t stride;
  const float* z;
  int z_ld, z_splits;
  size_t z_stride;
};

template <typename TX, int VEC>
__global__ __launch_bounds__(256) void moe_combine_kernel(float* __restrict__ stream, const float* __restrict__ y, int top, int N,
                                                          const int* __restrict__ ids, const float* __restrict__ weights,
                                                          const TX* __restrict__ x, int ldx, int real, const float* __restrict__ scale,
                                                          MoeExtra extra) {
  struct alignas(4 * VEC) Columns { float e[VEC]; };
  const int n = (blockIdx.x * blockDim.x + threadIdx.x) * VEC;
  if (n >= N) return;
  const size_t t = blockIdx.y;
  float acc[VEC];
#pragma unroll
  for (int i = 0; i < VEC; ++i) acc[i] = 0.f;
#pragma unroll 4
  for (int j = 0; j < top; ++j) {
    if (ids != nullptr && ids[t * top + j] >= real) {
      const float w = weights[t * top + j];
#pragma unroll
      for (int i = 0; i < VEC; ++i) acc[i] += w * to_f32(x[t * ldx + n + i]);
    } else {
      const Columns v = *reinterpret_cast<const Columns*>(y + (t * top + j) * N + n);
#pragma unroll
      for (int i = 0; i < VEC; ++i) acc[i] += v.e[i];
    }
  }
  if (extra.sum != nullptr) {
    const float g = extra.z != nullptr ? 1.f / (1.f + expf(-sum_splits(extra.z + t * extra.z_ld, extra.z_splits, extra.z_stride))) : 1.f;
    const float* p = extra.sum + t * N + n;
    if constexpr (VEC == 4) {
      const float4 v = add_splits4(p, extra.splits, extra.stride);
      acc[0] += g * v.x; acc[1] += g * v.y; acc[2] += g * v.z; acc[3] += g * v.w;
    } else {
      acc[0] += g * sum_splits(p, extra.splits, extra.stride);
    }
  }
  Columns* s = reinterpret_cast<Columns*>(stream + t * N + n);
  Columns v = *s;
#pragma unroll
  for (int i = 0; i < VEC; ++i) v.e[i] += scale ? acc[i] * scale[n + i] : acc[i];
  *s = v;
}

extern "C" int ms_moe_combine(float* stream, const float* y, int T, int top, int N, const int* ids, const float* weights,
                              const void* x, int x_is_bf16, int ldx, int real, const float* scale, const float* extra,
                              int extra_splits, long long extra_stride, const float* z, int z_ld, int z_splits, long long z_stride,
                              hipStream_t st) {
  if (T <= 0 || N <= 0) return MS_OK;
  if (stream == nullptr || y == nullptr || top < 1 || T > 65535 || (ids != nullptr && (weights == nullptr || x == nullptr || ldx < N)) ||
      (extra != nullptr && (extra_splits < 1 || (extra_splits > 1 && extra_stride < (long long)T * N))) ||
      (z != nullptr && (extra == nullptr || z_ld < 1 || z_splits < 1 || (z_splits > 1 && z_stride < (long long)T * z_ld))))
    return MS_BAD_ARG;
  const bool vec = N % 4 == 0 && (size_t)stream % 16 == 0 && (size_t)y % 16 == 0 && (size_t)extra % 16 == 0 &&
                   (extra == nullptr || extra_stride % 4 == 0);
  const int cols = vec ? 1024 : 256;
  const dim3 grid((N + cols - 1) / cols, T);
  const MoeExtra ex{extra, extra_splits, (size_t)extra_stride, z, z_ld, z_splits, (size_t)z_stride};
#define COMBINE(TX, V) moe_combine_kernel<TX, V><<<grid, 256, 0, st>>>(stream, y, top, N, ids, weights, (const TX*)x, ldx, real, scale, ex)
  if (x_is_bf16) { if (vec) COMBINE(bf16, 4); else COMBINE(bf16, 1); }
  else { if (vec) COMBINE(float, 4); else COMBINE(float, 1); }
#undef COMBINE
  return launch_status();
}
