// Attention of rows that bring several tokens, for bfloat16 storage, with softmax weights that meet the values unrounded:
// each float32 weight is cut into three bfloat16 pieces (its leading, middle and last eight bits: their sum is the weight),
// and the second product runs once per piece into the same float32 accumulators. Scores are float32 sums of exact products.
//
// The form follows the prefill kernel for rounded weights: a block owns 64 NQ query rows (tokens x the heads of a key head's
// group), walks tiles of 64 keys held in a ring of two LDS stages (global_load_lds, chunks permuted so that fragment reads touch
// every bank once, one barrier per tile), and takes both products transposed (S^T = K Q^T, O^T = V^T P^T), key rows in an
// order that leaves a lane with eight consecutive keys of its own query row: weights never move between lanes, and a lane holds
// the maximum and sum of the row whose outputs it holds. KSPLIT == 2: two waves share a group of rows, each takes half of every
// key tile, and they meet once at the end. What bounds it is the matrix cores beside the vector units: per 16 rows and 64 keys of
// 128 elements 16 products for the scores and 48 for the values, and some twenty vector instructions a weight.
//
// Two sources of keys and values:
//  * EXPANDED == false: the paged cache (keys [pages, Hkv, 16, DP], values [pages, Hkv / value_share, Dv, 16]).
//  * EXPANDED == true: a latent attention's keys and values multiplied out for the step (see latent_gather_kernel): keys
//    [S, H DP] beside a part [S, DR] that all heads share, values transposed [H DV, S]. A prompt then multiplies DP + DR + 3 DV
//    elements per head, query and key, where the latent itself as key and value takes C + DR + 3 C: with 128 + 64, 128 and a
//    latent of 512 a quarter, for two products of the latents with the weights more. One layer's attention, 16 heads, latent
//    512 + 64, expansion included, against attention over the latents with its two products per head: 2,000 tokens 94 against
//    761 us, 256 tokens 35 / 72, 16 tokens 24 / 27, 64 tokens behind 16,000 649 / 2,529.
// Over the cache, against the kernels it took the place of (keys and values straight from the pages into registers, weights through
// LDS): 2,048 tokens, 16 heads over 4, 128 elements 53 us against 242 (keys beside kept first ones) and 149 (sinks); two maps
// over values of 256, 1,201 and two shorter prompts, 69 against 125.
//
// Waves and rows, measured at those shapes before the maximum lagged: over the cache 64 rows with KSPLIT = 2 are 63 us where 64 rows
// of four waves take 65 and 128 rows 93 (too few blocks); 8,192 tokens of 32 heads 1,158, 1,098 and 947. Since then 53, - and 79;
// 980, - and 845. Expanded, the fragments of 192 elements leave
// KSPLIT = 2 (128 registers a lane) spilling: 116 us against 94 with four waves at 64 rows, 123 at 128 rows.
#include "common.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;
typedef __attribute__((__vector_size__(4 * sizeof(int)))) int i32x4;

#define PAGE 16
#define TK 64  // keys per tile

struct ExactArgs {
  const bf16* q;          // the rows' queries: token * q_stride + head * q_head
  int q_stride, q_head;
  const bf16* q_turned;   // DR > 0: the turned part, token * qt_stride + head * qt_head
  int qt_stride, qt_head;
  const bf16 *k, *v;      // pages, or (EXPANDED) keys [S, H DP] and values [H DV, S]
  const bf16* k_turned;   // EXPANDED: [S, DR]
  const int* block_table;
  int table_width;
  const int* key_base;    // EXPANDED: per row of the step, where its key 0 would lie in [0, S) (a multiple of 64, may be negative)
  int keys;               // EXPANDED: S
  const int *tile_first, *tile_count, *token_row, *pos;
  bf16* out;
  float* out32;           // the result unrounded, if given
  int Hq, Hkv, value_share, value_runs;
  float scale, softcap;
  int window, keep_first;
  const float* sinks;
  const float* gate;      // results times sigmoid(gate[token * gate_ld + gate_col + (gate_each ? head * Dv + e : head)])
  int gate_ld, gate_col, gate_each;
};

template <int N>
__device__ __forceinline__ void wait_loads() {
  static_assert(N >= 0 && N < 64, "vmcnt has six bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

__device__ __forceinline__ int pick(i32x4 v, int i) {
  int p = v[0];
  p = i == 1 ? v[1] : p;
  p = i == 2 ? v[2] : p;
  p = i == 3 ? v[3] : p;
  return p;
}

// tanh on the hardware's exp2 and reciprocal: 1 - 2 / (1 + e^(2x)).
__device__ __forceinline__ float tanh_fast(float x) {
  return 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(x * 2.885390081777927f));
}

// The upper halves of two floats as a pair of bfloat16 (a first).
__device__ __forceinline__ unsigned upper_halves(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ __forceinline__ float upper(float p) { return __uint_as_float(__float_as_uint(p) & 0xffff0000u); }

// Which permutation of its 16-byte chunks a key row lies in: the 16 lanes that read a chunk column together take key rows
// {0-3, 8-11, 16-19, 24-27} (+ 4, + 32), which must come to 16 different slots of 256 bytes (two rows of 128 bytes side by side).
template <int CHUNKS> __device__ __forceinline__ int key_swizzle(int R) {
  return CHUNKS == 16 ? ((R & 3) | ((R >> 1) & 12)) : (((R >> 1) & 1) | ((R >> 2) & 6));
}

// Values of keys that no row of a block sees become zeros: their weight is zero, and zero times an infinity or NaN (of another
// request in page 0, which stands in for entries without a page, or of whoever had the page before) is NaN. Only tiles at the ends
// of what is seen have such keys. (The other keys of a multiplied-out row are zeros, or its own.) The masks of four pairs of
// values at keys key .. key + 7; seen are those up to `last` but for a gap from `kept` to before `lo`.
struct ValueMask { unsigned u[4]; };
__device__ __forceinline__ ValueMask value_mask(int key, int last, int lo, int kept) {
  auto first_bits = [](int n) { return (1u << max(0, min(8, n))) - 1u; };
  const unsigned seen = first_bits(last + 1 - key) & ~(first_bits(lo - key) & ~first_bits(kept - key));
  ValueMask m;
#pragma unroll
  for (int i = 0; i < 4; ++i) m.u[i] = ((seen >> (2 * i)) & 1u) * 0xffffu | ((seen >> (2 * i + 1)) & 1u) * 0xffff0000u;
  return m;
}

template <int DP, int DR, int DV> constexpr int exact_stage_bytes() { return TK * DP * 2 + TK * DR * 2 + DV * TK * 2; }
template <int DP, int DR, int DV, int NQ, int KSPLIT> constexpr int exact_lds_bytes() {
  constexpr int merge = KSPLIT > 1 ? 4 * NQ * (16 * (DV + 1) + 32) * 4 : 0;
  return 2 * exact_stage_bytes<DP, DR, DV>() > merge ? 2 * exact_stage_bytes<DP, DR, DV>() : merge;
}

template <int DP, int DR, int DV, int NQ, int KSPLIT, bool EXPANDED>
__global__ __launch_bounds__(256 * KSPLIT, 2 * KSPLIT) void attn_exact_kernel(ExactArgs a) {
  constexpr int NW = 4 * KSPLIT;
  constexpr int KP = DP / 32, KR = DR / 32, KK = KP + KR, DB = DV / 16;
  constexpr int ROWS = 64 * NQ, WROWS = 16 * NQ;
  constexpr int WK = TK / KSPLIT, TB = WK / 16;
  constexpr int PCH = DP / 8, RCH = DR > 0 ? DR / 8 : 8;  // 16-byte chunks of a key row, of its turned part
  constexpr int PRPI = 64 / PCH, RRPI = 64 / RCH;         // rows a load instruction of a wave fills
  constexpr int PI = TK / PRPI / NW, RI = DR > 0 ? TK / RRPI / NW : 0, VI = DV / 8 / NW;
  constexpr int P_BYTES = TK * DP * 2, R_BYTES = TK * DR * 2, STAGE_BYTES = exact_stage_bytes<DP, DR, DV>();
  static_assert(PI >= 1 && PI * PRPI * NW == TK && VI >= 1 && VI * 8 * NW == DV && (DR == 0 || RI * RRPI * NW == TK), "sizes");
  static_assert((PCH == 8 || PCH == 16) && RCH == 8, "the swizzles know rows of 128 and 256 bytes");
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  const int G = a.Hq / a.Hkv;
  const int combos = a.Hkv * a.value_runs;
  const int combo = blockIdx.x % combos, tile = blockIdx.x / combos;  // (a pair of key head and run of values stays on few XCDs)
  const int kvh = combo / a.value_runs, e0 = (combo % a.value_runs) * DV;
  const int Dv = a.value_runs * DV, vh = kvh / a.value_share, Hv = a.Hkv / a.value_share;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
  const int rg = wave % 4, kg = wave / 4;
  const int r = lane % 16, g = lane / 16;
  const int first = a.tile_first[tile], count = a.tile_count[tile];
  const int pos0 = a.pos[first], last_pos = pos0 + count - 1;
  const int batch_row = a.token_row[first];
  const int* table = EXPANDED ? nullptr : a.block_table + (size_t)batch_row * a.table_width;
  const int base = EXPANDED ? a.key_base[batch_row] : 0;
  const int window = a.window;
  const int kv_lo = (window > 0 && pos0 - window + 1 > 0) ? pos0 - window + 1 : 0;
  const int kept = a.keep_first < kv_lo ? a.keep_first : kv_lo;

  int row_pos[NQ];
  bool row_ok[NQ];
  bf16x8 qf[NQ][KK];
#pragma unroll
  for (int b = 0; b < NQ; ++b) {
    const int row = rg * WROWS + b * 16 + r;
    const int tok = row / G;
    row_ok[b] = tok < count && row < (ROWS / G) * G;
    row_pos[b] = pos0 + tok;
    const int head = kvh * G + row % G;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      if (row_ok[b]) {
        const bf16* src = kk < KP ? a.q + (size_t)(first + tok) * a.q_stride + (size_t)head * a.q_head + kk * 32
                                  : a.q_turned + (size_t)(first + tok) * a.qt_stride + (size_t)head * a.qt_head + (kk - KP) * 32;
        qf[b][kk] = *reinterpret_cast<const bf16x8*>(src + g * 8);
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) qf[b][kk][i] = static_cast<bf16>(0.f);
      }
    }
  }
  const int grp_first_tok = (rg * WROWS) / G;
  const int grp_last_tok = min(count - 1, (rg * WROWS + WROWS - 1) / G);
  const bool grp_has_rows = grp_first_tok < count;
  const int grp_last_pos = pos0 + grp_last_tok, grp_first_pos = pos0 + grp_first_tok;

  // Over the cache the maximum that the exponents subtract may lag behind a row's own by up to 8 (in units of log2): the weights are exact
  // in float32 and reach the products unrounded, so nothing is lost by it, and the tiles that raise no row's maximum by more exchange
  // nothing between lanes and rescale nothing; each lane keeps its own share of a row's sum until the end (the error against 64 bits: 1
  // to 2 % less). A row renews its maximum by its own scores alone, so that its bits don't depend on the rows beside it; until it does so
  // its weights may be up to 256. Microseconds, 2,048 tokens of 16 heads over 4 of 128 behind a window of 2,048: 64 before, 53 now (128
  // rows: 96 and 79); 8,192 of 32 over 8: 1,160 and 980 (980 and 845). What must not grow is the lanes' state: a limit and a rescale
  // factor kept in registers spilled the form of 128 registers inside the loop and took 61; as it is, that form leaves 20 bytes a lane in
  // scratch memory, written ahead of the loop and read behind it. Multiplied out the lag saved 4 of 63; there the maximum stays the
  // row's own and sums are joined tile by tile, which keeps the results of the form before to the bit.
  constexpr bool LAGS = !EXPANDED;
  constexpr float LAG = LAGS ? 8.f : 0.f;
  float m_run[NQ], l_run[NQ];
  floatx4 o[NQ][DB];
#pragma unroll
  for (int b = 0; b < NQ; ++b) {
    m_run[b] = -INFINITY;
    l_run[b] = 0.f;
#pragma unroll
    for (int i = 0; i < DB; ++i) o[b][i] = floatx4{0.f, 0.f, 0.f, 0.f};
  }

  // The key tiles: those of the kept first keys, then those from the window's first key on. Number n starts at key tile_at(n).
  const int kept_tiles = (kept + TK - 1) / TK;
  const int window_tile = max(kv_lo / TK, kept_tiles);
  const int n_tiles = kept_tiles + (last_pos / TK - window_tile + 1);
  auto tile_at = [&](int n) { return (n < kept_tiles ? n : window_tile + n - kept_tiles) * TK; };

  // The first key from `from` on that no row of the block sees (see value_mask).
  auto first_unseen = [&](int from) { return from < kv_lo ? max(from, kept) : last_pos + 1; };
  // Masked in the fragments, that costs nothing but instructions; where these would spill, in LDS before the barrier. 3,000 tokens
  // behind a window of 128, 16 heads, with masks and without: heads of 64 22.9 us and 22.2, of 128 31.6 and 29.7 (in fragments 39.1).
  constexpr bool MASK_FRAGMENTS = !EXPANDED && !(DP == 128 && KSPLIT == 2);

  // What does not depend on the tile: the offset of the lane's chunk within its page (or from the tile's first key), and which
  // of the tile's four pages it comes from.
  int p_page[PI], v_page[VI];
  unsigned p_off[PI], r_off[RI > 0 ? RI : 1], v_off[VI];
#pragma unroll
  for (int j = 0; j < PI; ++j) {
    const int R = (wave * PI + j) * PRPI + lane / PCH, c = (lane % PCH) ^ key_swizzle<PCH>(R);
    p_page[j] = __builtin_amdgcn_readfirstlane(R / PAGE);  // the rows of one instruction lie in one page
    p_off[j] = EXPANDED ? (unsigned)(R * (a.Hkv * DP) + c * 8) : (unsigned)((kvh * PAGE + R % PAGE) * DP + c * 8);
  }
#pragma unroll
  for (int j = 0; j < RI; ++j) {
    const int R = (wave * RI + j) * RRPI + lane / RCH, c = (lane % RCH) ^ key_swizzle<RCH>(R);
    r_off[j] = (unsigned)(R * DR + c * 8);
  }
#pragma unroll
  for (int j = 0; j < VI; ++j) {
    const int d = (wave * VI + j) * 8 + lane / 8, c = (lane % 8) ^ ((d >> 1) & 7);  // chunk c: keys 8 c .. 8 c + 7 of the tile
    v_page[j] = c / 2;
    v_off[j] = EXPANDED ? (unsigned)(c * 8) : (unsigned)((vh * Dv + e0 + d) * PAGE + (c % 2) * 8);
  }
  const unsigned k_page_bytes = (unsigned)(a.Hkv * PAGE * DP * 2), v_page_bytes = (unsigned)(Hv * Dv * PAGE * 2);  // (the host checks that they fit)
  auto at_page = [](const bf16* base, int page, unsigned bytes, unsigned off) __attribute__((always_inline)) {
    return (const bf16*)((const char*)(base + off) + (unsigned long long)(unsigned)max(page, 0) * bytes);
  };
  auto load = [&](const bf16* src, unsigned char* to) __attribute__((always_inline)) {
    __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)src, (void __attribute__((address_space(3)))*)to, 16, 0, 0);
  };
  auto tile_pages = [&](int n) -> i32x4 {  // tiles past the last are clamped to it: what is fetched for them is never used
    if constexpr (EXPANDED) return i32x4{0, 0, 0, 0};
    else return *reinterpret_cast<const i32x4*>(table + tile_at(min(n, n_tiles - 1)) / PAGE);
  };
  auto issue = [&](int n, i32x4 pages) __attribute__((always_inline)) {
    unsigned char* stage = smem + (n % 2) * STAGE_BYTES;
    if constexpr (EXPANDED) {
      const int at = base + tile_at(min(n, n_tiles - 1));  // a multiple of 64, and the tile's 64 keys lie in [0, S)
      const bf16* kt = a.k + (size_t)at * (a.Hkv * DP) + kvh * DP;
      const bf16* rt = a.k_turned + (size_t)at * DR;
      const bf16* vt = a.v + (size_t)kvh * DV * a.keys + at;
#pragma unroll
      for (int j = 0; j < PI; ++j) load(kt + p_off[j], stage + (wave * PI + j) * 1024);
#pragma unroll
      for (int j = 0; j < RI; ++j) load(rt + r_off[j], stage + P_BYTES + (wave * RI + j) * 1024);
#pragma unroll
      for (int j = 0; j < VI; ++j)
        load(vt + (size_t)((wave * VI + j) * 8 + lane / 8) * a.keys + v_off[j], stage + P_BYTES + R_BYTES + (wave * VI + j) * 1024);
    } else {
      // entries without a page (past the last key, or given back behind a window) read page 0: their keys are masked, their values made zeros
#pragma unroll
      for (int j = 0; j < PI; ++j) load(at_page(a.k, pick(pages, p_page[j]), k_page_bytes, p_off[j]), stage + (wave * PI + j) * 1024);
#pragma unroll
      for (int j = 0; j < VI; ++j)
        load(at_page(a.v, pick(pages, v_page[j]), v_page_bytes, v_off[j]), stage + P_BYTES + R_BYTES + (wave * VI + j) * 1024);
    }
  };

  const float cap_in = a.softcap > 0.f ? a.scale / a.softcap : 0.f;
  const float cap_out = a.softcap * 1.44269504088896340736f;
  const float scale2 = a.softcap > 0.f ? 1.f : a.scale * 1.44269504088896340736f;  // scores in units of log2 (bounded ones are when made)
  i32x4 pages_next = tile_pages(0);
  {
    const i32x4 pages = pages_next;
    pages_next = tile_pages(1);
    issue(0, pages);
  }
  const int krow = (r < 8 ? 0 : 16) + (r % 4) + 8 * ((r / 4) % 2);
  const int vsw = (r >> 1) & 7;
  for (int n = 0; n < n_tiles; ++n) {
    const int t0 = tile_at(n);
    wait_loads<0>();
    if (!EXPANDED && !MASK_FRAGMENTS && t0 + TK > first_unseen(t0)) {  // a lane masks what it has fetched itself
#pragma unroll
      for (int j = 0; j < VI; ++j) {
        const int d = (wave * VI + j) * 8 + lane / 8;
        const ValueMask m = value_mask(t0 + 8 * ((lane % 8) ^ ((d >> 1) & 7)), last_pos, kv_lo, kept);
        uint4* v = reinterpret_cast<uint4*>(smem + (n % 2) * STAGE_BYTES + P_BYTES + R_BYTES + (wave * VI + j) * 1024 + lane * 16);
        const uint4 x = *v;
        *v = make_uint4(x.x & m.u[0], x.y & m.u[1], x.z & m.u[2], x.w & m.u[3]);
      }
    }
    __syncthreads();  // tile n has landed for every wave, and every wave is done with tile n - 1
    {
      const i32x4 pages = pages_next;
      pages_next = tile_pages(n + 2);
      issue(n + 1, pages);
    }
    const unsigned char* ks = smem + (n % 2) * STAGE_BYTES;
    const unsigned char* rs = ks + P_BYTES;
    const unsigned char* vs = rs + R_BYTES;
    const int w0 = t0 + kg * WK;  // this wave's keys of the tile: w0 .. w0 + WK - 1
    if (!grp_has_rows || w0 > grp_last_pos) continue;
    if (window > 0 && w0 + WK - 1 < grp_first_pos - window + 1 && w0 >= a.keep_first) continue;  // (the block may see as windowed what the wave sees as kept)

    floatx4 s[NQ][TB];
#pragma unroll
    for (int b = 0; b < NQ; ++b)
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) s[b][tb] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      bf16x8 kf[TB];
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) {
        const int R = kg * WK + (tb / 2) * 32 + krow + 4 * (tb % 2);
        kf[tb] = kk < KP ? *reinterpret_cast<const bf16x8*>(ks + R * (DP * 2) + (((kk * 4 + g) ^ key_swizzle<PCH>(R)) * 16))
                         : *reinterpret_cast<const bf16x8*>(rs + R * (DR * 2) + ((((kk - KP) * 4 + g) ^ key_swizzle<RCH>(R)) * 16));
      }
#pragma unroll
      for (int tb = 0; tb < TB; ++tb)
#pragma unroll
        for (int b = 0; b < NQ; ++b) s[b][tb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[tb], qf[b][kk], s[b][tb], 0, 0, 0);
    }
    if (a.softcap > 0.f) {
#pragma unroll
      for (int b = 0; b < NQ; ++b)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
          for (int i = 0; i < 4; ++i) s[b][tb][i] = cap_out * tanh_fast(s[b][tb][i] * cap_in);
    }
    // Masks only where the keys cross the diagonal, the window's edge or the end of the kept keys for some row of the group
    // (the same answer for the whole wave).
    const bool masked = __builtin_amdgcn_readfirstlane((int)(w0 + WK - 1 > grp_first_pos || (window > 0 && w0 <= grp_last_pos - window)));
    if (masked) {
#pragma unroll
      for (int b = 0; b < NQ; ++b)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int t = w0 + (tb / 2) * 32 + 8 * g + 4 * (tb % 2) + i;
            const bool seen = !row_ok[b] | ((t <= row_pos[b]) & ((window == 0) | (t > row_pos[b] - window) | (t < a.keep_first)));
            s[b][tb][i] = seen ? s[b][tb][i] : -INFINITY;
          }
    }
    union Piece { unsigned u[4]; bf16x8 v; } hi[NQ][TB / 2], mid[NQ][TB / 2], low[NQ][TB / 2];
#pragma unroll
    for (int b = 0; b < NQ; ++b) {
      float s_max = -INFINITY;
#pragma unroll
      for (int tb = 0; tb < TB; ++tb)
#pragma unroll
        for (int i = 0; i < 4; ++i) s_max = fmaxf(s_max, s[b][tb][i]);
      float corr = 1.f;
      if (__builtin_amdgcn_ballot_w64(s_max * scale2 > m_run[b] + LAG) != 0) {
        const float m_top = rows4_max(s_max) * scale2;
        const float m_new = m_top > m_run[b] + LAG ? m_top : m_run[b];  // each row by its own scores: its bits don't depend on the rows beside it
        corr = __builtin_amdgcn_exp2f(m_run[b] - (m_new == -INFINITY ? 0.f : m_new));
        if (LAGS) l_run[b] *= corr;
        m_run[b] = m_new;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[b][db][i] *= corr;
      }
      const float m_sub = m_run[b] == -INFINITY ? 0.f : m_run[b];  // a row that has seen no key yet
      float psum = 0.f;  // (of this tile by itself: added one by one to the longer sum, the weights lose more)
#pragma unroll
      for (int tb = 0; tb < TB; ++tb)
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
          const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[b][tb][i], scale2, -m_sub));
          const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[b][tb][i + 1], scale2, -m_sub));
          psum += p0;
          psum += p1;
          const float r0 = p0 - upper(p0), r1 = p1 - upper(p1);  // exact: what is left of 24 bits
          const int at = (tb % 2) * 2 + i / 2;
          hi[b][tb / 2].u[at] = upper_halves(p0, p1);
          mid[b][tb / 2].u[at] = upper_halves(r0, r1);
          low[b][tb / 2].u[at] = upper_halves(r0 - upper(r0), r1 - upper(r1));
        }
      l_run[b] = LAGS ? l_run[b] + psum : l_run[b] * corr + rows4_sum(psum);
    }
#pragma unroll
    for (int pr = 0; pr < TB / 2; ++pr) {
      bf16x8 vf[DB];
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const int c = (kg * WK + pr * 32) / 8 + g;
        vf[db] = *reinterpret_cast<const bf16x8*>(vs + (db * 16 + r) * (TK * 2) + ((c ^ vsw) * 16));
      }
      if (MASK_FRAGMENTS && w0 + WK > first_unseen(w0)) {
        const ValueMask m = value_mask(w0 + pr * 32 + 8 * g, last_pos, kv_lo, kept);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          Piece v;
          v.v = vf[db];
#pragma unroll
          for (int i = 0; i < 4; ++i) v.u[i] &= m.u[i];
          vf[db] = v.v;
        }
      }
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int b = 0; b < NQ; ++b) o[b][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[db], hi[b][pr].v, o[b][db], 0, 0, 0);
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int b = 0; b < NQ; ++b) o[b][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[db], mid[b][pr].v, o[b][db], 0, 0, 0);
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int b = 0; b < NQ; ++b) o[b][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[db], low[b][pr].v, o[b][db], 0, 0, 0);
    }
  }
  if (LAGS) {
#pragma unroll
    for (int b = 0; b < NQ; ++b) l_run[b] = rows4_sum(l_run[b]);
  }
  wait_loads<0>();  // the tile fetched ahead past the end must not land in memory that is used otherwise

  if (KSPLIT > 1) {
    // The second key group hands its running maximum, sum and output to the first through LDS.
    __syncthreads();
    float* mg = reinterpret_cast<float*>(smem);
    constexpr int PER = 16 * (DV + 1) + 32;
#pragma unroll
    for (int b = 0; b < NQ; ++b) {
      float* at = mg + (rg * NQ + b) * PER;
      if (kg == 1) {
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int i = 0; i < 4; ++i) at[r * (DV + 1) + db * 16 + 4 * g + i] = o[b][db][i];
        if (g == 0) {
          at[16 * (DV + 1) + r] = m_run[b];
          at[16 * (DV + 1) + 16 + r] = l_run[b];
        }
      }
    }
    __syncthreads();
    if (kg == 1) return;
#pragma unroll
    for (int b = 0; b < NQ; ++b) {
      const float* at = mg + (rg * NQ + b) * PER;
      const float m2 = at[16 * (DV + 1) + r], l2 = at[16 * (DV + 1) + 16 + r];
      const float m = fmaxf(m_run[b], m2);
      const float m_safe = m == -INFINITY ? 0.f : m;
      const float f1 = __builtin_amdgcn_exp2f(m_run[b] - m_safe), f2 = __builtin_amdgcn_exp2f(m2 - m_safe);
      l_run[b] = l_run[b] * f1 + l2 * f2;
      m_run[b] = m;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[b][db][i] = o[b][db][i] * f1 + at[r * (DV + 1) + db * 16 + 4 * g + i] * f2;
    }
  }

  // o[b][db][i] = O[row r of block b][e0 + db * 16 + 4 g + i]
#pragma unroll
  for (int b = 0; b < NQ; ++b) {
    const int row = rg * WROWS + b * 16 + r;
    const int tok = row / G;
    if (tok >= count || row >= (ROWS / G) * G) continue;
    const int head = kvh * G + row % G;
    float inv = 1.f / l_run[b];
    if (a.sinks) {  // exp(sink) joins the denominator: both are brought to the larger of the two maxima first
      const float sink2 = a.sinks[head] * 1.44269504088896340736f, m_all = fmaxf(m_run[b], sink2);
      const float c = __builtin_amdgcn_exp2f(m_run[b] - m_all);
      inv = c / (l_run[b] * c + __builtin_amdgcn_exp2f(sink2 - m_all));
    }
    const size_t at = ((size_t)(first + tok) * a.Hq + head) * Dv + e0 + 4 * g;
    const float* gr = a.gate ? a.gate + (size_t)(first + tok) * a.gate_ld + a.gate_col + (a.gate_each ? (size_t)head * Dv + e0 + 4 * g : (size_t)head) : nullptr;
    if (gr && !a.gate_each) inv *= 1.f / (1.f + expf(-gr[0]));
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      floatx4 v = o[b][db] * inv;
      if (gr && a.gate_each) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] *= 1.f / (1.f + expf(-gr[db * 16 + i]));
      }
      if (a.out32) {
        *reinterpret_cast<floatx4*>(a.out32 + at + db * 16) = v;
      } else {
        bf16x4 w;
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = static_cast<bf16>(v[i]);
        *reinterpret_cast<bf16x4*>(a.out + at + db * 16) = w;
      }
    }
  }
}

template <int DP, int DR, int DV, int NQ, int KSPLIT, bool EXPANDED>
static int launch_exact(unsigned grid, const ExactArgs& a, hipStream_t st) {
  constexpr int lds = exact_lds_bytes<DP, DR, DV, NQ, KSPLIT>();
  static_assert(2 * lds <= 160 * 1024, "two blocks share a CU");
  static bool ready = false;  // more than 64 KB of LDS has to be asked for once per kernel
  if (!ready) {
    if (hipFuncSetAttribute((const void*)attn_exact_kernel<DP, DR, DV, NQ, KSPLIT, EXPANDED>, hipFuncAttributeMaxDynamicSharedMemorySize, lds) !=
        hipSuccess)
      return MS_LAUNCH_FAILED;
    ready = true;
  }
  attn_exact_kernel<DP, DR, DV, NQ, KSPLIT, EXPANDED><<<grid, 256 * KSPLIT, lds, st>>>(a);
  return launch_status();
}

// The run of value elements a block owns (0: the kernel does not take the shape): keys of 64 or 128 elements, values a
// multiple of 64 or 128 elements respectively, up to 64 query heads per key head, 16-token pages.
extern "C" int ms_attention_exact_run(int group, int D, int Dv, int page_size) {
  if (page_size != PAGE || group < 1 || group > 64 || (D != 64 && D != 128) || Dv < D || Dv % D) return 0;
  return D;
}

// Rows that bring several tokens over the paged cache; tiles of rows_per_tile / group tokens, rows_per_tile 64 or 128 (64: two
// waves share a group of rows).
extern "C" int ms_attention_exact(const void* q, int q_stride, const void* k, const void* v, const int* block_table, int table_width,
                                  const int* tile_first, const int* tile_count, int tiles, int rows_per_tile, const int* token_row,
                                  const int* pos, void* out, int out_f32, int Hq, int Hkv, int D, int Dv, int page_size, float scale,
                                  int window, int keep_first, float softcap, const float* sinks, int value_share, hipStream_t st) {
  if (tiles <= 0) return MS_OK;
  if (Hq <= 0 || Hkv <= 0 || Hq % Hkv || window < 0 || keep_first < 0 || table_width <= 0 || table_width % 4 || q_stride < Hq * D ||
      q_stride % 8 || (size_t)q % 16 || (size_t)k % 16 || (size_t)v % 16 || (size_t)block_table % 16 || (size_t)out % 16 || !(softcap >= 0.f) ||
      value_share < 1 || Hkv % value_share || (rows_per_tile != 64 && rows_per_tile != 128) || Hq / Hkv > rows_per_tile)
    return MS_BAD_ARG;
  const int run = ms_attention_exact_run(Hq / Hkv, D, Dv, page_size);
  if (run == 0 || (long long)Hkv * PAGE * D * 2 > 2147483647LL || (long long)(Hkv / value_share) * PAGE * Dv * 2 > 2147483647LL) return MS_UNSUPPORTED;
  const long long blocks = (long long)tiles * Hkv * (Dv / run);
  if (blocks > 2147483647LL) return MS_BAD_ARG;
  ExactArgs a{};
  a.q = (const bf16*)q; a.q_stride = q_stride; a.q_head = D;
  a.k = (const bf16*)k; a.v = (const bf16*)v;
  a.block_table = block_table; a.table_width = table_width;
  a.tile_first = tile_first; a.tile_count = tile_count; a.token_row = token_row; a.pos = pos;
  a.out = (bf16*)out; a.out32 = out_f32 ? (float*)out : nullptr;
  a.Hq = Hq; a.Hkv = Hkv; a.value_share = value_share; a.value_runs = Dv / run;
  a.scale = scale; a.softcap = softcap; a.window = window; a.keep_first = window > 0 ? keep_first : 0; a.sinks = sinks;
  if (D == 128) return rows_per_tile == 128 ? launch_exact<128, 0, 128, 2, 1, false>((unsigned)blocks, a, st)
                                            : launch_exact<128, 0, 128, 1, 2, false>((unsigned)blocks, a, st);
  return rows_per_tile == 128 ? launch_exact<64, 0, 64, 2, 1, false>((unsigned)blocks, a, st)
                              : launch_exact<64, 0, 64, 1, 2, false>((unsigned)blocks, a, st);
}

// ---------------------------------------------------------------------------------------------
// The latents of a step's rows out of the cache pages [pages, 1, 16, C + R], 64 consecutive keys of one row a block: c [S, C]
// and the shared turned part [S, R], what the products that make keys and values read. blocks: per block the row, its first
// key's position and how many keys the row holds from there on (the rest of the 64 is zeros).
__global__ __launch_bounds__(256) void latent_gather_kernel(const bf16* __restrict__ pages, const int* __restrict__ block_table,
                                                            int table_width, const int* __restrict__ block_row,
                                                            const int* __restrict__ block_pos, const int* __restrict__ block_keys,
                                                            bf16* __restrict__ c, bf16* __restrict__ turned, int C, int R) {
  const int row = block_row[blockIdx.x], j0 = block_pos[blockIdx.x], keys = block_keys[blockIdx.x];
  const int* table = block_table + (size_t)row * table_width;
  const int runs = (C + R) / 8, c_runs = C / 8;
  for (int i = threadIdx.x; i < TK * runs; i += 256) {
    const int k = i / runs, run = i % runs, j = j0 + k;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (k < keys) {
      const int page = table[j / PAGE];
      if (page >= 0) v = *reinterpret_cast<const uint4*>(pages + ((size_t)page * PAGE + j % PAGE) * (C + R) + run * 8);
    }
    const size_t s = (size_t)blockIdx.x * TK + k;
    if (run < c_runs) *reinterpret_cast<uint4*>(c + s * C + run * 8) = v;
    else *reinterpret_cast<uint4*>(turned + s * R + (run - c_runs) * 8) = v;
  }
}

extern "C" int ms_latent_gather(const void* pages, const int* block_table, int table_width, const int* block_row, const int* block_pos,
                                const int* block_keys, int blocks, void* c, void* turned, int C, int R, hipStream_t st) {
  if (blocks <= 0) return MS_OK;
  if (table_width <= 0 || C <= 0 || R <= 0 || C % 8 || R % 8 || (size_t)pages % 16 || (size_t)c % 16 || (size_t)turned % 16) return MS_BAD_ARG;
  latent_gather_kernel<<<blocks, 256, 0, st>>>((const bf16*)pages, block_table, table_width, block_row, block_pos, block_keys, (bf16*)c,
                                               (bf16*)turned, C, R);
  return launch_status();
}

// 1 where the expanded form takes a latent attention's sizes.
extern "C" int ms_attention_expanded_ok(int Dn, int R, int Dv, int C, int page_size) {
  return page_size == PAGE && Dn == 128 && R == 64 && Dv == 128 && C % 8 == 0;
}

// Rows that bring several tokens over multiplied-out keys [keys, H Dn] (+ [keys, R] shared) and values [H Dv, keys]; tiles of
// rows_per_tile tokens. q: plain parts [T, H Dn]; q_turned: a token's turned parts, head h's R elements from h * qt_head on.
extern "C" int ms_attention_expanded(const void* q, const void* q_turned, int qt_stride, int qt_head, const void* k, const void* k_turned,
                                     const void* v, const int* key_base, int keys, const int* tile_first, const int* tile_count, int tiles,
                                     int rows_per_tile, const int* token_row, const int* pos, void* out, int H, int Dn, int R, int Dv,
                                     float scale, int window, const float* sinks, const float* gate, int gate_ld, int gate_col,
                                     int gate_each, hipStream_t st) {
  if (tiles <= 0) return MS_OK;
  if (H <= 0 || window < 0 || keys <= 0 || keys % TK || qt_stride % 8 || qt_head % 8 || qt_stride < H * qt_head || qt_head < R ||
      (size_t)q % 16 || (size_t)q_turned % 16 || (size_t)k % 16 || (size_t)k_turned % 16 || (size_t)v % 16 || (size_t)out % 16 ||
      (rows_per_tile != 64 && rows_per_tile != 128) || (gate && (gate_col < 0 || gate_ld < gate_col + (gate_each ? H * Dv : H))))
    return MS_BAD_ARG;
  if (!ms_attention_expanded_ok(Dn, R, Dv, 8, PAGE) || (long long)H * Dn * TK > 2147483647LL) return MS_UNSUPPORTED;
  const long long blocks = (long long)tiles * H;
  if (blocks > 2147483647LL) return MS_BAD_ARG;
  ExactArgs a{};
  a.q = (const bf16*)q; a.q_stride = H * Dn; a.q_head = Dn;
  a.q_turned = (const bf16*)q_turned; a.qt_stride = qt_stride; a.qt_head = qt_head;
  a.k = (const bf16*)k; a.k_turned = (const bf16*)k_turned; a.v = (const bf16*)v;
  a.key_base = key_base; a.keys = keys;
  a.tile_first = tile_first; a.tile_count = tile_count; a.token_row = token_row; a.pos = pos;
  a.out = (bf16*)out;
  a.Hq = H; a.Hkv = H; a.value_share = 1; a.value_runs = 1;
  a.scale = scale; a.window = window; a.sinks = sinks;
  a.gate = gate; a.gate_ld = gate_ld; a.gate_col = gate_col; a.gate_each = gate_each;
  return rows_per_tile == 128 ? launch_exact<128, 64, 128, 2, 1, true>((unsigned)blocks, a, st)
                              : launch_exact<128, 64, 128, 1, 1, true>((unsigned)blocks, a, st);
}
