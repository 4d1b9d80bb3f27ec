// Causal grouped-query attention in float32 over the paged cache (16-token pages, heads of 64 or 128 elements, all keys
// visible): the sums of the generic kernel with one order (attention.hip, four parts over the tiles of 64 keys) bit for bit,
// with keys and values brought into LDS by whole lines. There a lane reads its own key row from memory, 16 bytes at a time at a
// stride of 512, and a load instruction takes its 64 lines one after the other; that, and not the arithmetic, bounds it.
//
// Microseconds, 16 heads over 8 of 128 elements, keys from memory, the generic kernel and this one: six tokens at 23 to 333 keys 17.1,
// 11.1; one at 4,000 121, 66; 64 at 700 114, 68; prompts of 23 to 333 tokens (1,068 in all) 213, 47; one of 2,000 2,669, 354. Not where
// many single tokens see few keys (256 at 30: 23, 37), nor where a prompt has few query rows (40 tokens behind 3,000: 215, 249): the
// caller keeps the generic kernel there.
//
// What fixes a result, here and there: a score is one chain of fused multiply-adds over the elements in ascending order; tile t
// belongs to part t % 4; a part keeps a running maximum and sum over its tiles in ascending order and adds its values key by
// key; the parts meet in order. Which wave or block does it, and which other rows share the keys, changes nothing.
//
// Two forms:
//  * tokens: rows that bring one token. A block owns a token and a key head, its four waves a part each, for all heads of the
//    group: the chain of loads is what counts. A wave has 32 KB of LDS to itself, two regions of half a tile, and keeps one of
//    them under way while it works on the other (keys' first half, second half, values' first half, second half), so there is
//    no barrier before the parts meet.
//  * rows: rows that bring several tokens. A block owns 32 query rows (tokens x the heads of the group) of one key head, a wave
//    eight of them, and walks the tiles once. Two blocks a CU cover each other's loads.
//
// Values of pages that a row does not reach are left out (zero times an infinity is no zero), as in the generic kernel.
#include "common.h"

#include <utility>

#define TK 64
#define PAGE 16
#define PARTS 4
#define REGION 16384  // bytes: 64 keys of 64 elements, or 64 elements of 64 keys

#define LOAD_LDS(src, dst) \
  __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(src), (void __attribute__((address_space(3)))*)(dst), 16, 0, 0)

// At most N of this wave's loads under way, its LDS reads returned.
template <int N> __device__ __forceinline__ void landed() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory"); }
template <int N> __device__ __forceinline__ void landed_for_block() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// Memory that no kernel writes while this one runs, read at an address that all lanes share: through the scalar cache, whatever
// the compiler can show. (As vector loads, page ids would wait for every load of keys sent out before them.)
typedef const __attribute__((address_space(4))) int* scalar_ints;

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

struct Pages { int id[4]; };  // of a tile; entries behind the last visible key's page repeat that page
__device__ __forceinline__ Pages pages_of(scalar_ints table, int tile, int last) {
  Pages p;
#pragma unroll
  for (int u = 0; u < 4; ++u) p.id[u] = table[min(tile * 4 + u, last / PAGE)];
  return p;
}

// Load instruction i of 16 of a region: four key rows of 256 bytes, chunk c of key R in place c ^ (R & 15), so that the lanes that
// read one chunk column of 16 keys touch every bank once.
template <int D> __device__ __forceinline__ void load_keys(unsigned char* region, const float* __restrict__ kc, int page, int Hkv, int kvh, int half, int i, int lane) {
  const int R = i * 4 + lane / 16, c = (lane % 16) ^ (R & 15);
  LOAD_LDS(kc + (((size_t)page * Hkv + kvh) * PAGE + (R & 15)) * D + half * 64 + c * 4, region + i * 1024);
}
// The same for values: 16 elements of a page, 64 bytes each, chunk c of element e in place c ^ ((e >> 2) & 3).
template <int D> __device__ __forceinline__ void load_values(unsigned char* region, const float* __restrict__ vc, int page, int Hkv, int kvh, int half, int i, int lane) {
  const int e = (i % 4) * 16 + lane / 4, c = (lane % 4) ^ ((e >> 2) & 3);
  LOAD_LDS(vc + (((size_t)page * Hkv + kvh) * D + half * 64 + e) * PAGE + c * 4, region + i * 1024);
}

// Rows come in fours, the height of v_mfma_f32_4x4x1: sixteen products of 4 rows x 1 by 1 x 4 keys, one fused multiply-add to a result,
// so a lane's four results are its own key's (or value element's) with four rows, and the sums are those of fmaf. Its left operand is
// taken from four lanes (4 j .. 4 j + 3: rows 0 .. 3) for all sixteen: a register holds sixteen elements of four queries, or sixteen
// weights of four rows, and neither is read again.
#define ROWS_MFMA(a, b, c, j) __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 4, j, 0)

template <typename F, int... J> __device__ __forceinline__ void for_sixteen(F f, std::integer_sequence<int, J...>) {
  (f(std::integral_constant<int, J>{}), ...);
}

// dot[c] goes on over the 64 elements of a region; q[c][s]: elements 16 s .. + 15 of chain c's four rows.
template <int C> __device__ __forceinline__ void scores(floatx4 (&dot)[C], const float (&q)[C][4], const unsigned char* region, int lane) {
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    floatx4 k[4];
    float a[C];
#pragma unroll
    for (int u = 0; u < 4; ++u) k[u] = *reinterpret_cast<const floatx4*>(region + lane * 256 + (((s * 4 + u) ^ (lane & 15)) * 16));
#pragma unroll
    for (int c = 0; c < C; ++c) a[c] = q[c][s];
    auto one = [&](auto j) __attribute__((always_inline)) {
#pragma unroll
      for (int c = 0; c < C; ++c) dot[c] = ROWS_MFMA(a[c], k[decltype(j)::value / 4][decltype(j)::value % 4], dot[c], decltype(j)::value);
    };
    for_sixteen(one, std::make_integer_sequence<int, 16>{});
  }
}

// wave_max and wave_sum of common.h, the same pairs in the same order, by register moves: lanes l ^ 32, ^ 16, ^ 8, ^ 4, ^ 2, ^ 1.
template <int CTRL> __device__ __forceinline__ float moved(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <typename F> __device__ __forceinline__ float across_wave(float v, F f) {
  auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(a[0]), __uint_as_float(a[1]));
  auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(b[0]), __uint_as_float(b[1]));
  v = f(v, moved<0x128>(v));               // row_ror 8
  v = f(v, moved<0x1B>(moved<0x141>(v)));  // half rows mirrored, then quads
  v = f(v, moved<0x4E>(v));                // quads' pairs swapped
  return f(v, moved<0xB1>(v));             // pairs swapped
}

#define PS 80  // floats from a row's weights to the next row's: reads of four rows x sixteen keys touch every bank once

// One row's step of the softmax: the tile's weights to ps, its maximum and sum, and what the values so far are multiplied by.
// last: the row's last key, counted from the tile's first; negative: the row does not see the tile, and nothing changes.
__device__ __forceinline__ float soften(float dot, float scale, int last, float& m, float& l, float* ps, int lane) {
  const bool seen = lane <= last;
  const float s = seen ? dot * scale : -INFINITY;
  const float m_new = fmaxf(m, across_wave(s, [](float x, float y) { return fmaxf(x, y); }));
  const float p = seen ? expf(s - m_new) : 0.f;
  const float corr = last < 0 ? 1.f : expf(m - m_new);
  l = l * corr + across_wave(p, [](float x, float y) { return x + y; });
  m = m_new;
  ps[lane] = p;
  return corr;
}

// o[h][c] (four rows of this lane's element of half h) goes on over the pages that chain c's rows reach; last[c][i]: row i's last key
// counted from the tile's first. The halves' regions lie one behind the other.
// One page of them; w[c]: four rows' weights in four lanes each.
template <int H, int C>
__device__ __forceinline__ void add_page(floatx4 (&o)[H][C], const float (&w)[C], const floatx4 (&v)[H][4]) {
  auto one = [&](auto j) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int c = 0; c < C; ++c) o[h][c] = ROWS_MFMA(w[c], v[h][decltype(j)::value / 4][decltype(j)::value % 4], o[h][c], decltype(j)::value);
  };
  for_sixteen(one, std::make_integer_sequence<int, 16>{});
}
template <int H> __device__ __forceinline__ void read_page(floatx4 (&v)[H][4], const unsigned char* regions, int u, int lane) {
#pragma unroll
  for (int h = 0; h < H; ++h)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      v[h][i] = *reinterpret_cast<const floatx4*>(regions + h * REGION + u * 4096 + lane * 64 + ((i ^ ((lane >> 2) & 3)) * 16));
}
// One half, rows that all end at key `end`.
__device__ __forceinline__ void add_values(floatx4 (&o)[1][1], int end, const float* ps, const unsigned char* region, int lane) {
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    if (u * PAGE > end) break;
    floatx4 v[1][4];
    read_page(v, region, u, lane);
    const float w[1] = {ps[(lane % 4) * PS + u * PAGE + lane / 4]};
    add_page(o, w, v);
  }
}
// (The pages in a loop of their own: unrolled, with what follows where rows part ways, the code of a tile is so long that fetching
// it shows.)
template <int H, int C>
__device__ __forceinline__ void add_values(floatx4 (&o)[H][C], const int (&last)[C][4], const float* ps, const unsigned char* regions, int lane) {
  int most = -1, least = TK;
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int i = 0; i < 4; ++i) most = max(most, last[c][i]), least = min(least, last[c][i]);
  const int pages = min(most, TK - 1) / PAGE + (most >= 0);
#pragma unroll 1
  for (int u = 0; u < pages; ++u) {
    floatx4 v[H][4];
    read_page(v, regions, u, lane);
    if (least >= u * PAGE) {
      float w[C];
#pragma unroll
      for (int c = 0; c < C; ++c) w[c] = ps[(c * 4 + lane % 4) * PS + u * PAGE + lane / 4];
      add_page(o, w, v);
    } else {  // the rows part ways at this page
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (last[c][i] < u * PAGE) continue;
          float x[H];
#pragma unroll
          for (int h = 0; h < H; ++h) x[h] = o[h][c][i];
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const floatx4 w = *reinterpret_cast<const floatx4*>(ps + (c * 4 + i) * PS + u * PAGE + k * 4);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
              for (int h = 0; h < H; ++h) x[h] = fmaf(w[e], v[h][k][e], x[h]);
          }
#pragma unroll
          for (int h = 0; h < H; ++h) o[h][c][i] = x[h];
        }
    }
  }
}

// HEADS (up to four): heads of a group that a wave takes at once; a larger group takes more blocks.
template <int D, int HEADS>
__global__ __launch_bounds__(256, 1) void attention_f32_tokens_kernel(const float* __restrict__ q, int q_stride, const float* __restrict__ kc,
                                                                      const float* __restrict__ vc, const int* __restrict__ block_table,
                                                                      int table_width, const int* __restrict__ token_list,
                                                                      const int* __restrict__ token_row, const int* __restrict__ pos,
                                                                      float* __restrict__ out, int Hq, int Hkv, float scale) {
  constexpr int HALVES = D / 64, LOADS = 16;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];  // per wave two regions, and then:
  float* ps_all = reinterpret_cast<float*>(lds + PARTS * 2 * REGION);     // [PARTS][4][PS]
  float* os = ps_all + PARTS * 4 * PS;                                    // [PARTS][HEADS][D]
  float* ml = os + PARTS * HEADS * D;                                     // [PARTS][HEADS][2]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
  const int t = token_list ? token_list[blockIdx.x] : blockIdx.x, kvh = blockIdx.y, group = Hq / Hkv;
  const int first_head = blockIdx.z * HEADS, heads = min(HEADS, group - first_head);
  const int p = pos[t], tiles = p / TK + 1, parts = min(tiles, PARTS);
  const scalar_ints table = (scalar_ints)(block_table + (size_t)token_row[t] * table_width);
  unsigned char *a = lds + wave * 2 * REGION, *b = a + REGION;
  float* ps = ps_all + wave * 4 * PS;

  Pages pages = pages_of(table, min(wave, tiles - 1), p);
  if (wave < tiles) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) load_keys<D>(a, kc, pages.id[i / 4], Hkv, kvh, 0, i, lane);
    if (HALVES == 2) {
#pragma unroll
      for (int i = 0; i < LOADS; ++i) load_keys<D>(b, kc, pages.id[i / 4], Hkv, kvh, 1, i, lane);
    }
  }
  float qa[HALVES][1][4];
  {
    const float* qh = q + (size_t)t * q_stride + (size_t)(kvh * group + first_head + min(lane % 4, heads - 1)) * D + lane / 4;
#pragma unroll
    for (int s = 0; s < 4 * HALVES; ++s) qa[s / 4][0][s % 4] = qh[s * 16];
  }
  float m[HEADS], l[HEADS];
  floatx4 o[HALVES][1][1];
#pragma unroll
  for (int h = 0; h < HEADS; ++h) {
    m[h] = -INFINITY;
    l[h] = 0.f;
  }
#pragma unroll
  for (int half = 0; half < HALVES; ++half) o[half][0][0] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int h = HEADS; h < 4; ++h) ps[h * PS + lane] = 0.f;  // rows that stand for no head
  for (int tile = wave; tile < tiles; tile += PARTS) {
    const int next = tile + PARTS;
    const Pages after = pages_of(table, min(next, tiles - 1), p);
    floatx4 dot[1] = {floatx4{0.f, 0.f, 0.f, 0.f}};
    // A region is loaded anew when all that was in it has come out (landed<> waits for that too).
    if (HALVES == 2) {
      landed<LOADS>();
      scores(dot, qa[0], a, lane);
      landed<LOADS>();
#pragma unroll
      for (int i = 0; i < LOADS; ++i) load_values<D>(a, vc, pages.id[i / 4], Hkv, kvh, 0, i, lane);
      landed<LOADS>();
      scores(dot, qa[HALVES - 1], b, lane);
      landed<LOADS>();
#pragma unroll
      for (int i = 0; i < LOADS; ++i) load_values<D>(b, vc, pages.id[i / 4], Hkv, kvh, 1, i, lane);
    } else {
#pragma unroll
      for (int i = 0; i < LOADS; ++i) load_values<D>(b, vc, pages.id[i / 4], Hkv, kvh, 0, i, lane);
      landed<LOADS>();
      scores(dot, qa[0], a, lane);
      landed<LOADS>();
      if (next < tiles) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) load_keys<D>(a, kc, after.id[i / 4], Hkv, kvh, 0, i, lane);
      }
    }
    const int end = p - tile * TK;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int h = 0; h < HEADS; ++h) {
      const float corr = soften(dot[0][h], scale, end, m[h], l[h], ps + h * PS, lane);
#pragma unroll
      for (int half = 0; half < HALVES; ++half) o[half][0][0][h] *= corr;
    }
    __builtin_amdgcn_wave_barrier();
    if (HALVES == 2) {
      landed<LOADS>();
      add_values(o[0], end, ps, a, lane);
      if (next < tiles) {
        landed<LOADS>();
#pragma unroll
        for (int i = 0; i < LOADS; ++i) load_keys<D>(a, kc, after.id[i / 4], Hkv, kvh, 0, i, lane);
        landed<LOADS>();
      } else {
        landed<0>();
      }
      add_values(o[HALVES - 1], end, ps, b, lane);
      if (next < tiles) {
        landed<LOADS>();
#pragma unroll
        for (int i = 0; i < LOADS; ++i) load_keys<D>(b, kc, after.id[i / 4], Hkv, kvh, 1, i, lane);
      }
    } else {
      if (next < tiles) landed<LOADS>();
      else landed<0>();
      add_values(o[0], end, ps, b, lane);
      landed<LOADS>();
    }
    pages = after;
  }
  if (parts > 1 && wave < parts) {
#pragma unroll
    for (int h = 0; h < HEADS; ++h) {
      if (lane == 0) {
        ml[(wave * HEADS + h) * 2] = m[h];
        ml[(wave * HEADS + h) * 2 + 1] = l[h];
      }
#pragma unroll
      for (int half = 0; half < HALVES; ++half) os[(wave * HEADS + h) * D + half * 64 + lane] = o[half][0][0][h];
    }
  }
  __syncthreads();
#pragma unroll
  for (int h = 0; h < HEADS; ++h) {
    if (h >= heads || (parts > 1 ? h : 0) != wave) continue;  // one part: the first wave has it
    float ll = l[h], oo[HALVES];
#pragma unroll
    for (int half = 0; half < HALVES; ++half) oo[half] = o[half][0][0][h];
    if (parts > 1) {
      float mm = ml[h * 2];
      for (int w = 1; w < parts; ++w) mm = fmaxf(mm, ml[(w * HEADS + h) * 2]);
      ll = 0.f;
#pragma unroll
      for (int half = 0; half < HALVES; ++half) oo[half] = 0.f;
      for (int w = 0; w < parts; ++w) {
        const float c = expf(ml[(w * HEADS + h) * 2] - mm);
        ll = fmaf(ml[(w * HEADS + h) * 2 + 1], c, ll);
#pragma unroll
        for (int half = 0; half < HALVES; ++half) oo[half] = fmaf(os[(w * HEADS + h) * D + half * 64 + lane], c, oo[half]);
      }
    }
    const float inv = 1.f / ll;
    float* ov = out + ((size_t)t * Hq + kvh * group + first_head + h) * D;
#pragma unroll
    for (int half = 0; half < HALVES; ++half) ov[half * 64 + lane] = oo[half] * inv;
  }
}

#define CHAINS 2          // fours of query rows of a wave
#define WROWS (4 * CHAINS)
#define ROWS (4 * WROWS)  // of a block

template <int D>
__global__ __launch_bounds__(256, 2) void attention_f32_rows_kernel(const float* __restrict__ q, int q_stride, const float* __restrict__ kc,
                                                                    const float* __restrict__ vc, const int* __restrict__ block_table,
                                                                    int table_width, const int* __restrict__ tile_first,
                                                                    const int* __restrict__ tile_count, const int* __restrict__ token_row,
                                                                    const int* __restrict__ pos, float* __restrict__ out, int Hq, int Hkv,
                                                                    float scale) {
  constexpr int HALVES = D / 64, LOADS = 4 * HALVES;  // a wave's share of a tile's keys, and of its values
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];  // HALVES regions of keys, as many of values, then weights
  unsigned char* values = lds + HALVES * REGION;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
  float* ps = reinterpret_cast<float*>(lds + 2 * HALVES * REGION) + wave * WROWS * PS;
  const int kvh = blockIdx.y, group = Hq / Hkv;
  const int first = tile_first[blockIdx.x], count = tile_count[blockIdx.x], rows = count * group;
  const int p_first = pos[first], p_last = p_first + count - 1;
  const scalar_ints table = (scalar_ints)(block_table + (size_t)token_row[first] * table_width);
  const int tiles = p_last / TK + 1;
  // The rows' positions; -1: a wave without rows. Rows that are not there go along with the last one (its queries, its keys) and are
  // never stored: as rows that see nothing they would part ways with the others at every page. 12 heads over 4 of 128, 64 tokens
  // behind 3,000 that way 368 us, this way 251; 16 rows of 5 behind 700 101, 68.
  int p[CHAINS][4], p_wave = -1;
#pragma unroll
  for (int r = 0; r < WROWS; ++r) {
    p[r / 4][r % 4] = wave * WROWS < rows ? p_first + min(wave * WROWS + r, rows - 1) / group : -1;
    p_wave = max(p_wave, p[r / 4][r % 4]);
  }
  auto get_keys = [&](int page) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < LOADS; ++j) load_keys<D>(lds + (j / 4) * REGION, kc, page, Hkv, kvh, j / 4, wave * 4 + j % 4, lane);
  };
  auto get_values = [&](int page) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < LOADS; ++j) load_values<D>(values + (j / 4) * REGION, vc, page, Hkv, kvh, j / 4, wave * 4 + j % 4, lane);
  };
  auto page_of = [&](int tile) __attribute__((always_inline)) { return table[min(tile * 4 + wave, p_last / PAGE)]; };  // a wave loads a page of each tile
  int page = page_of(0);
  get_keys(page);
  float qa[HALVES][CHAINS][4];
#pragma unroll
  for (int c = 0; c < CHAINS; ++c) {
    const int row = min(wave * WROWS + c * 4 + lane % 4, rows - 1);
    const float* qh = q + (size_t)(first + row / group) * q_stride + (size_t)(kvh * group + row % group) * D + lane / 4;
#pragma unroll
    for (int s = 0; s < 4 * HALVES; ++s) qa[s / 4][c][s % 4] = qh[s * 16];
  }
  float m[WROWS], l[WROWS];            // of the part at work
  float m_part[WROWS], l_part[WROWS];  // lane w: of part w
  floatx4 o[HALVES][CHAINS], o_part[PARTS][HALVES][CHAINS];
#pragma unroll
  for (int r = 0; r < WROWS; ++r) {
    m_part[r] = -INFINITY;
    l_part[r] = 0.f;
  }
#pragma unroll
  for (int w = 0; w < PARTS; ++w)
#pragma unroll
    for (int half = 0; half < HALVES; ++half)
#pragma unroll
      for (int c = 0; c < CHAINS; ++c) o_part[w][half][c] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto of_part = [](float v, int w) __attribute__((always_inline)) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), w)); };
  for (int tile = 0; tile < tiles; ++tile) {
    const int after = page_of(min(tile + 1, tiles - 1));
    landed_for_block<0>();  // the keys are there, and nobody reads the values of the tile before
    get_values(page);
    const int part = tile % PARTS;
    const bool work = tile * TK <= p_wave;  // the same for the whole wave
    int last[CHAINS][4];
#pragma unroll
    for (int r = 0; r < WROWS; ++r) last[r / 4][r % 4] = p[r / 4][r % 4] - tile * TK;
    if (work) {
#pragma unroll
      for (int r = 0; r < WROWS; ++r) {
        m[r] = of_part(m_part[r], part);
        l[r] = of_part(l_part[r], part);
      }
#pragma unroll
      for (int w = 0; w < PARTS; ++w)
        if (part == w) {
#pragma unroll
          for (int half = 0; half < HALVES; ++half)
#pragma unroll
            for (int c = 0; c < CHAINS; ++c) o[half][c] = o_part[w][half][c];
        }
      floatx4 dot[CHAINS];
#pragma unroll
      for (int c = 0; c < CHAINS; ++c) dot[c] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int half = 0; half < HALVES; ++half) scores(dot, qa[half], lds + half * REGION, lane);
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int r = 0; r < WROWS; ++r) {
        const float corr = soften(dot[r / 4][r % 4], scale, last[r / 4][r % 4], m[r], l[r], ps + r * PS, lane);
#pragma unroll
        for (int half = 0; half < HALVES; ++half) o[half][r / 4][r % 4] *= corr;
      }
      __builtin_amdgcn_wave_barrier();
    }
    landed_for_block<0>();  // the values are there, and nobody reads this tile's keys any more
    if (tile + 1 < tiles) get_keys(after);
    if (work) {
      add_values(o, last, ps, values, lane);
#pragma unroll
      for (int w = 0; w < PARTS; ++w)
        if (part == w) {
#pragma unroll
          for (int half = 0; half < HALVES; ++half)
#pragma unroll
            for (int c = 0; c < CHAINS; ++c) o_part[w][half][c] = o[half][c];
        }
#pragma unroll
      for (int r = 0; r < WROWS; ++r) {
        m_part[r] = lane == part ? m[r] : m_part[r];
        l_part[r] = lane == part ? l[r] : l_part[r];
      }
    }
    page = after;
  }
#pragma unroll
  for (int r = 0; r < WROWS; ++r) {
    const int c = r / 4, i = r % 4, row = wave * WROWS + r;
    if (row >= rows) continue;
    const int parts = min(p[c][i] / TK + 1, PARTS);
    float ll = of_part(l_part[r], 0), oo[HALVES];
#pragma unroll
    for (int half = 0; half < HALVES; ++half) oo[half] = o_part[0][half][c][i];
    if (parts > 1) {
      float mm = of_part(m_part[r], 0);
#pragma unroll
      for (int w = 1; w < PARTS; ++w)
        if (w < parts) mm = fmaxf(mm, of_part(m_part[r], w));
      ll = 0.f;
#pragma unroll
      for (int half = 0; half < HALVES; ++half) oo[half] = 0.f;
#pragma unroll
      for (int w = 0; w < PARTS; ++w) {
        if (w >= parts) continue;
        const float e = expf(of_part(m_part[r], w) - mm);
        ll = fmaf(of_part(l_part[r], w), e, ll);
#pragma unroll
        for (int half = 0; half < HALVES; ++half) oo[half] = fmaf(o_part[w][half][c][i], e, oo[half]);
      }
    }
    const float inv = 1.f / ll;
    float* ov = out + ((size_t)(first + row / group) * Hq + kvh * group + row % group) * D;
#pragma unroll
    for (int half = 0; half < HALVES; ++half) ov[half * 64 + lane] = oo[half] * inv;
  }
}

// Query rows of a block of the form for rows of several tokens (0: neither form takes the shape).
extern "C" int ms_attention_f32_rows(int group, int D, int page_size) {
  return page_size == PAGE && (D == 64 || D == 128) && group >= 1 && group <= 16 ? ROWS : 0;
}

static int ask_lds(const void* kernel, int bytes) {
  return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess ? MS_OK : MS_LAUNCH_FAILED;
}

template <int D, int HEADS>
static int launch_tokens(const float* q, int q_stride, const float* kc, const float* vc, const int* block_table, int table_width,
                         const int* token_list, const int* token_row, const int* pos, float* out, int tokens, int Hq, int Hkv, float scale,
                         hipStream_t st) {
  constexpr int bytes = PARTS * 2 * REGION + PARTS * (4 * PS + HEADS * (D + 2)) * 4;
  static_assert(bytes <= 160 * 1024, "LDS of a CU");
  static const int ready = ask_lds((const void*)attention_f32_tokens_kernel<D, HEADS>, bytes);
  if (ready != MS_OK) return ready;
  const dim3 grid(tokens, Hkv, (Hq / Hkv + HEADS - 1) / HEADS);
  attention_f32_tokens_kernel<D, HEADS><<<grid, 256, bytes, st>>>(q, q_stride, kc, vc, block_table, table_width, token_list, token_row, pos, out, Hq, Hkv, scale);
  return launch_status();
}

// Tokens of rows that bring one (token_list: their flat indices, or null for tokens 0, 1, ...). Keys and values 16-byte aligned.
extern "C" int ms_attention_f32_tokens(const void* q, int q_stride, const void* kc, const void* vc, const int* block_table, int table_width,
                                       const int* token_list, const int* token_row, const int* pos, void* out, int tokens, int Hq, int Hkv,
                                       int D, int page_size, float scale, hipStream_t st) {
  if (tokens <= 0) return MS_OK;
  if (Hq <= 0 || Hkv <= 0 || Hq % Hkv || Hkv > 65535 || table_width <= 0 || q_stride < Hq * D || ((size_t)kc | (size_t)vc) % 16) return MS_BAD_ARG;
  const int group = Hq / Hkv;
  if (!ms_attention_f32_rows(group, D, page_size)) return MS_UNSUPPORTED;
#define GO(DIM, HEADS) \
  return launch_tokens<DIM, HEADS>((const float*)q, q_stride, (const float*)kc, (const float*)vc, block_table, table_width, token_list, token_row, pos, (float*)out, tokens, Hq, Hkv, scale, st)
  if (D == 128) {
    if (group == 1) GO(128, 1);
    if (group == 2) GO(128, 2);
    GO(128, 4);
  }
  if (group == 1) GO(64, 1);
  if (group == 2) GO(64, 2);
  GO(64, 4);
#undef GO
}

// Rows that bring several tokens: `tiles` runs of at most ROWS / group consecutive new tokens of one sequence.
extern "C" int ms_attention_f32(const void* q, int q_stride, const void* kc, const void* vc, const int* block_table, int table_width,
                                const int* tile_first, const int* tile_count, int tiles, const int* token_row, const int* pos, void* out,
                                int Hq, int Hkv, int D, int page_size, float scale, hipStream_t st) {
  if (tiles <= 0) return MS_OK;
  if (Hq <= 0 || Hkv <= 0 || Hq % Hkv || Hkv > 65535 || table_width <= 0 || q_stride < Hq * D || ((size_t)kc | (size_t)vc) % 16 ||
      tile_first == nullptr || tile_count == nullptr)
    return MS_BAD_ARG;
  if (!ms_attention_f32_rows(Hq / Hkv, D, page_size)) return MS_UNSUPPORTED;
  const dim3 grid(tiles, Hkv);
#define GO(DIM)                                                                                                                          \
  do {                                                                                                                                   \
    constexpr int bytes = 2 * (DIM / 64) * REGION + ROWS * PS * 4;                                                                       \
    static const int ready = ask_lds((const void*)attention_f32_rows_kernel<DIM>, bytes);                                                \
    if (ready != MS_OK) return ready;                                                                                                    \
    attention_f32_rows_kernel<DIM><<<grid, 256, bytes, st>>>((const float*)q, q_stride, (const float*)kc, (const float*)vc, block_table, \
                                                             table_width, tile_first, tile_count, token_row, pos, (float*)out, Hq, Hkv, scale); \
  } while (0)
  if (D == 128) GO(128);
  else GO(64);
#undef GO
  return launch_status();
}
