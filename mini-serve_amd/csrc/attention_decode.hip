// Decode attention for bfloat16: one query token per sequence over the paged cache, split over the
// keys so that a small batch still fills the chip, then a fixed-order reduction of the splits.
//
// Cache layouts (one KV head of one page is contiguous):
//   keys   K [pages, Hkv, page_size = 16, D]     a token's head is a row of D
//   values V [pages, Hkv, D, page_size = 16]     transposed within the page: the 16 tokens of one
//                                                head element are contiguous
// Both feed v_mfma_f32_16x16x32_bf16, the values straight from global memory with one vector load per lane, the keys through LDS or
// straight too:
//   scores  S^T[token, query] : A operand = K rows (i = token), B operand = Q (j = query head of the group)
//   output  O^T[d, query]     : A operand = V^T (i = d, k = token), B operand = P (j = query, k = token)
// The two score products of a 32-token chunk take their key rows in an order chosen so that a lane
// of the results holds 8 consecutive tokens of one page for one query (lane group g: page g / 2 of
// the chunk, tokens 8 (g % 2) .. + 7; four from each product). The MFMA's k index of the second
// product is mapped to tokens in the same way, so exactly these 8 values are the lane's P operand
// (probabilities never move between lanes) and its V^T operand is one 16-byte load.
//
// Grid: (Hkv, rows, splits). A block of 4 waves takes a contiguous range of 32-token chunks; its
// waves take a quarter of them each and are merged in LDS. splits == 1 writes the result directly.
#include "common.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

#define PAGE 16
#define CHUNK 32  // tokens per step of a wave: two pages

// One 32-token chunk as a wave holds it: the matrix operands themselves, 16 bytes a lane. Values are asked for as whole lines. Keys
// take one of two ways to their operands, with the same results:
//  * through LDS: a chunk's keys go there by whole lines, two chunks in a ring that belongs to the wave. Loaded as operands, a lane's
//    16 bytes belong to one row of 256 and a load touches sixteen rows, every line twice: a block that has a CU to itself gets
//    through a chunk in 1.8 us where it needs 1.2, which counts wherever the longest rows' chains of chunks are what takes the time.
//  * straight into registers: rows of one length whose pages lie in order walk through memory in step and keep meeting in the
//    same memory channels; there loads of many short pieces are the faster ones. Also for keys that do not start at a
//    multiple of 16 bytes.
// A block decides by its own length and that of four other rows (in_step). Microseconds, 32 heads over 8 KV heads of 128, all in registers,
// all through LDS, and so chosen: 128 rows of 4,100 tokens 325, 356, 325; of 2,048 167, 170, 169; of 600 60, 56, 56; of 418 to
// 4,049 215, 198, 200; 64 of 303 to 1,800 58, 53, 53; 48 of 309 to 2,789 69, 62, 62; 40 of 200 and one of 14,000 102, 77, 79; 8 of
// 4,080 29.3, 29.2, 28.9; 1 of 14,000 21.3, 20.6, 21.3; 1 of 217 9.7, 9.6, 9.6.
template <int D>
struct DecodeValues {
  bf16x8 v[D / 16];
};
template <int D>
struct DecodeTile : DecodeValues<D> {
  bf16x8 ka[D / 32], kb[D / 32];
};
constexpr int STEP_CHUNKS = 48;  // chunks of a block (1,536 tokens) from which rows in step matter

// LDS of a block: the four waves' rings (their first half carries the wave's output to the merge at the end), the queries, the new key and
// value, the waves' maxima and sums.
template <int D>
struct DecodeLds {
  static constexpr int CHUNK_BYTES = CHUNK * D * 2, RING = 2 * CHUNK_BYTES;
  static constexpr int QUERIES = 4 * RING, KV_NEW = QUERIES + 16 * D * 2, MAXIMA = KV_NEW + 2 * D * 2, SUMS = MAXIMA + 4 * 16 * 4;
  static constexpr int BYTES = SUMS + 4 * 16 * 4;
  static_assert(16 * (D + 4) * 4 <= RING, "a wave's output fits in its ring");
};

// The fused form takes, instead of finished queries and a cache that already holds the new token, the
// qkv projection as it leaves the small-M product: float partial sums [splits, tokens, (Hq + 2 Hkv) D].
// Every wave sums, norms and rotates the queries of its KV head's group itself (up to 256 floats; the
// block's waves share the work if there are more);
// the one wave whose chunks end with the sequence's last token does the same for the new key, takes
// the new value, stores both into the cache and puts them into its operands of that chunk in
// registers (what its loads brought from the not yet written slot is replaced, so no store has to be
// waited for). This is the work of the QK-norm / rotation / store kernel, which a step of single
// tokens then does not launch.
struct FusedQkv {
  const float* parts;      // [splits, tokens, row_width]
  int splits;
  long long split_stride;  // floats between splits
  int row_width;           // (Hq + 2 Hkv) D
  const bf16* q_weight;    // [D] each, or both nullptr: no norm
  const bf16* k_weight;
  float eps;
  const float* rope;       // [tokens, D]: cosines, then sines, of D / 2 angles; nullptr: no rotation
  int store;               // 0: another layer owns the cache, the new token is already in it
};

// Four consecutive elements d0 .. d0 + 3 of a head whose D / 4 holders are neighbouring lanes (an
// aligned group): RMSNorm over the head with weight w (if any), then rotation by the angles of
// `rope_row` (if any), element d paired with d +- D / 2. Every lane of the wave must call this.
// The weights and angles come in a HeadTerms that was asked for earlier.
struct HeadTerms {
  bf16 w[4];
  float4 c, s;
};
template <int D>
__device__ __forceinline__ void head_terms(HeadTerms& t, int d0, const bf16* __restrict__ w, const float* __restrict__ rope_row) {
  if (w != nullptr) {
#pragma unroll
    for (int e = 0; e < 4; ++e) t.w[e] = w[d0 + e];
  }
  if (rope_row != nullptr) {
    const int j0 = d0 % (D / 2);
    t.c = *reinterpret_cast<const float4*>(rope_row + j0);
    t.s = *reinterpret_cast<const float4*>(rope_row + D / 2 + j0);
  }
}
template <int D>
__device__ __forceinline__ void head_norm_rotate(float (&x)[4], int d0, const HeadTerms& t, bool norm, float eps, bool rotate) {
  if (norm) {
    float ss = x[0] * x[0] + x[1] * x[1] + x[2] * x[2] + x[3] * x[3];
    ss = group_sum<D / 4>(ss);
    const float rstd = rsqrtf(ss / (float)D + eps);
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = x[e] * rstd * to_f32(t.w[e]);
  }
  if (rotate) {
    const float cs[4] = {t.c.x, t.c.y, t.c.z, t.c.w}, ss[4] = {t.s.x, t.s.y, t.s.z, t.s.w};
    const bool low = d0 < D / 2;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float partner = lane_xor_f32<D / 8>(x[e]);
      x[e] = low ? x[e] * cs[e] - partner * ss[e] : x[e] * cs[e] + partner * ss[e];
    }
  }
}

// Sum over the splits, in ascending order, of four floats at `at` of each split; the first four splits' loads go out in
// ask_parts4, ahead of whatever the caller asks for next.
struct Parts4 { float4 v[4]; };
__device__ __forceinline__ void ask_parts4(Parts4& a, const float* __restrict__ parts, int s0, int splits, long long stride, size_t at) {
#pragma unroll
  for (int u = 0; u < 4; ++u) a.v[u] = *reinterpret_cast<const float4*>(parts + (size_t)(s0 + u < splits ? s0 + u : 0) * stride + at);
}
__device__ __forceinline__ void sum_parts4(float (&x)[4], Parts4& a, const float* __restrict__ parts, int splits, long long stride, size_t at) {
  x[0] = x[1] = x[2] = x[3] = 0.f;
  auto add = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (s0 + u >= splits) a.v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
      x[0] += a.v[u].x; x[1] += a.v[u].y; x[2] += a.v[u].z; x[3] += a.v[u].w;
    }
  };
  add(0);  // (outside the loop: in it, the wait for these four would be one for all that was asked for since)
  for (int s0 = 4; s0 < splits; s0 += 4) {
    ask_parts4(a, parts, s0, splits, stride, at);
    add(s0);
  }
}

// 16 bytes a lane from `offset` (in bytes, each lane's own) of a page's head, BYTES long, into 1 KB of LDS. A buffer load and not a global one: behind a
// global load into LDS the compiler makes every wait for a register a wait for all loads.
template <int BYTES>
__device__ __forceinline__ void page_to_lds(const void* page, int offset, unsigned char* to) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)page, 0, BYTES, 0x00020000),
                                           (void __attribute__((address_space(3)))*)to, 16, offset, 0, 0, LOAD_ONCE);
}

// MAY_STEP: the instance that has both ways for its keys; without it, through LDS alone (a twentieth faster where a call takes 10 us).
template <int D, bool FUSED, bool MAY_STEP>
__global__ __launch_bounds__(256, 2) void attn_decode_split_kernel(
    const bf16* __restrict__ q, int q_stride, bf16* kc_rw, bf16* vc_rw,
    const int* __restrict__ block_table, int table_width, const int* __restrict__ tokens,
    const int* __restrict__ token_row, const int* __restrict__ pos, bf16* __restrict__ out,
    float* __restrict__ part_o, float* __restrict__ part_ml, int G, float scale, int window, unsigned per_split, FusedQkv fin) {
  constexpr int KK = D / 32;  // k-steps of the score product
  constexpr int DB = D / 16;  // 16-wide blocks of the head
  const bf16* kc = kc_rw;
  const bf16* vc = vc_rw;
  // No division by a number that the compiler does not know (some 40 instructions each, one behind the other): the grid is (KV heads,
  // rows, splits), and per_split is 2^32 / splits rounded up (0: divide).
  const int kvh = blockIdx.x, b = blockIdx.y, Hkv = gridDim.x, Hq = G * Hkv;
  const int split = blockIdx.z, splits = gridDim.z;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
  const int r = lane % 16, g = lane / 16;
  const int tok = tokens ? tokens[b] : b;
  // Fused form: the group's queries (G * D floats, four a lane and round) need nothing but the token's number. They are asked for
  // before the position, which the table's entries wait for and the keys and values behind those: loads come back in the order in
  // which they went out, and behind the keys and values they would cost a round trip of their own.
  // Up to 256 floats (a lane's four of one round): every wave works its own copy out, no barrier.
  // More: the block's waves share the work (a wave takes whole heads) and meet once.
  const int gd = G * D;
  const bool together = gd > 4 * WAVE;
  const size_t qkv_row = FUSED ? (size_t)tok * fin.row_width : 0;
  const float* rope_row = FUSED && fin.rope ? fin.rope + (size_t)tok * D : nullptr;
  Parts4 q_parts;
  HeadTerms q_terms;
  if (FUSED) {
    const int e0 = (together ? tid : lane) * 4, ec = e0 < gd ? e0 : 0;
    ask_parts4(q_parts, fin.parts, 0, fin.splits, fin.split_stride, qkv_row + (size_t)kvh * gd + ec);
    head_terms<D>(q_terms, ec % D, fin.q_weight, rope_row);
  }
  const int kv_len = pos[tok] + 1;
  // (MAY_STEP) Rows in step: this row and four others have as many tokens within a 32nd.
  bool in_step = MAY_STEP;
  if (MAY_STEP) {
    const int rows = gridDim.y, apart[4] = {1, rows / 4, rows / 2, rows - 1};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int other = b + apart[i] < rows ? b + apart[i] : b + apart[i] - rows;
      in_step = in_step && abs(pos[tokens ? tokens[other] : other] + 1 - kv_len) * 32 <= kv_len;
    }
  }
  const int lo = (window > 0 && kv_len > window) ? kv_len - window : 0;
  const int lo_al = lo & ~(CHUNK - 1);
  const int n_chunks = (kv_len - lo_al + CHUNK - 1) / CHUNK;
  const int round_up = n_chunks + splits - 1;
  const int per = per_split ? (int)__umulhi((unsigned)round_up, per_split) : round_up / splits;
  const bool through_lds = !MAY_STEP || (reinterpret_cast<size_t>(kc_rw) % 16 == 0 && !(in_step && per >= STEP_CHUNKS));
  const int c_begin = split * per;
  const int c_end = min(n_chunks, c_begin + per);
  const int* table = block_table + (size_t)token_row[tok] * table_width;

  // Query operand: column r is query head kvh * G + r of the group (zero beyond the group).
  bf16x8 qf[KK];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) {
    if (!FUSED && r < G) {
      qf[kk] = *reinterpret_cast<const bf16x8*>(q + (size_t)tok * q_stride + (size_t)(kvh * G + r) * D + kk * 32 + g * 8);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) qf[kk][i] = static_cast<bf16>(0.f);
    }
  }

  // Scores are kept in units of log2 (exp2 is one instruction); maxima, also those handed to the
  // reduction kernel, are in the same units.
  const float scale2 = scale * 1.44269504088896340736f;
  float m_run = -INFINITY, l_run = 0.f;  // of query r (replicated over the four lane groups)
  floatx4 o[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i) o[i] = floatx4{0.f, 0.f, 0.f, 0.f};

  // Two chunks are in flight per wave: while one is multiplied the next one's keys and values are already on their way. Loads come
  // back in the order in which they go out, and what keeps the second chunk in flight is that no wait asks for more than it
  // needs: the wait for keys in LDS is counted by hand, the others the compiler counts, which it can where loop and branches
  // leave it one order of loads only; and page ids are not loaded chunk by chunk, as the wait for them, the newest loads of
  // all, would be a wait for everything.
  // A wave takes a contiguous quarter of the block's chunks (not every fourth chunk): with a request's
  // pages next to each other in memory, waves that step through every fourth chunk in lockstep keep
  // hitting the same few memory channels (measured on the address pattern alone: 5.1 -> 5.8 TB/s).
  const int per_wave = (c_end - c_begin + 3) / 4;
  const int w_begin = c_begin + wave * per_wave, w_end = min(c_end, w_begin + per_wave);
  // Fused form: this wave's chunks end with the sequence's last one, which holds the new token.
  const bool has_new = FUSED && fin.store && w_begin < w_end && w_end == n_chunks;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];  // DecodeLds<D>::BYTES
  typedef DecodeLds<D> Lds;
  unsigned char* ring = smem + wave * Lds::RING;
  bf16* kv_new = reinterpret_cast<bf16*>(smem + Lds::KV_NEW);  // the new key, then the new value
  // A wave's page ids, 64 at a time, one a lane: entry i is page i of the chunks from id_first on. Whether a chunk has a second page at all
  // is settled when its entries are used.
  int ids = 0, id_first = w_begin;
  auto fetch_ids = [&](int c) __attribute__((always_inline)) {
    id_first = c;
    ids = table[min((lo_al + c * CHUNK) / PAGE + lane, table_width - 1)];
    asm volatile("" : "+v"(ids));  // waited for here
  };
  constexpr int KCH = D / 8, RPI = 64 / KCH, LOADS = CHUNK / RPI;  // pieces of a key row, rows a load fills, loads a chunk
  // Piece c of row R lies in slot c ^ key_slot(R): the 16 lanes that read a piece together have rows {0-3, 8-11, 16-19, 24-27} (+ 4), which
  // differ in bits 0, 1, 3 and 4 (a row of 128 bytes has eight slots, and bit 0 picks the half of the banks).
  auto key_slot = [](int R) { return KCH == 16 ? ((R & 3) | ((R >> 1) & 12)) : (((R >> 1) & 1) | ((R >> 2) & 6)); };
  // Key rows: lane r feeds row r of both products. Product a takes tokens 0-3 and 8-11 of each page,
  // product b tokens 4-7 and 12-15 (rows 0-7 from the chunk's first page, 8-15 from its second).
  const int key_row = (r < 8 ? 0 : PAGE) + (r % 4) + 8 * ((r / 4) % 2);
  int key_off[LOADS];
#pragma unroll
  for (int j = 0; j < LOADS; ++j) {
    const int R = j * RPI + lane / KCH;  // row of the chunk: of its first page up to 15
    key_off[j] = (R % PAGE * D + ((lane % KCH) ^ key_slot(R)) * 8) * 2;
  }
  auto load = [&](auto& t, int c) __attribute__((always_inline)) {
    constexpr bool THROUGH_LDS = __is_same(decltype(t), DecodeValues<D>&);
    if (c - id_first >= WAVE / 2) fetch_ids(c);
    const int at = 2 * (c - id_first);
    const int p0 = max(__builtin_amdgcn_readlane(ids, at), 0);  // a page behind the window was given back: its tokens are masked below
    const int p1 = (lo_al + c * CHUNK + PAGE < kv_len) ? max(__builtin_amdgcn_readlane(ids, at + 1), 0) : p0;
    const bf16* page0 = kc + ((size_t)p0 * Hkv + kvh) * PAGE * D;
    const bf16* page1 = kc + ((size_t)p1 * Hkv + kvh) * PAGE * D;
    if constexpr (THROUGH_LDS) {
      // A page's 16 rows of the head are contiguous, 1 KB a load, each row's 16-byte pieces permuted (key_slot).
      unsigned char* stage = ring + ((c - w_begin) & 1) * Lds::CHUNK_BYTES;
#pragma unroll
      for (int j = 0; j < LOADS; ++j) page_to_lds<PAGE * D * 2>(j * RPI < PAGE ? page0 : page1, key_off[j], stage + j * 1024);
    } else {
      const bf16* k0 = (r < 8 ? page0 : page1) + key_row % PAGE * D + g * 8;
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        t.ka[kk] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(k0 + kk * 32));
        t.kb[kk] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(k0 + 4 * D + kk * 32));
      }
    }
    asm volatile("" ::: "memory");  // the values behind the keys: the waits below count on it
    __builtin_amdgcn_sched_barrier(0);
    // V^T operand: element d = db * 16 + r, tokens 8 (g % 2) .. + 7 of page g / 2.
    const bf16* v0 = vc + (((size_t)(g < 2 ? p0 : p1) * Hkv + kvh) * D + r) * PAGE + (g % 2) * 8;
#pragma unroll
    for (int db = 0; db < DB; ++db) t.v[db] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(v0 + (size_t)db * 16 * PAGE));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // LAST: the wave's last chunk; else the next one has been asked for as well.
  struct Last {};
  struct NotLast {};
  auto multiply = [&](auto& t, int c, auto which) __attribute__((always_inline)) {
    constexpr bool THROUGH_LDS = __is_same(decltype(t), DecodeValues<D>&);
    constexpr bool LAST = __is_same(decltype(which), Last);
    const int t0 = lo_al + c * CHUNK;
    bf16x8 ka[KK], kb[KK];
    if constexpr (THROUGH_LDS) {
      // The chunk's keys are there when at most its values and the next chunk are under way (the new key's stores, where there are any, are newer).
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LAST ? DB : 2 * DB + LOADS) : "memory");
      const unsigned char* stage = ring + ((c - w_begin) & 1) * Lds::CHUNK_BYTES;
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        ka[kk] = *reinterpret_cast<const bf16x8*>(stage + key_row * D * 2 + (((kk * 4 + g) ^ key_slot(key_row)) * 16));
        kb[kk] = *reinterpret_cast<const bf16x8*>(stage + (key_row + 4) * D * 2 + (((kk * 4 + g) ^ key_slot(key_row + 4)) * 16));
      }
    } else {
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) ka[kk] = t.ka[kk], kb[kk] = t.kb[kk];
    }
    if (FUSED && LAST && has_new) {
      // The new token is token j of this chunk: key row jt of page jp, that is row r_new of product a
      // or b; and element j % 8 of the value operands of lane group 2 jp + jt / 8.
      const int j = kv_len - 1 - t0, jp = j / PAGE, jt = j % PAGE;
      const int r_new = jp * 8 + (jt / 8) * 4 + jt % 4;
      const bool second = (jt / 4) & 1;
      if (r == r_new) {
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
          const bf16x8 kn = *reinterpret_cast<const bf16x8*>(&kv_new[kk * 32 + g * 8]);
          if (second) kb[kk] = kn;
          else ka[kk] = kn;
        }
      }
      // A chunk that ends in its first page reads that page for its second half as well (masked, but a
      // probability of 0 does not wipe out whatever the unwritten slot happens to hold).
      const bool twice = t0 + PAGE >= kv_len;
      if (g % 2 == jt / 8 && (g / 2 == jp || twice)) {
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          const bf16 vn = kv_new[D + db * 16 + r];
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (e == jt % 8) t.v[db][e] = vn;
        }
      }
    }
    floatx4 s0 = floatx4{0.f, 0.f, 0.f, 0.f}, s1 = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[kk], qf[kk], s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kb[kk], qf[kk], s1, 0, 0, 0);
    }
    if (!LAST && THROUGH_LDS)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the keys are read: the chunk after the next takes their place in the ring
    // This lane: tokens tl + i (s0) and tl + 4 + i (s1) of query r, tl = t0 + 16 (g / 2) + 8 (g % 2).
    const int tl = t0 + 8 * g;
    float sc[8];
    float m_new = m_run;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ta = tl + i, tb = ta + 4;
      sc[i] = (ta >= lo && ta < kv_len) ? s0[i] * scale2 : -INFINITY;
      sc[4 + i] = (tb >= lo && tb < kv_len) ? s1[i] * scale2 : -INFINITY;
      m_new = fmaxf(m_new, fmaxf(sc[i], sc[4 + i]));
    }
    m_new = rows4_max(m_new);
    // A chunk that holds no visible token at all cannot occur: chunks start at the window's first
    // token's chunk and end at the last token's.
    float psum = 0.f;
    bf16x8 pf;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float p = __builtin_amdgcn_exp2f(sc[i] - m_new);
      psum += p;
      pf[i] = static_cast<bf16>(p);
    }
    psum = rows4_sum(psum);
    const float corr = __builtin_amdgcn_exp2f(m_run - m_new);
    l_run = l_run * corr + psum;
    m_run = m_new;
    // O^T[d, query]: a lane's output values are all of its own query r.
#pragma unroll
    for (int db = 0; db < DB; ++db) {
#pragma unroll
      for (int i = 0; i < 4; ++i) o[db][i] *= corr;
      o[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(t.v[db], pf, o[db], 0, 0, 0);
    }
  };
  {
    DecodeValues<D> va, vb;
    int c = w_begin;
    // The wave that holds the new token asks for its key (lanes 0 .. D / 4 - 1) and value (lanes 32 ..
    // 32 + D / 4 - 1) ahead of the first chunk too.
    const bool is_k = lane < 32, kv_valid = lane % 32 < D / 4;
    const int kv_d0 = kv_valid ? (lane % 32) * 4 : 0;
    const size_t kv_at = qkv_row + (size_t)(is_k ? Hq + kvh : Hq + Hkv + kvh) * D + kv_d0;
    Parts4 kv_parts;
    HeadTerms k_terms;
    int new_page = 0;
    if (FUSED && has_new) {
      new_page = table[(kv_len - 1) / PAGE];
      ask_parts4(kv_parts, fin.parts, 0, fin.splits, fin.split_stride, kv_at);
      head_terms<D>(k_terms, kv_d0, fin.k_weight, rope_row);
    }
    auto queries = [&]() __attribute__((always_inline)) {
      const int step = together ? 4 * 256 : 4 * WAVE;
      bf16* q_lds = reinterpret_cast<bf16*>(smem + Lds::QUERIES) + (together ? 0 : wave * 4 * WAVE);  // (16 D hold four waves' 256 from D = 64 on)
      auto round = [&](int base) __attribute__((always_inline)) {
        const int e0 = base + (together ? tid : lane) * 4;
        const bool valid = e0 < gd;
        const int ec = valid ? e0 : 0;
        const size_t at = qkv_row + (size_t)kvh * gd + ec;
        if (base > 0) {
          ask_parts4(q_parts, fin.parts, 0, fin.splits, fin.split_stride, at);
          head_terms<D>(q_terms, ec % D, fin.q_weight, rope_row);
        }
        float x[4];
        sum_parts4(x, q_parts, fin.parts, fin.splits, fin.split_stride, at);
        head_norm_rotate<D>(x, ec % D, q_terms, fin.q_weight != nullptr, fin.eps, rope_row != nullptr);
        if (valid) {
          bf16x4 xb;
#pragma unroll
          for (int e = 0; e < 4; ++e) xb[e] = static_cast<bf16>(x[e]);
          *reinterpret_cast<bf16x4*>(q_lds + ec) = xb;
        }
      };
      round(0);  // (outside the loop for the same reason)
      for (int base = step; base < gd; base += step) round(base);
      if (together) __syncthreads();
      if (r < G) {
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) qf[kk] = *reinterpret_cast<const bf16x8*>(q_lds + r * D + kk * 32 + g * 8);
      }
      if (has_new) {
        // The new key and value: into the cache, and into LDS for this wave's last chunk.
        float xn[4];
        sum_parts4(xn, kv_parts, fin.parts, fin.splits, fin.split_stride, kv_at);
        float xk[4] = {xn[0], xn[1], xn[2], xn[3]};
        head_norm_rotate<D>(xk, kv_d0, k_terms, fin.k_weight != nullptr, fin.eps, rope_row != nullptr);
        const int p = kv_len - 1;
        const size_t page = (size_t)new_page;
        if (kv_valid && is_k) {
          bf16x4 xb;
#pragma unroll
          for (int e = 0; e < 4; ++e) xb[e] = static_cast<bf16>(xk[e]);
          *reinterpret_cast<bf16x4*>(&kv_new[kv_d0]) = xb;
          *reinterpret_cast<bf16x4*>(kc_rw + ((page * Hkv + kvh) * PAGE + p % PAGE) * D + kv_d0) = xb;
        }
        if (kv_valid && !is_k) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const bf16 vb = static_cast<bf16>(xn[e]);
            kv_new[D + kv_d0 + e] = vb;
            vc_rw[((page * Hkv + kvh) * D + kv_d0 + e) * PAGE + p % PAGE] = vb;
          }
        }
      }
    };
    // The page ids are the newest of what was asked for so far, so what the queries are made of is there as well; a wave without
    // chunks waits for it here, as behind a place where only some waves have waited the wait would be one for keys and values too.
    if (c < w_end) {
      fetch_ids(c);
      if (!FUSED) {
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) asm volatile("" : "+v"(qf[kk]));
      }
      if (through_lds) load(va, c);
    } else if (FUSED) {
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    }
    if (FUSED && (together || c < w_end)) queries();
    auto walk = [&](auto& ta, auto& tb) __attribute__((always_inline)) {
      for (; c + 2 < w_end; c += 2) {
        // (in step, heads of 64: with a second chunk on its way all the time 64 rows of 4,100 tokens, 32 heads, take 417 us, so 396)
        if (D == 64 && __is_same(decltype(ta), DecodeTile<D>&)) __builtin_amdgcn_s_waitcnt(0x0f70);
        load(tb, c + 1);
        multiply(ta, c, NotLast());
        load(ta, c + 2);
        multiply(tb, c + 1, NotLast());
      }
      if (c + 1 < w_end) {
        load(tb, c + 1);
        multiply(ta, c, NotLast());
        multiply(tb, c + 1, Last());
      } else {
        multiply(ta, c, Last());
      }
    };
    if (c < w_end && through_lds) {
      walk(va, vb);
    } else if (MAY_STEP && c < w_end) {
      DecodeTile<D> ta, tb;
      load(ta, c);
      walk(ta, tb);
    }
  }

  // Merge the block's four waves: per query (m, l) and O[query][D].
  float (*sm)[16] = reinterpret_cast<float (*)[16]>(smem + Lds::MAXIMA), (*sl)[16] = reinterpret_cast<float (*)[16]>(smem + Lds::SUMS);
  auto so = [&](int w) { return reinterpret_cast<float*>(smem + w * Lds::RING); };  // [16][D + 4]: the wave is done with its keys
  if (g == 0) {
    sm[wave][r] = m_run;
    sl[wave][r] = l_run;
  }
  if (r < G) {  // the group's queries alone
#pragma unroll
    for (int db = 0; db < DB; ++db) *reinterpret_cast<floatx4*>(so(wave) + r * (D + 4) + db * 16 + 4 * g) = o[db];
  }
  __syncthreads();
  for (int e = tid; e < G * D; e += 256) {
    const int qh = e / D, d = e % D;
    float M = fmaxf(fmaxf(sm[0][qh], sm[1][qh]), fmaxf(sm[2][qh], sm[3][qh]));
    float L = 0.f, O = 0.f;
    if (M > -INFINITY) {
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float f = __builtin_amdgcn_exp2f(sm[w][qh] - M);  // 0 for a wave that saw nothing
        L += sl[w][qh] * f;
        O += so(w)[qh * (D + 4) + d] * f;
      }
    }
    const int head = kvh * G + qh;
    if (splits == 1) {
      out[((size_t)tok * Hq + head) * D + d] = static_cast<bf16>(O / L);
    } else {
      const size_t at = ((size_t)b * Hq + head) * splits + split;
      part_o[at * D + d] = O;
      if (d == 0) {
        part_ml[at * 2] = M;
        part_ml[at * 2 + 1] = L;
      }
    }
  }
}

// Reduction of the splits in ascending order: grid (rows, Hq), D threads. Loads go out 32 splits at
// a time (all of them, for most shapes), so that their latencies overlap; the order of the sums is
// the order of the splits whatever the batching.
template <int D>
__global__ __launch_bounds__(D) void attn_decode_reduce_kernel(const float* __restrict__ part_o,
                                                                const float* __restrict__ part_ml,
                                                                const int* __restrict__ tokens, bf16* __restrict__ out,
                                                                int Hq, int splits) {
  constexpr int NB = 32;
  const int b = blockIdx.x, head = blockIdx.y, d = threadIdx.x;
  const size_t base = ((size_t)b * Hq + head) * splits;
  const float2* ml = reinterpret_cast<const float2*>(part_ml) + base;
  float M = -INFINITY, L = 0.f, O = 0.f;
  if (splits <= NB) {
    // One round: everything is asked for before the maximum is known.
    float2 q[NB];
    float o[NB];
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const bool in = u < splits;
      q[u] = in ? ml[u] : make_float2(-INFINITY, 0.f);
      o[u] = in ? part_o[(base + u) * D + d] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < NB; ++u) M = fmaxf(M, q[u].x);
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const float f = q[u].x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(q[u].x - M);  // an empty or absent split adds nothing
      L += q[u].y * f;
      O += o[u] * f;
    }
  } else {
    for (int s0 = 0; s0 < splits; s0 += NB) {
      float m[NB];
#pragma unroll
      for (int u = 0; u < NB; ++u) m[u] = s0 + u < splits ? ml[s0 + u].x : -INFINITY;
#pragma unroll
      for (int u = 0; u < NB; ++u) M = fmaxf(M, m[u]);
    }
    for (int s0 = 0; s0 < splits; s0 += NB) {
      float2 q[NB];
      float o[NB];
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        const bool in = s0 + u < splits;
        q[u] = in ? ml[s0 + u] : make_float2(-INFINITY, 0.f);
        o[u] = in ? part_o[(base + s0 + u) * D + d] : 0.f;
      }
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        const float f = q[u].x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(q[u].x - M);
        L += q[u].y * f;
        O += o[u] * f;
      }
    }
  }
  const int tok = tokens ? tokens[b] : b;
  out[((size_t)tok * Hq + head) * D + d] = static_cast<bf16>(O / L);
}

// rows decode tokens (tokens[i] = flat token index, or nullptr for the identity). part_o holds
// rows * Hq * splits * D floats, part_ml rows * Hq * splits * 2 (unused when splits == 1).
template <bool FUSED>
static int launch_decode(const bf16* q, int q_stride, bf16* kc, bf16* vc, const int* block_table, int table_width,
                         const int* tokens, const int* token_row, const int* pos, bf16* out, float* part_o, float* part_ml,
                         int rows, int splits, int Hq, int Hkv, int D, float scale, int window, FusedQkv fin, hipStream_t st,
                         bool reduce = true) {
  // round_up * per_split >> 32 is the quotient where round_up * splits < 2^32 (per_split exceeds 2^32 / splits by less than one):
  // for fewer than 64 splits always, as there are fewer than 2^26 chunks of 32 tokens.
  const unsigned per_split = splits > 1 && splits < 64 ? (unsigned)(((1ULL << 32) + splits - 1) / splits) : 0;
  static bool ready = false;  // more than 64 KB of LDS has to be asked for once per kernel
  if (!ready) {
    if (hipFuncSetAttribute((const void*)attn_decode_split_kernel<128, FUSED, false>, hipFuncAttributeMaxDynamicSharedMemorySize, DecodeLds<128>::BYTES) != hipSuccess ||
        hipFuncSetAttribute((const void*)attn_decode_split_kernel<128, FUSED, true>, hipFuncAttributeMaxDynamicSharedMemorySize, DecodeLds<128>::BYTES) != hipSuccess)
      return MS_LAUNCH_FAILED;
    ready = true;
  }
  // Whether a block may have STEP_CHUNKS chunks, as far as the table's width tells.
  const bool may_step = (size_t)kc % 16 != 0 || (long long)table_width * PAGE >= (long long)STEP_CHUNKS * CHUNK * splits;
  // A grid's second dimension ends at 65,535: more rows go in runs of that many, each with its own part of everything that goes by rows.
  for (int first = 0; first < rows; first += 65535) {
    const int n = rows - first < 65535 ? rows - first : 65535;
    dim3 grid(Hkv, n, splits);
#define LAUNCH_AS(DD, MAY_STEP)                                                                                         \
    attn_decode_split_kernel<DD, FUSED, MAY_STEP><<<grid, 256, DecodeLds<DD>::BYTES, st>>>(q, q_stride, kc, vc, block_table, table_width, tokens, \
                                                              token_row, pos, out, part_o, part_ml, Hq / Hkv, scale,     \
                                                              window, per_split, fin)
#define LAUNCH(DD)                                                                                                      \
    if (may_step) LAUNCH_AS(DD, true); else LAUNCH_AS(DD, false);                                                       \
    if (splits > 1 && reduce) attn_decode_reduce_kernel<DD><<<dim3(n, Hq), DD, 0, st>>>(part_o, part_ml, tokens, out, Hq, splits)
    if (D == 128) { LAUNCH(128); } else { LAUNCH(64); }
#undef LAUNCH
#undef LAUNCH_AS
    if (tokens) {
      tokens += n;
    } else {
      if (q) q += (size_t)n * q_stride;
      if (out) out += (size_t)n * Hq * D;
      if (FUSED) fin.parts += (size_t)n * fin.row_width;
      if (FUSED && fin.rope) fin.rope += (size_t)n * D;
      token_row += n;
      pos += n;
    }
    if (splits > 1) {
      part_o += (size_t)n * Hq * splits * D;
      part_ml += (size_t)n * Hq * splits * 2;
    }
  }
  return launch_status();
}

extern "C" int ms_attention_decode_bf16(const void* q, int q_stride, const void* kc, const void* vc,
                                        const int* block_table, int table_width, const int* tokens,
                                        const int* token_row, const int* pos, void* out, float* part_o, float* part_ml,
                                        int rows, int splits, int Hq, int Hkv, int D, int page_size, float scale,
                                        int window, hipStream_t st) {
  if (rows <= 0) return MS_OK;
  if (page_size != PAGE || (D != 64 && D != 128)) return MS_UNSUPPORTED;
  if (Hq <= 0 || Hkv <= 0 || Hq % Hkv || Hq / Hkv > 16 || splits < 1 || splits > 65535 || window < 0 || table_width <= 0 ||
      q_stride < Hq * D || q_stride % 8 || (splits > 1 && (!part_o || !part_ml)))
    return MS_BAD_ARG;
  return launch_decode<false>((const bf16*)q, q_stride, (bf16*)kc, (bf16*)vc, block_table, table_width, tokens, token_row,
                              pos, (bf16*)out, part_o, part_ml, rows, splits, Hq, Hkv, D, scale, window, FusedQkv{}, st);
}

// The same over the qkv projection's partial sums `parts` [qkv_splits, tokens, (Hq + 2 Hkv) D] (floats,
// qkv_split_stride apart) of a step whose rows bring one token each: per-head RMSNorm of q and k with
// bfloat16 weights [D] (both nullptr: none), rotation over the whole head by the table `rope`
// [tokens, D] (nullptr: none) in pairs (j, j + D/2) (rope_pairing must be MS_ROPE_HALVES: the kernel's lanes
// hold the halves of a head side by side; any other pairing is MS_UNSUPPORTED), and, with store != 0, the new token's key and value written to its place
// in the cache (its page is taken from the block table at pos).
extern "C" int ms_attention_decode_fused_bf16(const float* parts, int qkv_splits, long long qkv_split_stride,
                                              const void* q_weight, const void* k_weight, float eps, const float* rope,
                                              int rope_pairing, int store, void* kc, void* vc, const int* block_table, int table_width,
                                              const int* tokens, const int* token_row, const int* pos, void* out,
                                              float* part_o, float* part_ml, int rows, int splits, int Hq, int Hkv, int D,
                                              int page_size, float scale, int window, int reduce, hipStream_t st) {
  if (rows <= 0) return MS_OK;
  if (page_size != PAGE || (D != 64 && D != 128) || (rope != nullptr && rope_pairing != MS_ROPE_HALVES)) return MS_UNSUPPORTED;
  if (Hq <= 0 || Hkv <= 0 || Hq % Hkv || Hq / Hkv > 16 || splits < 1 || splits > 65535 || window < 0 || table_width <= 0 ||
      (splits > 1 && (!part_o || !part_ml)) || (splits > 1 && reduce && out == nullptr) || (splits == 1 && out == nullptr) ||
      parts == nullptr || qkv_splits < 1 || qkv_split_stride % 4 ||
      (q_weight == nullptr) != (k_weight == nullptr))
    return MS_BAD_ARG;
  FusedQkv fin;
  fin.parts = parts;
  fin.splits = qkv_splits;
  fin.split_stride = qkv_split_stride;
  fin.row_width = (Hq + 2 * Hkv) * D;
  fin.q_weight = (const bf16*)q_weight;
  fin.k_weight = (const bf16*)k_weight;
  fin.eps = eps;
  fin.rope = rope;
  fin.store = store;
  return launch_decode<true>(nullptr, 0, (bf16*)kc, (bf16*)vc, block_table, table_width, tokens, token_row, pos, (bf16*)out,
                             part_o, part_ml, rows, splits, Hq, Hkv, D, scale, window, fin, st, reduce != 0);
}

// ---------------------------------------------------------------------------------------------
// The reduction of the splits and the output projection in one kernel, for up to 16 rows that bring one
// token each: Y[m, n] = sum over heads h, d of out[m, h, d] W[n, h D + d], out being what the reduction
// kernel above would have written. A block owns HB heads (a slice of K) and NW * 16 rows of W, one wave
// per 16 rows. Its waves first ask for their weights, then merge the splits of the block's heads for every
// row (a wave per (row, head): a lane per split finds the maximum and the weights by wave reductions;
// then every thread sums its elements over the splits in ascending order), leave the merged rows in LDS
// as bfloat16, and multiply. K is split over the grid by heads: block column c writes the float partial
// sums P[c, m, n], which the reader of the residual stream adds up as it does for the other products
// of few rows. At most 64 splits (a lane each).
#define MERGE_MAX_SPLITS 64
#define MERGE_MAX_HB 4
// HB heads per block; every wave takes NPW blocks of 16 rows of W (so that a wide W does not mean many
// blocks that each merge the same splits again).
template <int D, int HB, int NPW>
__global__ __launch_bounds__(256) void attn_merge_project_kernel(const float* __restrict__ part_o,
                                                                 const float* __restrict__ part_ml,
                                                                 const bf16* __restrict__ W, float* __restrict__ P, int rows,
                                                                 int Hq, int splits, int N, int SG, int per, unsigned per_element) {
  constexpr int NW = 4, KB = HB * D, STEPS = KB / 64;
  __shared__ float fw[HB][16][MERGE_MAX_SPLITS];                 // weight of split s in row m of head j
  __shared__ __attribute__((aligned(16))) bf16 xs[16][KB + 8];   // merged rows; rows beyond `rows` are zero
  __shared__ float4 psum[NW * WAVE];
  const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE;
  const int r = lane % 16, g = lane / 16;
  const int h0 = blockIdx.x * HB;  // first head of this block
  const int K = Hq * D;            // columns of W
  const int nb0 = (blockIdx.y * NW + wave) * NPW * 16;
  // Loads come back in the order in which they went out, so what is needed first is asked for first: the splits' maxima and sums of
  // the wave's first two (row, head) pairs, then the first eight splits of the thread's element, both from the cache, then the weights,
  // which come from memory.
  const int pairs = rows * HB;
  auto pair_ml = [&](int p) { return reinterpret_cast<const float2*>(part_ml) + ((size_t)(p / HB) * Hq + h0 + p % HB) * splits; };
  float2 ml_first[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) ml_first[u] = pair_ml(min(wave + u * NW, pairs - 1))[min(lane, splits - 1)];
  // Merged rows. An element is four consecutive d of one (row, head); there are E = rows * HB * D / 4 of
  // them. With fewer elements than threads the splits of an element are shared out among SG threads
  // (contiguous ranges, each summed in ascending order, the ranges then added in ascending order), so
  // that one row's 64 splits are not one thread's 64 dependent loads.
  const int E = rows * HB * (D / 4);
  constexpr int threads = NW * WAVE;
  const int quot = SG == 1 ? 0 : (int)((tid * per_element) >> 16);  // tid / E
  const int my_e = min(tid - quot * E, E - 1), my_sg = min(quot, SG - 1);
  float4 o_first[8];
  {
    const int m = my_e / (HB * (D / 4)), c = my_e % (HB * (D / 4));
    const float* po = part_o + (((size_t)m * Hq + h0 + c / (D / 4)) * splits) * D + (c % (D / 4)) * 4;
#pragma unroll
    for (int u = 0; u < 8; ++u) o_first[u] = *reinterpret_cast<const float4*>(po + (size_t)min(my_sg * per + u, splits - 1) * D);
  }
  union Chunk { uint4 u; bf16x8 v; };
  Chunk a[NPW][STEPS][2];
#pragma unroll
  for (int q = 0; q < NPW; ++q) {
    const bf16* wp = W + (size_t)min(nb0 + q * 16 + r, N - 1) * K + (size_t)h0 * D + g * 16;
#pragma unroll
    for (int u = 0; u < STEPS; ++u) {
      a[q][u][0].u = load_once(wp + u * 64);
      a[q][u][1].u = load_once(wp + u * 64 + 8);
    }
  }
  for (int e = tid; e < 16 * (KB / 4); e += NW * WAVE)  // rows beyond `rows` read as zero
    *reinterpret_cast<uint2*>(&xs[e / (KB / 4)][(e % (KB / 4)) * 4]) = make_uint2(0, 0);
  // the weights of the splits: wave w takes the (row, head) pairs w, w + NW, ...
  for (int p = wave; p < rows * HB; p += NW) {
    const int m = p / HB, j = p % HB;
    float2 q = p == wave ? ml_first[0] : p == wave + NW ? ml_first[1] : pair_ml(p)[min(lane, splits - 1)];
    if (lane >= splits) q = make_float2(-INFINITY, 0.f);
    const float mx = wave_max(q.x);
    const float f = q.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(q.x - mx);  // an empty or absent split adds nothing
    const float total = wave_sum(q.y * f);
    fw[j][m][lane] = f / total;
  }
  __syncthreads();
  for (int base = 0; base < E * SG; base += threads) {
    const int item = base + tid;
    const bool live = item < E * SG;
    const int e = SG == 1 ? (live ? item : 0) : my_e, sg = SG == 1 ? 0 : my_sg;  // (SG > 1: one round)
    const int m = e / (HB * (D / 4)), c = e % (HB * (D / 4));
    const int j = c / (D / 4), d = (c % (D / 4)) * 4;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    const int s_end = min(splits, (sg + 1) * per);
    if (live) {
      const float* po = part_o + (((size_t)m * Hq + h0 + j) * splits) * D + d;
      for (int s0 = sg * per; s0 < s_end; s0 += 8) {
        float4 t[8];
        if (base == 0 && s0 == sg * per) {
#pragma unroll
          for (int u = 0; u < 8; ++u) t[u] = o_first[u];
        } else {
#pragma unroll
          for (int u = 0; u < 8; ++u) t[u] = *reinterpret_cast<const float4*>(po + (size_t)min(s0 + u, splits - 1) * D);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const float f = s0 + u < s_end ? fw[j][m][s0 + u] : 0.f;
          acc.x += t[u].x * f; acc.y += t[u].y * f; acc.z += t[u].z * f; acc.w += t[u].w * f;
        }
      }
    }
    if (SG > 1) {  // then E * SG <= threads: one round
      psum[tid] = acc;
      __syncthreads();
      if (tid < E) {
        acc = psum[tid];
        for (int q = 1; q < SG; ++q) {
          const float4 t = psum[q * E + tid];
          acc.x += t.x; acc.y += t.y; acc.z += t.z; acc.w += t.w;
        }
      }
    }
    if (live && sg == 0) {
      union { uint2 u; bf16 b[4]; } o;
      o.b[0] = static_cast<bf16>(acc.x); o.b[1] = static_cast<bf16>(acc.y);
      o.b[2] = static_cast<bf16>(acc.z); o.b[3] = static_cast<bf16>(acc.w);
      *reinterpret_cast<uint2*>(&xs[m][j * D + d]) = o.u;
    }
  }
  __syncthreads();
  bf16x8 x[STEPS][2];
#pragma unroll
  for (int u = 0; u < STEPS; ++u) {
    const bf16* xp = &xs[r][u * 64 + g * 16];
    x[u][0] = *reinterpret_cast<const bf16x8*>(xp);
    x[u][1] = *reinterpret_cast<const bf16x8*>(xp + 8);
  }
#pragma unroll
  for (int q = 0; q < NPW; ++q) {
    floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < STEPS; ++u) {
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[q][u][0].v, x[u][0], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[q][u][1].v, x[u][1], acc, 0, 0, 0);
    }
    // acc[e] = Y[m = r][n = nb + 4 g + e] of this block's heads
    const int nb = nb0 + q * 16;
    if (r < rows && nb + 16 <= N)
      *reinterpret_cast<float4*>(P + ((size_t)blockIdx.x * rows + r) * N + nb + 4 * g) = make_float4(acc[0], acc[1], acc[2], acc[3]);
  }
}

// Heads per block so that the output projection's partial sums number at most 16: 1, 2, 3 or 4 (a block's
// slice of K, HB * D, is then a whole number of 64-element steps for both head sizes).
static int merge_project_heads_per_block(int Hq) {
  const int hb = (Hq + 15) / 16;
  return hb < 1 || hb > MERGE_MAX_HB || Hq % hb ? 0 : hb;
}

// How many partial sums ms_attention_merge_project leaves for this shape, or -1 where it has no kernel and
// the reduction kernel and the output projection must run apart. The one place that decides it: the launch
// below asks the same function, so a caller that sizes its buffers by the answer is never refused afterwards.
extern "C" int ms_attention_merge_project_splits(int rows, int Hq, int D, int splits, int N) {
  const int hb = merge_project_heads_per_block(Hq);
  if (hb == 0 || rows < 1 || rows > 16 || splits < 1 || splits > MERGE_MAX_SPLITS || (D != 64 && D != 128) || N <= 0 || N % 64)
    return -1;
  return Hq / hb;
}

// P [ms_attention_merge_project_splits(...), rows, N] (float partial sums) from the split attention's
// partial results of `rows` <= 16 single-token rows (part_o, part_ml as the decode kernels leave them)
// and the output projection's weight W [N, Hq * D]. MS_UNSUPPORTED exactly where that function says -1.
// The widest instance (D 128, 4 heads, 256 rows of W per block) has 256 registers of weights and moves 116 values through the
// accumulation registers; nothing goes to scratch memory. Microseconds (weights from memory, 1 and 8 rows): 16 heads and 1,024
// columns 4.3 -> 3.7 and 4.8 -> 3.5, 32 heads and 4,096 columns 10.5 -> 10.0 and 13.2 -> 11.5, since loads go out in the order of
// their use and a wave's sums no longer pass through LDS.
extern "C" int ms_attention_merge_project(const float* part_o, const float* part_ml, const void* W, float* P, int rows,
                                          int Hq, int D, int splits, int N, hipStream_t st) {
  if (rows <= 0 || N <= 0) return MS_OK;
  if (part_o == nullptr || part_ml == nullptr || W == nullptr || P == nullptr || Hq <= 0 || splits < 1) return MS_BAD_ARG;
  const int out_splits = ms_attention_merge_project_splits(rows, Hq, D, splits, N);
  if (out_splits < 1) return MS_UNSUPPORTED;
  const int hb = Hq / out_splits;
  // Rows of W per block: 64, or 256 where that still leaves a block for every CU.
  const int npw = (N % 256 == 0 && (long)out_splits * (N / 256) >= 256) ? 4 : 1;
  dim3 grid(out_splits, N / (64 * npw));
  const bf16* w = (const bf16*)W;
  // How many threads share an element's splits, how many splits each takes, and 2^16 / elements rounded up (at most 128 elements where it
  // is used: 256 threads times the rounding stays below 2^16). Divisions done here, once.
  const int elements = rows * hb * (D / 4), sg = elements >= 256 ? 1 : 256 / elements, per = (splits + sg - 1) / sg;
  const unsigned per_element = (65536 + elements - 1) / elements;
#define LAUNCH(DD, HB, NPW) \
  attn_merge_project_kernel<DD, HB, NPW><<<grid, 256, 0, st>>>(part_o, part_ml, w, P, rows, Hq, splits, N, sg, per, per_element)
#define LAUNCH_HB(DD, NPW)                                                                                              \
  if (hb == 1) LAUNCH(DD, 1, NPW);                                                                                      \
  else if (hb == 2) LAUNCH(DD, 2, NPW);                                                                                 \
  else if (hb == 3) LAUNCH(DD, 3, NPW);                                                                                 \
  else LAUNCH(DD, 4, NPW)
  if (D == 128 && npw == 4) { LAUNCH_HB(128, 4); }
  else if (D == 128) { LAUNCH_HB(128, 1); }
  else if (npw == 4) { LAUNCH_HB(64, 4); }
  else { LAUNCH_HB(64, 1); }
#undef LAUNCH_HB
#undef LAUNCH
  return launch_status();
}
