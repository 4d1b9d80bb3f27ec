// Linear recurrences over a matrix state per (request, head), token by token:
//     S_t = a_t S_(t-1) + b_t k_t v_t^T,   o_t = S_t^T q_t          (S: [D, E], k, q: [D], v: [E])
// in forms that differ in where a_t and b_t come from:
//   MS_REC_DECAY: a_t = decay[head] (a constant per head), b_t = 1; o_t as above.
//   MS_REC_EXP_GATES: a log input gate i_t and a log forget gate f_t per head and token, made bounded by a soft cap,
//       i = cap tanh((x_i + bias_i) / cap), f = logsigmoid(cap tanh((x_f + bias_f) / cap)), and a running maximum
//       m_t = max(f_t + m_(t-1), i_t) (m starts at 0) that keeps the exponentials in range:
//       a_t = exp(f_t + m_(t-1) - m_t), b_t = exp(i_t - m_t); a vector n_t = a_t n_(t-1) + b_t k_t beside S;
//       o_t = S_t^T q_t / (max(|n_t . q_t|, exp(-m_t)) + 1e-6).
//   MS_REC_WKV: a decay per key channel and token, w_t [D] (its logarithm is row t of the float32 matrix `w`, columns h D ..), and a bonus
//       u [H, D] that only the current token gets: o_t = (S_(t-1) + diag(u) k_t v_t^T)^T q_t, and only then
//       S_t = diag(w_t) S_(t-1) + k_t v_t^T.
//   MS_REC_STEP: both from one step size per head and token, d_t = softplus(w_t + bias) (column h of the matrix `w`):
//       a_t = exp(decay[head] d_t), b_t = d_t; a share of the value joins the output, o_t = S_t^T q_t + u[head] v_t. `share`
//       consecutive heads read the same q and k.
// q, k, v (and the gates' inputs) are columns of one float32 matrix x [tokens, ld] (the layer's projections);
// an activation (none or SiLU) is applied to q, k and v on the way in, q is then scaled by q_scale. Everything
// is float32. The state lives in S [slots, H, D, E] (and n [slots, H, D], m [slots, H]); a row whose
// sequence starts in this step (starts[row] == 0) begins from zero, every other row from its slot; the state after
// the row's last token is written back.
//
// One block of 256 threads per (row, head, run of EB value columns) walks the row's tokens in order with the state
// in registers (the columns of S are independent of one another, so few rows still fill the chip):
// thread (s, e) holds S[d][e] for d = s, s + NS, ... (NS = 256 / EP slices, EP the power of two that holds EB),
// adds its part of o_t[e], and the slices' parts meet in LDS in ascending s. What an output element is summed
// from, and in which order, depends on D alone: a token's result does not depend on how the sequence was
// cut into steps or batched.
#include "common.h"

#define MS_REC_DECAY 0
#define MS_REC_EXP_GATES 1
#define MS_REC_WKV 2
#define MS_REC_STEP 3

struct RecurrenceArgs {
  const float* x;
  int ld, q_off, k_off, v_off, i_off, f_off;
  int H, D, E, act, mode;
  float q_scale, cap;
  const float* decay;
  const void* i_bias;
  const void* f_bias;
  int bias_is_bf16;
  float* S;
  float* n;
  float* m;
  const int* row_start;
  const int* starts;
  const int* state_slots;
  float* out;
  const float* w;  // MS_REC_WKV: the decays' logarithms [tokens, ld_w], head h's D channels from column h D on; MS_REC_STEP: the steps [tokens, ld_w]
  int ld_w;
  const float* u;  // MS_REC_WKV: the bonus [H, D]; MS_REC_STEP: the value's share of the output [H]
  int share;       // heads that read the same q and k (1 but for MS_REC_STEP)
  float* kept;     // MS_REC_EXP_GATES with several runs of value columns: [rows, H, D + 1], n and m until every block has read them
};

__device__ __forceinline__ float rec_act(float v, int act) { return act ? v / (1.f + expf(-v)) : v; }
__device__ __forceinline__ float rec_bias(const void* b, int is_bf16, int h) {
  if (b == nullptr) return 0.f;
  return is_bf16 ? to_f32(((const bf16*)b)[h]) : ((const float*)b)[h];
}
__device__ __forceinline__ float log_sigmoid(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }

template <int PM>
__global__ __launch_bounds__(256) void gated_recurrence_kernel(RecurrenceArgs a, int EP, int EB) {
  __shared__ float qs[2][256], ks[2][256], ws[2][256], us[256];
  __shared__ float red[256];
  __shared__ float wred[2][4];
  const int b = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int D = a.D, E = a.E;
  const int NS = 256 / EP, s = tid / EP;
  const int e = blockIdx.z * EB + tid % EP;  // this thread's column; columns beyond the block's run or beyond E are idle
  const bool col = tid % EP < EB && e < E;
  const int per = (D + NS - 1) / NS;
  const int t0 = a.row_start[b], t1 = a.row_start[b + 1];
  const bool fresh = a.starts[b] == 0;
  const size_t slot = (size_t)a.state_slots[b];
  float* Sg = a.S + (slot * a.H + h) * (size_t)D * E;
  const bool gates = a.mode == MS_REC_EXP_GATES, wkv = a.mode == MS_REC_WKV, steps = a.mode == MS_REC_STEP;
  const int hq = steps ? h / a.share : h;
  if (wkv && tid < D) us[tid] = a.u[h * D + tid];  // read behind the first token's barrier
  float S[PM];
#pragma unroll
  for (int i = 0; i < PM; ++i) {
    const int d = s + i * NS;
    S[i] = (!fresh && i < per && d < D && col) ? Sg[(size_t)d * E + e] : 0.f;
  }
  float nv = 0.f, m = 0.f;
  if (gates && !fresh) {
    if (tid < D) nv = a.n[(slot * a.H + h) * D + tid];
    m = a.m[slot * a.H + h];
  }
  const float decay = (gates || wkv) ? 0.f : a.decay[h];
  const float bi = (gates || steps) ? rec_bias(a.i_bias, a.bias_is_bf16, h) : 0.f;
  const float bf = gates ? rec_bias(a.f_bias, a.bias_is_bf16, h) : 0.f;
  for (int t = t0; t < t1; ++t) {
    const float* xr = a.x + (size_t)t * a.ld;
    const int buf = (t - t0) & 1;
    float fs = decay, is = 1.f;
    if (gates) {
      const float gi = a.cap * tanhf((xr[a.i_off + h] + bi) / a.cap);
      const float gf = log_sigmoid(a.cap * tanhf((xr[a.f_off + h] + bf) / a.cap));
      const float m_new = fmaxf(gf + m, gi);
      fs = expf(gf + m - m_new);
      is = expf(gi - m_new);
      m = m_new;
    }
    if (steps) {
      is = softplus(a.w[(size_t)t * a.ld_w + h] + bi);
      fs = expf(decay * is);
    }
    float kd = 0.f, qd = 0.f;
    if (tid < D) {
      qd = rec_act(xr[a.q_off + hq * D + tid], a.act) * a.q_scale;
      kd = rec_act(xr[a.k_off + hq * D + tid], a.act);
      qs[buf][tid] = qd;
      ks[buf][tid] = kd;
      if (wkv) ws[buf][tid] = expf(a.w[(size_t)t * a.ld_w + h * D + tid]);
    }
    if (gates) {
      nv = fs * nv + is * kd;  // threads beyond D carry zeros
      const float part = wave_sum(nv * qd);
      if (tid % WAVE == 0) wred[buf][tid / WAVE] = part;
    }
    const float v = col ? rec_act(xr[a.v_off + h * E + e], a.act) : 0.f;
    __syncthreads();
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < PM; ++i) {
      const int d = s + i * NS;
      if (i < per && d < D) {
        if (wkv) {
          const float kv = ks[buf][d] * v;
          acc += (S[i] + us[d] * kv) * qs[buf][d];
          S[i] = ws[buf][d] * S[i] + kv;
        } else {
          S[i] = fs * S[i] + is * ks[buf][d] * v;
          acc += S[i] * qs[buf][d];
        }
      }
    }
    if (NS > 1) {
      __syncthreads();  // the previous token's sums have been read
      red[tid] = acc;
      __syncthreads();
      if (s == 0) {
        acc = red[tid];
        for (int j = 1; j < NS; ++j) acc += red[j * EP + tid];
      }
    }
    if (s == 0 && col) {
      if (gates) {
        const float nq = (wred[buf][0] + wred[buf][1]) + (wred[buf][2] + wred[buf][3]);
        acc = acc / (fmaxf(fabsf(nq), expf(-m)) + 1e-6f);
      }
      if (steps) acc += a.u[h] * v;
      a.out[(size_t)t * (a.H * E) + h * E + e] = acc;
    }
  }
#pragma unroll
  for (int i = 0; i < PM; ++i) {
    const int d = s + i * NS;
    if (i < per && d < D && col) Sg[(size_t)d * E + e] = S[i];
  }
  if (gates && blockIdx.z == 0) {  // every run of columns has formed the same n and m
    // A block of another run may not have started yet: it must still find the old ones, so the new ones wait elsewhere.
    float* to = a.kept ? a.kept + ((size_t)b * a.H + h) * (D + 1) : a.n + (slot * a.H + h) * D;
    if (tid < D) to[tid] = nv;
    if (tid == 0) *(a.kept ? to + D : a.m + slot * a.H + h) = m;
  }
}

// n and m of a step's rows into the state. grid (rows, H).
__global__ __launch_bounds__(256) void rec_commit_kernel(RecurrenceArgs a) {
  const int b = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, D = a.D;
  const size_t at = (size_t)a.state_slots[b] * a.H + h;
  const float* from = a.kept + ((size_t)b * a.H + h) * (D + 1);
  if (tid < D) a.n[at * D + tid] = from[tid];
  if (tid == 0) a.m[at] = from[D];
}

extern "C" int ms_gated_recurrence(const float* x, int ld, int q_off, int k_off, int v_off, int i_off, int f_off, int H, int D,
                                   int E, int act, int mode, float q_scale, float cap, const float* decay, const void* i_bias,
                                   const void* f_bias, int bias_is_bf16, float* S, float* n, float* m, const int* row_start,
                                   const int* starts, const int* state_slots, float* out, int rows, const float* w, int ld_w,
                                   const float* u, int share, float* kept, hipStream_t st) {
  if (rows <= 0) return MS_OK;
  if (H <= 0 || D <= 0 || E <= 0 || x == nullptr || S == nullptr || out == nullptr || row_start == nullptr || starts == nullptr ||
      state_slots == nullptr || (act != 0 && act != 1) || q_off < 0 || k_off < 0 || v_off < 0)
    return MS_BAD_ARG;
  // (q, k and v may lie in later rows of the matrix that x is the top of: their columns are then counted past ld, and the
  // caller answers for the rows being there)
  if (mode == MS_REC_DECAY) {
    if (decay == nullptr) return MS_BAD_ARG;
  } else if (mode == MS_REC_EXP_GATES) {
    if (n == nullptr || m == nullptr || !(cap > 0.f) || i_off < 0 || f_off < 0 || i_off + H > ld || f_off + H > ld) return MS_BAD_ARG;
  } else if (mode == MS_REC_WKV) {
    if (w == nullptr || u == nullptr || ld_w < H * D) return MS_BAD_ARG;
  } else if (mode == MS_REC_STEP) {
    if (decay == nullptr || w == nullptr || u == nullptr || ld_w < H || share < 1 || H % share) return MS_BAD_ARG;
  } else {
    return MS_BAD_ARG;
  }
  if (D > 256 || E > 256 || H > 65535) return MS_UNSUPPORTED;
  // Runs of 32 value columns, always: the order of an output's sum then depends on D alone.
  const int EB = E < 32 ? E : 32, EP = 32;
  const int per = (D + 256 / EP - 1) / (256 / EP);
  RecurrenceArgs a{x, ld, q_off, k_off, v_off, i_off, f_off, H, D, E, act, mode, q_scale, cap, decay, i_bias, f_bias, bias_is_bf16,
                   S, n, m, row_start, starts, state_slots, out, w, ld_w, u, share, nullptr};
  const dim3 grid(rows, H, (E + EB - 1) / EB);
  if (mode == MS_REC_EXP_GATES && grid.z > 1) {
    if (kept == nullptr) return MS_BAD_ARG;
    a.kept = kept;
  }
  if (per <= 4) gated_recurrence_kernel<4><<<grid, 256, 0, st>>>(a, EP, EB);
  else if (per <= 16) gated_recurrence_kernel<16><<<grid, 256, 0, st>>>(a, EP, EB);
  else if (per <= 64) gated_recurrence_kernel<64><<<grid, 256, 0, st>>>(a, EP, EB);
  else if (per <= 128) gated_recurrence_kernel<128><<<grid, 256, 0, st>>>(a, EP, EB);
  else return MS_UNSUPPORTED;
  if (a.kept != nullptr) rec_commit_kernel<<<dim3(rows, H), 256, 0, st>>>(a);
  return launch_status();
}

// ---------------------------------------------------------------------------------------------
// The same recurrences for rows that bring many tokens, in chunks of REC_CHUNK tokens and three passes, so
// that the work is matrix products over a chunk and every chunk of every row and head has a block of its own:
//   1. per chunk: the chunk's own contribution to the state at its end, U = sum_j w_j k_j v_j^T (and u = sum_j
//      w_j k_j), w_j = exp(B - b_j + i_j - a) with b_j the log forget gates summed from the chunk's start through
//      j, B = b_last, and a = max_j (B - b_j + i_j) (a = 0 for the constant decay, whose weights cannot grow);
//   2. per (row, head), chunk after chunk: m' = max(B + m, a), S' = exp(B + m - m') S + exp(a - m') U; the state
//      *before* each chunk takes U's place in the buffer, m and n before it are kept beside it; the state after
//      the last chunk goes to the slot;
//   3. per chunk: with the state S0 (n0, m0) before it, m_t by its own recurrence from m0,
//      o_t = g_t S0^T q_t + sum_(j <= t) P_tj v_j,  P_tj = (q_t . k_j) exp(b_t - b_j + i_j - m_t),  g_t = exp(b_t + m0 - m_t),
//      n_t . q_t = g_t n0 . q_t + sum_j P_tj, and the normaliser as above.
// Every exponent is at most zero by the definition of the maxima. All float32; sums are reassociated against the
// token-by-token kernel, nothing else differs. Head sizes up to REC_CHUNK_MAX_DIM; larger ones take the other kernel.
#define REC_CHUNK 64
#define REC_CHUNK_MAX_DIM 128

struct ChunkArgs {
  RecurrenceArgs r;
  float* U;    // [chunks, H, D * E]
  float* u;    // [chunks, H, D]
  double* cs;  // [chunks, H, 4]: B, a, m before the chunk, m after the row's last (double: B may be in the hundreds where B + m is small)
  int rows;
};

// The chunk `c` of the step: its row, first token and token count; *base = index of the row's first chunk.
__device__ __forceinline__ void find_chunk(const int* __restrict__ row_start, int rows, int c, int* row, int* first, int* count,
                                           int* base) {
  int b = 0, at = 0;
  for (; b < rows - 1; ++b) {
    const int nc = (row_start[b + 1] - row_start[b] + REC_CHUNK - 1) / REC_CHUNK;
    if (c < at + nc) break;
    at += nc;
  }
  *row = b;
  *base = at;
  *first = row_start[b] + (c - at) * REC_CHUNK;
  const int left = row_start[b + 1] - *first;
  *count = left < REC_CHUNK ? left : REC_CHUNK;
}

// All three passes multiply in float32 on the matrix cores (v_mfma_f32_16x16x4_f32: 32-bit operands, products and sums). Layout
// (lane l, g = l / 16, r = l % 16): A operand A[i = r][k = g], B operand B[k = g][j = r], result D[i = 4 g + 0..3][j = r].
// Two choices of which number an index stands for save every exchange between lanes:
//   * a sum's index k may run in any order that both operands share. A lane that holds elements 8 g .. 8 g + 7 of a row feeds
//     them to eight products in turn; a lane that holds the scores of keys 4 g + x of its token feeds them to the product with
//     values as they are.
//   * value columns: a lane reads the four columns 4 r .. 4 r + 3 at once and feeds them to four products q. As the first operand
//     (outputs): the lane's results x of the products q are then columns 16 g + 4 x + q, sixteen in a row. As the second (summary): they
//     are columns 4 r + q of row 4 g + x, so that a store writes 256 bytes of a row of U (28 us; as the first operand 16-byte
//     pieces of sixteen rows, 33. The outputs gain nothing from it: their rows' factors would have to change lanes).
// Head sizes are padded to DS runs of 32 (keys) and EH runs of 64 (values) with zeros. 2,048 tokens, 16 heads of 128 x 128:
// summary 28 us, scan 18, output 40 (with a branch around every load 33 and 57; on the vector units 73, 50 and 162); the bytes alone take
// about 11, 11 and 17, and all blocks load at the same time, then multiply.
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

// Four columns col .. col + 3 of a row of `width` columns, zeros from the width on. vec: rows 16-byte aligned, width a multiple of 4.
__device__ __forceinline__ floatx4 load4(const float* __restrict__ row, int col, int width, bool vec) {
  if (vec) return col < width ? *reinterpret_cast<const floatx4*>(row + col) : floatx4{0.f, 0.f, 0.f, 0.f};
  floatx4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = col + i < width ? row[col + i] : 0.f;
  return v;
}
__device__ __forceinline__ void store4(float* __restrict__ row, int col, int width, bool vec, floatx4 v) {
  if (vec) {
    if (col < width) *reinterpret_cast<floatx4*>(row + col) = v;
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (col + i < width) row[col + i] = v[i];
}
__device__ __forceinline__ floatx4 rec_act4(floatx4 v, int act) {
  if (act) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = rec_act(v[i], act);
  }
  return v;
}

// What the chunk's log gates are made of, a lane of the first wave for each token (the other waves load the same): asked for ahead of
// everything else, since loads come back in order.
struct GateInputs {
  float i, f;
  unsigned i_bias, f_bias;  // as they are stored: a conversion would wait for them
};
__device__ __forceinline__ unsigned bias_bits(const void* b, int is_bf16, int h) {
  if (b == nullptr) return 0;
  return is_bf16 ? (unsigned)((const unsigned short*)b)[h] : ((const unsigned*)b)[h];
}
__device__ __forceinline__ float bias_value(unsigned bits, int is_bf16) { return __uint_as_float(is_bf16 ? bits << 16 : bits); }
__device__ __forceinline__ GateInputs load_gates(const RecurrenceArgs& a, int h, int first, int count) {
  GateInputs in{0.f, 0.f, 0, 0};
  if (a.mode == MS_REC_EXP_GATES) {
    const float* xr = a.x + (size_t)(first + min((int)threadIdx.x % REC_CHUNK, count - 1)) * a.ld + h;
    in.i = xr[a.i_off];
    in.f = xr[a.f_off];
    in.i_bias = bias_bits(a.i_bias, a.bias_is_bf16, h);
    in.f_bias = bias_bits(a.f_bias, a.bias_is_bf16, h);
  } else {
    in.f = a.decay[h];
  }
  return in;
}

// Log gates of the chunk's tokens, a lane of the first wave each: gi[], and the running sums of the log forget gates in bs[].
// The sums are kept in double precision: the kernels need their differences, which may be small where the sums are in the
// hundreds, and in float32 such a difference would carry the sums' rounding. With `mt` (the running maximum before the chunk
// is m0): m_t = max(f_t + m_(t-1), i_t) = b_t + max(m0, max over s <= t of i_s - b_s). The caller's next barrier makes them known.
__device__ __forceinline__ void chunk_gates(const RecurrenceArgs& a, const GateInputs& in, int count, float* gi, double* bs,
                                            float* mt = nullptr, double m0 = 0.0) {
  const int tid = threadIdx.x;
  static_assert(REC_CHUNK == WAVE, "a lane per token");
  if (tid < REC_CHUNK) {
    const bool gates = a.mode == MS_REC_EXP_GATES;
    float i = 0.f, f = 0.f;
    if (tid < count) {
      if (gates) {
        i = a.cap * tanhf((in.i + bias_value(in.i_bias, a.bias_is_bf16)) / a.cap);
        f = log_sigmoid(a.cap * tanhf((in.f + bias_value(in.f_bias, a.bias_is_bf16)) / a.cap));
      } else {
        f = logf(in.f);
      }
    }
    double b = (double)f;
#pragma unroll
    for (int off = 1; off < WAVE; off <<= 1) {
      const double v = __shfl_up(b, off, WAVE);
      if (tid >= off) b += v;
    }
    gi[tid] = i;
    bs[tid] = b;
    if (mt != nullptr) {
      double top = tid < count ? (double)i - b : -INFINITY;
#pragma unroll
      for (int off = 1; off < WAVE; off <<= 1) {
        const double v = __shfl_up(top, off, WAVE);
        if (tid >= off) top = fmax(top, v);
      }
      mt[tid] = gates ? (float)(b + fmax(m0, top)) : 0.f;
    }
  }
}

// A thread's share of the chunk's rows of 4 N4 floats (column `off` of x on): all loads go out together, rows past
// the chunk's end read its last one and become zeros when they are put into LDS, rows `stride` floats apart.
template <int N4> struct ChunkRows {
  static constexpr int PER = REC_CHUNK * N4 / 256;
  static_assert(REC_CHUNK * N4 % 256 == 0, "");
  floatx4 v[PER];
  __device__ __forceinline__ void load(const RecurrenceArgs& a, int first, int count, int off) {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int i = threadIdx.x + u * 256;
      v[u] = *reinterpret_cast<const floatx4*>(a.x + (size_t)(first + min(i / N4, count - 1)) * a.ld + off + i % N4 * 4);
    }
  }
  __device__ __forceinline__ void put(float* to, int stride, int count, int act) {
    if (act) {
#pragma unroll
      for (int u = 0; u < PER; ++u) v[u] = rec_act4(v[u], act);
    }
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int i = threadIdx.x + u * 256;
      const float live = i / N4 < count ? 1.f : 0.f;
      floatx4 x;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = live != 0.f ? v[u][e] : 0.f;
      *reinterpret_cast<floatx4*>(to + i / N4 * stride + i % N4 * 4) = x;
    }
  }
};

// FULL (here and below): heads fill the runs they are padded to, in 16-byte aligned columns, so that no load needs a branch around
// it. A branch makes the next wait one for every load: a block's 24 loads into LDS and its queries then came one after another.
template <int DS, int EH, bool FULL>
__global__ __launch_bounds__(256) void rec_chunk_summary_kernel(ChunkArgs c, bool vec_v) {
  constexpr int ES = EH * 64, TW = (2 * DS + 3) / 4;  // TW: 16-row groups of U a wave owns (number wave, wave + 4)
  __shared__ __attribute__((aligned(16))) float V[REC_CHUNK * ES];
  __shared__ double bs[REC_CHUNK];
  __shared__ float gi[REC_CHUNK], wt[REC_CHUNK];
  const RecurrenceArgs& a = c.r;
  const int D = a.D, E = a.E, h = blockIdx.y, tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE;
  const int r = lane % 16, g = lane / 16;
  int row, first, count, base;
  find_chunk(a.row_start, c.rows, blockIdx.x, &row, &first, &count, &base);
  const GateInputs gate_in = load_gates(a, h, first, count);
  // a lane's keys: tokens 4 s + g, elements 16 (wave + 4 i) + r
  float k[TW][REC_CHUNK / 4];
  if constexpr (FULL) {
    ChunkRows<ES / 4> v;
    v.load(a, first, count, a.v_off + h * E);
#pragma unroll
    for (int i = 0; i < TW; ++i)
#pragma unroll
      for (int s = 0; s < REC_CHUNK / 4; ++s)  // (past the last group of elements, or the chunk's end: others, whose results are not stored or which count as zero)
        k[i][s] = a.x[(size_t)(first + min(4 * s + g, count - 1)) * a.ld + a.k_off + h * D + min((wave + 4 * i) * 16 + r, D - 1)];
    v.put(V, ES, count, a.act);
  } else {
#pragma unroll
    for (int i = 0; i < TW; ++i)
#pragma unroll
      for (int s = 0; s < REC_CHUNK / 4; ++s) {
        const int j = 4 * s + g, d = (wave + 4 * i) * 16 + r;
        k[i][s] = j < count && d < D ? a.x[(size_t)(first + j) * a.ld + a.k_off + h * D + d] : 0.f;
      }
    for (int i = tid; i < REC_CHUNK * (ES / 4); i += 256) {
      const int j = i / (ES / 4), e = (i % (ES / 4)) * 4;
      const floatx4 v = j < count ? load4(a.x + (size_t)(first + j) * a.ld + a.v_off + h * E, e, E, vec_v) : floatx4{0.f, 0.f, 0.f, 0.f};
      *reinterpret_cast<floatx4*>(V + j * ES + e) = rec_act4(v, a.act);
    }
  }
  chunk_gates(a, gate_in, count, gi, bs);
  __syncthreads();
  const double B = bs[count - 1];
  const bool gates = a.mode == MS_REC_EXP_GATES;
  float amax = 0.f;
  if (gates) {  // every wave finds the chunk's maximum for itself
    float w = lane < count ? (float)(B - bs[lane]) + gi[lane] : -INFINITY;
    amax = wave_max(w);
  }
  if (tid < REC_CHUNK) wt[tid] = tid < count ? expf((float)(B - bs[tid]) + gi[tid] - amax) : 0.f;
  __syncthreads();
  floatx4 acc[TW][EH][4];
#pragma unroll
  for (int i = 0; i < TW; ++i)
#pragma unroll
    for (int e = 0; e < EH; ++e)
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[i][e][q] = floatx4{0.f, 0.f, 0.f, 0.f};
  float ksum[TW];
#pragma unroll
  for (int i = 0; i < TW; ++i) ksum[i] = 0.f;
#pragma unroll
  for (int s = 0; s < REC_CHUNK / 4; ++s) {
    if (4 * s >= count) continue;
    const float w = wt[4 * s + g];
    floatx4 v[EH];
#pragma unroll
    for (int e = 0; e < EH; ++e) v[e] = *reinterpret_cast<const floatx4*>(V + (4 * s + g) * ES + e * 64 + 4 * r);
#pragma unroll
    for (int i = 0; i < TW; ++i) {
      const float kw = w * (4 * s + g < count ? rec_act(k[i][s], a.act) : 0.f);  // (zero times an infinite key would be no number)
      ksum[i] += kw;
#pragma unroll
      for (int e = 0; e < EH; ++e)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[i][e][q] = __builtin_amdgcn_mfma_f32_16x16x4f32(kw, v[e][q], acc[i][e][q], 0, 0, 0);
    }
  }
  const size_t at = (size_t)blockIdx.x * a.H + h;
  const bool vec = E % 4 == 0;
#pragma unroll
  for (int i = 0; i < TW; ++i) {
    const int d0 = (wave + 4 * i) * 16;
    if (gates) {
      const float sum = rows4_sum(ksum[i]);
      if (g == 0 && d0 + r < D) c.u[at * D + d0 + r] = sum;
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int d = d0 + 4 * g + x;
      if (d >= D) continue;
#pragma unroll
      for (int e = 0; e < EH; ++e)
        store4(c.U + (at * D + d) * E, e * 64 + 4 * r, E, vec, floatx4{acc[i][e][0][x], acc[i][e][1][x], acc[i][e][2][x], acc[i][e][3][x]});
    }
  }
  if (tid == 0) {
    double* o = c.cs + at * 4;
    o[0] = B;
    o[1] = (double)amax;
  }
}

// Pass 2. grid (rows, H, slices): a thread owns VN consecutive elements of the state and walks the row's chunks with the next
// AHEAD of them under way: each waits for memory once, but they wait together.
template <int VN>
__global__ __launch_bounds__(256) void rec_chunk_scan_kernel(ChunkArgs c) {
  constexpr int AHEAD = 8;
  struct alignas(VN * 4) Vec { float e[VN]; };
  const RecurrenceArgs& a = c.r;
  const int b = blockIdx.x, h = blockIdx.y, z = blockIdx.z, tid = threadIdx.x;
  const int DE = a.D * a.E;
  int base = 0;
  for (int r = 0; r < b; ++r) base += (a.row_start[r + 1] - a.row_start[r] + REC_CHUNK - 1) / REC_CHUNK;
  const int nc = (a.row_start[b + 1] - a.row_start[b] + REC_CHUNK - 1) / REC_CHUNK;
  const bool fresh = a.starts[b] == 0;
  const bool gates = a.mode == MS_REC_EXP_GATES;
  const size_t slot = (size_t)a.state_slots[b];
  const int idx = (z * 256 + tid) * VN;
  const bool own = idx < DE;
  float* Sg = a.S + (slot * a.H + h) * (size_t)DE + idx;
  Vec S, next[AHEAD];
#pragma unroll
  for (int i = 0; i < VN; ++i) S.e[i] = 0.f;
  if (own && !fresh) S = *reinterpret_cast<const Vec*>(Sg);
  const bool own_n = gates && z == 0 && tid < a.D;
  float nv = (own_n && !fresh) ? a.n[(slot * a.H + h) * a.D + tid] : 0.f;
  double m = (gates && !fresh) ? (double)a.m[slot * a.H + h] : 0.0;
  double bn[AHEAD], an[AHEAD];
  float un[AHEAD];
  auto fetch = [&](int k, int u) __attribute__((always_inline)) {
    const size_t at = (size_t)(base + min(k, nc - 1)) * a.H + h;  // (beyond the last chunk: read again, not used)
    if (own) next[u] = *reinterpret_cast<const Vec*>(c.U + at * DE + idx);
    bn[u] = c.cs[at * 4];
    an[u] = c.cs[at * 4 + 1];
    un[u] = own_n ? c.u[at * a.D + tid] : 0.f;
  };
  for (int k0 = 0; k0 < nc; k0 += AHEAD) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) fetch(k0 + u, u);
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      if (k0 + u >= nc) continue;
      const size_t at = (size_t)(base + k0 + u) * a.H + h;
      float alpha, beta;
      if (gates) {
        const double m_new = fmax(bn[u] + m, an[u]);
        alpha = expf((float)(bn[u] + m - m_new));
        beta = expf((float)(an[u] - m_new));
        if (z == 0 && tid == 0) c.cs[at * 4 + 2] = m;
        m = m_new;
      } else {
        alpha = expf((float)bn[u]);
        beta = 1.f;
      }
      if (own) *reinterpret_cast<Vec*>(c.U + at * DE + idx) = S;
#pragma unroll
      for (int i = 0; i < VN; ++i) S.e[i] = alpha * S.e[i] + beta * next[u].e[i];
      if (own_n) {
        c.u[at * a.D + tid] = nv;
        nv = alpha * nv + beta * un[u];
      }
    }
  }
  if (own) *reinterpret_cast<Vec*>(Sg) = S;
  if (own_n) a.n[(slot * a.H + h) * a.D + tid] = nv;
  // (not into the state yet: a block of another slice may not have read the old one; the third pass puts it there)
  if (gates && z == 0 && tid == 0 && nc > 0) c.cs[((size_t)(base + nc - 1) * a.H + h) * 4 + 3] = m;
}

// Pass 3. A wave owns 16 of the chunk's tokens; lane (g, r) holds token r's queries 32 s + 8 g + j, its scores of keys 16 tb + 4 g + x,
// and its outputs. Keys (rows KS apart, so that 16 rows touch every bank once) and values go through LDS, the state before the
// chunk comes straight from memory, a run of 32 rows ahead.
template <int DS, int EH>
constexpr size_t rec_output_lds() { return sizeof(float) * (REC_CHUNK * (DS * 32 + 4) + REC_CHUNK * EH * 64); }

template <int DS, int EH, bool FULL>
__global__ __launch_bounds__(256, 2) void rec_chunk_output_kernel(ChunkArgs c, bool vec_qk, bool vec_v) {
  constexpr int KS = DS * 32 + 4, ES = EH * 64;
  extern __shared__ __attribute__((aligned(16))) float sm[];
  float* K = sm;                    // [REC_CHUNK][KS]
  float* V = K + REC_CHUNK * KS;    // [REC_CHUNK][ES]
  __shared__ double bs[REC_CHUNK];
  __shared__ float gi[REC_CHUNK], mt[REC_CHUNK];
  const RecurrenceArgs& a = c.r;
  const int D = a.D, E = a.E, h = blockIdx.y, tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE;
  const int r = lane % 16, g = lane / 16;
  int row, first, count, base;
  find_chunk(a.row_start, c.rows, blockIdx.x, &row, &first, &count, &base);
  const bool gates = a.mode == MS_REC_EXP_GATES;
  const size_t at = (size_t)blockIdx.x * a.H + h;
  const double m0 = gates ? c.cs[at * 4 + 2] : 0.0;
  if (gates && tid == 0 && first + count == a.row_start[row + 1]) a.m[(size_t)a.state_slots[row] * a.H + h] = (float)c.cs[at * 4 + 3];
  const int t = wave * 16 + r;  // this lane's token
  const GateInputs gate_in = load_gates(a, h, first, count);
  const float* S0 = c.U + at * (size_t)D * E;
  const bool vec_s = E % 4 == 0;
  floatx4 state[2][8][EH];
  auto fetch = [&](int s) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int e = 0; e < EH; ++e) {
        const int d = s * 32 + 8 * g + j;
        if constexpr (FULL) state[s % 2][j][e] = *reinterpret_cast<const floatx4*>(S0 + (size_t)d * E + e * 64 + 4 * r);
        else state[s % 2][j][e] = d < D ? load4(S0 + (size_t)d * E, e * 64 + 4 * r, E, vec_s) : floatx4{0.f, 0.f, 0.f, 0.f};
      }
  };
  float q[DS][8];
  const float* qr = a.x + (size_t)(first + (t < count ? t : 0)) * a.ld + a.q_off + h * D;
  if constexpr (FULL) {
    floatx4 qv[DS][2];
    ChunkRows<DS * 8> kv;
    ChunkRows<ES / 4> vv;
#pragma unroll
    for (int s = 0; s < DS; ++s)
#pragma unroll
      for (int u = 0; u < 2; ++u) qv[s][u] = *reinterpret_cast<const floatx4*>(qr + s * 32 + 8 * g + 4 * u);
    kv.load(a, first, count, a.k_off + h * D);
    vv.load(a, first, count, a.v_off + h * E);
    fetch(0);
    kv.put(K, KS, count, a.act);
    vv.put(V, ES, count, a.act);
    if (a.act) {
#pragma unroll
      for (int s = 0; s < DS; ++s)
#pragma unroll
        for (int u = 0; u < 2; ++u) qv[s][u] = rec_act4(qv[s][u], a.act);
    }
#pragma unroll
    for (int s = 0; s < DS; ++s)
#pragma unroll
      for (int i = 0; i < 8; ++i) q[s][i] = t < count ? qv[s][i / 4][i % 4] * a.q_scale : 0.f;
  } else {
#pragma unroll
    for (int s = 0; s < DS; ++s)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const floatx4 v = rec_act4(t < count ? load4(qr, s * 32 + 8 * g + 4 * u, D, vec_qk) : floatx4{0.f, 0.f, 0.f, 0.f}, a.act);
#pragma unroll
        for (int i = 0; i < 4; ++i) q[s][4 * u + i] = v[i] * a.q_scale;
      }
    for (int i = tid; i < REC_CHUNK * DS * 8; i += 256) {
      const int j = i / (DS * 8), d = (i % (DS * 8)) * 4;
      const floatx4 v = j < count ? load4(a.x + (size_t)(first + j) * a.ld + a.k_off + h * D, d, D, vec_qk) : floatx4{0.f, 0.f, 0.f, 0.f};
      *reinterpret_cast<floatx4*>(K + j * KS + d) = rec_act4(v, a.act);
    }
    for (int i = tid; i < REC_CHUNK * (ES / 4); i += 256) {
      const int j = i / (ES / 4), e = (i % (ES / 4)) * 4;
      const floatx4 v = j < count ? load4(a.x + (size_t)(first + j) * a.ld + a.v_off + h * E, e, E, vec_v) : floatx4{0.f, 0.f, 0.f, 0.f};
      *reinterpret_cast<floatx4*>(V + j * ES + e) = rec_act4(v, a.act);
    }
    fetch(0);
  }
  chunk_gates(a, gate_in, count, gi, bs, mt, m0);

  // what the state before the chunk gives
  floatx4 acc[EH][4];
#pragma unroll
  for (int e = 0; e < EH; ++e)
#pragma unroll
    for (int u = 0; u < 4; ++u) acc[e][u] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < DS; ++s) {
    if (s + 1 < DS) fetch(s + 1);
    __builtin_amdgcn_sched_barrier(0);  // else the loads move down to their use
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int e = 0; e < EH; ++e)
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[e][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(state[s % 2][j][e][u], q[s][j], acc[e][u], 0, 0, 0);
  }
  __syncthreads();  // the gates, which the first wave made while the others were at the products above, and keys and values
  const double bt = bs[t];
  const float m = mt[t];
  const float from_before = expf((float)(bt + m0 - (double)m));
#pragma unroll
  for (int e = 0; e < EH; ++e)
#pragma unroll
    for (int u = 0; u < 4; ++u) acc[e][u] *= from_before;
  float n_dot = 0.f;
  if (gates) {
    const float* n0 = c.u + at * D;
#pragma unroll
    for (int s = 0; s < DS; ++s)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int d = s * 32 + 8 * g + j;
        if (FULL || d < D) n_dot = fmaf(n0[d], q[s][j], n_dot);
      }
    n_dot *= from_before;
  }
  // the chunk's own keys, 16 at a time, up to the wave's tokens
  for (int tb = 0; tb <= wave; ++tb) {
    if (tb * 16 >= count) break;
    floatx4 p = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      const float* kr = K + (tb * 16 + r) * KS + s * 32 + 8 * g;
      const floatx4 k0 = *reinterpret_cast<const floatx4*>(kr), k1 = *reinterpret_cast<const floatx4*>(kr + 4);
#pragma unroll
      for (int j = 0; j < 8; ++j) p = __builtin_amdgcn_mfma_f32_16x16x4f32(j < 4 ? k0[j] : k1[j - 4], q[s][j], p, 0, 0, 0);
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int j = tb * 16 + 4 * g + x;
      p[x] = j <= t && t < count ? p[x] * expf((float)(bt - bs[j]) + gi[j] - m) : 0.f;
      n_dot += p[x];
    }
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int e = 0; e < EH; ++e) {
        const floatx4 v = *reinterpret_cast<const floatx4*>(V + (tb * 16 + 4 * g + x) * ES + e * 64 + 4 * r);
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[e][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[u], p[x], acc[e][u], 0, 0, 0);
      }
  }
  float inv = 1.f;
  if (gates) inv = 1.f / (fmaxf(fabsf(rows4_sum(n_dot)), expf(-m)) + 1e-6f);
  if (t >= count) return;
  float* o = a.out + (size_t)(first + t) * (a.H * E) + h * E;
#pragma unroll
  for (int e = 0; e < EH; ++e)
#pragma unroll
    for (int x = 0; x < 4; ++x)
      store4(o, e * 64 + 16 * g + 4 * x, E, vec_s, floatx4{acc[e][0][x], acc[e][1][x], acc[e][2][x], acc[e][3][x]} * inv);
}

template <int DS, int EH>
static int launch_rec_chunks(const ChunkArgs& c, int chunks, hipStream_t st) {
  const RecurrenceArgs& a = c.r;
  constexpr size_t lds = rec_output_lds<DS, EH>();
  static bool ready = false;
  if (!ready) {
    for (const void* fn : {(const void*)rec_chunk_output_kernel<DS, EH, true>, (const void*)rec_chunk_output_kernel<DS, EH, false>})
      if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) return MS_LAUNCH_FAILED;
    ready = true;
  }
  const bool rows = (size_t)a.x % 16 == 0 && a.ld % 4 == 0;  // rows 16-byte aligned; then the heads' columns have to be
  const bool vec_qk = rows && a.D % 4 == 0 && a.q_off % 4 == 0 && a.k_off % 4 == 0, vec_v = rows && a.E % 4 == 0 && a.v_off % 4 == 0;
  const bool full = a.D == DS * 32 && a.E == EH * 64 && vec_qk && vec_v;
  if (full) rec_chunk_summary_kernel<DS, EH, true><<<dim3(chunks, a.H), 256, 0, st>>>(c, vec_v);
  else rec_chunk_summary_kernel<DS, EH, false><<<dim3(chunks, a.H), 256, 0, st>>>(c, vec_v);
  const int DE = a.D * a.E;
  if (DE % 4 == 0) rec_chunk_scan_kernel<4><<<dim3(c.rows, a.H, (DE + 1023) / 1024), 256, 0, st>>>(c);
  else rec_chunk_scan_kernel<1><<<dim3(c.rows, a.H, (DE + 255) / 256), 256, 0, st>>>(c);
  if (full) rec_chunk_output_kernel<DS, EH, true><<<dim3(chunks, a.H), 256, lds, st>>>(c, vec_qk, vec_v);
  else rec_chunk_output_kernel<DS, EH, false><<<dim3(chunks, a.H), 256, lds, st>>>(c, vec_qk, vec_v);
  return launch_status();
}

// Floats of scratch per chunk and head that ms_gated_recurrence_chunked needs for U; u takes D and cs 4 per chunk and head.
extern "C" int ms_gated_recurrence_chunk_tokens() { return REC_CHUNK; }
extern "C" int ms_gated_recurrence_chunk_max_dim() { return REC_CHUNK_MAX_DIM; }

// As ms_gated_recurrence, in chunks. `chunks` = sum over the rows of ceil(tokens / REC_CHUNK) (the host knows the rows'
// lengths); U [chunks, H, D * E], u [chunks, H, D] (float) and cs [chunks, H, 4] (double) are scratch.
extern "C" int ms_gated_recurrence_chunked(const float* x, int ld, int q_off, int k_off, int v_off, int i_off, int f_off, int H, int D,
                                           int E, int act, int mode, float q_scale, float cap, const float* decay,
                                           const void* i_bias, const void* f_bias, int bias_is_bf16, float* S, float* n, float* m,
                                           const int* row_start, const int* starts, const int* state_slots, float* out, int rows,
                                           int chunks, float* U, float* u, double* cs, hipStream_t st) {
  if (rows <= 0 || chunks <= 0) return MS_OK;
  if (H <= 0 || D <= 0 || E <= 0 || x == nullptr || S == nullptr || out == nullptr || row_start == nullptr || starts == nullptr ||
      state_slots == nullptr || U == nullptr || cs == nullptr || (act != 0 && act != 1) || q_off < 0 || k_off < 0 || v_off < 0 ||
      q_off + H * D > ld || k_off + H * D > ld || v_off + H * E > ld)
    return MS_BAD_ARG;
  if (mode == MS_REC_DECAY) {
    if (decay == nullptr) return MS_BAD_ARG;
  } else if (mode == MS_REC_EXP_GATES) {
    if (n == nullptr || m == nullptr || u == nullptr || !(cap > 0.f) || i_off < 0 || f_off < 0 || i_off + H > ld || f_off + H > ld)
      return MS_BAD_ARG;
  } else {
    return MS_BAD_ARG;
  }
  if (D > REC_CHUNK_MAX_DIM || E > REC_CHUNK_MAX_DIM || H > 65535 || rows > 65535) return MS_UNSUPPORTED;
  ChunkArgs c{{x, ld, q_off, k_off, v_off, i_off, f_off, H, D, E, act, mode, q_scale, cap, decay, i_bias, f_bias, bias_is_bf16, S, n,
               m, row_start, starts, state_slots, out},
              U, u, cs, rows};
  const int ds = (D + 31) / 32;
  if (E <= 64) {
    if (ds == 1) return launch_rec_chunks<1, 1>(c, chunks, st);
    if (ds == 2) return launch_rec_chunks<2, 1>(c, chunks, st);
    if (ds == 3) return launch_rec_chunks<3, 1>(c, chunks, st);
    return launch_rec_chunks<4, 1>(c, chunks, st);
  }
  if (ds == 1) return launch_rec_chunks<1, 2>(c, chunks, st);
  if (ds == 2) return launch_rec_chunks<2, 2>(c, chunks, st);
  if (ds == 3) return launch_rec_chunks<3, 2>(c, chunks, st);
  return launch_rec_chunks<4, 2>(c, chunks, st);
}
