// True float32 matrix product C[M, N] = A[M, K] * W[N, K]^T on the matrix cores' 32-bit form
// (v_mfma_f32_16x16x4_f32: float32 operands, products and sums; no reduced precision).
//
// Every output element is the sum of at most sixteen partial sums, added in ascending order to zero; partial sum c covers
// k = c * chunk .. (c + 1) * chunk - 1 with chunk = 64 * ceil(K / 1024), as one accumulator's chain over slabs of 32 k in
// ascending order and, inside a slab, over j = 0 .. 7 of the four products k = 8 g + j, g = 0 .. 3. That order depends on K
// alone. Both kernels below keep it, so results do not depend on how rows are batched.
//
// Operand roles as in the bfloat16 products: the weight rows are the A operand (row index i = n), the activation rows the B
// operand (column index j = m), so a lane holds four consecutive n of one m. Layout of v_mfma_f32_16x16x4_f32 (lane l,
// g = l / 16, r = l % 16): A operand A[i = r][k = g], B operand B[k = g][j = r], result D[i = 4 g + 0..3][j = r]. A lane reads
// the eight consecutive k = 8 g .. 8 g + 7 of its row with two 16-byte loads and feeds them to eight products in turn.
//
//  * few rows (gemm_f32_few_kernel): what bounds it is the weights' bytes. A block owns 16 weight rows and up to 32 rows of
//    A; each of its waves streams one chunk of K straight from global memory into registers, or, where STREAM has it, through LDS, all
//    of it asked for before the first product where the chunk is short (K up to 3072), and the waves' partial sums meet in LDS.
//    6 rows x 1,024 x 3,072: 11.7 us, 1.1 TB/s (tiles of 64 x 64 on the vector units, which this replaces: 189 us); through LDS
//    6 rows x 4,096 x 1,024: 5.8 us (registers 7.3); 6 rows x 151,936 x 1,024: 100 us, 6.2 TB/s (134; vector units 261).
//  * many rows (gemm_f32_rows_kernel): tiles of 16 to 128 rows x 64, bound by the matrix cores (157 TFLOP/s nominal). Against the
//    kernel below, which these products ran in: 1,068 x 4,096 x 1,024 115 -> 86 us, 1,068 x 1,024 x 3,072 119 -> 67, 300 x 1,024 x
//    3,072 68 -> 33, 2,120 x 6,144 x 4,096 1,039 -> 892 (120 TFLOP/s), 2,048 x 6,144 x 1,024 214 -> 216.
//  * many rows, other K or alignment, or a short K (gemm_f32_tile_kernel): tiles of 64 x 64 or 128 x 128, slabs of 32 k with a last
//    one cut off, two blocks a CU.
// f32_few_rows and f32_tile_height have the lines between them.
#include "common.h"

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

#define F32_SLAB 32
#define F32_CHUNKS 16  // partial sums of an output element, at most

static __host__ __device__ __forceinline__ int f32_chunk(int K) { return 64 * ((K + 1023) / 1024); }

__device__ __forceinline__ float f32_at(const float4& lo, const float4& hi, int j) {
  return j == 0 ? lo.x : j == 1 ? lo.y : j == 2 ? lo.z : j == 3 ? lo.w : j == 4 ? hi.x : j == 5 ? hi.y : j == 6 ? hi.z : hi.w;
}

// mode 0: C = sum (float)   mode 1: C += sum (float)   mode 2: C = bf16(sum)
__device__ __forceinline__ void f32_store(void* __restrict__ C, int mode, size_t at, float v) {
  if (mode == 0) ((float*)C)[at] = v;
  else if (mode == 1) ((float*)C)[at] += v;
  else ((bf16*)C)[at] = static_cast<bf16>(v);
}

// ---------------------------------------------------------------------------------------------
// MT: 16-row groups of A a block owns (gridDim.y blocks share the rows of A). One wave per chunk of K.
// SLABS > 0: K is a multiple of 64, rows are 16-byte aligned and a chunk has at most SLABS slabs: all of a wave's loads go out
// at once, in straight code (a load behind a test of its own k is a branch, and the compiler waits between them). SLABS = 0:
// the same with a chunk of any length, two slabs at a time, the next two under way. SLABS < 0: any K, any alignment.
// PARTS: a block is one wave, blockIdx.z its chunk, and the partial sums go to C [chunks, M, N] for the next kernel to add.
// STREAM (SLABS > 0): the weights come through LDS. A lane's operand is 16 bytes of one row, so a load into registers touches sixteen rows;
// a load into LDS takes whole lines of 128 bytes and may say that they are read once (ONCE: one block reads them), which a stream of
// them is 10 to 20 % faster by. All of a wave's slabs are under way at once, as in registers.
template <int MT, int SLABS, bool PARTS = false, bool STREAM = false, bool ONCE = false>
__global__ __launch_bounds__(PARTS ? WAVE : F32_CHUNKS * WAVE) void gemm_f32_few_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                                         void* __restrict__ C, int mode, int M, int N, int K, int lda,
                                                                         int ldc, int chunk) {
  static_assert(!STREAM || SLABS > 0, "");
  constexpr int SUMS = MT * 16 * 17;  // floats a wave leaves for the block's other threads: [MT * 16][16 + 1]
  constexpr int RING = SLABS * 16 * 128;  // STREAM: bytes of a wave's slabs, 16 rows of 128 each; its sums take their place
  static_assert(!STREAM || PARTS || SUMS * 4 <= RING, "");
  __shared__ float parts[PARTS || STREAM ? 1 : F32_CHUNKS * SUMS];
  extern __shared__ __attribute__((aligned(1024))) unsigned char few_ring[];
  auto sums_of = [&](int w) { return STREAM ? reinterpret_cast<float*>(few_ring + w * RING) : parts + w * SUMS; };
  constexpr int SET = SLABS > 0 ? SLABS : SLABS == 0 ? 2 : 1, SETS = SLABS == 0 ? 2 : 1;  // slabs whose loads go out together
  const int wave = PARTS ? blockIdx.z : __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
  const int r = lane % 16, g = lane / 16;
  const int n0 = blockIdx.x * 16, m0 = blockIdx.y * (MT * 16);
  const int k_lo = wave * chunk, k_hi = min(K, k_lo + chunk);
  const float* wrow = W + (size_t)min(n0 + r, N - 1) * K + 8 * g;  // rows beyond the edge repeat the last one and are not stored
  const float* arow[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) arow[i] = A + (size_t)min(m0 + i * 16 + r, M - 1) * lda + 8 * g;

  floatx4 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};
  float4 w[SETS][SET][2], a[SETS][SET][MT][2];
  auto load8 = [&](const float* row, int k, float4 (&to)[2]) __attribute__((always_inline)) {
    if constexpr (SLABS >= 0) {
      to[0] = *reinterpret_cast<const float4*>(row + k);
      to[1] = *reinterpret_cast<const float4*>(row + k + 4);
    } else {
      float e[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) e[i] = k + 8 * g + i < k_hi ? row[k + i] : 0.f;
      to[0] = make_float4(e[0], e[1], e[2], e[3]);
      to[1] = make_float4(e[4], e[5], e[6], e[7]);
    }
  };
  auto fetch = [&](int set, int s, int k) __attribute__((always_inline)) {
    load8(wrow, k, w[set][s]);
#pragma unroll
    for (int i = 0; i < MT; ++i) load8(arow[i], k, a[set][s][i]);
  };
  auto multiply = [&](int set, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int i = 0; i < MT; ++i)
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(f32_at(w[set][s][0], w[set][s][1], j), f32_at(a[set][s][i][0], a[set][s][i][1], j),
                                                      acc[i], 0, 0, 0);
  };
  if constexpr (STREAM) {
    unsigned char* ring = few_ring + (PARTS ? 0 : wave * RING);
    // A's rows first: they come from the cache, and loads come back in the order in which they went out.
#pragma unroll
    for (int s = 0; s < SLABS; ++s)
#pragma unroll
      for (int i = 0; i < MT; ++i) load8(arow[i], min(k_lo + s * F32_SLAB, k_hi - F32_SLAB), a[0][s][i]);
#pragma unroll
    for (int s = 0; s < SLABS; ++s)
#pragma unroll
      for (int j = 0; j < 2; ++j) {  // eight rows a load; 16-byte piece c of row R lies in slot c ^ ((R >> 1) & 7)
        const int R = j * 8 + lane / 8, c = (lane % 8) ^ ((R >> 1) & 7);
        const float* src = W + (size_t)min(n0 + R, N - 1) * K + min(k_lo + s * F32_SLAB, k_hi - F32_SLAB) + c * 4;
        __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)src,
                                         (void __attribute__((address_space(3)))*)(ring + s * 2048 + j * 1024), 16, 0, ONCE ? LOAD_ONCE : 0);
      }
    auto slab = [&](int s) __attribute__((always_inline)) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        union { floatx4 v; float4 f; } x;
        x.v = *reinterpret_cast<const floatx4*>(ring + s * 2048 + r * 128 + (((2 * g + h) ^ (r >> 1)) * 16));
        w[0][s][h] = x.f;
      }
      if (k_lo + s * F32_SLAB < k_hi) multiply(0, s);
    };
    // For all slabs at once: behind global loads into LDS the compiler makes the wait for a register, here one of A's, a wait for
    // every load. A's rows pass through the statements below, or the compiler moves the first slab's loads into the branch of their
    // use, behind the wait (6 rows, us, so and as it is: x 4,096 x 1,024 6.2, 5.8; x 3,072 x 1,024 5.6, 5.2; x 2,048 x 1,024 in parts 4.2, 4.1).
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < SLABS; ++s)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) asm volatile("" : "+v"(reinterpret_cast<floatx4&>(a[0][s][i][h])));
#pragma unroll
    for (int s = 0; s < SLABS; ++s) slab(s);
  } else if constexpr (SLABS > 0) {
#pragma unroll
    for (int s = 0; s < SLABS; ++s) fetch(0, s, min(k_lo + s * F32_SLAB, k_hi - F32_SLAB));  // (the last chunk may be shorter)
#pragma unroll
    for (int s = 0; s < SLABS; ++s)
      if (k_lo + s * F32_SLAB < k_hi) multiply(0, s);
  } else if constexpr (SLABS == 0) {
    constexpr int STEP = 2 * F32_SLAB;
    fetch(0, 0, k_lo);
    fetch(0, 1, k_lo + F32_SLAB);
    for (int k0 = k_lo; k0 < k_hi; k0 += 2 * STEP) {
      const int k1 = min(k0 + STEP, k_hi - STEP), k2 = min(k0 + 2 * STEP, k_hi - STEP);  // beyond the chunk: loaded again, not used
      fetch(1, 0, k1);
      fetch(1, 1, k1 + F32_SLAB);
      multiply(0, 0);
      multiply(0, 1);
      fetch(0, 0, k2);
      fetch(0, 1, k2 + F32_SLAB);
      if (k0 + STEP < k_hi) {
        multiply(1, 0);
        multiply(1, 1);
      }
    }
  } else {
    for (int k0 = k_lo; k0 < k_hi; k0 += F32_SLAB) {  // from K on there are zeros: they change nothing
      fetch(0, 0, k0);
      multiply(0, 0);
    }
  }
  if constexpr (PARTS) {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int m = m0 + i * 16 + r, n = n0 + 4 * g;
      if (m >= M) continue;
      float* to = (float*)C + ((size_t)wave * M + m) * N + n;
      if (N % 4 == 0) {
        if (n < N) *reinterpret_cast<floatx4*>(to) = acc[i];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) to[e] = acc[i][e];
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) sums_of(wave)[(i * 16 + r) * 17 + 4 * g + e] = acc[i][e];
  __syncthreads();
  const int chunks = blockDim.x / WAVE;
  for (int o = threadIdx.x; o < MT * 256; o += blockDim.x) {
    const int m = o / 16, n = o % 16;
    if (m0 + m >= M || n0 + n >= N) continue;
    float sum = 0.f;
    for (int c = 0; c < chunks; ++c) sum += sums_of(c)[m * 17 + n];
    f32_store(C, mode, (size_t)(m0 + m) * ldc + n0 + n, sum);
  }
}

// The gated feed-forward's input for up to 16 rows in one kernel: out[m, i] = act(x . gate_i) * (x . up_i) for W [2 inter, K] of
// alternating runs of 16 gate rows and 16 up rows. A block owns one run of each and all of K, a wave a chunk of 64 k for both, as in
// the kernel above with STREAM; the sums are the same ones, and so are the products' activations: what it spares is the launch and the
// trip of the product through memory (3,072 outputs of 1,024, us in two kernels and in one: 1 row 11.2, 8.0; 6 rows 10.5, 8.0; 16 rows 11.1,
// 8.4).
__global__ __launch_bounds__(F32_CHUNKS * WAVE) void gemm_f32_few_gated_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                                               float* __restrict__ out, int M, int inter, int K, int lda,
                                                                               int act, float limit) {
  constexpr int SLABS = 2, SUMS = 16 * 17, RING = 2 * SLABS * 2048;  // per wave: gate rows' slabs, then up rows'; the sums take their place
  extern __shared__ __attribute__((aligned(1024))) unsigned char gated_ring[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE, r = lane % 16, g = lane / 16;
  const int k_lo = wave * SLABS * F32_SLAB;
  unsigned char* ring = gated_ring + wave * RING;
  const float* arow = A + (size_t)min(r, M - 1) * lda + k_lo + 8 * g;
  float4 a[SLABS][2];
#pragma unroll
  for (int s = 0; s < SLABS; ++s) {
    a[s][0] = *reinterpret_cast<const float4*>(arow + s * F32_SLAB);
    a[s][1] = *reinterpret_cast<const float4*>(arow + s * F32_SLAB + 4);
  }
#pragma unroll
  for (int s = 0; s < SLABS; ++s)
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int R = j * 8 + lane / 8, c = (lane % 8) ^ ((R >> 1) & 7);
        const float* src = W + ((size_t)blockIdx.x * 32 + u * 16 + R) * K + k_lo + s * F32_SLAB + c * 4;
        __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)src,
                                         (void __attribute__((address_space(3)))*)(ring + (u * SLABS + s) * 2048 + j * 1024), 16, 0, LOAD_ONCE);
      }
  floatx4 acc[2] = {floatx4{0.f, 0.f, 0.f, 0.f}, floatx4{0.f, 0.f, 0.f, 0.f}};
  auto slab = [&](int s) __attribute__((always_inline)) {
    float4 w[2][2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        union { floatx4 v; float4 f; } x;
        x.v = *reinterpret_cast<const floatx4*>(ring + (u * SLABS + s) * 2048 + r * 128 + (((2 * g + h) ^ (r >> 1)) * 16));
        w[u][h] = x.f;
      }
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int u = 0; u < 2; ++u)
        acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(f32_at(w[u][0], w[u][1], j), f32_at(a[s][0], a[s][1], j), acc[u], 0, 0, 0);
  };
  // The first slab's products wait for both slabs (as above); what its own wait brings is that its weights are read from LDS while
  // the other slab's come (6 rows, 2,048 outputs of 1,024: 7.0 us, with one wait for both 7.3).
  asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
  slab(0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  slab(1);
  float* sums = reinterpret_cast<float*>(ring);
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int e = 0; e < 4; ++e) sums[u * SUMS + r * 17 + 4 * g + e] = acc[u][e];
  __syncthreads();
  const int chunks = blockDim.x / WAVE;
  for (int o = threadIdx.x; o < 256; o += blockDim.x) {
    const int m = o / 16, n = o % 16;
    if (m >= M) continue;
    float gate = 0.f, up = 0.f;
    for (int c = 0; c < chunks; ++c) {
      const float* of = reinterpret_cast<const float*>(gated_ring + c * RING) + m * 17 + n;
      gate += of[0];
      up += of[SUMS];
    }
    out[(size_t)m * inter + blockIdx.x * 16 + n] = gated_value(gate, up, act, limit);
  }
}

// ---------------------------------------------------------------------------------------------
// B x B tiles, four waves of B / 2 x B / 2. A tile row of a slab is 128 bytes; its 16-byte chunk c lies in slot
// c ^ ((row >> 1) & 7), so a fragment's 16 rows touch every bank once. DMA: rows 16-byte aligned and K a multiple of 4, slabs
// straight into LDS, chunks from K on from four zeros (1,000 x 5,120 x 1,500: 274 -> 154 us); otherwise through registers.
__device__ const float4 f32_zeros = {0.f, 0.f, 0.f, 0.f};
static __host__ __device__ constexpr int f32_stages(int B) { return B == 64 ? 4 : 2; }  // 64 x 64: few blocks, each alone with its loads

template <int B, bool DMA>
__global__ __launch_bounds__(256, 2) void gemm_f32_tile_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                               void* __restrict__ C, int mode, int M, int N, int K, int lda, int ldc,
                                                               int chunk, bool vec_store) {
  constexpr int F = B / 32;                // 16-row fragments of a wave tile, each way
  constexpr int STAGE = 2 * B * 128;       // bytes: B rows of A, then B rows of W
  constexpr int LOADS = B / 32;            // load instructions per wave, operand and slab (eight rows each)
  constexpr int STAGES = f32_stages(B);
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];  // STAGES * STAGE
  const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE;
  const int r = lane % 16, g = lane / 16;
  const int m0 = blockIdx.y * B, n0 = blockIdx.x * B;
  const int wm = (wave / 2) * (B / 2), wn = (wave % 2) * (B / 2);
  const int lrow = lane / 8, lslot = lane % 8;
  const float *asrc[LOADS], *wsrc[LOADS];
  int koff[LOADS];
#pragma unroll
  for (int j = 0; j < LOADS; ++j) {
    const int R = (wave * LOADS + j) * 8 + lrow;
    koff[j] = (lslot ^ ((R >> 1) & 7)) * 4;
    asrc[j] = A + (size_t)min(m0 + R, M - 1) * lda + koff[j];
    wsrc[j] = W + (size_t)min(n0 + R, N - 1) * K + koff[j];
  }
  auto issue = [&](int slab) __attribute__((always_inline)) {
    unsigned char* stage = lds + (slab % STAGES) * STAGE;
    const int k = slab * F32_SLAB;
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      const int at = (wave * LOADS + j) * 1024;
      if constexpr (DMA) {
        // In assembly: behind the builtin the compiler waits for every load under way ahead of the next read of LDS.
        const unsigned to = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(__attribute__((address_space(3))) unsigned char*)(stage + at));
        const float *as = asrc[j] + k, *ws = wsrc[j] + k;
        if (k + F32_SLAB > K && k + koff[j] >= K) as = ws = reinterpret_cast<const float*>(&f32_zeros);
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %3, off"
                     ::"s"(to), "v"(as), "s"(to + B * 128), "v"(ws) : "memory");
      } else {
        float4 a, w;
        float* ae = reinterpret_cast<float*>(&a);
        float* we = reinterpret_cast<float*>(&w);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bool in = k + koff[j] + e < K;
          ae[e] = in ? asrc[j][k + e] : 0.f;
          we[e] = in ? wsrc[j][k + e] : 0.f;
        }
        *reinterpret_cast<float4*>(stage + at + lane * 16) = a;
        *reinterpret_cast<float4*>(stage + B * 128 + at + lane * 16) = w;
      }
    }
  };
  floatx4 acc[F][F], total[F][F];
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) acc[i][j] = total[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int sw = (r >> 1) & 7;
  const int c0 = ((2 * g) ^ sw) * 16, c1 = ((2 * g + 1) ^ sw) * 16;
  const int slabs = (K + F32_SLAB - 1) / F32_SLAB, per_chunk = chunk / F32_SLAB;

#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < slabs) issue(s);
  for (int s = 0; s < slabs; ++s) {
    // This wave's part of slab s has landed (loads return in order; later slabs may still be in flight), and behind the
    // barrier everyone's; everyone has also read the stage that is filled next.
    if (!DMA) __syncthreads();
    else if (s + STAGES - 1 > slabs) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((STAGES - 2) * 2 * LOADS) : "memory");
    if (s + STAGES - 1 < slabs) issue(s + STAGES - 1);
    const unsigned char* stage = lds + (s % STAGES) * STAGE;
    float4 w[F][2], a[F][2];
#pragma unroll
    for (int i = 0; i < F; ++i) {
      const unsigned char* row = stage + B * 128 + (wn + i * 16 + r) * 128;
      w[i][0] = *reinterpret_cast<const float4*>(row + c0);
      w[i][1] = *reinterpret_cast<const float4*>(row + c1);
    }
#pragma unroll
    for (int j = 0; j < F; ++j) {
      const unsigned char* row = stage + (wm + j * 16 + r) * 128;
      a[j][0] = *reinterpret_cast<const float4*>(row + c0);
      a[j][1] = *reinterpret_cast<const float4*>(row + c1);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(f32_at(w[i][0], w[i][1], e), f32_at(a[j][0], a[j][1], e), acc[i][j], 0, 0, 0);
    if ((s + 1) % per_chunk == 0 || s + 1 == slabs) {
#pragma unroll
      for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j) {
          total[i][j] += acc[i][j];
          acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
  }
#pragma unroll
  for (int j = 0; j < F; ++j) {
    const int m = m0 + wm + j * 16 + r;
    if (m >= M) continue;
#pragma unroll
    for (int i = 0; i < F; ++i) {
      const int n = n0 + wn + i * 16 + 4 * g;
      const size_t at = (size_t)m * ldc + n;
      const floatx4 v = total[i][j];
      if (vec_store && mode != 2 && n + 3 < N) {
        float4 o = make_float4(v[0], v[1], v[2], v[3]);
        if (mode == 1) {
          const float4 c = *reinterpret_cast<const float4*>((const float*)C + at);
          o = make_float4(c.x + o.x, c.y + o.y, c.z + o.z, c.w + o.w);
        }
        *reinterpret_cast<float4*>((float*)C + at) = o;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) f32_store(C, mode, at + e, v[e]);
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Many rows, K a multiple of 32 and rows 16-byte aligned: tiles of 16 FM rows x 64 columns, one block a CU, a wave 16 columns. The
// products bound it (256 FM clocks a slab; fragment reads take LDS a third of that), so a tile may have any height in steps of 16,
// and f32_tile_height takes the one that leaves the least of the chip idle in the last round. With one wave per SIMD nothing covers a
// wait but the wave's own order: slabs come straight into a ring of LDS stages, four or more under way; the eight k of a lane are
// two sets of fragments, one multiplied while the other is read; a slab's place is loaded anew, an instruction at a time between
// the products, when every wave has read its second set.
static __host__ __device__ constexpr int f32_ring(int FM) { return (84 * 1024 + (FM * 16 + 64) * 128 - 1) / ((FM * 16 + 64) * 128); }  // more than half a CU's LDS

// Block barrier after which at most n slabs of LOADS loads each are in flight, n up to MOST, and this wave's LDS reads have returned.
template <int MOST, int LOADS>
__device__ __forceinline__ void f32_wait_slabs(int n) {
  if constexpr (MOST > 0) {
    if (n < MOST) return f32_wait_slabs<MOST - 1, LOADS>(n);
  }
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(MOST * LOADS) : "memory");
}

template <int FM>
__global__ __launch_bounds__(256, 2) void gemm_f32_rows_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                               void* __restrict__ C, int mode, int M, int N, int K, int lda, int ldc,
                                                               int chunk, bool vec_store) {
  constexpr int BM = 16 * FM, STAGE = (BM + 64) * 128, STAGES = f32_ring(FM);
  constexpr int INSTR = 2 * FM + 8, LOADS = (INSTR + 3) / 4;  // load instructions of a slab (eight rows each), of a wave
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];  // STAGES * STAGE: BM rows of A, then 64 of W
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
  const int r = lane % 16, g = lane / 16;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * 64;
  const float* src[LOADS];  // this lane's part of the next slab to load
#pragma unroll
  for (int j = 0; j < LOADS; ++j) {
    const int i = min(wave + 4 * j, INSTR - 1);  // (the last may be loaded by several waves, the same bytes to the same place)
    const int R = i * 8 + lane / 8;
    src[j] = (i < 2 * FM ? A + (size_t)min(m0 + R, M - 1) * lda : W + (size_t)min(n0 + R - BM, N - 1) * K) + ((lane % 8) ^ ((R >> 1) & 7)) * 4;
  }
  auto issue_one = [&](int stage, int j) __attribute__((always_inline)) {
    __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)src[j],
                                     (void __attribute__((address_space(3)))*)(lds + stage + min(wave + 4 * j, INSTR - 1) * 1024), 16, 0, 0);
    src[j] += F32_SLAB;
  };
  floatx4 acc[FM], total[FM];
#pragma unroll
  for (int i = 0; i < FM; ++i) acc[i] = total[i] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int sw = (r >> 1) & 7;
  const unsigned char *w_row = lds + (BM + wave * 16 + r) * 128, *a_row = lds + r * 128;
  const int off[2] = {((2 * g) ^ sw) * 16, ((2 * g + 1) ^ sw) * 16};
  const int slabs = K / F32_SLAB, per_chunk = chunk / F32_SLAB;
  floatx4 w[2], a[2][FM];
  auto read_one = [&](int set, int stage, int q) __attribute__((always_inline)) {
    if (q == 0) w[set] = *reinterpret_cast<const floatx4*>(w_row + (stage + off[set]));
    else a[set][q > 0 ? q - 1 : 0] = *reinterpret_cast<const floatx4*>(a_row + (stage + off[set]) + (q - 1) * 16 * 128);
  };
  // The products of one set, k = 8 g + 4 set + 0 .. 3; between them the reads of the other set and, in a slab's second half, the
  // loads. fresh: a chunk begins, and the sums of the one before join the total while its first products run.
  auto step = [&](int set, int read_stage, int load_stage, bool loads, bool fresh) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < 4 * FM; ++p) {
      if (fresh && p < FM) {
        const floatx4 before = acc[p % FM];
        acc[p % FM] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[set][0], a[set][p % FM][0], floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        total[p % FM] += before;
      } else {
        acc[p % FM] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[set][p / FM], a[set][p % FM][p / FM], acc[p % FM], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (p < FM + 1) read_one(1 - set, read_stage, p);
      if (loads) {
#pragma unroll
        for (int j = 0; j < LOADS; ++j)
          if (j * 4 * FM / LOADS == p) issue_one(load_stage, j);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  for (int s = 0; s < min(STAGES, slabs); ++s)
#pragma unroll
    for (int j = 0; j < LOADS; ++j) issue_one(s * STAGE, j);
  f32_wait_slabs<STAGES - 1, LOADS>(slabs - 1);
#pragma unroll
  for (int q = 0; q < FM + 1; ++q) read_one(0, 0, q);
  int stage = 0, in_chunk = 0;  // the slab's place in the ring, and in its chunk
  for (int s = 0; s < slabs; ++s) {
    const int next = stage + STAGE == STAGES * STAGE ? 0 : stage + STAGE;
    if (in_chunk == 0) step(0, stage, 0, false, true);
    else step(0, stage, 0, false, false);
    in_chunk = in_chunk + 1 == per_chunk ? 0 : in_chunk + 1;
    // Slab s + 1 is there for every wave, and every wave has read all of slab s. (Behind the last slab what is read lies in the
    // ring and is not used.)
    if (s + STAGES < slabs) {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((STAGES - 2) * LOADS) : "memory");
      step(1, next, stage, true, false);
    } else {
      f32_wait_slabs<STAGES - 2, LOADS>(slabs - 2 - s);
      step(1, next, 0, false, false);
    }
    stage = next;
  }
#pragma unroll
  for (int i = 0; i < FM; ++i) total[i] += acc[i];
#pragma unroll
  for (int j = 0; j < FM; ++j) {
    const int m = m0 + j * 16 + r, n = n0 + wave * 16 + 4 * g;
    if (m >= M) continue;
    const size_t to = (size_t)m * ldc + n;
    const floatx4 v = total[j];
    if (vec_store && mode != 2 && n + 3 < N) {
      float4 o = make_float4(v[0], v[1], v[2], v[3]);
      if (mode == 1) {
        const float4 c = *reinterpret_cast<const float4*>((const float*)C + to);
        o = make_float4(c.x + o.x, c.y + o.y, c.z + o.z, c.w + o.w);
      }
      *reinterpret_cast<float4*>((float*)C + to) = o;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < N) f32_store(C, mode, to + e, v[e]);
    }
  }
}

template <int FM>
static int launch_f32_rows(const float* A, const float* W, void* C, int mode, int M, int N, int K, int lda, int ldc, int chunk,
                           bool vec_store, hipStream_t st) {
  constexpr int bytes = f32_ring(FM) * (16 * FM + 64) * 128;
  static const bool ready = hipFuncSetAttribute((const void*)gemm_f32_rows_kernel<FM>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess;
  if (!ready) return MS_LAUNCH_FAILED;
  const dim3 grid((N + 63) / 64, (M + 16 * FM - 1) / (16 * FM));
  if (grid.y > 65535) return MS_BAD_ARG;
  gemm_f32_rows_kernel<FM><<<grid, 256, bytes, st>>>(A, W, C, mode, M, N, K, lda, ldc, chunk, vec_store);
  return launch_status();
}

// Partial sums that a product of few rows leaves where the caller's next kernel adds them (0: none, the product is finished by
// ms_gemm_f32). They are the sums of the chunks, so adding them in ascending order to zero gives the finished product's bits.
// Up to 2,048 columns: a block that owns 16 of them and all of K leaves most of the chip idle then, a wave per chunk does not
// (with the RMS norm that adds the parts, 6 rows, microseconds: 1,024 x 2,048 11.2 finished, 7.4 in parts; 1,024 x 3,072 13.9,
// 8.4). At 4,096 columns and more the blocks fill the chip and the parts only cost (4,096 x 1,024: 6.5 and 6.3 without the
// consumer, which then reads sixteen times the product).
extern "C" int ms_gemm_f32_parts_count(int M, int N, int K) {
  if (M <= 0 || M > 16 || N <= 0 || K <= 0 || N > 2048) return 0;
  const int chunk = f32_chunk(K);
  return (K + chunk - 1) / chunk;
}

// P [ms_gemm_f32_parts_count(M, N, K), M, N] = the partial sums of A [M, K] * W [N, K]^T.
extern "C" int ms_gemm_f32_parts(const float* A, const float* W, float* P, int M, int N, int K, int lda, hipStream_t st) {
  const int count = ms_gemm_f32_parts_count(M, N, K);
  if (count == 0 || lda < K || (size_t)P % 16) return MS_BAD_ARG;
  const int chunk = f32_chunk(K);
  const bool vec = K % 64 == 0 && lda % 4 == 0 && (size_t)A % 16 == 0 && (size_t)W % 16 == 0;
  const int slabs = vec ? chunk / F32_SLAB : -1;
  const dim3 grid((N + 15) / 16, 1, count);
#define FEW_PARTS(SLABS) gemm_f32_few_kernel<1, SLABS, true><<<grid, WAVE, 0, st>>>(A, W, P, 0, M, N, K, lda, N, chunk)
#define FEW_PARTS_STREAM(SLABS) gemm_f32_few_kernel<1, SLABS, true, true, true><<<grid, WAVE, SLABS * 2048, st>>>(A, W, P, 0, M, N, K, lda, N, chunk)
  if (slabs < 0) FEW_PARTS(-1);
  else if (slabs == 2) FEW_PARTS_STREAM(2);
  else if (slabs == 4) FEW_PARTS_STREAM(4);
  else if (slabs == 6) FEW_PARTS_STREAM(6);
  else FEW_PARTS(0);
#undef FEW_PARTS
#undef FEW_PARTS_STREAM
  return launch_status();
}

// out [M, inter] = act(A gate^T) * (A up^T) (act: an MS_ACT_* number; limit: the bound of MS_ACT_SWIGLU_CLAMPED), gate and up rows in W in
// alternating runs of 16: what ms_gemm_f32 and ms_act_mul make of it, bit for bit. MS_UNSUPPORTED where no kernel takes the shape: more
// than 16 rows, K no multiple of 64 or beyond 1,024 (a chunk is then more than two slabs), up to 2,048 columns (a product of those leaves
// its chunks' sums, which fill the chip better), more blocks than fit on the chip at once (6 rows, 9,728 outputs of 960: 19.6 us in two
// kernels, 20.1), rows that are not 16-byte aligned.
extern "C" int ms_gemm_f32_gated(const float* A, const float* W, float* out, int M, int inter, int K, int lda, int act, float limit, hipStream_t st) {
  if (M <= 0 || inter <= 0) return MS_OK;
  if (K <= 0 || lda < K || act < 0 || act >= MS_GATED_COUNT || (act == MS_ACT_SWIGLU_CLAMPED && !(limit > 0.f))) return MS_BAD_ARG;
  if (M > 16 || inter % 16 || inter <= 1024 || K % 64 || K > 1024 || lda % 4 || (size_t)A % 16 || (size_t)W % 16) return MS_UNSUPPORTED;
  const int waves = K / 64, bytes = waves * 4 * 2048;
  if (inter / 16 > 256 * (160 * 1024 / bytes)) return MS_UNSUPPORTED;
  static bool ready = false;  // more than 64 KB of LDS has to be asked for once
  if (!ready) {
    if (hipFuncSetAttribute((const void*)gemm_f32_few_gated_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 16 * 4 * 2048) != hipSuccess)
      return MS_LAUNCH_FAILED;
    ready = true;
  }
  gemm_f32_few_gated_kernel<<<inter / 16, waves * WAVE, bytes, st>>>(A, W, out, M, inter, K, lda, act, limit);
  return launch_status();
}

// Which of the two older kernels; microseconds, few rows and tiles. K a multiple of 64: the first up to 80 tiles of 64 x 64 (256 x
// 1,024 x 3,072, 64 tiles: 46, 65; at 80 tiles 68, 65), up to 32 rows whatever the columns, up to 64 rows until 128 tiles: 64 x 6,144 x
// 1,024 (96) 19, 28; 64 x 8,192 x 2,048 (128) 52, 52; 64 x 37,984 x 1,024 103, 67. Other K: its loads wait slab by slab, so it
// pays for little work alone: 8 x 8,192 x 1,000 23, 28; 32 x 8,192 x 1,000 45, 28; 32 x 60,000 x 1,000 314, 84. Where the
// tiles too load element by element (K or the rows' distance not a multiple of 4, other bases): 16 x 5,200 x 777 17, 35;
// 48 x 8,192 x 777 52, 44; 16 x 60,000 x 777 119, 111.
static bool f32_few_rows(int M, int N, int K, bool vec) {
  const long long columns = (N + 63) / 64, tiles = columns * ((M + 63) / 64);
  if (vec && K % 64 == 0) return M <= 32 || tiles <= (M <= 64 ? 128 : 80);
  const long long work = columns * (16 + M);
  return vec ? work <= (M <= 32 ? 2900 : 2300) : M <= 10 || work <= (M <= 32 ? 7000 : 5600);
}

// Tiles of the kernel for tiles that are 64 or 128 each way.
static int f32_square_tile(int M, int N) { return (long long)((M + 127) / 128) * ((N + 127) / 128) >= 512 ? 128 : 64; }

// Predicted microseconds where K is a multiple of 32 and rows are 16-byte aligned: a part per launch, per round of blocks (256, one
// a CU; of the square tiles 512, a last round of up to 256 counting less) and per slab of it. Fits to 9,429 products of 1 to 4,096
// rows, 16 to 60,000 columns and K of 32 to 5,000, each timed in every form, weights from memory: half within 6 %, nine in ten within 17 %.
static float f32_rounds(long long blocks) { return (float)((blocks + 255) / 256); }
static float f32_rows_us(int fm, int M, int N, int K) {
  return 1.5f + f32_rounds((long long)((M + 16 * fm - 1) / (16 * fm)) * ((N + 63) / 64)) * (1.19f + 0.377f * fm + K / F32_SLAB * (0.153f + 0.112f * fm));
}
static float f32_older_us(int M, int N, int K) {
  if (f32_few_rows(M, N, K, true)) {
    const float rounds = f32_rounds((long long)((N + 15) / 16) * (M <= 16 ? 1 : (M + 31) / 32)), k = K / 1000.f;
    if (K % 64 == 0) return 3.2f + rounds * (0.38f + 5.6f * k);
    return M <= 16 ? 2.8f + rounds * (0.11f + 9.5f * k) : 3.55f + rounds * (0.45f + 18.7f * k);
  }
  const int b = f32_square_tile(M, N);
  const long long tiles = (long long)((M + b - 1) / b) * ((N + b - 1) / b), rest = tiles % 512;
  const float full = (float)(tiles / 512 + (rest > 256)), last = rest > 0 && rest <= 256 ? 1.f : 0.f, slabs = (float)(K / F32_SLAB);
  return b == 64 ? 0.4f + (full + last) * 2.83f + slabs * (full * 1.30f + last * 0.77f) : (full + last) * 4.74f + slabs * (full * 4.76f + last * 2.23f);
}

// The height, in steps of 16 rows, of the tiles that take such a product in the older kernels' place; 0: none, they keep it. Tiles of
// any height need 7 % less predicted time. Over the 9,429 products they then take 17 % less than the older kernels alone (269 ms for
// 326, the best of each 267), and 0.8 % of the products take 3 % longer or more. Microseconds, older and tiles of any height: 300 x
// 1,024 x 3,072 68, 33; 24 x 12,288 x 4,096 87, 52; 16 x 531 x 3,488 51, 29. A short K or little work stays: 1,000 x 12,288 x 64 24, 31;
// 64 x 60,000 x 544 52, 57; 17 x 437 x 3,072 19, 26. Up to 16 rows of a K that is a multiple of 64 the weights' bytes bound both,
// and the kernel for few rows reads them faster (6 x 4,096 x 4,096 22, 30).
static int f32_tile_height(int M, int N, int K) {
  if (M <= 16 && K % 64 == 0) return 0;
  int best = 0;
  float least = 0.93f * f32_older_us(M, N, K);
  for (int fm = 8; fm >= 1; --fm) {
    const float t = f32_rows_us(fm, M, N, K);
    if (t < least) least = t, best = fm;
  }
  return best;
}

// Rows of the tiles that a product of contiguous 16-byte aligned operands runs in over gemm_f32_rows_kernel, 0 where another kernel
// takes it. For tests that must know which instance they have reached.
extern "C" int ms_gemm_f32_tile_rows(int M, int N, int K) {
  return M <= 0 || N <= 0 || K <= 0 || K % F32_SLAB ? 0 : 16 * f32_tile_height(M, N, K);
}

extern "C" int ms_gemm_f32(const float* A, const float* W, void* C, int mode, int M, int N, int K, int lda, int ldc,
                           hipStream_t st) {
  if (M <= 0 || N <= 0) return MS_OK;
  if (K <= 0 || lda < K || ldc < N || mode < 0 || mode > 2) return MS_BAD_ARG;
  const int chunk = f32_chunk(K);
  const int waves = (K + chunk - 1) / chunk;
  const bool vec = K % 4 == 0 && lda % 4 == 0 && (size_t)A % 16 == 0 && (size_t)W % 16 == 0;
  const bool whole = vec && K % F32_SLAB == 0;  // no slab cut off
  const int fm = whole ? f32_tile_height(M, N, K) : 0;
  if (!fm && f32_few_rows(M, N, K, vec)) {
    const int mt = M <= 16 ? 1 : 2;
    const int slabs = vec && K % 64 == 0 ? chunk / F32_SLAB : -1;
    dim3 grid((N + 15) / 16, (M + mt * 16 - 1) / (mt * 16));
    if (grid.y > 65535) return MS_BAD_ARG;
#define FEW(MT, SLABS) gemm_f32_few_kernel<MT, SLABS><<<grid, waves * WAVE, 0, st>>>(A, W, C, mode, M, N, K, lda, ldc, chunk)
    if (mt == 1) {
      if (slabs < 0) FEW(1, -1);
      else if (slabs == 2) gemm_f32_few_kernel<1, 2, false, true, true><<<grid, waves * WAVE, waves * 2 * 2048, st>>>(A, W, C, mode, M, N, K, lda, ldc, chunk);
      else if (slabs == 4) FEW(1, 4);
      else if (slabs == 6) FEW(1, 6);
      else FEW(1, 0);
    } else {
      if (slabs < 0) FEW(2, -1);
      else if (slabs == 2) FEW(2, 2);
      else if (slabs == 4) FEW(2, 4);
      else FEW(2, 0);
    }
#undef FEW
    return launch_status();
  }
  const bool dma = vec;
  const bool vec_store = ldc % 4 == 0 && (size_t)C % 16 == 0;
  switch (fm) {
#define ROWS(FM) case FM: return launch_f32_rows<FM>(A, W, C, mode, M, N, K, lda, ldc, chunk, vec_store, st)
    ROWS(1); ROWS(2); ROWS(3); ROWS(4); ROWS(5); ROWS(6); ROWS(7); ROWS(8);
#undef ROWS
    default: break;
  }
  const int b = f32_square_tile(M, N);
  dim3 grid((N + b - 1) / b, (M + b - 1) / b);
  if (grid.y > 65535) return MS_BAD_ARG;
#define TILE(B) do { constexpr int bytes = f32_stages(B) * 2 * B * 128; \
                     if (dma) gemm_f32_tile_kernel<B, true><<<grid, 256, bytes, st>>>(A, W, C, mode, M, N, K, lda, ldc, chunk, vec_store); \
                     else gemm_f32_tile_kernel<B, false><<<grid, 256, bytes, st>>>(A, W, C, mode, M, N, K, lda, ldc, chunk, vec_store); } while (0)
  if (b == 128) TILE(128);
  else TILE(64);
#undef TILE
  return launch_status();
}
