// Shared device helpers for the gfx950 kernels: element types, conversions, wave and block reductions.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef __bf16 bf16;

#define WAVE 64

// Error codes returned by every extern "C" entry point (0 = launched).
#define MS_OK 0
#define MS_BAD_ARG 1
#define MS_UNSUPPORTED 2
#define MS_LAUNCH_FAILED 3

__device__ __forceinline__ float to_f32(float x) { return x; }
__device__ __forceinline__ float to_f32(bf16 x) { return static_cast<float>(x); }

template <typename T> __device__ __forceinline__ T from_f32(float x);
template <> __device__ __forceinline__ float from_f32<float>(float x) { return x; }
template <> __device__ __forceinline__ bf16 from_f32<bf16>(float x) { return static_cast<bf16>(x); }

// A lane's value from another lane of its row of 16, in the instruction that uses it (DPP): no trip through LDS, which costs
// some 100 clocks a step where a wave has a SIMD nearly to itself, as in a decode step. CTRL: quad_perm with lanes 1 or 2 apart
// exchanged, rows or halves of rows mirrored (lanes l ^ 15, l ^ 7), rows rotated by 4 or 8.
#define DPP_XOR1 0xB1
#define DPP_XOR2 0x4E
#define DPP_XOR3 0x1B
#define DPP_HALF_MIRROR 0x141
#define DPP_MIRROR 0x140
#define DPP_ROR4 0x124
#define DPP_ROR8 0x128
template <int CTRL> __device__ __forceinline__ int dpp_i32(int x) { return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xf, 0xf, true); }
template <int CTRL> __device__ __forceinline__ float dpp_f32(float x) { return __int_as_float(dpp_i32<CTRL>(__float_as_int(x))); }

// Both values of a pair of lanes 16 (32) apart, the same two in both lanes.
__device__ __forceinline__ float2 swap16_f32(float v) {
  auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return make_float2(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
__device__ __forceinline__ float2 swap32_f32(float v) {
  auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return make_float2(__uint_as_float(a[0]), __uint_as_float(a[1]));
}

// The value of lane l ^ OFF.
template <int OFF> __device__ __forceinline__ float lane_xor_f32(float v) {
  static_assert(OFF == 1 || OFF == 2 || OFF == 4 || OFF == 8 || OFF == 16, "");
  if constexpr (OFF == 1) return dpp_f32<DPP_XOR1>(v);
  else if constexpr (OFF == 2) return dpp_f32<DPP_XOR2>(v);
  else if constexpr (OFF == 4) return dpp_f32<DPP_XOR3>(dpp_f32<DPP_HALF_MIRROR>(v));
  else if constexpr (OFF == 8) return dpp_f32<DPP_ROR8>(v);
  else {
    const float2 p = swap16_f32(v);  // rows 0 and 2 hold the first, rows 1 and 3 the second
    return (threadIdx.x & 16) ? p.x : p.y;
  }
}

// Sum over aligned groups of N lanes, in pairs 1, 2, 4, ... apart: a lane adds the sum of its partner's group to its own (from step 4 on
// any lane of that group will do, all hold the same).
template <int N> __device__ __forceinline__ float group_sum(float v) {
  static_assert(N == 4 || N == 8 || N == 16 || N == 32, "");
  v += dpp_f32<DPP_XOR1>(v);
  v += dpp_f32<DPP_XOR2>(v);
  if constexpr (N >= 8) v += dpp_f32<DPP_HALF_MIRROR>(v);
  if constexpr (N >= 16) v += dpp_f32<DPP_MIRROR>(v);
  if constexpr (N >= 32) {
    const float2 p = swap16_f32(v);
    v = p.x + p.y;
  }
  return v;
}

// Sum / maximum over the wave, in pairs 32, 16, 8, ... apart (from 4 on a rotation does for the exchange: lanes 8 apart hold the same).
__device__ __forceinline__ float wave_sum(float v) {
  float2 p = swap32_f32(v);
  v = p.x + p.y;
  p = swap16_f32(v);
  v = p.x + p.y;
  v += dpp_f32<DPP_ROR8>(v);
  v += dpp_f32<DPP_ROR4>(v);
  v += dpp_f32<DPP_XOR2>(v);
  v += dpp_f32<DPP_XOR1>(v);
  return v;
}

__device__ __forceinline__ float wave_max(float v) {
  float2 p = swap32_f32(v);
  v = fmaxf(p.x, p.y);
  p = swap16_f32(v);
  v = fmaxf(p.x, p.y);
  v = fmaxf(v, dpp_f32<DPP_ROR8>(v));
  v = fmaxf(v, dpp_f32<DPP_ROR4>(v));
  v = fmaxf(v, dpp_f32<DPP_XOR2>(v));
  v = fmaxf(v, dpp_f32<DPP_XOR1>(v));
  return v;
}

// Maximum / sum over the four lanes l, l ^ 16, l ^ 32, l ^ 48 (one element of each 16-lane row), the
// same bits in all four: v_permlane16_swap and v_permlane32_swap hand a lane its partner's value
// without a trip through LDS. The sum is (row 0 + row 1) + (row 2 + row 3) for every lane.
__device__ __forceinline__ float rows4_max(float v) {
  auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float rows4_sum(float v) {
  auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Sum over a block of NT threads (NT a multiple of 64, at most 1024). `red` holds NT / 64 floats.
// Every thread receives the total; the order of additions is fixed by NT alone.
template <int NT> __device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int i = 0; i < NT / WAVE; ++i) total += red[i];
  return total;
}

// Sum of `splits` floats spaced `stride` apart, added in ascending order. Loads are issued eight at a
// time so that they overlap; absent splits contribute an exact zero.
__device__ __forceinline__ float sum_splits(const float* __restrict__ p, int splits, size_t stride) {
  float acc = 0.f;
  for (int s0 = 0; s0 < splits; s0 += 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = (s0 + u < splits) ? p[(size_t)(s0 + u) * stride] : 0.f;
#pragma unroll
    for (int u = 0; u < 8; ++u) acc += v[u];
  }
  return acc;
}

// acc += parts of splits s0 .. s0 + B - 1 (those below `splits`), four floats each, in ascending order;
// the B loads are issued before the first sum.
template <int B>
__device__ __forceinline__ void add_splits(float4& acc, const float* __restrict__ p, int s0, int splits, size_t split_stride) {
  float4 t[B];
#pragma unroll
  for (int u = 0; u < B; ++u) {
    const bool in = s0 + u < splits;
    t[u] = *reinterpret_cast<const float4*>(p + (size_t)(in ? s0 + u : 0) * split_stride);
    if (!in) t[u] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
#pragma unroll
  for (int u = 0; u < B; ++u) {
    acc.x += t[u].x; acc.y += t[u].y; acc.z += t[u].z; acc.w += t[u].w;
  }
}

// 16 bytes that this launch reads once: a matrix's weights in a step of few rows. Marked so, they do not push what the step's small
// kernels hand one another out of the L2 (28 layers of 1,024 columns, a step of one row 980 -> 936 us).
__device__ __forceinline__ uint4 load_once(const void* p) {
  typedef __attribute__((__vector_size__(4 * sizeof(unsigned)))) unsigned u32x4_once;
  union { u32x4_once v; uint4 u; } x;
  x.v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_once*>(p));
  return x.u;
}

#define LOAD_ONCE 2  // the same for loads straight into LDS: their cache policy

// Four consecutive weights in one load (w + i is aligned to four elements), kept as loaded: what uses
// them comes after the block's sum, and a conversion right after the load would wait for it there.
template <typename TW> struct Weights4;
template <> struct Weights4<float> {
  float4 v;
  __device__ __forceinline__ void load(const float* w) { v = *reinterpret_cast<const float4*>(w); }
  __device__ __forceinline__ float at(int e) const { return e == 0 ? v.x : e == 1 ? v.y : e == 2 ? v.z : v.w; }
};
template <> struct Weights4<bf16> {
  union { uint2 u; bf16 e[4]; } v;
  __device__ __forceinline__ void load(const bf16* w) { v.u = *reinterpret_cast<const uint2*>(w); }
  __device__ __forceinline__ float at(int e) const { return to_f32(v.e[e]); }
};

// The sum of `splits` slices, four floats each, in ascending order. The loads of a batch of splits go out together; few
// splits (a tile product's two to four) take a batch of their own size, so that no load is issued for nothing.
__device__ __forceinline__ float4 add_splits4(const float* __restrict__ p, int splits, size_t split_stride) {
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  if (splits == 1) {
    add_splits<1>(acc, p, 0, splits, split_stride);
  } else if (splits <= 2) {
    add_splits<2>(acc, p, 0, splits, split_stride);
  } else if (splits <= 4) {
    add_splits<4>(acc, p, 0, splits, split_stride);
  } else if (splits <= 8) {
    add_splits<8>(acc, p, 0, splits, split_stride);
  } else {  // the products of a decode step leave 12 to 16: one round trip, not two
    for (int s0 = 0; s0 < splits; s0 += 16) add_splits<16>(acc, p, s0, splits, split_stride);
  }
  return acc;
}

// Which elements of a head make pair j of a rotary position encoding: (j, j + rot/2) or (2j, 2j + 1).
#define MS_ROPE_HALVES 0
#define MS_ROPE_ADJACENT 1

// Activations of the gated feed-forward, by the number the host passes: out = act(gate) * up, in float32.
#define MS_ACT_SILU 0
#define MS_ACT_GELU_TANH 1
// A gated feed-forward with bounded inputs: g = min(gate, limit), u = clamp(up, -limit, limit),
// out = g sigmoid(1.702 g) (u + 1). Not of the form act(gate) * up: it takes `limit` beside the number.
#define MS_ACT_SWIGLU_CLAMPED 2
#define MS_GATED_COUNT 3  // what a gated feed-forward may run: the matrix kernels' epilogues and the activation kernels know them
// The square of max(x, 0): only as the activation of a feed-forward without a gate.
#define MS_ACT_RELU_SQUARED 3
// The hyperbolic tangent: between the two steps of a small projection, never in a feed-forward's gate.
#define MS_ACT_TANH 4
static __host__ __device__ __forceinline__ bool ms_act_ungated_ok(int act) {
  return act == MS_ACT_SILU || act == MS_ACT_GELU_TANH || act == MS_ACT_RELU_SQUARED || act == MS_ACT_TANH;
}
__device__ __forceinline__ float activate(float x, int act) {
  if (act == MS_ACT_RELU_SQUARED) { const float r = fmaxf(x, 0.f); return r * r; }
  if (act == MS_ACT_TANH) return tanhf(x);
  if (act == MS_ACT_GELU_TANH) return 0.5f * x * (1.f + tanhf(0.7978845608028654f * (x + 0.044715f * x * x * x)));
  return x / (1.f + expf(-x));
}
// log(1 + exp(z)) without overflow.
__device__ __forceinline__ float softplus(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }
// What a gated feed-forward makes of one gate and one up value, float32.
__device__ __forceinline__ float gated_value(float gate, float up, int act, float limit) {
  if (act == MS_ACT_SWIGLU_CLAMPED) {
    const float g = fminf(gate, limit);
    const float u = fminf(fmaxf(up, -limit), limit);
    return g / (1.f + expf(-1.702f * g)) * (u + 1.f);
  }
  return activate(gate, act) * up;
}

static inline int launch_status() { return hipGetLastError() == hipSuccess ? MS_OK : MS_LAUNCH_FAILED; }
