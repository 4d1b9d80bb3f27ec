// A plain decoder layer's launches for a step that brings prompts, or portions of them, in one call: norm, query/key/value product, head norm with rotation and
// cache store, attention, output product, norm, gated product, down product. It launches the kernels that the calls one by one
// launch, picked the same way, into one workspace: the same results. What it spares is the host's work between them, which
// bounds short prompts. 28 layers of 1,024 columns, milliseconds a step, one by one and in one call: five prompts of 19 to 211 tokens
// 2.45, 2.32; three of 33 to 75 2.66, 1.51; one of 71 2.62, 1.43; five of two to four 2.65, 1.42.
#include "common.h"

extern "C" {
int ms_rmsnorm(float*, const void*, int, void*, int, const int*, int, int, float, const float*, int, long long, const float*, hipStream_t);
int ms_gemm_bf16_small_splits(int, int, int);
int ms_gemm_bf16_small(const void*, const void*, float*, void*, int, int, int, int, int, int, int, hipStream_t);
int ms_gemm_bf16_tile_splits(int, int, int);
int ms_gemm_bf16(const void*, const void*, void*, int, int, int, int, int, int, int, hipStream_t);
int ms_gemm_bf16_gated(const void*, const void*, void*, int, int, int, int, int, float, hipStream_t);
int ms_act_mul(const void*, void*, int, int, int, int, int, float, hipStream_t);
int ms_act_mul_parts(const float*, int, long long, void*, int, int, int, int, int, float, hipStream_t);
int ms_qk_norm_rope_store(const void*, const float*, int, long long, void*, int, int, const int*, const void*, const void*, int, float,
                          const float*, int, int, void*, void*, int, int, int, int, int, hipStream_t);
int ms_attention_decode_bf16(const void*, int, const void*, const void*, const int*, int, const int*, const int*, const int*, void*, float*,
                             float*, int, int, int, int, int, int, float, int, hipStream_t);
int ms_attention_prefill_bf16(const void*, int, const void*, const void*, const int*, int, const int*, const int*, int, int, const int*,
                              const int*, void*, int, int, int, int, float, int, hipStream_t);
int ms_attention_prefill_parts_bf16(const void*, int, const void*, const void*, const int*, int, const int*, int, int, float*, float*, int,
                                    const int*, const int*, void*, int, int, int, int, float, hipStream_t);
}

#define SMALL_ROWS 64  // up to here a product leaves partial sums whatever its columns

// Mirrored by DenseLayerCall in ops.py: pointers first, then numbers.
struct DenseLayer {
  // of the step
  float* residual;
  unsigned char* workspace;  // dense_layer_bytes of it
  const float* rope;
  const int *slots, *block_table, *token_row, *pos, *tile_first, *tile_count, *plan;
  float *part_o, *part_ml;
  const int* decode_tokens;  // flat indices of the rows that bring one token
  float *decode_o, *decode_ml;
  // of the layer
  const float* pending;  // partial sums to add to the residual stream first
  const void *mixer_norm, *qkv, *q_norm, *k_norm, *o, *ffn_norm, *gate_up, *down;
  void *k_cache, *v_cache;
  int tokens, width, heads, kv_heads, dim, inter, rot, pairing, table_width, tiles, tile_rows, entries, merges, act;
  int pending_splits, mixer_norm_bf16, qk_norm_bf16, ffn_norm_bf16, decode_rows, decode_splits;
  float limit, mixer_eps, qk_eps, ffn_eps, scale;
};

struct Layout {
  size_t x, qkv, q, out, parts_o, gate, act, down, end;
  int qkv_splits, o_splits, gate_splits, down_splits;
};

// 0: the product is finished where it is made; else the partial sums it leaves.
static int left_splits(int M, int N, int K) {
  if (M <= SMALL_ROWS) return ms_gemm_bf16_small_splits(M, N, K);
  const int s = ms_gemm_bf16_tile_splits(M, N, K);
  return s > 1 ? s : 0;
}

static Layout layout_of(int M, int width, int heads, int kv_heads, int dim, int inter) {
  const int qkv_n = (heads + 2 * kv_heads) * dim, q_n = heads * dim;
  Layout l;
  l.qkv_splits = left_splits(M, qkv_n, width);
  l.o_splits = left_splits(M, width, q_n);
  l.gate_splits = left_splits(M, 2 * inter, width);
  l.down_splits = left_splits(M, width, inter);
  // What is read before the other is written shares a place: query/key/value and gate/up, attention's output and the activation, the
  // output product's partial sums and the down product's.
  const auto most = [](size_t a, size_t b) { return a > b ? a : b; };
  size_t at = 0;
  auto take = [&](size_t bytes) { const size_t here = at; at = (at + bytes + 255) / 256 * 256; return here; };
  l.x = take((size_t)M * width * 2);
  l.qkv = l.gate = take(most((size_t)M * qkv_n * (l.qkv_splits ? 4 * (size_t)l.qkv_splits : 2),
                             (size_t)M * 2 * inter * (l.gate_splits ? 4 * (size_t)l.gate_splits : 2)));
  l.q = take(l.qkv_splits ? (size_t)M * q_n * 2 : 0);
  l.out = l.act = take(most((size_t)M * q_n * 2, (size_t)M * inter * 2));
  l.parts_o = l.down = take((size_t)M * width * 4 * most(l.o_splits, l.down_splits));
  l.end = at;
  return l;
}

// The workspace's bytes, where in it the down product's partial sums lie and how many there are (0: it is added into the stream).
extern "C" int ms_dense_layer_plan(int M, int width, int heads, int kv_heads, int dim, int inter, long long* bytes, long long* down_at, int* down_splits) {
  if (M <= 0 || width <= 0 || heads <= 0 || kv_heads <= 0 || dim <= 0 || inter <= 0) return MS_BAD_ARG;
  const Layout l = layout_of(M, width, heads, kv_heads, dim, inter);
  *bytes = (long long)l.end;
  *down_at = (long long)l.down;
  *down_splits = l.down_splits;
  return MS_OK;
}

// x [M, K] W^T: partial sums at `to` where there are splits, else bfloat16 at `to`, or added into `into`.
static int product(const void* x, const void* w, void* to, float* into, int splits, int M, int N, int K, hipStream_t st) {
  if (M <= SMALL_ROWS) return ms_gemm_bf16_small(x, w, (float*)to, nullptr, 1, 0, M, N, K, K, N, st);
  if (splits) return ms_gemm_bf16(x, w, to, 1, M, N, K, K, N, splits, st);
  return into ? ms_gemm_bf16(x, w, into, 2, M, N, K, K, N, 1, st) : ms_gemm_bf16(x, w, to, 0, M, N, K, K, N, 1, st);
}

extern "C" int ms_dense_layer(const DenseLayer* d, hipStream_t st) {
  const int M = d->tokens, W = d->width, qkv_n = (d->heads + 2 * d->kv_heads) * d->dim, q_n = d->heads * d->dim;
  const Layout l = layout_of(M, W, d->heads, d->kv_heads, d->dim, d->inter);
  unsigned char* ws = d->workspace;
  void *x = ws + l.x, *qkv = ws + l.qkv, *out = ws + l.out, *gate = ws + l.gate, *act = ws + l.act;
  void* q = l.qkv_splits ? (void*)(ws + l.q) : qkv;
  const int q_stride = l.qkv_splits ? q_n : qkv_n;
#define DO(call) do { const int rc = (call); if (rc != MS_OK) return rc; } while (0)
  DO(ms_rmsnorm(d->residual, d->mixer_norm, d->mixer_norm_bf16, x, 1, nullptr, M, W, d->mixer_eps, d->pending, d->pending_splits,
                d->pending ? (long long)M * W : 0, nullptr, st));
  DO(product(x, d->qkv, qkv, nullptr, l.qkv_splits, M, qkv_n, W, st));
  DO(ms_qk_norm_rope_store(l.qkv_splits ? nullptr : qkv, l.qkv_splits ? (const float*)qkv : nullptr, l.qkv_splits,
                           l.qkv_splits ? (long long)M * qkv_n : 0, q, q_stride, 1, d->slots, d->q_norm, d->k_norm, d->qk_norm_bf16, d->qk_eps,
                           d->rope, d->rot, d->pairing, d->k_cache, d->v_cache, M, d->heads, d->kv_heads, d->dim, 16, st));
  if (d->decode_rows)
    DO(ms_attention_decode_bf16(q, q_stride, d->k_cache, d->v_cache, d->block_table, d->table_width, d->decode_tokens, d->token_row, d->pos, out,
                                d->decode_o, d->decode_ml, d->decode_rows, d->decode_splits, d->heads, d->kv_heads, d->dim, 16, d->scale, 0, st));
  if (d->plan)
    DO(ms_attention_prefill_parts_bf16(q, q_stride, d->k_cache, d->v_cache, d->block_table, d->table_width, d->plan, d->entries, d->merges,
                                       d->part_o, d->part_ml, d->tile_rows, d->token_row, d->pos, out, d->heads, d->kv_heads, d->dim, 16,
                                       d->scale, st));
  else
    DO(ms_attention_prefill_bf16(q, q_stride, d->k_cache, d->v_cache, d->block_table, d->table_width, d->tile_first, d->tile_count, d->tiles,
                                 d->tile_rows, d->token_row, d->pos, out, d->heads, d->kv_heads, d->dim, 16, d->scale, 0, st));
  DO(product(out, d->o, ws + l.parts_o, d->residual, l.o_splits, M, W, q_n, st));
  DO(ms_rmsnorm(d->residual, d->ffn_norm, d->ffn_norm_bf16, x, 1, nullptr, M, W, d->ffn_eps, l.o_splits ? (const float*)(ws + l.parts_o) : nullptr,
                l.o_splits, l.o_splits ? (long long)M * W : 0, nullptr, st));
  const int fused = ms_gemm_bf16_gated(x, d->gate_up, act, M, d->inter, W, W, d->act, d->limit, st);
  if (fused == MS_UNSUPPORTED) {
    DO(product(x, d->gate_up, gate, nullptr, l.gate_splits, M, 2 * d->inter, W, st));
    if (l.gate_splits)
      DO(ms_act_mul_parts((const float*)gate, l.gate_splits, (long long)M * 2 * d->inter, act, 1, M, d->inter, 16, d->act, d->limit, st));
    else
      DO(ms_act_mul(gate, act, 1, M, d->inter, 16, d->act, d->limit, st));
  } else if (fused != MS_OK) {
    return fused;
  }
  return product(act, d->down, ws + l.down, d->residual, l.down_splits, M, W, d->inter, st);
#undef DO
}
