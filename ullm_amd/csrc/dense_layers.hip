// The launches of a run of alike pre-norm layers (grouped-query attention and a gated feed-forward, bfloat16) over one batch with
// prompt portions in it, one after the other from native code (the layer: ullm/models/qwen3.py:159-178).  No kernel of its own: the
// launches, their order and their arguments are those of the parts' own forward passes, whose checks and choices the caller
// has made once for all layers.
//
// What bounded such steps of small models was the host: ten launches a layer cost the interpreter 160 us, the kernels of a 0.6B
// layer take 60 (300 tokens) to 110 us (800).  From here a launch is 2 to 3 us.
#include "common.h"
#include "launchers.h"

// How a product is made: by the panels kernel (`shape`, `slices`) in `mode`, or by the large tiles (`shape` 64-row groups).
struct DenseProduct {
  int tiles, mode, shape, slices;
};

// One layer's tensors.
struct DenseLayer {
  const float *norm1, *q_gain, *k_gain, *cos_sin, *b_qkv, *norm2;
  const void *w_qkv, *w_o, *w_gate_up, *w_down;
  void *k_pool, *v_pool;
  const int* block_table;
  long long bt_stride, write_kv;
};

struct DenseStep {
  decltype(&ullm_add_rmsnorm) add_rmsnorm;
  decltype(&ullm_sum_stacks) sum_stacks;
  decltype(&ullm_qk_norm_rope_write) qk_norm_rope_write;
  decltype(&ullm_qk_norm_rope_write_sums) qk_norm_rope_write_sums;
  decltype(&ullm_gemm_panels) panels;
  decltype(&ullm_gemm_tiles) tiles;
  decltype(&ullm_attention_decode) decode;
  decltype(&ullm_attention_prefill) prefill;
  decltype(&ullm_attention_mixed) mixed_attention;
  // the stream, and room for what lies between two launches (sums: q|k|v in slices; mixed, fed: what the two halves add to the stream)
  float* residual;
  void *normed, *qkv, *q, *attended, *act;
  float *sums, *decode_parts;
  void *mixed, *fed;
  const int *positions, *token_entry, *decode_tokens, *prompt_tiles, *wide_tiles;
  long long tile_keys_total, wide_keys_total, decode_keys_total;
  DenseProduct into, out, gate_up, down;
  int tokens, width, heads, kv_heads, head_dim, inner, table_rows, rot, style, page_size, window;
  int num_decode, decode_splits, decode_waves, num_tiles, tile_keys_max, num_wide, wide_keys_max, decode_keys_max;
  float eps1, eps2, qk_eps, scale;
};

// C = A W^T (gated: silu of the first half of W's rows times the second), [M, N] or sums [slices, M, N]
static int dense_product(const DenseStep& s, const DenseProduct& p, const void* a, int K, const void* w, const float* bias, void* out, int N,
                         int gated, hipStream_t stream) {
  const int ldo = gated ? N / 2 : N;
  return p.tiles ? s.tiles(a, K, w, K, bias, out, ldo, s.tokens, N, K, p.mode, p.shape, 0.f, 0.f, stream)
                 : s.panels(a, K, w, K, bias, out, ldo, s.tokens, N, K, p.mode, p.shape, p.slices, 0.f, 0.f, 0, stream);
}

#define STEP(call) do { const int rc = (call); if (rc != 0) return rc; } while (0)

// Bytes of a step and of a layer, which the caller lays out by hand.
extern "C" int ullm_dense_step_bytes(void) { return (int)sizeof(DenseStep); }
extern "C" int ullm_dense_layer_bytes(void) { return (int)sizeof(DenseLayer); }

// Runs the layers from the stream as it is; the last one's `fed` is left to be added.
extern "C" int ullm_dense_layers(const DenseStep* step, const DenseLayer* layers, int n_layers, hipStream_t stream) {
  const DenseStep& s = *step;
  const int T = s.tokens, H = s.width, q_width = s.heads * s.head_dim, qkv_width = (s.heads + 2 * s.kv_heads) * s.head_dim;
  enum { FLOAT = 2 };                                     // both products' mode that leaves 32-bit sums
  // what is still to be added to the stream, as add_rmsnorm takes it
  const void* pending = nullptr;
  int pending_dtype = ULLM_BF16, pending_count = 1;
  long long pending_stride = 0;
  auto norm = [&](const float* gain, float eps) {
    return s.add_rmsnorm(pending, s.residual, gain, eps, s.normed, nullptr, T, H, pending_dtype, ULLM_BF16, 1, pending_count, pending_stride,
                         stream);
  };
  auto leave = [&](const DenseProduct& p, const void* branch) {
    pending = branch;
    pending_dtype = p.mode == FLOAT ? ULLM_F32 : ULLM_BF16;
    pending_count = p.mode == FLOAT ? p.slices : 1;
    pending_stride = pending_count > 1 ? (long long)T * H : 0;
  };
  for (int i = 0; i < n_layers; ++i) {
    const DenseLayer& l = layers[i];
    STEP(norm(l.norm1, s.eps1));
    int written = ULLM_ERR_UNSUPPORTED;
    if (s.into.mode == FLOAT) {
      STEP(dense_product(s, s.into, s.normed, H, l.w_qkv, nullptr, s.sums, qkv_width, 0, stream));
      // the heads' kernel adds the slices up, where it can
      written = s.qk_norm_rope_write_sums(s.sums, s.into.slices, l.b_qkv, qkv_width, s.q, q_width, l.q_gain, l.k_gain, s.qk_eps, l.cos_sin,
                                          s.table_rows, s.rot, s.style, s.positions, s.token_entry, l.block_table, (int)l.bt_stride, l.k_pool,
                                          l.v_pool, s.page_size, T, s.heads, s.kv_heads, s.head_dim, (int)l.write_kv, stream);
      if (written != ULLM_ERR_UNSUPPORTED) STEP(written);
      else STEP(s.sum_stacks(s.sums, s.into.slices, l.b_qkv, s.qkv, T, qkv_width, ULLM_BF16, stream));
    } else {
      STEP(dense_product(s, s.into, s.normed, H, l.w_qkv, l.b_qkv, s.qkv, qkv_width, 0, stream));
    }
    if (written != 0)
      STEP(s.qk_norm_rope_write(s.qkv, qkv_width, s.q, q_width, l.q_gain, l.k_gain, s.qk_eps, l.cos_sin, s.table_rows, s.rot, s.style,
                                s.positions, s.token_entry, l.block_table, (int)l.bt_stride, l.k_pool, l.v_pool, s.page_size, T, s.heads,
                                s.kv_heads, s.head_dim, (int)l.write_kv, s.heads + s.kv_heads, s.head_dim, ULLM_BF16, stream));
    // both kinds of tokens in one launch, where that is the better way
    int together = ULLM_ERR_UNSUPPORTED;
    if (s.num_decode > 0 && s.num_tiles > 0) {
      together = s.mixed_attention(s.q, q_width, s.attended, q_width, l.k_pool, l.v_pool, s.decode_tokens, s.num_decode, s.decode_keys_total,
                                   s.decode_keys_max, s.prompt_tiles, s.num_tiles, s.positions, s.token_entry, l.block_table, (int)l.bt_stride,
                                   s.page_size, s.heads, s.kv_heads, s.head_dim, s.scale, s.window, s.tile_keys_total, s.tile_keys_max,
                                   s.wide_tiles, s.num_wide, s.wide_keys_total, s.wide_keys_max, 0, stream);
      if (together != ULLM_ERR_UNSUPPORTED) STEP(together);
    }
    if (together != 0 && s.num_decode > 0)
      STEP(s.decode(s.q, q_width, s.attended, q_width, l.k_pool, l.v_pool, s.decode_tokens, s.num_decode, s.positions, s.token_entry,
                    l.block_table, (int)l.bt_stride, s.page_size, s.heads, s.kv_heads, s.head_dim, s.scale, s.window, s.decode_splits,
                    s.decode_waves, s.decode_parts, stream));
    if (together != 0 && s.num_tiles > 0)
      STEP(s.prefill(s.q, q_width, s.attended, q_width, l.k_pool, l.v_pool, s.prompt_tiles, s.num_tiles, s.positions, s.token_entry,
                     l.block_table, (int)l.bt_stride, s.page_size, s.heads, s.kv_heads, s.head_dim, s.scale, s.window, 0,
                     s.tile_keys_total, s.tile_keys_max, s.wide_tiles, s.num_wide, s.wide_keys_total, s.wide_keys_max, stream));
    STEP(dense_product(s, s.out, s.attended, q_width, l.w_o, nullptr, s.mixed, H, 0, stream));
    leave(s.out, s.mixed);
    STEP(norm(l.norm2, s.eps2));
    STEP(dense_product(s, s.gate_up, s.normed, H, l.w_gate_up, nullptr, s.act, 2 * s.inner, 1, stream));
    STEP(dense_product(s, s.down, s.act, s.inner, l.w_down, nullptr, s.fed, H, 0, stream));
    leave(s.down, s.fed);
  }
  return 0;
}
