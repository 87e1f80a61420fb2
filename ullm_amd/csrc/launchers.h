// The entry points of other families that dense_layers.hip calls through pointers: declared once, so that the compiler holds a
// family's definition to what the caller passes.
#pragma once
#include <hip/hip_runtime.h>

extern "C" {
int ullm_add_rmsnorm(const void* branch, float* residual, const float* gain, float eps, void* y, const int* rows, int n_rows, int H,
                     int branch_dtype, int y_dtype, int write_res, int n_branch, long long branch_stride, hipStream_t stream);
int ullm_sum_stacks(const float* stacks, int n_stacks, const float* bias, void* out, int M, int N, int dtype, hipStream_t stream);
int ullm_qk_norm_rope_write(const void* qkv, int qkv_stride, void* q_out, int q_out_stride, const float* q_gain, const float* k_gain,
                            float eps, const float* cos_sin, int table_rows, int rot, int style, const int* positions,
                            const int* token_entry, const int* block_table, int bt_stride, void* k_pool, void* v_pool, int page_size,
                            int T_, int nq, int nkv, int hd, int write_kv, int v_head0, int norm_dim, int dtype, hipStream_t stream);
int ullm_qk_norm_rope_write_sums(const float* sums, int slices, const float* bias, int stride, void* q_out, int q_out_stride,
                                 const float* q_gain, const float* k_gain, float eps, const float* cos_sin, int table_rows, int rot, int style,
                                 const int* positions, const int* token_entry, const int* block_table, int bt_stride, void* k_pool,
                                 void* v_pool, int page_size, int T_, int nq, int nkv, int hd, int write_kv, hipStream_t stream);
int ullm_gemm_panels(const void* x, int ldx, const void* w, int ldw, const float* bias, void* out, int ldo, int M, int N, int K, int mode,
                     int shape, int slices, float limit, float alpha, int act, hipStream_t stream);
int ullm_gemm_tiles(const void* x, int ldx, const void* w, int ldw, const float* bias, void* out, int ldo, int M, int N, int K, int mode,
                    int row_groups, float limit, float alpha, hipStream_t stream);
int ullm_attention_decode(const void* q, int q_stride, void* out, int out_stride, const void* k_pool, const void* v_pool,
                          const int* token_list, int n_items, const int* positions, const int* token_entry, const int* block_table,
                          int bt_stride, int page_size, int nq, int nkv, int hd, float scale, int window, int num_splits, int waves,
                          float* workspace, hipStream_t stream);
int ullm_attention_prefill(const void* q, int q_stride, void* out, int out_stride, const void* k_pool, const void* v_pool,
                           const int* tiles, int n_tiles, const int* positions, const int* token_entry, const int* block_table,
                           int bt_stride, int page_size, int nq, int nkv, int hd, float scale, int window, int halves,
                           long long keys_total, int keys_max, const int* wide_tiles, int n_wide, long long wide_total, int wide_max,
                           hipStream_t stream);
int ullm_attention_mixed(const void* q, int q_stride, void* out, int out_stride, const void* k_pool, const void* v_pool, const int* decode_tokens,
                         int n_decode, long long decode_keys, int decode_keys_max, const int* tiles, int n_tiles, const int* positions,
                         const int* token_entry, const int* block_table, int bt_stride, int page_size, int nq, int nkv, int hd, float scale,
                         int window, long long keys_total, int keys_max, const int* wide_tiles, int n_wide, long long wide_total, int wide_max,
                         int way, hipStream_t stream);
}
