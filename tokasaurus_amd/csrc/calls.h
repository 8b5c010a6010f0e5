// The entry points that block_calls.hip calls one after the other.  Included where each is defined as well: two declarations of one
// C name that differ do not compile, where a declaration by hand would be linked with, or called through, whatever is there.
#pragma once

#include "common.h"

struct GemmExtra;

// of the same library
TK_API int tk_gemm_skinny_bf16(const void* A, int lda, const void* W, void* C, int ldc, const void* residual, int ldr, const GemmExtra* extra, int M,
                               int N, int K, int epi, int waves_k, int tiles, int staged, int tile_rows, int fold, hipStream_t stream);
TK_API int tk_split_linear_add_rmsnorm(const void* A, int lda, const void* W, float* part, int M, int N, int K, int cuts, const void* residual,
                                       const void* w, int w_f32, void* stream_out, void* out, float eps, int once, hipStream_t stream);
TK_API int tk_split_linear_rope_append(const void* A, int lda, const void* W, float* part, int M, int K, int cuts, void* q, const int* positions,
                                       const int* token_req, const int* block_table, int table_stride, const float* cos_t, const float* sin_t,
                                       void* kcache, void* vcache, int nq, int nkv, int d, int P, hipStream_t stream);
TK_API int tk_gemm_tiles_bf16(const void* A, int lda, const void* W, void* C, int ldc, int M, int N, int K, int glu, int shape, hipStream_t stream);
TK_API int tk_paged_attention_mfma(const void* q, int q_stride, void* out, int out_stride, const void* kcache, const void* vcache,
                                   const int* block_table, int table_stride, const int* q_start, const int* kv_len, const int* tile_req,
                                   const int* tile_row0, const int* tile_row1, int n_tiles, int row_tiles, int nq, int nkv, int d, int P,
                                   int window, float scale, int split, int waves, int grid_splits, int max_splits, float* part_o, float* part_ml,
                                   unsigned* tickets, int grouped, int even, hipStream_t stream);

// of the other libraries, called by their addresses
TK_API int tk_rope_append(int dt, void* qkv, int row_stride, const int* positions, const int* token_req, const int* block_table, int table_stride,
                          const float* cos_t, const float* sin_t, void* kcache, void* vcache, int n_tokens, int nq, int nkv, int d, int rot, int P,
                          int write_cache, hipStream_t stream);
TK_API int tk_add_rmsnorm(int dt, const void* x, const void* residual, const void* w, int w_f32, void* stream_out, void* out, int rows, int hidden,
                          float eps, hipStream_t stream);
TK_API int tk_swiglu(int dt, const void* gate_up, void* out, int rows, int inter, hipStream_t stream);
TK_API int tk_gemm_library_bf16(const void* x, int ldx, const void* w, int ldw, void* out, int ldo, int M, int N, int K, int f32_out, void* workspace,
                                size_t workspace_bytes, hipStream_t stream);
