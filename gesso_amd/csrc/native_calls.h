// The entry points that host.cpp calls, declared once for both sides: a definition that differs from its declaration here does not
// compile, and the pointers in host.cpp have these types.
#pragma once

#define GS_ABI_VERSION 15               // of all entry points together

typedef struct ihipStream_t* hipStream_t;

extern "C" {
int gs_abi_version();
const char* gs_last_error();
int gs_add_rmsnorm(float* res, const void* delta, int delta_dtype, const float* w, float eps, void* out, int out_dtype, const int* rows,
                   int n_out, int H, hipStream_t stream);
int gs_gemm_skinny(const void* X, int ldx, int x_tiled, const float* res, const float* ssq, int nb, const float* norm_w, float eps,
                   const void* W, const void* Wt, void* Y, int y_dtype, int ldy, int M, int N, int K, int epilogue, int y_tiled,
                   hipStream_t stream);
int gs_gemm_mid_takes(int M, int N, int K, int epilogue);
int gs_gemm_mid(const void* X, int ldx, const void* Wt, void* Y, int ldy, int M, int N, int K, int epilogue, hipStream_t stream);
int gs_gemm_mid_swiglu_scaled(const void* X, int ldx, const float* ssq, int nssq, float eps, const void* Wt, void* Y, int ldy, int M, int N,
                              int K, hipStream_t stream);
int gs_gemm_mid_residual_sums(int M, int N, int K);
int gs_gemm_mid_residual(const void* X, int ldx, const void* Wt, float* res, const float* next_weight, void* rows, float* ssq, int M, int N,
                         int K, hipStream_t stream);
int gs_gemm_mid_parts(const void* X, int ldx, const void* Wt, float* part, int parts, int M, int N, int K, hipStream_t stream);
int gs_residual_from_parts(const float* part, int parts, float* res, float* ssq, const float* next_w, float eps, void* normed,
                           int normed_dtype, int normed_tiled, int M, int N, hipStream_t stream);
int gs_short_conv(const void* bcx, int dtype, const float* taps, const float* bias, float* state, const int* seq_of_token, const int* q_start,
                  const int* slots, void* out, int ntok, int nseq, int H, int W, int all_single, hipStream_t stream);
int gs_qknorm_rope_kv(void* qkv, int dtype, const float* qw, const float* kw, float eps, const float* cos_t, const float* sin_t, int rotary_dim,
                      int interleaved, int max_position, const int* positions, const int* seq_of_token, const int* block_table, int max_blocks,
                      int page_size, void* kcache, void* vcache, int ntok, int nh, int nkv, int d, int write_kv, int vd, const float* vcos,
                      const float* vsin, int ld, int plain_norm, const void* v_first, int ldf, const float* mix, int maps, hipStream_t stream);
int gs_attention_prefill(const void* q, int q_stride, const void* kcache, const void* vcache, const int* positions, const int* tile_seq,
                         const int* tile_row, const int* tile_n, int ntiles, const int* block_table, int max_blocks, int page_size, int window,
                         float scale, void* out, int nh, int nkv, int d, int tile_rows, int chunk, int sink, float softcap, int keep_first,
                         const float* sinks, hipStream_t stream);
}
