/*
 * gdn_rows.h -- the chunked prefill and the decode on q, k, v that are column
 * slices of wider tensors (a Qwen3-Next layer splits its convolution's output
 * [B, T, 2 Hqk K + Hv V] into them, modeling_qwen3_next.py:641-648), read in
 * place instead of through contiguous copies.
 *
 * As gdn_chunk_fwd / gdn_chunk_fwd_gating (gdn.h, gdn_layer.h) and
 * gdn_recurrent_fwd / _indexed / _gating, with q_row, k_row, v_row: elements
 * from one token's rows to the next's (token b T + t of a batch at b T + t
 * rows; a token's heads contiguous).  A row is at least its heads long, a
 * multiple of 8 elements and under 2^23; q, k, v are 16-byte aligned.  The
 * gates come from (A_log, a, b, dt_bias) when A_log is non-NULL, else from g
 * and beta.  gdn_recurrent_fwd_rows: state_indices nullable (num_slots is
 * then N).
 */
#ifndef AVELANG_AMD_GDN_ROWS_H
#define AVELANG_AMD_GDN_ROWS_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

int gdn_chunk_fwd_rows(const void* q, const void* k, const void* v,
                       long long q_row, long long k_row, long long v_row,
                       const float* g, const float* beta,
                       const void* A_log, const void* a, const void* b, const void* dt_bias,
                       int a_dtype, int b_dtype, int p_dtype, float sp_beta, float sp_threshold,
                       const float* h0, float* ht, void* o, const int32_t* cu_seqlens,
                       int B, int T, int Hqk, int Hv, int K, int V, int N,
                       float scale, int use_qk_l2norm,
                       void* workspace, size_t workspace_bytes, void* stream);

int gdn_recurrent_fwd_rows(const void* q, const void* k, const void* v,
                           long long q_row, long long k_row, long long v_row,
                           const float* g, const float* beta,
                           const void* A_log, const void* a, const void* b, const void* dt_bias,
                           int a_dtype, int b_dtype, int p_dtype, float sp_beta,
                           float sp_threshold,
                           const float* h0, float* ht, void* o, const int32_t* cu_seqlens,
                           const int32_t* state_indices,
                           int B, int T, int Hqk, int Hv, int K, int V, int N, int num_slots,
                           float scale, int use_qk_l2norm, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* AVELANG_AMD_GDN_ROWS_H */
