// The argument checks of the prefill entry points over contiguous K/V (host), for the entry
// points that launch something of their own before the attention.
#pragma once

#include <stdint.h>

// NIA_OK or the status nia_prefill (with `mask`: nia_prefill_masked) refuses the call with;
// `empty`: an accepted call without query rows.
int32_t check_prefill_args(const void* out, int64_t out_tok_stride, int64_t out_head_stride,
                           const void* q, int64_t q_tok_stride, int64_t q_head_stride,
                           const void* k, int64_t k_tok_stride, int64_t k_head_stride,
                           const void* v, int64_t v_tok_stride, int64_t v_head_stride,
                           const int32_t* q_start, const int32_t* q_len, const int32_t* k_start,
                           const int32_t* k_len, int32_t num_seqs, int32_t max_q_len,
                           int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, float scale,
                           int32_t causal, int32_t dtype, const float* mask,
                           int64_t mask_seq_stride, int64_t mask_head_stride,
                           int64_t mask_q_stride, bool& empty);
