// attn_bf16x3.hpp — flash attention for prompts on bf16 MFMA, every F32 value
// as three exact bf16 pieces (attn_bf16x3.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "ikv_common.hpp"

namespace ikv {

// Shapes it takes: head_dim a multiple of 4 up to 128, 16-byte aligned
// operands, sizes that index in int.
bool attn_bf16x3_supported(const void *q, const void *k, const void *v, const void *out, int n_head,
                           int n_head_kv, int head_dim, int64_t n_q, int64_t n_kv, int64_t n_past);

// Arguments as ikv_attn_prefill_f32 (n_q, n_kv > 0, n_past >= 0, n_head a
// multiple of n_head_kv, already checked); pages: NULL, or the cache's table.
int attn_bf16x3(const float *q, const float *k, const float *v, const Pages *pages, float *out,
                int n_head, int n_head_kv, int head_dim, int64_t n_q, int64_t n_kv, int64_t n_past,
                float scale, hipStream_t s);

}  // namespace ikv
