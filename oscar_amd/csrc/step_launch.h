// The short-step write (step_write.hip) as the other sources launch it.
#pragma once

#include "oscar_common.h"

namespace oscar {

// q_rot [n_tokens][num_heads][D] fp32 = query @ R_k, query bf16
// [n_tokens][q_stride]; q_rot and rot_k 16-byte aligned, n_tokens >= 1.
int launch_rotate_queries(const uint16_t* q, int64_t q_stride, int32_t n_tokens, int32_t num_heads, const float* rot_k,
                          float* q_rot, hipStream_t stream);

// oscar_step_write, with the request layout in host arrays, or
// (layout_on_device) in device arrays that are read on the stream.
int step_write(bool layout_on_device, const void* query_bf16, int64_t query_token_stride, const void* key_bf16,
               const void* value_bf16, int64_t kv_token_stride, int32_t num_tokens, int32_t num_heads,
               int32_t num_kv_heads, int32_t head_size, const float* rot_k, const float* rot_v,
               const int64_t* slot_mapping, const int32_t* query_start_loc, const int32_t* seq_lens,
               int32_t num_requests, void* k_cache, void* v_cache, int32_t block_size, int64_t num_pages,
               int64_t k_stride_page, int64_t k_stride_token, int64_t k_stride_head, int64_t v_stride_page,
               int64_t v_stride_token, int64_t v_stride_head, int32_t clip_index_k, int32_t clip_index_v,
               float* stage_k, float* stage_v, int64_t* stage_owner, void* stage_k_image, void* stage_v_image,
               int32_t stage_rows, int32_t sink_eff, int32_t recent, float* q_rot, float* k_rot, float* v_rot,
               hipStream_t stream);

}  // namespace oscar
