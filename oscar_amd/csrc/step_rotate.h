// The fp32 rotations of the short-step write, without its write (step_write.hip).
#pragma once

#include "oscar_common.h"

namespace oscar {

// q_rot [n_tokens][num_heads][D] fp32 = query @ R_k, query bf16
// [n_tokens][q_stride]; q_rot and rot_k 16-byte aligned, n_tokens >= 1.
int launch_rotate_queries(const uint16_t* q, int64_t q_stride, int32_t n_tokens, int32_t num_heads, const float* rot_k,
                          float* q_rot, hipStream_t stream);

}  // namespace oscar
