// The bulk write's kernel arguments (quant_write.hip): its own launch's, or
// those of a write that waits to share a launch with the prefill read's
// operand rotation.
#pragma once

#include "oscar_common.h"

namespace oscar {

struct CacheArgs {
  uint8_t* k_cache;
  uint8_t* v_cache;
  int64_t k_page, k_tok, k_head;     // byte strides
  int64_t v_page, v_tok, v_head;
  int32_t block_size;
  int64_t num_slots;                 // pages * block_size (< 2^31); larger slots are skipped
  FastDiv bs_div;                    // block_size
};

// The window arena of a bulk write (rows = 0: none).
struct WindowArgs {
  const int32_t* query_start;   // [num_requests + 1] on the device
  const int32_t* seq_lens;      // [num_requests]
  int32_t num_requests;
  int32_t rows;
  int32_t sink_eff, recent;
  int32_t num_kv_heads;
  float* stage_k;               // [rows][bs][Hk][D] fp32
  float* stage_v;
  int64_t* owner;               // [rows][bs]
  int64_t* winner;              // seat winners (read after this call's pass)
  _Float16* kimg;               // operand images, or null
  _Float16* vimg;
};

struct FusedWriteArgs {
  const uint16_t* key;
  const uint16_t* value;
  int64_t n_tokens, token_stride;
  const uint8_t* rot_k;         // operands
  const uint8_t* rot_v;
  const int64_t* slots;
  CacheArgs c;
  int32_t clip_k, clip_v;
  WindowArgs w;
  int32_t token_blocks, num_kv_heads;   // workgroups: token_blocks x (kv head, side)
};

}  // namespace oscar
