// What the sources launch of one another in a step's forward.
#pragma once

#include "bulk_write.h"
#include "oscar_common.h"
#include "../../include/oscar_amd.h"

namespace oscar {

// q_rot [n_tokens][num_heads][D] fp32 = query @ R_k, query bf16
// [n_tokens][q_stride]; q_rot and rot_k 16-byte aligned, n_tokens >= 1.
int launch_rotate_queries(const uint16_t* q, int64_t q_stride, int32_t n_tokens, int32_t num_heads, const float* rot_k,
                          float* q_rot, hipStream_t stream);

// Runs of consecutive tokens, packed: token p of the packed order, pos[r] <= p
// < pos[r + 1], is token tok[r] + p - pos[r] of the step.
constexpr int kMaxTokenRuns = 64;
struct TokenRuns {
  int32_t n;                          // runs
  int32_t tokens;                     // of all runs
  int32_t pos[kMaxTokenRuns];
  int32_t tok[kMaxTokenRuns];
};

// q_rot [tokens][num_heads][D], k_rot / v_rot [tokens][num_kv_heads][D] fp32 of
// the runs' tokens (step_write.hip).
int launch_rotate_runs(const uint16_t* q, int64_t q_stride, const uint16_t* k, const uint16_t* v, int64_t kv_stride,
                       const TokenRuns& runs, int32_t num_heads, int32_t num_kv_heads, const float* rot_k,
                       const float* rot_v, float* q_rot, float* k_rot, float* v_rot, hipStream_t stream);

// The paged read of the requests of 1 .. spans query tokens of a step, from
// their packed rotated q / k / v to their rows of the step's bf16 output
// (paged_decode.hip).
struct DecodeSpans {
  const float* q_rot;                 // [packed tokens][Hq][D]
  const float* k_rot;
  const float* v_rot;
  const int32_t* query_start_loc;     // host, the step's
  const int32_t* seq_lens;            // host
  int32_t num_requests;               // of the step
  int32_t spans;                      // most query tokens of a request that is read
  int32_t max_query_len;              // of those requests
  int64_t max_history;
  const int32_t* block_table;
  int64_t block_table_stride;
  int32_t block_table_cols;
};
// (check_only: the arguments' checks alone, nothing enqueued)
int launch_decode_spans(const oscar_mtp_layer& layer, const DecodeSpans& d, void* out_bf16, int64_t out_token_stride,
                        void* workspace, size_t workspace_size, bool check_only, hipStream_t stream);

// oscar_quant_write_window (stage_rows > 0) or oscar_quant_write of a step
// whose request layout is in host arrays; layout: 2 num_requests + 1 ints of
// device scratch (quant_write.hip).  With `later`, a write of the bulk kernel is
// not launched: its arguments are left there, *waits is set, and the caller
// hands it to prefill_rotated.
int quant_write_step(const oscar_mtp_layer& layer, const void* rot_k_operand, const void* rot_v_operand,
                     int64_t* seat_winner, const void* key_bf16, const void* value_bf16, int64_t kv_token_stride,
                     int32_t num_tokens, const int64_t* slot_mapping, const int32_t* query_start_loc,
                     const int32_t* seq_lens, int32_t num_requests, int32_t* layout, FusedWriteArgs* later, bool* waits,
                     hipStream_t stream);

// oscar_prefill_rotated, whose first launch also carries out the write in
// `write`, if there is one (prefill.hip).  check_only: the arguments' checks
// alone, nothing enqueued.
int prefill_rotated(
    const void* query_bf16, int64_t query_token_stride, const void* key_bf16, const void* value_bf16,
    int64_t kv_token_stride, int32_t num_requests, const int32_t* first_tokens, const int32_t* new_tokens,
    const int64_t* cached_lens, const int32_t* table_rows, int32_t num_heads, int32_t num_kv_heads,
    int32_t head_size, const void* rot_k_operand, const void* rot_v_operand, const void* rot_v_t_operand,
    const void* k_cache, const void* v_cache, int32_t block_size, int64_t num_pages, int64_t k_stride_page,
    int64_t k_stride_token, int64_t k_stride_head, int64_t v_stride_page, int64_t v_stride_token,
    int64_t v_stride_head, const int32_t* block_table, int64_t block_table_stride, int32_t block_table_cols,
    const float* stage_k, const float* stage_v, const int64_t* stage_owner, int32_t stage_rows, float scale,
    void* out_bf16, void* workspace, size_t workspace_size, const FusedWriteArgs* write, bool check_only,
    hipStream_t stream);

// The read of one request over its fp32 rows by whole row blocks of
// kPrefillSmallTile rows (prefill_rows.hip); the arguments have been checked.
constexpr int kPrefillSmallTile = 128;
struct PrefillRows {
  const float* q;        // [N][Hq][D]
  const float* k_new;    // [N][Hk][D]
  const float* v_new;
  int32_t n_new;
  int32_t num_heads, num_kv_heads, group;
  const uint8_t* k_cache;
  const uint8_t* v_cache;
  int64_t k_page, k_tok, k_head, v_page, v_tok, v_head;
  int32_t block_size;
  FastDiv bs_div;        // block_size
  FastDiv rows_div;      // stage_rows (1 without an arena)
  int64_t num_pages;
  const int32_t* bt;     // the request's block-table row
  int32_t bt_cols;
  int64_t cached;        // C
  const float* stage_k;
  const float* stage_v;
  const int64_t* owner;
  int32_t stage_rows;
  float scale_log2;
  float* out;
};
int launch_prefill_rows(const PrefillRows& a, hipStream_t stream);

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
