// The forward of one layer for a step with long requests (gfx950): one call
// enqueues what the step needs, in the order of the reference's forward
// (oscar_ascend/backend.py:239-319, 361-415):
//   1. the INT2 write of every token and, with an arena, the window write
//      (quant_write_step: a seat-winner pass that also carries the request
//      layout to the device, then the fused write, which shares a launch with
//      step 3's operand rotation);
//   2. the short requests' q / k / v rotated in fp32, packed (one launch);
//   3. the long requests: operand rotation, prefill read, merge, R_v^T;
//   4. the short requests' paged read, whose merge writes their output rows.
// The rotated short queries are taken before anything is written to the
// output.  The long requests' scratch is free again when the short read's
// partials take its place (one stream).
//
// A step of 7 x 4 + 1024 tokens took 424 us of host time for 26 launches when
// Python drove the parts (gathers, library products, conversions and copies
// between them) around 175 us of GPU work; it takes 120 in nine launches now.
#include "prefill_operands.h"
#include "step_launch.h"

namespace oscar {
namespace {

struct StepPlan {
  int32_t shorts, short_tokens, max_query_len;
  int64_t max_history;
  size_t layout, q_rot, k_rot, v_rot, rest, total;   // workspace offsets; rest: prefill scratch, then partials
  size_t rest_bytes;
};

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// The long requests of one prefill launch.
struct LongBatch {
  int32_t n;
  int32_t first[kMaxPrefillItems], fresh[kMaxPrefillItems], row[kMaxPrefillItems];
  int64_t cached[kMaxPrefillItems];
};

// Fills b with the next long requests from request i on; false when none is left.
bool next_batch(LongBatch& b, int32_t& i, int32_t num_requests, const int32_t* qsl, const int32_t* seqs,
                int32_t max_short) {
  b.n = 0;
  for (; i < num_requests && b.n < kMaxPrefillItems; ++i) {
    const int32_t nq = qsl[i + 1] - qsl[i];
    if (nq <= max_short || nq <= 0) continue;
    b.first[b.n] = qsl[i];
    b.fresh[b.n] = nq;
    b.cached[b.n] = (int64_t)seqs[i] - nq;
    b.row[b.n++] = i;
  }
  return b.n > 0;
}

int plan_step(StepPlan& p, int32_t num_requests, const int32_t* qsl, const int32_t* seqs, int32_t num_heads,
              int32_t num_kv_heads, int32_t max_short) {
  p = StepPlan{};
  if (num_requests <= 0 || !qsl || !seqs || num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads ||
      max_short < 0 || qsl[0] != 0)
    return kErrInvalidArgument;
  for (int32_t i = 0; i < num_requests; ++i) {
    const int32_t nq = qsl[i + 1] - qsl[i];
    if (nq < 0 || seqs[i] < nq) return kErrInvalidArgument;
    if (nq == 0 || nq > max_short) continue;
    ++p.shorts;
    p.short_tokens += nq;
    p.max_query_len = nq > p.max_query_len ? nq : p.max_query_len;
    p.max_history = seqs[i] - nq > p.max_history ? seqs[i] - nq : p.max_history;
  }
  size_t o = align256((2 * (size_t)num_requests + 1) * sizeof(int32_t));
  p.q_rot = o;
  o = align256(o + (size_t)p.short_tokens * num_heads * kHeadDim * sizeof(float));
  p.k_rot = o;
  o = align256(o + (size_t)p.short_tokens * num_kv_heads * kHeadDim * sizeof(float));
  p.v_rot = o;
  o = align256(o + (size_t)p.short_tokens * num_kv_heads * kHeadDim * sizeof(float));
  p.rest = o;
  if (p.shorts > 0) {
    p.rest_bytes = oscar_paged_decode_workspace_bytes(p.shorts, num_kv_heads, num_heads, p.max_query_len,
                                                      p.max_history, 0);
    if (p.rest_bytes == 0) return kErrInvalidArgument;
  }
  LongBatch b;
  for (int32_t i = 0; next_batch(b, i, num_requests, qsl, seqs, max_short);) {
    const size_t n = oscar_prefill_rotated_workspace_bytes(b.n, b.fresh, b.cached, num_heads, num_kv_heads);
    if (n == 0) return kErrInvalidArgument;
    p.rest_bytes = n > p.rest_bytes ? n : p.rest_bytes;
  }
  p.total = o + p.rest_bytes;
  return kOk;
}

}  // namespace
}  // namespace oscar

using namespace oscar;

extern "C" size_t oscar_step_forward_workspace_bytes(int32_t num_requests, const int32_t* query_start_loc,
                                                     const int32_t* seq_lens, int32_t num_heads, int32_t num_kv_heads,
                                                     int32_t max_short) {
  StepPlan p;
  return plan_step(p, num_requests, query_start_loc, seq_lens, num_heads, num_kv_heads, max_short) == kOk ? p.total
                                                                                                          : 0;
}

extern "C" int oscar_step_forward(const oscar_mtp_layer* layer, const void* rot_k_operand, const void* rot_v_operand,
                                  const void* rot_v_t_operand, int64_t* seat_winner, const void* query_bf16,
                                  int64_t query_token_stride, const void* key_bf16, const void* value_bf16,
                                  int64_t kv_token_stride, const int64_t* slot_mapping, const int32_t* block_table,
                                  int64_t block_table_stride, int32_t block_table_cols,
                                  const int32_t* query_start_loc, const int32_t* seq_lens, int32_t num_requests,
                                  int32_t max_short, void* out_bf16, void* workspace, size_t workspace_size,
                                  hipStream_t stream) {
  if (!layer) return kErrInvalidArgument;
  const oscar_mtp_layer& L = *layer;
  if (L.head_size != kHeadDim) return kErrUnsupportedHeadDim;
  StepPlan p;
  int rc = plan_step(p, num_requests, query_start_loc, seq_lens, L.num_heads, L.num_kv_heads, max_short);
  if (rc != kOk) return rc;
  const int32_t num_tokens = query_start_loc[num_requests];
  if (num_tokens == 0) return kOk;
  const int64_t width = (int64_t)L.num_heads * kHeadDim;
  if (!rot_k_operand || !rot_v_operand || !rot_v_t_operand || !L.rot_k || !L.rot_v || !L.rot_v_t || !query_bf16 ||
      !key_bf16 || !value_bf16 || !slot_mapping || !block_table || !out_bf16 || query_token_stride < width ||
      kv_token_stride < (int64_t)L.num_kv_heads * kHeadDim || block_table_cols <= 0 || L.block_size <= 0 ||
      L.num_pages <= 0 || L.stage_rows < 0 || L.sink_eff < 0 || L.recent < 0)
    return kErrInvalidArgument;
  if ((query_token_stride & 7) || (kv_token_stride & 7) || (reinterpret_cast<uintptr_t>(query_bf16) & 15) ||
      (reinterpret_cast<uintptr_t>(key_bf16) & 15) || (reinterpret_cast<uintptr_t>(value_bf16) & 15) ||
      (reinterpret_cast<uintptr_t>(out_bf16) & 15) || (reinterpret_cast<uintptr_t>(workspace) & 15) ||
      (reinterpret_cast<uintptr_t>(L.rot_k) & 15) || (reinterpret_cast<uintptr_t>(L.rot_v) & 15))
    return kErrInvalidArgument;
  if (L.stage_rows > 0 && (!L.stage_k || !L.stage_v || !L.stage_owner || !L.stage_k_image || !L.stage_v_image ||
                           !seat_winner || (reinterpret_cast<uintptr_t>(L.stage_k) & 15) ||
                           (reinterpret_cast<uintptr_t>(L.stage_v) & 15) ||
                           (reinterpret_cast<uintptr_t>(L.stage_k_image) & 15) ||
                           (reinterpret_cast<uintptr_t>(L.stage_v_image) & 15)))
    return kErrInvalidArgument;
  if (L.block_size % 32) return kErrUnsupportedGeometry;
  if (workspace == nullptr || workspace_size < p.total) return kErrWorkspaceTooSmall;
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  const uint16_t* q = static_cast<const uint16_t*>(query_bf16);
  const uint16_t* k = static_cast<const uint16_t*>(key_bf16);
  const uint16_t* v = static_cast<const uint16_t*>(value_bf16);

  float* q_rot = reinterpret_cast<float*>(ws + p.q_rot);
  float* k_rot = reinterpret_cast<float*>(ws + p.k_rot);
  float* v_rot = reinterpret_cast<float*>(ws + p.v_rot);
  auto read_long = [&](const LongBatch& b, const FusedWriteArgs* write, bool check_only) {
    return prefill_rotated(query_bf16, query_token_stride, key_bf16, value_bf16, kv_token_stride, b.n, b.first, b.fresh,
                           b.cached, b.row, L.num_heads, L.num_kv_heads, L.head_size, rot_k_operand, rot_v_operand,
                           rot_v_t_operand, L.k_cache, L.v_cache, L.block_size, L.num_pages, L.k_stride_page,
                           L.k_stride_token, L.k_stride_head, L.v_stride_page, L.v_stride_token, L.v_stride_head,
                           block_table, block_table_stride, block_table_cols,
                           L.stage_rows > 0 ? L.stage_k : nullptr, L.stage_rows > 0 ? L.stage_v : nullptr,
                           L.stage_rows > 0 ? L.stage_owner : nullptr, L.stage_rows, L.scale, out_bf16, ws + p.rest,
                           p.rest_bytes, write, check_only, stream);
  };
  auto read_short = [&](bool check_only) {
    return launch_decode_spans(L, DecodeSpans{q_rot, k_rot, v_rot, query_start_loc, seq_lens, num_requests, max_short,
                                              p.max_query_len, p.max_history, block_table, block_table_stride,
                                              block_table_cols},
                               out_bf16, width, ws + p.rest, p.rest_bytes, check_only, stream);
  };

  // Whatever a part of the step refuses is refused before the first launch
  // (the write's own checks precede its launches, which come first).
  LongBatch b;
  int32_t next = 0;
  while (next_batch(b, next, num_requests, query_start_loc, seq_lens, max_short))
    if ((rc = read_long(b, nullptr, true)) != kOk) return rc;
  if (p.shorts > 0 && (rc = read_short(true)) != kOk) return rc;

  next = 0;
  const bool any_long = next_batch(b, next, num_requests, query_start_loc, seq_lens, max_short);
  FusedWriteArgs write;
  bool waits = false;
  rc = quant_write_step(L, rot_k_operand, rot_v_operand, seat_winner, key_bf16, value_bf16, kv_token_stride,
                        num_tokens, slot_mapping, query_start_loc, seq_lens, num_requests,
                        reinterpret_cast<int32_t*>(ws + p.layout), any_long ? &write : nullptr, &waits, stream);
  if (rc != kOk) return rc;

  if (p.shorts > 0) {
    TokenRuns runs{};
    int64_t done = 0;                                // packed tokens of earlier launches
    auto flush = [&]() {
      const int64_t kv = done * L.num_kv_heads * kHeadDim;
      const int st = launch_rotate_runs(q, query_token_stride, k, v, kv_token_stride, runs, L.num_heads,
                                        L.num_kv_heads, L.rot_k, L.rot_v, q_rot + done * width, k_rot + kv,
                                        v_rot + kv, stream);
      done += runs.tokens;
      runs = TokenRuns{};
      return st;
    };
    for (int32_t i = 0; i < num_requests; ++i) {
      const int32_t tok = query_start_loc[i], nq = query_start_loc[i + 1] - tok;
      if (nq <= 0 || nq > max_short) continue;
      const int32_t r = runs.n - 1;
      if (r < 0 || runs.tok[r] + (runs.tokens - runs.pos[r]) != tok) {      // no run that ends here
        if (runs.n == kMaxTokenRuns && (rc = flush()) != kOk) return rc;
        runs.pos[runs.n] = runs.tokens;
        runs.tok[runs.n++] = tok;
      }
      runs.tokens += nq;
    }
    if (runs.n > 0 && (rc = flush()) != kOk) return rc;
  }

  for (bool more = any_long; more;
       more = next_batch(b, next, num_requests, query_start_loc, seq_lens, max_short)) {
    if ((rc = read_long(b, waits ? &write : nullptr, false)) != kOk) return rc;
    waits = false;
  }

  return p.shorts > 0 ? read_short(false) : (int)kOk;
}
