// MFMA operands of the prefill read's new tokens (gfx950): what the rotation
// (or the fp32 conversion) writes to HBM and the prefill kernel reads.
//
//   q16  [rows][256] fp16, row = compact token * Hq + head; 16-byte chunk
//        c = 2m + g of a row is the Q^T operand of k-step m, lane half g:
//        positions 8g .. 8g + 7 of the step's 16 features (k_feature order);
//   qsum [rows] fp32, the sum of a row's fp16 values;
//   kimg [tile][Hk][32 tokens][256] fp16, vimg [tile][Hk][256 features][32
//        tokens] fp16: a 32-token key block exactly as the kernel keeps it in
//        LDS (16 KB each), so that a block is a straight copy.  A request's
//        tiles start at its own first token; tokens past its last repeat it.
//
// LDS tiles, shared with the history tiles the kernel builds from codes:
//   K: row = token (512 bytes), chunk c of a token at k_chunk(c, token): the
//      sixteen tokens that an operand read takes together, and the sixteen
//      chunks that sixteen threads of one token store together, fall into
//      sixteen different 16-byte slots of the 64 banks.
//   V: row = feature (64 bytes), chunk 2mm + g holds the eight tokens
//      16mm + 8e + 4g + i (e = 0, 1; i = 0 .. 3) that lane half g multiplies
//      in PV k-step mm, at v_chunk(2mm + g, feature): one 16-byte read per
//      operand, conflict-free along features.
#pragma once

#include "bulk_write.h"
#include "oscar_common.h"

namespace oscar {

constexpr int kKeyBlk = 32;                                 // keys per block
constexpr int kKeyTileHalfs = kKeyBlk * kHeadDim;           // one K or V tile: 16 KB

__host__ __device__ __forceinline__ constexpr int k_chunk(int c, int token) {
  return (c & 16) | ((c & 15) ^ (c >> 4) ^ (token & 15));
}
__host__ __device__ __forceinline__ constexpr int v_chunk(int c, int feature) { return c ^ ((feature >> 2) & 3); }

// Position p of a 16-feature group is feature (p >> 1) + 8 (p & 1): one shift
// and mask of a code dword yields a pair.
__host__ __device__ __forceinline__ constexpr int k_feature(int p) { return (p >> 1) + 8 * (p & 1); }

// The long requests of a launch, in the kernel arguments.
constexpr int kMaxPrefillItems = 48;
struct OperandItem {
  int32_t tok0;     // first new token in the inputs
  int32_t n_new;    // new tokens
  int32_t ctok0;    // first compact token (q16 / qsum rows)
  int32_t tile0;    // first key tile
};
struct OperandItems {
  int32_t n;
  int32_t tokens, tiles;     // compact tokens and key tiles of all items
  OperandItem it[kMaxPrefillItems];
};

struct PrefillOperands {
  _Float16* q16;
  float* qsum;
  _Float16* kimg;
  _Float16* vimg;
};

// quant_write.hip: operands from bf16 query / key / value, rotated on MFMA,
// and in the same launch the bulk write in `write`, if there is one.
int launch_rotate_operands(const uint16_t* q, int64_t q_stride, const uint16_t* k, const uint16_t* v,
                           int64_t kv_stride, int32_t num_heads, int32_t num_kv_heads, const uint8_t* rot_k,
                           const uint8_t* rot_v, const OperandItems& items, const PrefillOperands& o,
                           const FusedWriteArgs* write, hipStream_t stream);

}  // namespace oscar
