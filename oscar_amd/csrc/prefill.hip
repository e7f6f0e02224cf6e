// Prefill continuation: causal attention of the new tokens of one or more
// requests over each request's C cached INT2 tokens plus themselves (gfx950,
// f16 MFMA).
//
// Semantics (reference dense path): keys 0 .. C-1 are the dequantized history
// (owner-matched FP32 staging values override INT2), keys C .. C+N-1 are the
// new tokens; new token j (absolute position C + j) sees keys 0 .. C + j.
// MFMA operands are rounded to fp16: the same MFMA rate as bf16 (the
// reference runs this attention in the model's bf16 dtype) with 3 more
// mantissa bits, which keeps softmax-weight rounding below the bf16 output
// tolerance even on x8 outlier channels.  Accumulation and softmax are fp32.
// Rotated domain in, rotated-V domain out (fp32).
//
// Work: a row is (new token j, head in group) of one kv head; a workgroup of
// eight wavefronts takes 256 consecutive rows (32 per wavefront) and walks
// their keys in 32-key blocks, history blocks first, then new-token blocks
// (from the request's first new token).
//
// Split (oscar_prefill_* with a workspace): the launch's row blocks, each as
// long as its key blocks, form one line of units; every workgroup (one per CU)
// takes an equal share of it, whatever row blocks that cuts.  A row block that
// lies in one share is finished there; of a cut one each share writes fp32
// partials (m, l, unnormalised O), which prefill_merge_kernel combines.  Reads of
// fp32 rows without a workspace, or of few key blocks, take whole row blocks
// instead (prefers_rows, prefers_rows_shares).
//
// A block is two phases of a wavefront:
//   M (matrix): O^T += V^T P^T of block i - 1 and S^T = K Q^T of block i (16
//     MFMA 32x32x16 each), and under them this wave's part of the tiles K of
//     block i + 1 and V of block i, built from codes loaded a block ahead
//     (new-token tiles are copied to LDS as they are, prefill_operands.h);
//   S (softmax): base-2 online softmax of block i with a lazily raised running
//     max, in registers.
// One barrier per block, after S for wavefronts 0-3 and after M for 4-7: in
// the interval between two barriers the former run M then S, the latter S
// then M, so that on every SIMD one wave's MFMAs run under the other's
// softmax.  K and V tiles are double-buffered in LDS (16 KB each); Q^T's first
// kQReg k-steps stay in registers, the rest in LDS.
//
// What bounds it: the operand reads' LDS latency.  A phase M issues its 32
// MFMAs in 2300 cycles where they need 1024 (timestamps), reads two pairs
// ahead being what 256 registers hold; S takes 1100-1400.  Without a tile's
// build, its loads, its exponentials or its PV it is 8-13 % faster each.  Two
// barriers per block with the wavefronts 4-7 a phase behind (1.19x slower),
// operand rows that two of sixteen lanes read from one bank slot (LDS active
// 45 % against 29 % of the time), and workgroups of four wavefronts, two per
// CU (1.25x slower) were left behind.  Before and after its blocks a piece
// takes about 5 and 2.5 us: unit, pages and Q^T, first words, first tile; and
// the partial.  One request, 6 heads, D = 256, this kernel: 9256 tokens over
// 15360 1988 -> 1200 us, 77 over 20011 1016 -> 34 us, 3001 alone 170 -> 50 us.
#include <algorithm>
#include <type_traits>
#include <utility>

#include "prefill_operands.h"
#include "step_launch.h"
#include "../../include/oscar_amd.h"

namespace oscar {
namespace {

constexpr int kBlk = kKeyBlk;
constexpr int kRowsPerWave = 32;
constexpr int kWaves = 8;
constexpr int kTileRows = kWaves * kRowsPerWave;
constexpr int kQReg = 4;              // k-steps whose Q^T operand stays in registers
constexpr int kAhead = 2;             // operand reads ahead of their MFMAs, in pairs
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLazy = 8.f;          // log2 headroom before a running max is raised
constexpr float kVsMax = 240.f;       // p vs stays below 2^kLazy * 240 < 65504 (fp16) under the lazy max
constexpr int kPartRows = kTileRows;
constexpr size_t kPartFloats = (size_t)kPartRows * (kHeadDim + 2);   // O rows, then m, then l
constexpr int kShares = 256;          // workgroups resident at once: one per CU
// A piece of a row block costs as much as this many of its key blocks before
// and after them (page lookup, Q^T, first tile; output or partial, which the
// output pass reads again): 7.5 us and that pass against 2.1 us a block.  (4
// to 7 are within 2 us of each other on the cases timed.)
constexpr int kPieceCost = 5;
constexpr int kMinShare = 5;          // units a share takes at least (see plan_share)
constexpr int kMergeManyPieces = 6;   // partials a row from which its merge takes four waves

struct PrefillItem {
  int64_t unit0;       // first unit of the item: kPieceCost, then one per key block, for each row block of
                       // each kv head
  int64_t head_units;  // units per kv head
  int32_t n_new;       // N
  int32_t cached;      // C
  int32_t req;         // block-table row
  int32_t tok0;        // first token in q / k_new / v_new / out (fp32 inputs: of the whole call)
  int32_t tile0;       // first new-token key tile
  int32_t rb0;         // first row block of the item (kv heads x row blocks)
  int32_t out0;        // first token in the step's output (rotated output)
};

struct PrefillArgs {
  const _Float16* q16;   // operands (prefill_operands.h), or null: the fp32 rows below
  const float* qsum;
  const _Float16* kimg;
  const _Float16* vimg;
  const float* q;        // [N][Hq][D]
  const float* k_new;    // [N][Hk][D]
  const float* v_new;
  int32_t num_heads, num_kv_heads, group;
  const uint8_t* k_cache;
  const uint8_t* v_cache;
  int64_t k_page, k_tok, k_head, v_page, v_tok, v_head;
  int32_t block_size;
  FastDiv bs_div;        // block_size
  FastDiv rows_div;      // stage_rows (1 without an arena)
  int64_t num_pages;
  const int32_t* bt;
  int64_t bt_stride;
  int32_t bt_cols;
  const float* stage_k;
  const float* stage_v;
  const int64_t* owner;
  int32_t stage_rows;
  float scale_log2;
  float* out;
  float* part;           // partial slots (two per share), or null: a workgroup takes a whole row block
  int64_t share;         // units per workgroup
  int64_t units;
  int32_t nitems;
  PrefillItem items[kMaxPrefillItems];
};

struct PrefillLds {
  _Float16 k[2][kKeyTileHalfs];         // K of block i in k[i & 1], V in v[i & 1]
  _Float16 v[2][kKeyTileHalfs];
  __attribute__((aligned(16))) _Float16 q[kWaves][16 - kQReg][64 * 8];   // Q^T operands of the k-steps past kQReg
};
constexpr size_t kPrefillLds = sizeof(PrefillLds);
static_assert(kPrefillLds <= 160 * 1024, "LDS of one workgroup");

__device__ __forceinline__ _Float16 to_h(float x) { return (_Float16)x; }

__device__ __forceinline__ void wave_sync_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// s_barrier without __syncthreads' memory fence (which would also wait for
// the outstanding global loads); LDS writes are complete at lgkmcnt(0).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt(0xC07F);       // lgkmcnt(0); vmcnt and expcnt left at their maxima
  asm volatile("s_barrier" ::: "memory");
}

// ... and with every copy to LDS of this wave complete (vmcnt(0)).
__device__ __forceinline__ void copy_barrier() {
  __builtin_amdgcn_s_waitcnt(0x0070);       // vmcnt(0), lgkmcnt(0), expcnt left at its maximum
  asm volatile("s_barrier" ::: "memory");
}

__device__ __forceinline__ int row_blocks(const PrefillItem& it, int group) {
  return (int)(((int64_t)it.n_new * group + kTileRows - 1) / kTileRows);
}
__device__ __forceinline__ int hist_blocks(const PrefillItem& it) { return (it.cached + kBlk - 1) / kBlk; }
// Key blocks of row block rb: its last row's token sees new tokens 0 .. that token.
__device__ __forceinline__ int key_blocks(const PrefillItem& it, int group, int rb) {
  const int64_t last = min((int64_t)(rb + 1) * kTileRows, (int64_t)it.n_new * group) - 1;
  return hist_blocks(it) + (int)(last / group) / kBlk + 1;
}

__device__ __forceinline__ int rb_units(const PrefillItem& it, int group, int rb) {
  return kPieceCost + key_blocks(it, group, rb);
}

// Sum over the lanes up to and including this one (wave-wide, DPP).
__device__ __forceinline__ uint32_t wave_scan(uint32_t x) {
  auto up = [](uint32_t v, auto ctrl, auto rows) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, decltype(ctrl)::value, decltype(rows)::value, 0xF, false);
  };
  using std::integral_constant;
  x += up(x, integral_constant<int, 0x111>{}, integral_constant<int, 0xF>{});     // row_shr:1, 2, 4, 8
  x += up(x, integral_constant<int, 0x112>{}, integral_constant<int, 0xF>{});
  x += up(x, integral_constant<int, 0x114>{}, integral_constant<int, 0xF>{});
  x += up(x, integral_constant<int, 0x118>{}, integral_constant<int, 0xF>{});
  x += up(x, integral_constant<int, 0x142>{}, integral_constant<int, 0xA>{});     // row_bcast:15 into rows 1 and 3
  x += up(x, integral_constant<int, 0x143>{}, integral_constant<int, 0xC>{});     // row_bcast:31 into rows 2 and 3
  return x;
}

// The sum of 64 row blocks' units as a wave scan, in two 32-bit halves: a row
// block has less than 2^28 units, so 16 low bits of each sum below 2^22 and
// the rest below 2^18.
__device__ __forceinline__ int64_t units_scan(int n) {
  return ((int64_t)wave_scan((uint32_t)n >> 16) << 16) + wave_scan((uint32_t)n & 0xFFFFu);
}
__device__ __forceinline__ int64_t lane64(int64_t x, int lane) {
  return (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(x >> 32), lane) << 32) |
                   (uint32_t)__builtin_amdgcn_readlane((int)x, lane));
}

// Units of the item's row blocks before rb (every lane of the wave calls it
// with the same rb).
__device__ __forceinline__ int64_t units_before(const PrefillItem& it, int group, int rb, int lane) {
  int64_t n = 0;
  for (int base = 0; base < rb; base += 64)
    n += lane64(units_scan(base + lane < rb ? rb_units(it, group, base + lane) : 0), 63);
  return n;
}

// Row block of unit u (relative to the kv head's first), and u within it: a
// wave-wide scan over 64 row blocks a time.
__device__ __forceinline__ void locate_unit(const PrefillItem& it, int group, int64_t u, int lane, int& rb,
                                            int& at_unit) {
  const int nrb = row_blocks(it, group);
  for (int base = 0;; base += 64) {
    const int b = base + lane;
    const int n = b < nrb ? rb_units(it, group, b) : 0;
    const int64_t incl = units_scan(n);
    const int64_t total = lane64(incl, 63);
    if (u < total || base + 64 >= nrb) {
      const int at = min(__popcll(__ballot(incl <= u)), 63);
      rb = base + at;
      at_unit = (int)(u - (lane64(incl, at) - __builtin_amdgcn_readlane(n, at)));
      return;
    }
    u -= total;
  }
}

// A V slot's code word and four fp32 values where the caller's strides and
// addresses promise less than their size (any V stride; an output or an arena
// aligned to its elements): the same one instruction each.
typedef uint32_t u32_any __attribute__((aligned(1)));
typedef floatx4 floatx4_any __attribute__((aligned(4)));

// Raw bytes of one history block for one thread of wave w: K role (token 4w +
// lane / 16, code word lane % 16: features 16 (lane % 16) .. +15) and owner
// tag of token lane % 32; V role (token 4w + lane % 4, code word lane / 4);
// meta of the key whose parameters this lane holds (par_key).  Every thread
// issues its loads whatever the block holds (tokens past C and invalid pages
// read an in-bounds slot, masked later).
struct KLoad {
  uint32_t kc;
  int32_t own;
};

// Score register q of lane half g is key 8 (q / 4) + 4g + q % 4 of the block:
// lane q of each 16-lane row of half g holds that key's parameters.
__device__ __forceinline__ int par_key(int lane) { return 8 * ((lane >> 2) & 3) + 4 * (lane >> 5) + (lane & 3); }

// What the block loop reads every block, per segment (uniform).  The rest of
// the arguments (the window arena's values) is read where it is needed,
// through cold_args: kept in registers it spilled others of the loop.
struct Hot {
  const uint8_t* kbase;      // this kv head's slots of page 0
  const uint8_t* vbase;
  int64_t k_page, v_page;
  uint32_t ktok, vtok;
  const int64_t* owner;      // null: no arena
  const int32_t* bt_row;
  int32_t num_pages, bt_cols, cached, block_size;
  FastDiv bs_div, rows_div;
  float scale_log2;
};

typedef __attribute__((address_space(4))) const PrefillArgs const_args;
__device__ __forceinline__ const const_args* cold_args() {
  const const_args* p = (const const_args*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
}

// A thread's byte offsets: into a page's slots (ko, vo, mo), of its chunks in
// the tiles it builds (ks, vs) and of the operands it reads (kr, vr).  The
// tile offsets differ between chunks by bit flips only (see k_chunk, v_chunk),
// so one register each serves all of them.
struct Roles {
  uint32_t ko, vo, mo;
  uint32_t ks, vs, kr, vr;
};

// Keeps a loop-invariant value from being expanded into one register per use.
__device__ __forceinline__ uint32_t opaque(uint32_t x) {
  asm volatile("" : "+v"(x));
  return x;
}

__device__ __forceinline__ Roles make_roles(uint32_t k_tok, uint32_t v_tok, int w, int lane) {
  Roles r;
  const int t32 = lane & 31, ktt = 4 * w + (lane >> 4), par = (lane >> 2) & 3;
  r.ko = (uint32_t)ktt * k_tok + kKCodeOff + 4 * (lane & 15);
  r.vo = (uint32_t)(4 * w + (lane & 3)) * v_tok + 4 * (lane >> 2);
  r.mo = (uint32_t)par_key(lane) * k_tok;
  r.ks = ktt * 512 + 16 * k_chunk(2 * (lane & 15), ktt);
  // tokens 4w .. 4w + 3 of feature 4 lane + par (see v_slot)
  r.vs = (4 * lane + par) * 64 + 16 * v_chunk(2 * (w >> 2) + (w & 1), 4 * lane) + 8 * ((w >> 1) & 1);
  r.kr = t32 * 512 + 16 * ((lane >> 5) ^ (lane & 15));
  r.vr = t32 * 64 + 16 * v_chunk(lane >> 5, t32);
  return r;
}

// Pages of the 64 history blocks from block b on, one a lane (negative: none);
// checked against the pool where they are taken out.
__device__ __forceinline__ int32_t load_pages(const Hot& h, int b, int lane) {
  const uint32_t k0 = (uint32_t)(b + lane) * kBlk, pidx = fast_div(k0, h.bs_div);
  const bool ok = k0 < (uint32_t)h.cached && pidx < (uint32_t)h.bt_cols;
  const int32_t p = h.bt_row[ok ? pidx : 0];
  return ok ? p : -1;
}
__device__ __forceinline__ int32_t valid_page(const Hot& h, int32_t page) { return page < h.num_pages ? page : -1; }

__device__ __forceinline__ KLoad load_k(const Hot& h, int k0, int32_t page, const Roles& r, int lane) {
  KLoad L;
  const int64_t pg = page >= 0 ? page : 0;
  const uint32_t prow0 = fast_mod((uint32_t)k0, h.bs_div);
  const uint8_t* kp = h.kbase + pg * h.k_page + (uint64_t)prow0 * h.ktok;
  L.kc = *reinterpret_cast<const uint32_t*>(kp + r.ko);
  // Owner tags are pages (< 2^31) or -1: the low word of the little-endian
  // int64 identifies them.  Without an arena the slots' own bytes stand in.
  const uint8_t* op = h.owner != nullptr
                          ? reinterpret_cast<const uint8_t*>(
                                h.owner + (int64_t)fast_mod((uint32_t)pg, h.rows_div) * h.block_size + prow0)
                          : kp;
  L.own = *reinterpret_cast<const int32_t*>(op + 8 * (lane & 31));
  return L;
}

__device__ __forceinline__ u32x2 load_meta(const Hot& h, int k0, int32_t page, const Roles& r) {
  const int64_t pg = page >= 0 ? page : 0;
  return *reinterpret_cast<const u32x2*>(h.kbase + pg * h.k_page +
                                         (uint64_t)fast_mod((uint32_t)k0, h.bs_div) * h.ktok + r.mo);
}

__device__ __forceinline__ uint32_t load_v(const Hot& h, int k0, int32_t page, const Roles& r) {
  const int64_t pg = page >= 0 ? page : 0;
  const uint8_t* vp = h.vbase + pg * h.v_page + (uint64_t)fast_mod((uint32_t)k0, h.bs_div) * h.vtok;
  return *reinterpret_cast<const u32_any*>(vp + r.vo);
}

// fp16 pair (1 + c/4) of the codes at bits [sh, sh + 2) and [sh + 16, sh + 18)
// of w (exact: 1, 1.25, 1.5, 1.75).
__device__ __forceinline__ uint32_t magic_pair(uint32_t w, int sh) {
  const uint32_t x = sh < 8 ? (w << (8 - sh)) : (w >> (sh - 8));
  return (x & 0x03000300u) | 0x3C003C00u;
}

typedef _Float16 half4 __attribute__((ext_vector_type(4)));

// A thread's two K chunks and its four V features (feature 4 lane + f holds
// tokens 4w .. +3) in the tiles.
__device__ __forceinline__ half8* k_slot(_Float16* kt, uint32_t ks, int e) {
  return reinterpret_cast<half8*>(reinterpret_cast<uint8_t*>(kt) + (ks ^ (16u * e)));
}
// f stands for feature f ^ par of the lane's four, par = (lane / 4) % 4, so
// that sixteen lanes store into sixteen different 16-byte slots of the banks.
__device__ __forceinline__ void* v_slot(_Float16* vt, uint32_t vs, int f) {
  return reinterpret_cast<uint8_t*>(vt) + (vs ^ (64u * f));
}

// A thread's 16 K values (features 16 k16 .. +15, fp32) into its token's row.
__device__ __forceinline__ void store_k_values(const floatx4 (&x)[4], uint32_t ks, _Float16* kt) {
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    half8 h;
#pragma unroll
    for (int e = 0; e < 8; ++e) h[e] = to_h(x[k_feature(8 * g + e) >> 2][k_feature(8 * g + e) & 3]);
    *k_slot(kt, ks, g) = h;
  }
}

// History tiles as code operands: K' = V' = 1 + c/4 (exact in fp16) with the
// token's scale and zero moved into per-key parameters: k = 4s K' + (z - 4s),
// so a score is ta (K'.q) + tb sum(q) with ta = 4 s_k, tb = z_k - 4 s_k (times
// the softmax scale), and v = vs V' + vz with vs = 4 s_v, vz = z_v - 4 s_v.
// Tokens the staging arena owns (rare: the sink / recent window) keep their
// FP32 values (rounded to fp16) with ta = scale, tb = 0, vs = 1, vz = 0.  Keys
// past C or on an unmapped page get all-zero parameters (an unmapped page
// reads as zeros; keys past C are masked by the consumer).

// Bits of the block's window-owned tokens; live: live tokens of the block.
__device__ __forceinline__ uint32_t window_mask(const Hot& h, int32_t own, int live, int32_t page, int lane) {
  return (uint32_t)__ballot(h.owner != nullptr && (lane & 31) < live && own == page);
}

__device__ __forceinline__ int live_tokens(const Hot& h, int k0, int32_t page) {
  return page >= 0 ? h.cached - k0 : 0;
}

__device__ __forceinline__ const float* stage_row(bool value, int32_t page, int k0, int t, int kvh) {
  const const_args* a = cold_args();
  const FastDiv rows{a->rows_div.d, a->rows_div.m, a->rows_div.l}, bs{a->bs_div.d, a->bs_div.m, a->bs_div.l};
  const int64_t seat = (int64_t)fast_mod((uint32_t)page, rows) * a->block_size + fast_mod((uint32_t)k0, bs) + t;
  return (value ? a->stage_v : a->stage_k) + (seat * a->num_kv_heads + kvh) * kHeadDim;
}

// This thread's part of the K tile from its code word: chunk e ...
__device__ __forceinline__ void build_k(uint32_t w, uint32_t ks, _Float16* kt, int e) {
  *k_slot(kt, ks, e) = __builtin_bit_cast(half8, u32x4{magic_pair(w, 8 * e), magic_pair(w, 8 * e + 2),
                                                       magic_pair(w, 8 * e + 4), magic_pair(w, 8 * e + 6)});
}

// ... and of the V tile: the four tokens' code words of a lane quad, byte
// transposed (lane j of the quad gets byte j of each), then the codes of its
// byte's four features as fp16 of the four tokens.
template <int kCtrl>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kCtrl, 0xF, 0xF, true);
}
__device__ __forceinline__ uint32_t quad_transpose(uint32_t x, int lane) {
  const uint32_t q0 = dpp_u32<0x00>(x), q1 = dpp_u32<0x55>(x), q2 = dpp_u32<0xAA>(x), q3 = dpp_u32<0xFF>(x);
  const uint32_t sel = 0x0400u + 0x0101u * (uint32_t)(lane & 3);      // byte j of both words
  const uint32_t lo = __builtin_amdgcn_perm(q1, q0, sel), hi = __builtin_amdgcn_perm(q3, q2, sel);
  return __builtin_amdgcn_perm(hi, lo, 0x05040100u);
}
__device__ __forceinline__ void build_v(uint32_t w, uint32_t vs, _Float16* vt, int f) {     // w: quad_transpose
  const uint32_t y = ((w >> (((vs >> 5) & 6u) ^ (2u * f))) & 0x03030303u) | 0x3C3C3C3Cu;
  // bytes {0, y.b0, 0, y.b1} and {0, y.b2, 0, y.b3}
  *reinterpret_cast<u32x2*>(v_slot(vt, vs, f)) =
      u32x2{__builtin_amdgcn_perm(0u, y, 0x010C000Cu), __builtin_amdgcn_perm(0u, y, 0x030C020Cu)};
}

// Window-owned tokens (rare), over what the builds above stored: their FP32
// values rounded to fp16, those of a K tile (kmask, page kpage, keys from k0)
// and of a V tile (vmask, its code words in x, page vpage, keys from v0).  The
// loads of both go out before either is waited for: a wait of its own for
// each cost a block 1 us.  (opaque: nothing of this is worth a register in the
// loop.)
__device__ __forceinline__ void window_tiles(uint32_t kmask, int32_t kpage, int k0, _Float16* kt, uint32_t vmask,
                                             uint32_t x, int32_t vpage, int v0, _Float16* vt, int kvh, const Roles& r,
                                             int w, int lane_) {
  const int lane = (int)opaque((uint32_t)lane_), t = 4 * w + (lane >> 4);
  const bool mine = ((kmask >> t) & 1u) != 0u;
  const uint32_t nib = (vmask >> (4 * w)) & 15u;
  floatx4 xk[4] = {}, y[4];
  if (mine) {
    const floatx4_any* src = reinterpret_cast<const floatx4_any*>(stage_row(false, kpage, k0, t, kvh) + 16 * (lane & 15));
#pragma unroll
    for (int e = 0; e < 4; ++e) xk[e] = src[e];
  }
  if (nib != 0u) {
    const uint32_t codes = quad_transpose(x, lane);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if ((nib >> k) & 1u)
        y[k] = *reinterpret_cast<const floatx4_any*>(stage_row(true, vpage, v0, 4 * w + k, kvh) + 4 * lane);
      else
#pragma unroll
        for (int e = 0; e < 4; ++e) y[k][e] = 1.f + 0.25f * (float)((codes >> (8 * k + 2 * e)) & 3u);
    }
  }
  if (mine) store_k_values(xk, opaque(r.ks), kt);
  if (nib != 0u) {
    const uint32_t vs = opaque(r.vs) ^ (64u * ((lane >> 2) & 3));      // (v_slot's f is then the feature)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      *reinterpret_cast<half4*>(v_slot(vt, vs, e)) = half4{to_h(y[0][e]), to_h(y[1][e]), to_h(y[2][e]), to_h(y[3][e])};
  }
}

// A value held by lane r of each 16-lane row, in every lane of the row.
template <int kLane>
__device__ __forceinline__ float row_bcast(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x150 + kLane, 0xF, 0xF, true));
}
// x[r] += y * (c of lane r of the row), r = 0 .. 15, and z += sum_r p[r] * (c of
// lane r): fused multiply-adds that take the broadcast as they read it (the
// compiler folds it into multiplies only and spends a move per broadcast
// otherwise).  The two wait states are those a DPP read needs after a VALU
// write of its source, which the compiler cannot see inside.
#define OSCAR_FMAC(dst, c, y, r) "v_fmac_f32_dpp " dst ", " c ", " y " row_newbcast:" #r " row_mask:0xf bank_mask:0xf\n\t"
__device__ __forceinline__ void fmac_bcast(float (&x)[16], float c, float y) {
  asm("s_nop 1\n\t"
      OSCAR_FMAC("%0", "%16", "%17", 0) OSCAR_FMAC("%1", "%16", "%17", 1) OSCAR_FMAC("%2", "%16", "%17", 2)
      OSCAR_FMAC("%3", "%16", "%17", 3) OSCAR_FMAC("%4", "%16", "%17", 4) OSCAR_FMAC("%5", "%16", "%17", 5)
      OSCAR_FMAC("%6", "%16", "%17", 6) OSCAR_FMAC("%7", "%16", "%17", 7) OSCAR_FMAC("%8", "%16", "%17", 8)
      OSCAR_FMAC("%9", "%16", "%17", 9) OSCAR_FMAC("%10", "%16", "%17", 10) OSCAR_FMAC("%11", "%16", "%17", 11)
      OSCAR_FMAC("%12", "%16", "%17", 12) OSCAR_FMAC("%13", "%16", "%17", 13) OSCAR_FMAC("%14", "%16", "%17", 14)
      OSCAR_FMAC("%15", "%16", "%17", 15)
      : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(x[4]), "+v"(x[5]), "+v"(x[6]), "+v"(x[7]), "+v"(x[8]),
        "+v"(x[9]), "+v"(x[10]), "+v"(x[11]), "+v"(x[12]), "+v"(x[13]), "+v"(x[14]), "+v"(x[15])
      : "v"(c), "v"(y));
}
__device__ __forceinline__ float dot_bcast(const float (&p)[16], float c, float z) {
  asm("s_nop 1\n\t"
      OSCAR_FMAC("%0", "%1", "%2", 0) OSCAR_FMAC("%0", "%1", "%3", 1) OSCAR_FMAC("%0", "%1", "%4", 2)
      OSCAR_FMAC("%0", "%1", "%5", 3) OSCAR_FMAC("%0", "%1", "%6", 4) OSCAR_FMAC("%0", "%1", "%7", 5)
      OSCAR_FMAC("%0", "%1", "%8", 6) OSCAR_FMAC("%0", "%1", "%9", 7) OSCAR_FMAC("%0", "%1", "%10", 8)
      OSCAR_FMAC("%0", "%1", "%11", 9) OSCAR_FMAC("%0", "%1", "%12", 10) OSCAR_FMAC("%0", "%1", "%13", 11)
      OSCAR_FMAC("%0", "%1", "%14", 12) OSCAR_FMAC("%0", "%1", "%15", 13) OSCAR_FMAC("%0", "%1", "%16", 14)
      OSCAR_FMAC("%0", "%1", "%17", 15)
      : "+v"(z)
      : "v"(c), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]), "v"(p[6]), "v"(p[7]), "v"(p[8]),
        "v"(p[9]), "v"(p[10]), "v"(p[11]), "v"(p[12]), "v"(p[13]), "v"(p[14]), "v"(p[15]));
  return z;
}
#undef OSCAR_FMAC
template <typename F, int... kI>
__device__ __forceinline__ void each16(F&& f, std::integer_sequence<int, kI...>) {
  (f(std::integral_constant<int, kI>{}), ...);
}

// New-token tiles copied as they are: kCopyWaves waves take equal parts.
typedef __attribute__((address_space(3))) void lds_void;
template <int kCopyWaves>
__device__ __forceinline__ void copy_tile(const _Float16* img, int64_t tile, _Float16* lds, int wave, int lane) {
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(img + tile * kKeyTileHalfs), (short)0, (int)(kKeyTileHalfs * sizeof(_Float16)), 0x00020000);
#pragma unroll
  for (int i = 0; i < 16 / kCopyWaves; ++i) {
    const int blk = 16 / kCopyWaves * wave + i;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void*)(lds + blk * 512), 16, (blk * 64 + lane) * 16, 0, 0, 0);
  }
}

// ... or, for callers without operands, rounded from the fp32 rows.
__device__ __forceinline__ void store_new_k(const PrefillArgs& a, const PrefillItem& it, int j0, int kvh,
                                            const Roles& r, int w, int lane, _Float16* kt) {
  const int j = min(j0 + 4 * w + (lane >> 4), it.n_new - 1);
  const floatx4* src = reinterpret_cast<const floatx4*>(
      a.k_new + ((int64_t)(it.tok0 + j) * a.num_kv_heads + kvh) * kHeadDim + 16 * (lane & 15));
  const floatx4 x[4] = {src[0], src[1], src[2], src[3]};
  store_k_values(x, r.ks, kt);
}
__device__ __forceinline__ void store_new_v(const PrefillArgs& a, const PrefillItem& it, int j0, int kvh,
                                            const Roles& r, int w, int lane, _Float16* vt) {
  const uint32_t vs = r.vs ^ (64u * ((lane >> 2) & 3));
  floatx4 x[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int j = min(j0 + 4 * w + k, it.n_new - 1);
    x[k] = *reinterpret_cast<const floatx4*>(
        a.v_new + ((int64_t)(it.tok0 + j) * a.num_kv_heads + kvh) * kHeadDim + 4 * lane);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    *reinterpret_cast<half4*>(v_slot(vt, vs, e)) = half4{to_h(x[0][e]), to_h(x[1][e]), to_h(x[2][e]), to_h(x[3][e])};
}

template <bool kImages>
__global__ __launch_bounds__(512, 2) void prefill_kernel(PrefillArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem_raw[];
  PrefillLds& S = *reinterpret_cast<PrefillLds*>(smem_raw);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5;
  const int col = lane & 31;
  const bool second = wave >= kWaves / 2;     // its barrier comes between M and S
  const Roles r = make_roles((uint32_t)a.k_tok, (uint32_t)a.v_tok, wave, lane);

  // ---- the workgroup's units [u, u1) ----
  int64_t u, u1;
  int item = 0, kvh, rb, ub;            // ub: u within row block rb
  if (a.part == nullptr) {
    // whole row blocks of one request, later ones (more keys) first
    const int nrb = row_blocks(a.items[0], a.group);
    kvh = (int)blockIdx.y;
    rb = nrb - 1 - (int)blockIdx.x;
    ub = 0;
    u = 0;
    u1 = rb_units(a.items[0], a.group, rb);
  } else {
    u = (int64_t)blockIdx.x * a.share;
    u1 = min(u + a.share, a.units);
    while (item + 1 < a.nitems && a.items[item + 1].unit0 <= u) ++item;
    const int64_t rel = u - a.items[item].unit0;
    kvh = rel < a.items[item].head_units ? 0 : (int)(rel / a.items[item].head_units);
    locate_unit(a.items[item], a.group, rel - (int64_t)kvh * a.items[item].head_units, lane, rb, ub);
  }

#pragma unroll 1
  while (u < u1) {
    const PrefillItem it = a.items[item];
    // this piece: units ub .. ub + take - 1 of the row block, key blocks kb .. kend - 1
    const int nblk = key_blocks(it, a.group, rb);
    const int take = (int)min((int64_t)(kPieceCost + nblk - ub), u1 - u);
    const int kb = max(ub - kPieceCost, 0), kend = ub + take - kPieceCost;
    const int64_t start = u + max(kPieceCost - ub, 0);    // unit of key block kb
    u += take;
    const int rb_now = rb, kvh_now = kvh;
    const bool rb_done = kend == nblk;
    ub = 0;
    if (rb_done && ++rb == row_blocks(it, a.group)) {
      rb = 0;
      if (++kvh == a.num_kv_heads) {
        kvh = 0;
        ++item;
      }
    }
    if (kend <= kb) continue;             // the share ends before the row block's first key block
    const int nh = hist_blocks(it);
    const int rows_total = it.n_new * a.group;
    const int row0 = rb_now * kTileRows;
    const int wrow0 = row0 + wave * kRowsPerWave;
    const bool wave_on = wrow0 < rows_total;
    const int row = wrow0 + col;
    const int rowc = min(row, rows_total - 1);
    const int my_tok = rowc / a.group;                    // sees new tokens 0 .. my_tok
    const int head = kvh_now * a.group + (rowc - my_tok * a.group);
    const int first_tok = min(wrow0, rows_total - 1) / a.group;              // of the wave's rows
    const int last_tok = (min(wrow0 + kRowsPerWave, rows_total) - 1) / a.group;

    const Hot h{a.k_cache + (int64_t)kvh_now * a.k_head, a.v_cache + (int64_t)kvh_now * a.v_head, a.k_page, a.v_page,
                (uint32_t)a.k_tok, (uint32_t)a.v_tok, a.stage_rows > 0 ? a.owner : nullptr,
                a.bt + (int64_t)it.req * a.bt_stride, (int32_t)min(a.num_pages, (int64_t)INT32_MAX), a.bt_cols,
                it.cached, a.block_size, a.bs_div, a.rows_div, a.scale_log2};

    // ---- first blocks' loads, then the wave's Q^T operands.  In phase M of
    // block i: lk holds block i + 1's words, lv block i's; pages p0 and p1
    // are those of blocks i and i + 1; meta (and cur) are block i's in phase S. ----
    struct Block {
      uint32_t win;       // window-owned tokens
      int live;           // tokens in the history, from the first
    };
    KLoad lk{};
    u32x2 meta{};
    uint32_t lv = 0;
    Block cur{0u, 0}, next{0u, 0};
    int32_t p0 = -1, p1 = -1;
    // (pages come from registers: a table read in the loop would be waited
    // for with the LDS reads at the next barrier)
    int pbase = kb;
    int32_t pgv = -1;
    auto page_at = [&](int i) { return valid_page(h, __builtin_amdgcn_readlane(pgv, i - pbase)); };
    if (kb < nh) pgv = load_pages(h, kb, lane);
    half8 qreg[kQReg], qlds[16 - kQReg];
    float qsum = 0.f;
    if constexpr (kImages) {
      const int64_t qrow = (int64_t)(it.tok0 + my_tok) * a.num_heads + head;
      const half8* qp = reinterpret_cast<const half8*>(a.q16 + qrow * kHeadDim) + g;
#pragma unroll
      for (int m = 0; m < kQReg; ++m) qreg[m] = qp[2 * m];
#pragma unroll
      for (int m = kQReg; m < 16; ++m) qlds[m - kQReg] = qp[2 * m];
      qsum = a.qsum[qrow];
    }
    __builtin_amdgcn_sched_barrier(0);      // (pages and queries in one round)
    if (kb < nh) {
      p1 = page_at(kb);
      lk = load_k(h, kb * kBlk, p1, r, lane);
      lv = load_v(h, kb * kBlk, p1, r);
      meta = load_meta(h, kb * kBlk, p1, r);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kImages) {
#pragma unroll
      for (int m = kQReg; m < 16; ++m) *reinterpret_cast<half8*>(&S.q[wave][m - kQReg][lane * 8]) = qlds[m - kQReg];
    } else {
      const float* qp = a.q + ((int64_t)(it.tok0 + my_tok) * a.num_heads + head) * kHeadDim + 4 * g;
      float qs = 0.f;
#pragma unroll
      for (int m = 0; m < 16; ++m) {
        const floatx4 x0 = *reinterpret_cast<const floatx4*>(qp + 16 * m);
        const floatx4 x1 = *reinterpret_cast<const floatx4*>(qp + 16 * m + 8);
        const half8 v = half8{to_h(x0[0]), to_h(x1[0]), to_h(x0[1]), to_h(x1[1]),
                              to_h(x0[2]), to_h(x1[2]), to_h(x0[3]), to_h(x1[3])};
#pragma unroll
        for (int e = 0; e < 8; ++e) qs += (float)v[e];
        if (m < kQReg) qreg[m < kQReg ? m : 0] = v;
        else *reinterpret_cast<half8*>(&S.q[wave][m < kQReg ? 0 : m - kQReg][lane * 8]) = v;
      }
      qsum = qs + shfl_xor_f32(qs, 32);
    }

    // the loop's waits must not count the loads above
#pragma unroll
    for (int m = 0; m < kQReg; ++m) asm volatile("" ::"v"(qreg[m]));
    asm volatile("" ::"v"(qsum));

    floatx16 acc[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) acc[t] = floatx16{};
    // Scores are taken relative to m_base, the row's lazily raised maximum (0
    // until the row has seen a key); raise: what a block's maximum has to
    // exceed to raise it.
    float m_base = 0.f, raise = -__builtin_inff();
    float l_run = 0.f, z_run = 0.f;     // this lane's keys' sums of p and p vz

    // K tile of block i (its words in lk, page p1) and V tile of block i (its
    // words in lv, page p0), with their window tokens.
    auto tile_k = [&](int i) { return S.k[i & 1]; };
    auto tile_v = [&](int i) { return S.v[i & 1]; };
    auto block_of = [&](int i) {
      const int live = live_tokens(h, i * kBlk, p1);
      return Block{window_mask(h, lk.own, live, p1, lane), live};
    };
    auto hist_k = [&](int i) {
      next = block_of(i);
      const uint32_t ks = opaque(r.ks);
      build_k(lk.kc, ks, tile_k(i), 0);
      build_k(lk.kc, ks, tile_k(i), 1);
      if (next.win != 0u)
        window_tiles(next.win, p1, i * kBlk, tile_k(i), 0u, 0u, -1, 0, tile_v(i), kvh_now, r, wave, lane);
    };
    auto hist_v = [&](int i) {
      const uint32_t vs = opaque(r.vs), w = quad_transpose(lv, lane);
#pragma unroll
      for (int f = 0; f < 4; ++f) build_v(w, vs, tile_v(i), f);
      if (cur.win != 0u)
        window_tiles(0u, -1, 0, tile_k(i), cur.win, lv, p0, i * kBlk, tile_v(i), kvh_now, r, wave, lane);
    };
    auto new_k = [&](int i, auto copy_waves) {
      constexpr int kCw = decltype(copy_waves)::value;
      if constexpr (kImages) {
        if (wave < kCw) copy_tile<kCw>(a.kimg, (int64_t)(it.tile0 + i - nh) * a.num_kv_heads + kvh_now, tile_k(i), wave, lane);
      } else {
        store_new_k(a, it, (i - nh) * kBlk, kvh_now, r, wave, lane, tile_k(i));
      }
    };
    auto new_v = [&](int i) {
      if constexpr (kImages) {
        if (!second) copy_tile<4>(a.vimg, (int64_t)(it.tile0 + i - nh) * a.num_kv_heads + kvh_now, tile_v(i), wave, lane);
      } else {
        store_new_v(a, it, (i - nh) * kBlk, kvh_now, r, wave, lane, tile_v(i));
      }
    };
    // The words of block i + 1's V and block i + 2's K, while those exist.
    auto load_next = [&](int i) {
      p0 = p1;
      if (i + 2 - pbase >= 64) {
        pbase = i + 2;
        pgv = load_pages(h, pbase, lane);
      }
      p1 = page_at(i + 2);
      if (i + 1 < min(kend, nh)) lv = load_v(h, (i + 1) * kBlk, p0, r);
      if (i + 2 < min(kend, nh)) lk = load_k(h, (i + 2) * kBlk, p1, r, lane);
    };
    // Blocks before kseen are seen by a row of the wave.
    const int kseen = !wave_on ? kb : min(kend, nh + last_tok / kBlk + 1);

    floatx16 s;
    half8 pb[2] = {half8{}, half8{}};

    // ---- phase M: O^T += V^T P^T of block i - 1 (zero weights before the
    // first block) and, with kQk, S^T = K Q^T of block i, MFMA by MFMA in
    // turn, operand reads kAhead pairs ahead ----
    auto matrix = [&](int i, auto qk_tag, auto&& piece) {
      constexpr bool kQk = decltype(qk_tag)::value;
      const uint32_t kr = opaque(r.kr), vr = opaque(r.vr);
      const uint8_t* qb =
          reinterpret_cast<const uint8_t*>(S.q) + opaque((uint32_t)(wave * (int)sizeof(S.q[0]) + 16 * lane));
      const uint8_t* kt = reinterpret_cast<const uint8_t*>(tile_k(i));
      const uint8_t* vt = reinterpret_cast<const uint8_t*>(tile_v(i - 1));
      auto read_k = [&](int m) {
        return *reinterpret_cast<const half8*>(kt + (kr ^ (16u * ((2 * m & 14) ^ (m >> 3)))) + 256 * (m >> 3));
      };
      // k-steps with Q^T in LDS first, then those in registers
      auto read_q = [&](int m) { return *reinterpret_cast<const half8*>(qb + 1024 * (m - kQReg)); };
      auto order = [](int n) { return n < 16 - kQReg ? n + kQReg : n - (16 - kQReg); };
      // feature block n & 7 of PV k-step n >> 3
      auto read_v = [&](int n) {
        return *reinterpret_cast<const half8*>(vt + (vr ^ (32u * (n >> 3))) + 2048 * (n & 7));
      };
      half8 ka[kAhead], qa[kAhead], va[kAhead];
      if constexpr (kQk) s = floatx16{};
#pragma unroll
      for (int n = 0; n < kAhead; ++n) {
        va[n] = read_v(n);
        if constexpr (kQk) {
          ka[n] = read_k(order(n));
          qa[n] = read_q(order(n));
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < 16; ++n) {
        // (the order below is the schedule: the compiler's own hoists the
        // operand reads and spills)
        const int nn = n + kAhead;
        acc[n & 7] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[n % kAhead], pb[n >> 3], acc[n & 7], 0, 0, 0);
        if (nn < 16) va[n % kAhead] = read_v(nn);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (kQk) {
          s = __builtin_amdgcn_mfma_f32_32x32x16_f16(
              ka[n % kAhead], order(n) < kQReg ? qreg[order(n) < kQReg ? order(n) : 0] : qa[n % kAhead], s, 0, 0, 0);
          if (nn < 16) {
            ka[n % kAhead] = read_k(order(nn));
            if (order(nn) >= kQReg) qa[n % kAhead] = read_q(order(nn));
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        piece(n);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    auto nothing = [](int) {};

    // ---- phase S: softmax of block i ----
    auto softmax = [&](int i, bool hist) {
      // This lane's key's parameters: score = par[0] (K'.q) + par[1] sum(q),
      // v = par[2] V' + par[3]; eager: some key has vs above kVsMax.
      floatx4 par{h.scale_log2, 0.f, 1.f, 0.f};
      bool eager = false;
      if (hist) {
        const int key = par_key(lane);
        const bool lv_ = key < cur.live, code = lv_ && ((cur.win >> key) & 1u) == 0u;
        const float ks = 4.f * f16_bits_to_f32(meta[0]), kz = f16_bits_to_f32(meta[0] >> 16);
        const float vs = 4.f * f16_bits_to_f32(meta[1]), vz = f16_bits_to_f32(meta[1] >> 16);
        par[0] = code ? ks * h.scale_log2 : (lv_ ? h.scale_log2 : 0.f);
        par[1] = code ? (kz - ks) * h.scale_log2 : 0.f;
        par[2] = code ? vs : (lv_ ? 1.f : 0.f);
        par[3] = code ? vz - vs : 0.f;
        eager = __ballot(code && vs > kVsMax) != 0ull;
        if (i + 1 < min(kend, nh)) meta = load_meta(h, (i + 1) * kBlk, p0, r);      // (p0: block i + 1's page by now)
      }
      constexpr auto regs = std::make_integer_sequence<int, 16>{};
      // x = score - m_base; key 8 jj + 4g + e of the block is register 4 jj + e
      float x[16];
      each16([&](auto reg) {
        constexpr int q = decltype(reg)::value;
        x[q] = row_bcast<q>(par[0]) * s[q];
      }, regs);
      fmac_bcast(x, par[1], qsum);
#pragma unroll
      for (int q = 0; q < 16; ++q) x[q] -= m_base;
      // Keys past C in the history's last block, causality in the new-token
      // blocks; a block every row of the wave sees whole skips the test.
      const int j0 = (i - nh) * kBlk;                     // first new token of a new-token block
      const bool whole = hist ? (i + 1) * kBlk <= h.cached : j0 + kBlk - 1 <= first_tok;
      if (!whole) {
        const int lim = (hist ? h.cached - i * kBlk - 1 : my_tok - j0) - 4 * g;      // last visible key
#pragma unroll
        for (int q = 0; q < 16; ++q) x[q] = 8 * (q >> 2) + (q & 3) <= lim ? x[q] : -__builtin_inff();
      }
      float mb = x[0];
#pragma unroll
      for (int q = 1; q < 16; ++q) mb = fmaxf(mb, x[q]);
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_int(mb), __float_as_int(mb), false, false);
      mb = fmaxf(__int_as_float(sw[0]), __int_as_float(sw[1]));
      // Lazy running max: raised only when a block exceeds it by more than
      // 2^kLazy (p vs stays in fp16 range), or by any amount when a key of
      // the block has vs above kVsMax, or when the row has seen no key yet
      // (which needs no rescale).
      const bool need = mb > (eager ? fminf(raise, 0.f) : raise);
      if (__ballot(need)) {
        const float delta = need ? mb : 0.f;
        const float alpha = raise == -__builtin_inff() ? 1.f : __builtin_amdgcn_exp2f(-delta);
#pragma unroll
        for (int t = 0; t < 8; ++t) acc[t] *= alpha;
        l_run *= alpha;
        z_run *= alpha;
#pragma unroll
        for (int q = 0; q < 16; ++q) x[q] -= delta;
        m_base += delta;
        raise = need ? kLazy : raise;
      }
      float psum = 0.f;
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        x[q] = __builtin_amdgcn_exp2f(x[q]);
        psum += x[q];
      }
      l_run += psum;
      z_run = dot_bcast(x, par[3], z_run);
      each16([&](auto reg) {
        constexpr int q = decltype(reg)::value;
        pb[q >> 3][q & 7] = to_h(row_bcast<q>(par[2]) * x[q]);
      }, regs);
    };

    // ---- first K tile (and a zero V tile before it), then M and S per block ----
    {
      floatx4* z = reinterpret_cast<floatx4*>(tile_v(kb - 1));
      z[tid] = floatx4{};
      z[tid + 64 * kWaves] = floatx4{};
      static_assert(2 * 64 * kWaves * sizeof(floatx4) == kKeyTileHalfs * sizeof(_Float16), "the tile");
    }
    if (kb < nh) {
      hist_k(kb);
      cur = next;
      p0 = p1;
      p1 = page_at(kb + 1);
      if (kb + 1 < min(kend, nh)) lk = load_k(h, (kb + 1) * kBlk, p1, r, lane);
      lds_barrier();
    } else {
      new_k(kb, std::integral_constant<int, kWaves>{});
      copy_barrier();
    }
    int i = kb;
    // blocks i and i + 1 in the history, i seen: builds under the MFMAs
    const int hot = min(kseen, min(kend, nh) - 1);
#pragma unroll 1
    for (; i < hot; ++i) {
      // (at the end of the phase, where the words have had longest to arrive)
      uint32_t w = 0;
      matrix(i, std::true_type{}, [&](int n) {
        if (n == 9) w = quad_transpose(lv, lane);
        if (n >= 10 && n < 14) build_v(w, opaque(r.vs), tile_v(i), n - 10);
        if (n >= 14) build_k(lk.kc, opaque(r.ks), tile_k(i + 1), n - 14);
      });
      next = block_of(i + 1);
      if ((next.win | cur.win) != 0u) {
        window_tiles(next.win, p1, (i + 1) * kBlk, tile_k(i + 1), cur.win, lv, p0, i * kBlk, tile_v(i), kvh_now, r,
                     wave, lane);
      }
      load_next(i);
      if (second) lds_barrier();
      softmax(i, true);
      cur = next;
      if (!second) lds_barrier();
    }
    // the history's last block and the new-token blocks
    auto builds = [&](int i) {
      if (i < nh) hist_v(i);
      else new_v(i);
      if (i + 1 < kend) {
        if (i + 1 < nh) hist_k(i + 1);
        else new_k(i + 1, std::integral_constant<int, 4>{});
      }
      if (i < nh) load_next(i);
    };
    // (a first-half wave's copies have had both phases)
    auto first_end = [&](int i) {
      if (kImages && i + 1 >= nh) copy_barrier();
      else lds_barrier();
    };
#pragma unroll 1
    for (; i < kseen; ++i) {
      builds(i);
      matrix(i, std::true_type{}, nothing);
      if (second) lds_barrier();
      softmax(i, i < nh);
      cur = next;
      if (!second) first_end(i);
    }
    // the last PV, then blocks that only other waves see
    if (i < kend) builds(i);
    matrix(i, std::false_type{}, nothing);
#pragma unroll 1
    while (i < kend) {
      if (second) lds_barrier();
      else first_end(i);
      cur = next;
      if (++i < kend) builds(i);
    }
    lds_barrier();              // the tiles are free

    // ---- the row block's output, or this share's partial of it ----
    const float l_tot = l_run + shfl_xor_f32(l_run, 32);
    const float z_tot = z_run + shfl_xor_f32(z_run, 32);
    // A lane holds quarters of 16-byte pieces of one row; through the wave's
    // own Q^T area (its last scores are done), 64 features of its 32 rows at a
    // time, they leave as whole 256-byte runs.  (Straight from the registers,
    // 32 bytes of 32 rows an instruction, a partial took 3.8 us.)  The lane's
    // row recomputed, so that nothing of it lives through the loop.
    const int elane = (int)opaque((uint32_t)lane);
    const int er = elane & 31, eg = elane >> 5;
    const bool whole_rb = kb == 0 && kend == nblk;
    const float inv = whole_rb ? (l_tot > 0.f ? 1.f / l_tot : 0.f) : 1.f;
    float* base = a.out;
    if (!whole_rb) {
      const int64_t slot = 2 * (int64_t)blockIdx.x + (start != (int64_t)blockIdx.x * a.share ? 1 : 0);
      base = a.part + slot * (int64_t)kPartFloats;
      if (eg == 0 && wrow0 + er < rows_total) {
        const int pr = wave * kRowsPerWave + er;
        base[kPartRows * kHeadDim + pr] = raise == -__builtin_inff() ? raise : m_base;
        base[kPartRows * (kHeadDim + 1) + pr] = l_tot;
      }
    }
    // rows 4 i + lane / 16 of the wave, piece lane % 16 of a run
    uint32_t off[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r8 = 4 * i + (elane >> 4), erow = wrow0 + r8;
      const int etok = erow / a.group, ehead = kvh_now * a.group + (erow - etok * a.group);
      const int64_t o = whole_rb ? (int64_t)(it.tok0 + etok) * a.num_heads + ehead : wave * kRowsPerWave + r8;
      off[i] = erow < rows_total ? (uint32_t)o : ~0u;
    }
    floatx4* T = reinterpret_cast<floatx4*>(S.q[wave]);
    static_assert(sizeof(S.q[0]) >= 32 * 64 * sizeof(float), "64 features of 32 rows");
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      wave_sync_lds();
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          const floatx16& c = acc[2 * p + tt];
          T[16 * er + ((8 * tt + 2 * jj + eg) ^ (er & 15))] =
              floatx4{(c[4 * jj] + z_tot) * inv, (c[4 * jj + 1] + z_tot) * inv, (c[4 * jj + 2] + z_tot) * inv,
                      (c[4 * jj + 3] + z_tot) * inv};
        }
      wave_sync_lds();
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int r8 = 4 * i + (elane >> 4);
        const floatx4 x = T[16 * r8 + ((elane & 15) ^ (r8 & 15))];
        if (off[i] != ~0u)
          *reinterpret_cast<floatx4_any*>(base + (uint64_t)off[i] * kHeadDim + 64 * p + 4 * (elane & 15)) = x;
      }
    }
  }
}

// Row pr of a row block from its n partials (slot(p)), LSE-combined and
// normalised: lane l's features 4l .. 4l + 3.  With kWavesPerRow waves (the
// workgroup's all), wave `first` takes partials first, first + kWavesPerRow,
// ...; the (m, l) come in one lane-parallel round per 64 partials.
template <int kWavesPerRow, class Slot>
__device__ __forceinline__ floatx4 merge_row(const Slot& slot, int n, int pr, int first, int lane) {
  float mx = -__builtin_inff();
  for (int p = lane; p < n; p += 64) mx = fmaxf(mx, slot(p)[kPartRows * kHeadDim + pr]);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  // partials first, first + kWavesPerRow, ... of the row
  const int mine = (n - first + kWavesPerRow - 1) / kWavesPerRow;
  floatx4 acc = floatx4{};
  float l = 0.f;
  constexpr int kBatch = 8;
  for (int p0 = 0; p0 < mine; p0 += 64) {
    const int p = first + (p0 + lane) * kWavesPerRow;
    float w = 0.f;
    if (p < n) {
      const float m = slot(p)[kPartRows * kHeadDim + pr];
      w = m == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(m - mx);
      l = fmaf(w, slot(p)[kPartRows * (kHeadDim + 1) + pr], l);
    }
    const int cnt = min(64, mine - p0);
    for (int b = 0; b < cnt; b += kBatch) {
      floatx4 x[kBatch];
#pragma unroll
      for (int k = 0; k < kBatch; ++k)
        x[k] = *reinterpret_cast<const floatx4*>(slot(first + (p0 + min(b + k, cnt - 1)) * kWavesPerRow) +
                                                 pr * kHeadDim + 4 * lane);
#pragma unroll
      for (int k = 0; k < kBatch; ++k) {
        const float wk = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), (b + k) & 63));
        if (b + k < cnt) acc += wk * x[k];
      }
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) l += __shfl_xor(l, o, 64);
  if constexpr (kWavesPerRow > 1) {
    __shared__ floatx4 osum[kWavesPerRow][64];
    __shared__ float lsum[kWavesPerRow];
    osum[first][lane] = acc;
    if (lane == 0) lsum[first] = l;
    __syncthreads();
    acc = osum[0][lane];
    l = lsum[0];
#pragma unroll
    for (int k = 1; k < kWavesPerRow; ++k) {
      acc += osum[k][lane];
      l += lsum[k];
    }
  }
  return acc * (l > 0.f ? 1.f / l : 0.f);
}

// Rows of the row blocks that the shares cut: their partials LSE-combined and
// normalised.  kWavesPerRow waves share a row's partials (one where a row has
// few of them, four where the work of few rows is spread over the GPU).
// grid.x = row blocks x kTileRows x
// kWavesPerRow / 4, 256 threads.
template <int kWavesPerRow>
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillArgs a) {
  constexpr int kRows = 4 / kWavesPerRow;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int grb = (int)blockIdx.x / (kTileRows / kRows);
  int item = 0;
  while (item + 1 < a.nitems && a.items[item + 1].rb0 <= grb) ++item;
  const PrefillItem it = a.items[item];
  const int nrb = row_blocks(it, a.group);
  const int kvh = (grb - it.rb0) / nrb, rb = (grb - it.rb0) - kvh * nrb;
  const int pr = ((int)blockIdx.x % (kTileRows / kRows)) * kRows + wave / kWavesPerRow;
  const int row = rb * kTileRows + pr;
  if (row >= it.n_new * a.group) return;
  // units of the row block's first and last key block
  const int64_t lo = it.unit0 + (int64_t)kvh * it.head_units + units_before(it, a.group, rb, lane) + kPieceCost;
  const int64_t hi = lo + key_blocks(it, a.group, rb) - 1;
  const int64_t w0 = lo / a.share, w1 = hi / a.share;
  if (w0 == w1) return;                       // written whole by its share
  const int n = (int)(w1 - w0) + 1;
  auto slot = [&](int p) {
    return a.part + (2 * (w0 + p) + (p == 0 && lo != w0 * a.share ? 1 : 0)) * (int64_t)kPartFloats;
  };
  const floatx4 o = merge_row<kWavesPerRow>(slot, n, pr, wave % kWavesPerRow, lane);
  if (wave % kWavesPerRow != 0) return;
  const int tok = row / a.group, head = kvh * a.group + (row - tok * a.group);
  *reinterpret_cast<floatx4_any*>(a.out + ((int64_t)(it.tok0 + tok) * a.num_heads + head) * kHeadDim + 4 * lane) = o;
}

// The read's bf16 output: rows merged where the shares cut their row block
// (merged: that is done, the rows are in a.out), multiplied by R_v^T and
// rounded.  A workgroup takes 32 rows of a row block.  Its eight waves first
// combine four rows each (lane l: features 4l .. 4l + 3), all rows' (m, l) in
// one load where a row has at most 16 pieces, and leave them in LDS as the
// bf16 high and low parts of MFMA operands; then wave t computes output
// features {128 h + 16 t + i} of every row, its operand fragments of R_v^T
// (rotation_operand's, high and low parts) straight from L2, kOutAhead steps
// ahead of their use.  Products and their order are rotate_rows_kernel's:
// R high x high, R low x high, R high x low.
// Reading the partials (83 MB at 3001 tokens) bounds it from below; two
// workgroups a CU overlap one's reads with the other's products.  The merge
// and the rotation of the merged rows took 18 + 18 us (3001 tokens), 23 + 16
// (1024 over 4K), 9 + 15 (77 over 20K) and 48 + 35 (9256 over 15K) as kernels
// of their own; this takes 27, 22, 9 + 8.5 and 51.  64 rows a workgroup, whose
// registers leave one to a CU, took 28, -, 9 + 11 and 55.
constexpr int kOutAhead = 4;
constexpr int kOutRows = 32;          // rows of a workgroup
constexpr int kOutMine = kOutRows / 8;

__global__ __launch_bounds__(512, 4) void prefill_output_kernel(PrefillArgs a, int merged,
                                                                const uint8_t* __restrict__ rop,
                                                                uint16_t* __restrict__ out) {
  // [part][k-step][row ^ k-step, half][8]: chunk rows swizzled so that a
  // wave's 16 k-steps of one row fall on different banks
  __shared__ __attribute__((aligned(16))) __bf16 xs[2][16][64][8];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int grb = (int)blockIdx.x / (kTileRows / kOutRows);
  const int pr0 = ((int)blockIdx.x % (kTileRows / kOutRows)) * kOutRows;
  int item = 0;
  while (item + 1 < a.nitems && a.items[item + 1].rb0 <= grb) ++item;
  const PrefillItem it = a.items[item];
  const int nrb = row_blocks(it, a.group);
  const int kvh = (grb - it.rb0) / nrb, rb = (grb - it.rb0) - kvh * nrb;
  const int rows = it.n_new * a.group;
  if (rb * kTileRows + pr0 >= rows) return;

  const u32x4* frag = reinterpret_cast<const u32x4*>(rop) + wave * 64 + lane;
  auto load_r = [&](int m, int p) { return __builtin_bit_cast(bf16x8, frag[(m * 16 + p * 8) * 64]); };
  bf16x8 f[kOutAhead][2];
#pragma unroll
  for (int m = 0; m < kOutAhead; ++m) {
    f[m][0] = load_r(m, 0);
    f[m][1] = load_r(m, 1);
  }

  // ---- rows pr0 + mine0 .. + kOutMine - 1 of the row block ----
  const int mine0 = kOutMine * wave;
  int n = 1;
  int64_t w0 = 0;
  bool second = false;                        // the first piece is its share's second partial
  if (!merged) {
    const int64_t lo = it.unit0 + (int64_t)kvh * it.head_units + units_before(it, a.group, rb, lane) + kPieceCost;
    const int64_t hi = lo + key_blocks(it, a.group, rb) - 1;
    w0 = lo / a.share;
    n = (int)(hi / a.share - w0) + 1;
    second = lo != w0 * a.share;
  }
  auto slot = [&](int p) { return a.part + (2 * (w0 + p) + (p == 0 && second ? 1 : 0)) * (int64_t)kPartFloats; };
  auto put = [&](int i, const floatx4& x) {
    const int rr = mine0 + i, m = (lane & 31) >> 1;
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    bf16x4 h, l;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      h[e] = (__bf16)x[e];
      l[e] = (__bf16)(x[e] - (float)h[e]);
    }
    const int at = (rr ^ m) + (lane & 32), sub = 4 * (lane & 1);
    *reinterpret_cast<bf16x4*>(&xs[0][m][at][sub]) = h;
    *reinterpret_cast<bf16x4*>(&xs[1][m][at][sub]) = l;
  };
  const int row0 = rb * kTileRows + pr0 + mine0;
  const int left = min(kOutMine, rows - row0);   // (<= 0: none of the wave's rows)
  constexpr int kFew = 64 / kOutMine, kBatch = 8;
  if (n == 1) {
    floatx4 x[kOutMine];
#pragma unroll
    for (int i = 0; i < kOutMine; ++i) {
      const int row = row0 + (i < left ? i : 0), tok = row / a.group, head = kvh * a.group + (row - tok * a.group);
      x[i] = floatx4{};
      if (i < left)
        x[i] = *reinterpret_cast<const floatx4*>(a.out + ((int64_t)(it.tok0 + tok) * a.num_heads + head) * kHeadDim +
                                                 4 * lane);
    }
#pragma unroll
    for (int i = 0; i < kOutMine; ++i) put(i, x[i]);
  } else if (n <= kFew) {
    // lane kFew i + p: piece p of row i
    const int wi = lane / kFew, wp = lane % kFew;
    float mp = -__builtin_inff(), lp = 0.f;
    if (wp < n && wi < left) {
      const float* part = slot(wp) + kPartRows * kHeadDim + pr0 + mine0 + wi;
      mp = part[0];
      lp = part[kPartRows];
    }
    // the rows' pieces in batches, the next batch requested before one is used
    constexpr int kSteps = kOutMine * (kFew / kBatch);
    floatx4 x[2][kBatch];
    auto load_batch = [&](int s) {
      const int i = s / (kFew / kBatch), p0 = kBatch * (s % (kFew / kBatch));
      if (p0 >= n) return;
#pragma unroll
      for (int k = 0; k < kBatch; ++k) {
        x[s & 1][k] = floatx4{};
        if (p0 + k < n && i < left)
          x[s & 1][k] =
              *reinterpret_cast<const floatx4*>(slot(p0 + k) + (int64_t)(pr0 + mine0 + i) * kHeadDim + 4 * lane);
      }
    };
    load_batch(0);
    float mx = mp;
#pragma unroll
    for (int o = kFew / 2; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    const float w = mp == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(mp - mx);
    float l = w * lp;
#pragma unroll
    for (int o = kFew / 2; o >= 1; o >>= 1) l += __shfl_xor(l, o, 64);
    const float inv = l > 0.f ? 1.f / l : 0.f;
    floatx4 acc = floatx4{};
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      const int i = s / (kFew / kBatch), p0 = kBatch * (s % (kFew / kBatch));
      if (s + 1 < kSteps) load_batch(s + 1);
      if (p0 < n) {
#pragma unroll
        for (int k = 0; k < kBatch; ++k)
          if (p0 + k < n)
            acc += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), kFew * i + p0 + k)) * x[s & 1][k];
      }
      if (p0 + kBatch == kFew) {
        put(i, acc * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(inv), kFew * i)));
        acc = floatx4{};
      }
    }
  } else {
#pragma unroll 1
    for (int i = 0; i < kOutMine; ++i) put(i, i < left ? merge_row<1>(slot, n, pr0 + mine0 + i, 0, lane) : floatx4{});
  }
  __syncthreads();

  floatx16 acc = floatx16{};
#pragma unroll
  for (int m = 0; m < 16; ++m) {
    const bf16x8 rh = f[m % kOutAhead][0], rl = f[m % kOutAhead][1];
    if (m + kOutAhead < 16) {
      f[m % kOutAhead][0] = load_r(m + kOutAhead, 0);
      f[m % kOutAhead][1] = load_r(m + kOutAhead, 1);
    }
    const int at = ((lane & 31) ^ m) + (lane & 32);
    const bf16x8 h = *reinterpret_cast<const bf16x8*>(&xs[0][m][at][0]);
    const bf16x8 l = *reinterpret_cast<const bf16x8*>(&xs[1][m][at][0]);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(rh, h, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(rl, h, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(rh, l, acc, 0, 0, 0);
  }
  const int row = rb * kTileRows + pr0 + (lane & 31);
  if (row >= rows) return;
  const int tok = row / a.group, head = kvh * a.group + (row - tok * a.group);
  __bf16* d = reinterpret_cast<__bf16*>(out) + ((int64_t)(it.out0 + tok) * a.num_heads + head) * kHeadDim +
              128 * (lane >> 5) + 16 * wave;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    bf16x8 o;
#pragma unroll
    for (int u = 0; u < 8; ++u) o[u] = (__bf16)acc[8 * q + u];
    reinterpret_cast<bf16x8*>(d)[q] = o;
  }
}

// Operands (prefill_operands.h) of rotated fp32 rows: one 16-byte chunk per
// thread; query rows first (32 threads per row), then key tiles, then value
// tiles.  Compact tokens are the inputs' tokens here.
struct ConvertArgs {
  const float* q;
  const float* k;
  const float* v;
  int32_t num_heads, num_kv_heads;
  PrefillOperands o;
  int64_t q_chunks, kv_chunks;
  OperandItems items;
};

__global__ __launch_bounds__(256) void convert_operands_kernel(ConvertArgs a) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx < a.q_chunks) {                      // a multiple of 256 or the tail's whole 32-thread rows
    const int64_t row = idx >> 5;
    const int c = (int)idx & 31;
    const float* src = a.q + row * kHeadDim + 16 * (c >> 1) + 4 * (c & 1);
    half8 o;
    float qs = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      o[e] = to_h(src[(e >> 1) + 8 * (e & 1)]);
      qs += (float)o[e];
    }
    reinterpret_cast<half8*>(a.o.q16)[idx] = o;
#pragma unroll
    for (int s = 16; s >= 1; s >>= 1) qs += __shfl_xor(qs, s, 64);
    if (c == 0) a.o.qsum[row] = qs;
    return;
  }
  int64_t r = idx - a.q_chunks;
  const bool value = r >= a.kv_chunks;
  if (value) r -= a.kv_chunks;
  if (r >= a.kv_chunks) return;
  const int64_t unit = r >> 10;                // (tile, kv head): 1024 chunks
  const int tile = (int)(unit / a.num_kv_heads), head = (int)(unit - (int64_t)tile * a.num_kv_heads);
  int i = 0;
  while (i + 1 < a.items.n && a.items.it[i + 1].tile0 <= tile) ++i;
  const OperandItem it = a.items.it[i];
  const int j0 = (tile - it.tile0) * kBlk;
  auto rowp = [&](const float* x, int t) {
    return x + ((int64_t)(it.tok0 + min(j0 + t, it.n_new - 1)) * a.num_kv_heads + head) * kHeadDim;
  };
  half8 o;
  if (!value) {
    const int token = (int)(r >> 5) & 31, c = (int)r & 31;
    const float* src = rowp(a.k, token) + 16 * (c >> 1) + 4 * (c & 1);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = to_h(src[(e >> 1) + 8 * (e & 1)]);
    reinterpret_cast<half8*>(a.o.kimg)[unit * 1024 + token * 32 + k_chunk(c, token)] = o;
  } else {
    const int f = (int)r & 255, c = (int)(r >> 8) & 3;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = to_h(rowp(a.v, 16 * (c >> 1) + 8 * (e >> 2) + 4 * (c & 1) + (e & 3))[f]);
    reinterpret_cast<half8*>(a.o.vimg)[unit * 1024 + f * 4 + v_chunk(c, f)] = o;
  }
}

std::atomic<uint64_t> g_lds_set[2] = {{0}, {0}};   // dynamic-LDS attribute set, one bit per device

// ---- host side ----

// Row blocks of `tile` rows of one kv head, and all their key blocks.
int64_t host_row_blocks(int64_t n_new, int64_t group, int tile) { return (n_new * group + tile - 1) / tile; }
int64_t host_key_blocks(int64_t n_new, int64_t cached, int64_t group, int tile) {
  const int64_t rows = n_new * group, nrb = host_row_blocks(n_new, group, tile);
  int64_t n = nrb * ((cached + kBlk - 1) / kBlk);
  for (int64_t rb = 0; rb < nrb; ++rb) {
    const int64_t last = ((rb + 1) * tile < rows ? (rb + 1) * tile : rows) - 1;
    n += last / group / kBlk + 1;
  }
  return n;
}

int64_t host_head_units(int64_t n_new, int64_t cached, int64_t group) {
  return host_row_blocks(n_new, group, kTileRows) * kPieceCost + host_key_blocks(n_new, cached, group, kTileRows);
}

// Units per workgroup: one round of kShares workgroups, of at least kMinShare
// units each (a partial of 256 rows is 264 KB, written and read again: 77
// tokens over 20K take 41 us + merge 10.7 in shares of 8, 36 + 12.9 of 6, 34 +
// 14 of 5, 34 + 14.4 of 4).
int64_t plan_share(int64_t units) {
  const int64_t s = (units + kShares - 1) / kShares;
  return s < kMinShare ? kMinShare : s;
}

struct Layout {          // byte offsets into the workspace
  size_t q16, qsum, kimg, vimg, out, part, total;
};

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

Layout workspace_layout(int64_t tokens, int64_t tiles, int64_t units, int32_t hq, int32_t hk, bool with_out) {
  Layout w;
  size_t o = 0;
  w.q16 = o;
  o = align256(o + (size_t)tokens * hq * kHeadDim * sizeof(_Float16));
  w.qsum = o;
  o = align256(o + (size_t)tokens * hq * sizeof(float));
  w.kimg = o;
  o = align256(o + (size_t)tiles * hk * kKeyTileHalfs * sizeof(_Float16));
  w.vimg = o;
  o = align256(o + (size_t)tiles * hk * kKeyTileHalfs * sizeof(_Float16));
  w.out = o;
  if (with_out) o = align256(o + (size_t)tokens * hq * kHeadDim * sizeof(float));
  w.part = o;
  const int64_t share = plan_share(units);
  o += (size_t)(2 * ((units + share - 1) / share)) * kPartFloats * sizeof(float);
  w.total = o;
  return w;
}

// The cache, block table, arena and geometry half of the arguments, checked
// (of a call without new tokens, `empty`, only the counts).
int fill_common(PrefillArgs& a, bool empty, int32_t num_heads, int32_t num_kv_heads, int32_t head_size, const void* k_cache,
                const void* v_cache, int32_t block_size, int64_t num_pages, int64_t k_stride_page,
                int64_t k_stride_token, int64_t k_stride_head, int64_t v_stride_page, int64_t v_stride_token,
                int64_t v_stride_head, const int32_t* block_table, int64_t block_table_stride,
                int32_t block_table_cols, const float* stage_k, const float* stage_v, const int64_t* stage_owner,
                int32_t stage_rows, float scale) {
  if (head_size != kHeadDim) return kErrUnsupportedHeadDim;
  if (num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads || block_size <= 0 || num_pages <= 0 ||
      stage_rows < 0 || block_table_cols < 0)
    return kErrInvalidArgument;
  if (empty) return kOk;
  if (!k_cache || !v_cache) return kErrInvalidArgument;
  if (stage_rows > 0 && (!stage_k || !stage_v || !stage_owner)) return kErrInvalidArgument;
  if (k_stride_head < kKCodeOff + kCodeBytes || v_stride_head < kCodeBytes || (k_stride_head & 7) ||
      (k_stride_token & 7) || (k_stride_page & 7) || block_size % kBlk != 0)
    return kErrUnsupportedGeometry;
  a.num_heads = num_heads;
  a.num_kv_heads = num_kv_heads;
  a.group = num_heads / num_kv_heads;
  a.k_cache = static_cast<const uint8_t*>(k_cache);
  a.v_cache = static_cast<const uint8_t*>(v_cache);
  a.k_page = k_stride_page;
  a.k_tok = k_stride_token;
  a.k_head = k_stride_head;
  a.v_page = v_stride_page;
  a.v_tok = v_stride_token;
  a.v_head = v_stride_head;
  a.block_size = block_size;
  a.bs_div = make_fast_div((uint32_t)block_size);
  a.rows_div = make_fast_div(stage_rows > 0 ? (uint32_t)stage_rows : 1u);
  a.num_pages = num_pages;
  a.bt = block_table;
  a.bt_stride = block_table_stride;
  a.bt_cols = block_table_cols;
  a.stage_k = stage_k;
  a.stage_v = stage_v;
  a.owner = stage_owner;
  a.stage_rows = stage_rows;
  a.scale_log2 = scale * kLog2e;
  return kOk;
}

// One request's sizes: positions and rows are handled in 32 bits in the kernel.
int check_request(int64_t n_new, int64_t cached, int32_t num_heads, int32_t block_size, const int32_t* table,
                  int32_t cols) {
  if (n_new < 0 || cached < 0 || cached + n_new >= ((int64_t)1 << 31) || n_new * num_heads >= ((int64_t)1 << 31))
    return kErrInvalidArgument;
  if (cached > 0 && (!table || (cached + block_size - 1) / block_size > cols)) return kErrInvalidArgument;
  return kOk;
}

void add_item(PrefillArgs& a, OperandItems& ops, int32_t n_new, int64_t cached, int32_t req, int32_t in_tok0) {
  PrefillItem& it = a.items[a.nitems];
  it.unit0 = a.units;
  it.head_units = host_head_units(n_new, cached, a.group);
  it.n_new = n_new;
  it.cached = (int32_t)cached;
  it.req = req;
  it.tok0 = ops.tokens;
  it.out0 = in_tok0;
  it.tile0 = ops.tiles;
  it.rb0 = 0;
  if (a.nitems > 0) {
    const PrefillItem& p = a.items[a.nitems - 1];
    it.rb0 = p.rb0 + (int32_t)(((int64_t)p.n_new * a.group + kTileRows - 1) / kTileRows) * a.num_kv_heads;
  }
  ops.it[ops.n++] = OperandItem{in_tok0, n_new, ops.tokens, ops.tiles};
  ops.tokens += n_new;
  ops.tiles += (n_new + kBlk - 1) / kBlk;
  a.units += it.head_units * a.num_kv_heads;
  ++a.nitems;
}

// Row blocks of a launch.
int64_t launch_row_blocks(const PrefillArgs& a) {
  const PrefillItem& p = a.items[a.nitems - 1];
  return p.rb0 + (((int64_t)p.n_new * a.group + kTileRows - 1) / kTileRows) * a.num_kv_heads;
}

// The read over operands in the workspace by shares; returns their number in
// wgs.
int launch_shares(PrefillArgs& a, int64_t& wgs, hipStream_t stream) {
  a.share = plan_share(a.units);
  wgs = (a.units + a.share - 1) / a.share;
  if (set_dynamic_lds(reinterpret_cast<const void*>(prefill_kernel<true>), (int)kPrefillLds, g_lds_set[1]) != kOk)
    return kErrLaunch;
  hipLaunchKernelGGL((prefill_kernel<true>), dim3((unsigned)wgs), dim3(64 * kWaves), kPrefillLds, stream, a);
  return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}

// A read of one request by whole row blocks of `tile` rows, in key blocks walked
// one after the other: the last row block's, and a CU's mean of all of them.
struct WholeLength {
  double last, mean;
  int64_t workgroups;
};
WholeLength whole_length(const PrefillArgs& a, int tile) {
  const PrefillItem& it = a.items[0];
  const int64_t last = ((int64_t)it.cached + kBlk - 1) / kBlk + (it.n_new - 1) / kBlk + 1;
  const int64_t all = host_key_blocks(it.n_new, it.cached, a.group, tile) * a.num_kv_heads;
  return WholeLength{(double)last, (double)all / kShares, host_row_blocks(it.n_new, a.group, tile) * a.num_kv_heads};
}

// Whether that read takes row blocks of 128 rows (prefill_rows.hip), not of 256
// (prefill_kernel<false>): of history, a key block of the latter takes a third
// longer for twice the rows; new tokens' fp32 rows are fetched ahead by the
// former only.  us, 128 against 256 rows: 6 heads, 17 tokens over 100 19.4 / 20.2,
// 100 over 800 56 / 69, 1500 alone 88 / 128, 6000 alone 305 / 462; 16 heads of two
// kv heads, 3000 over 2400 379 / 367; 64 of eight, 600 over 400 106 / 88, 1000
// alone 129 / 97; 32 heads, 3000 over 2400 636 / 500.
bool prefers_rows(const PrefillArgs& a) {
  const WholeLength w1 = whole_length(a, kPrefillSmallTile), w2 = whole_length(a, kTileRows);
  return 0.85 * std::max(w1.last, 1.3 * w1.mean) < std::max(w2.last, 1.3 * w2.mean);
}

// Whether a read of one request with a workspace takes row blocks of 128 rows
// whole all the same: one launch instead of three, without operands and
// partials.  In us beside what both take: 1.6 a key block (of every round of the
// CUs where several kv heads are one after the other) against 1.6 a unit of a
// share, 0.25 a row block (operands, partials) and 10 for the launches.  Of 423
// shapes it picks the slower one by 13 % at most, by 0.1 on average.  us, whole
// against shares: 6 heads, 17 tokens alone 14.1 / 22, over 100 19.4 / 24.7, over 400
// 35 / 26.6, 200 alone 23 / 29.5, over 300 39 / 32; 32 heads, 1500 alone 91 / 108;
// 64 of eight kv heads, 400 over 100 44 / 61, 600 over 400 106 / 92.
bool prefers_rows_shares(const PrefillArgs& a) {
  const WholeLength w = whole_length(a, kPrefillSmallTile);
  const int64_t rounds = a.num_kv_heads > 1 ? (w.workgroups + kShares - 1) / kShares : 1;
  const int64_t rbs = host_row_blocks(a.items[0].n_new, a.group, kTileRows) * a.num_kv_heads;
  return 1.6 * std::max(w.last * (double)rounds, 1.15 * w.mean) <
         10. + 1.6 * (double)plan_share(a.units) + 0.25 * (double)rbs;
}

constexpr size_t kRowsWorkspace = 16;   // that such a read asks for (it uses none; zero means a refused shape)

// That read (prefill_rows.hip).
int launch_rows(const PrefillArgs& a, const float* q_rot, const float* k_new, const float* v_new, float* out,
                hipStream_t stream) {
  const PrefillItem& it = a.items[0];
  return launch_prefill_rows(PrefillRows{q_rot, k_new, v_new, it.n_new, a.num_heads, a.num_kv_heads, a.group,
                                         a.k_cache, a.v_cache, a.k_page, a.k_tok, a.k_head, a.v_page, a.v_tok,
                                         a.v_head, a.block_size, a.bs_div, a.rows_div, a.num_pages, a.bt, a.bt_cols,
                                         it.cached, a.stage_k, a.stage_v, a.owner, a.stage_rows, a.scale_log2, out},
                             stream);
}

// Few row blocks in many shares: a workgroup per row merges them.
bool many_pieces(const PrefillArgs& a, int64_t wgs) { return launch_row_blocks(a) * kMergeManyPieces <= wgs; }

int launch_merge(const PrefillArgs& a, int64_t wgs, hipStream_t stream) {
  if (wgs <= 1) return kOk;
  const int64_t rbs = launch_row_blocks(a);
  if (many_pieces(a, wgs))
    hipLaunchKernelGGL((prefill_merge_kernel<4>), dim3((unsigned)(rbs * kTileRows)), dim3(256), 0, stream, a);
  else
    hipLaunchKernelGGL((prefill_merge_kernel<1>), dim3((unsigned)(rbs * kTileRows / 4)), dim3(256), 0, stream, a);
  return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}

// The bf16 output of the shares: merge and rotation in one pass, unless rows
// average more pieces than a wave's one round of (m, l) takes: a workgroup per
// row then merges them first (77 tokens over 20K: two row blocks of 128
// pieces, which the 16 workgroups of the output pass could not read quickly).
int launch_output(const PrefillArgs& a, int64_t wgs, const void* rop, void* out_bf16, hipStream_t stream) {
  const int64_t rbs = launch_row_blocks(a);
  const bool many = wgs > 1 && rbs * (64 / kOutMine) <= wgs;
  if (many) {
    const int st = launch_merge(a, wgs, stream);
    if (st != kOk) return st;
  }
  const uint8_t* r = static_cast<const uint8_t*>(rop);
  uint16_t* o = static_cast<uint16_t*>(out_bf16);
  hipLaunchKernelGGL(prefill_output_kernel, dim3((unsigned)(rbs * (kTileRows / kOutRows))), dim3(512), 0, stream, a,
                     (int)many, r, o);
  return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}

void bind_workspace(PrefillArgs& a, PrefillOperands& o, const Layout& w, uint8_t* ws) {
  o.q16 = reinterpret_cast<_Float16*>(ws + w.q16);
  o.qsum = reinterpret_cast<float*>(ws + w.qsum);
  o.kimg = reinterpret_cast<_Float16*>(ws + w.kimg);
  o.vimg = reinterpret_cast<_Float16*>(ws + w.vimg);
  a.q16 = o.q16;
  a.qsum = o.qsum;
  a.kimg = o.kimg;
  a.vimg = o.vimg;
  a.part = reinterpret_cast<float*>(ws + w.part);
}

}  // namespace
}  // namespace oscar

using namespace oscar;

extern "C" size_t oscar_prefill_workspace_bytes(int32_t num_new, int32_t num_heads, int32_t num_kv_heads,
                                                int64_t cached_len) {
  if (num_new <= 0 || num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads || cached_len < 0) return 0;
  if (cached_len + num_new >= ((int64_t)1 << 31)) return 0;
  PrefillArgs a{};
  a.num_kv_heads = num_kv_heads;
  a.group = num_heads / num_kv_heads;
  OperandItems ops{};
  add_item(a, ops, num_new, cached_len, 0, 0);
  if (prefers_rows_shares(a)) return kRowsWorkspace;
  return workspace_layout(ops.tokens, ops.tiles, a.units, num_heads, num_kv_heads, false).total;
}

extern "C" int oscar_prefill_continuation_split(
    const float* q_rot, const float* k_new, const float* v_new, int32_t num_new, int32_t num_heads,
    int32_t num_kv_heads, int32_t head_size, const void* k_cache, const void* v_cache,
    int32_t block_size, int64_t num_pages, int64_t k_stride_page, int64_t k_stride_token,
    int64_t k_stride_head, int64_t v_stride_page, int64_t v_stride_token, int64_t v_stride_head,
    const int32_t* block_table_row, int32_t block_table_cols, int64_t cached_len,
    const float* stage_k, const float* stage_v, const int64_t* stage_owner, int32_t stage_rows,
    float scale, float* out, void* workspace, size_t workspace_size, hipStream_t stream) {
  PrefillArgs a{};
  if (num_new < 0 || cached_len < 0) return kErrInvalidArgument;
  int st = fill_common(a, num_new == 0, num_heads, num_kv_heads, head_size, k_cache, v_cache, block_size, num_pages,
                       k_stride_page, k_stride_token, k_stride_head, v_stride_page, v_stride_token, v_stride_head,
                       block_table_row, 0, block_table_cols, stage_k, stage_v, stage_owner, stage_rows, scale);
  if (st != kOk || num_new == 0) return st;
  if ((st = check_request(num_new, cached_len, num_heads, block_size, block_table_row, block_table_cols)) != kOk)
    return st;
  if (!q_rot || !k_new || !v_new || !out || !workspace || (reinterpret_cast<uintptr_t>(workspace) & 15))
    return kErrInvalidArgument;
  OperandItems ops{};
  add_item(a, ops, num_new, cached_len, 0, 0);
  if (prefers_rows_shares(a))
    return workspace_size < kRowsWorkspace ? (int)kErrWorkspaceTooSmall
                                           : launch_rows(a, q_rot, k_new, v_new, out, stream);
  const Layout w = workspace_layout(ops.tokens, ops.tiles, a.units, num_heads, num_kv_heads, false);
  if (workspace_size < w.total) return kErrWorkspaceTooSmall;
  ConvertArgs c{q_rot, k_new, v_new, num_heads, num_kv_heads, PrefillOperands{}, 0, 0, ops};
  bind_workspace(a, c.o, w, static_cast<uint8_t*>(workspace));
  a.out = out;
  c.q_chunks = (int64_t)ops.tokens * num_heads * (kHeadDim / 8);
  c.kv_chunks = (int64_t)ops.tiles * num_kv_heads * (kKeyTileHalfs / 8);
  const int64_t blocks = (c.q_chunks + 2 * c.kv_chunks + 255) / 256;
  hipLaunchKernelGGL(convert_operands_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, c);
  if (hipGetLastError() != hipSuccess) return kErrLaunch;
  int64_t wgs = 0;
  if ((st = launch_shares(a, wgs, stream)) != kOk) return st;
  return launch_merge(a, wgs, stream);
}

extern "C" int oscar_prefill_continuation(
    const float* q_rot, const float* k_new, const float* v_new, int32_t num_new, int32_t num_heads,
    int32_t num_kv_heads, int32_t head_size, const void* k_cache, const void* v_cache,
    int32_t block_size, int64_t num_pages, int64_t k_stride_page, int64_t k_stride_token,
    int64_t k_stride_head, int64_t v_stride_page, int64_t v_stride_token, int64_t v_stride_head,
    const int32_t* block_table_row, int32_t block_table_cols, int64_t cached_len,
    const float* stage_k, const float* stage_v, const int64_t* stage_owner, int32_t stage_rows,
    float scale, float* out, hipStream_t stream) {
  PrefillArgs a{};
  if (num_new < 0 || cached_len < 0) return kErrInvalidArgument;
  int st = fill_common(a, num_new == 0, num_heads, num_kv_heads, head_size, k_cache, v_cache, block_size, num_pages,
                       k_stride_page, k_stride_token, k_stride_head, v_stride_page, v_stride_token, v_stride_head,
                       block_table_row, 0, block_table_cols, stage_k, stage_v, stage_owner, stage_rows, scale);
  if (st != kOk || num_new == 0) return st;
  if ((st = check_request(num_new, cached_len, num_heads, block_size, block_table_row, block_table_cols)) != kOk)
    return st;
  if (!q_rot || !k_new || !v_new || !out) return kErrInvalidArgument;
  a.q = q_rot;
  a.k_new = k_new;
  a.v_new = v_new;
  a.out = out;
  OperandItems ops{};
  add_item(a, ops, num_new, cached_len, 0, 0);
  if (prefers_rows(a)) return launch_rows(a, q_rot, k_new, v_new, out, stream);
  const int64_t rows = (int64_t)num_new * a.group;
  const dim3 grid((unsigned)((rows + kTileRows - 1) / kTileRows), (unsigned)num_kv_heads);
  if (set_dynamic_lds(reinterpret_cast<const void*>(prefill_kernel<false>), (int)kPrefillLds, g_lds_set[0]) != kOk)
    return kErrLaunch;
  hipLaunchKernelGGL((prefill_kernel<false>), grid, dim3(64 * kWaves), kPrefillLds, stream, a);
  return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}

extern "C" size_t oscar_prefill_rotated_workspace_bytes(int32_t num_requests, const int32_t* new_tokens,
                                                        const int64_t* cached_lens, int32_t num_heads,
                                                        int32_t num_kv_heads) {
  if (num_requests <= 0 || !new_tokens || !cached_lens || num_heads <= 0 || num_kv_heads <= 0 ||
      num_heads % num_kv_heads)
    return 0;
  size_t most = 0;
  for (int32_t r0 = 0; r0 < num_requests; r0 += kMaxPrefillItems) {     // one launch's requests
    int64_t tokens = 0, tiles = 0, units = 0;
    for (int32_t i = r0; i < num_requests && i < r0 + kMaxPrefillItems; ++i) {
      if (new_tokens[i] < 0 || cached_lens[i] < 0) return 0;
      tokens += new_tokens[i];
      tiles += (new_tokens[i] + kBlk - 1) / kBlk;
      units += host_head_units(new_tokens[i], cached_lens[i], num_heads / num_kv_heads) * num_kv_heads;
    }
    const size_t n = workspace_layout(tokens, tiles, units, num_heads, num_kv_heads, true).total;
    most = n > most ? n : most;
  }
  return most;
}

namespace oscar {

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
    hipStream_t stream) {
  PrefillArgs base{};
  int st = fill_common(base, false, num_heads, num_kv_heads, head_size, k_cache, v_cache, block_size, num_pages,
                       k_stride_page, k_stride_token, k_stride_head, v_stride_page, v_stride_token, v_stride_head,
                       block_table, block_table_stride, block_table_cols, stage_k, stage_v, stage_owner, stage_rows,
                       scale);
  if (st != kOk) return st;
  if (num_requests < 0) return kErrInvalidArgument;
  if (num_requests == 0) return kOk;
  if (!query_bf16 || !key_bf16 || !value_bf16 || !first_tokens || !new_tokens || !cached_lens || !table_rows ||
      !rot_k_operand || !rot_v_operand || !rot_v_t_operand || !out_bf16 || !workspace)
    return kErrInvalidArgument;
  // 16-byte vector accesses: every (token, head) row start 16-byte aligned
  if (query_token_stride < (int64_t)num_heads * kHeadDim || kv_token_stride < (int64_t)num_kv_heads * kHeadDim ||
      (query_token_stride & 7) || (kv_token_stride & 7) || (reinterpret_cast<uintptr_t>(query_bf16) & 15) ||
      (reinterpret_cast<uintptr_t>(key_bf16) & 15) || (reinterpret_cast<uintptr_t>(value_bf16) & 15) ||
      (reinterpret_cast<uintptr_t>(out_bf16) & 15) || (reinterpret_cast<uintptr_t>(rot_k_operand) & 15) ||
      (reinterpret_cast<uintptr_t>(rot_v_operand) & 15) || (reinterpret_cast<uintptr_t>(rot_v_t_operand) & 15) ||
      (reinterpret_cast<uintptr_t>(workspace) & 15))
    return kErrInvalidArgument;
  for (int32_t i = 0; i < num_requests; ++i) {
    if (first_tokens[i] < 0 || table_rows[i] < 0) return kErrInvalidArgument;
    if ((st = check_request(new_tokens[i], cached_lens[i], num_heads, block_size, block_table, block_table_cols)) !=
        kOk)
      return st;
  }
  if (workspace_size < oscar_prefill_rotated_workspace_bytes(num_requests, new_tokens, cached_lens, num_heads,
                                                             num_kv_heads))
    return kErrWorkspaceTooSmall;
  if (check_only) return kOk;
  for (int32_t r0 = 0; r0 < num_requests; r0 += kMaxPrefillItems) {
    PrefillArgs a = base;
    OperandItems ops{};
    for (int32_t i = r0; i < num_requests && i < r0 + kMaxPrefillItems; ++i)
      if (new_tokens[i] > 0) add_item(a, ops, new_tokens[i], cached_lens[i], table_rows[i], first_tokens[i]);
    if (a.nitems == 0) continue;
    const Layout w = workspace_layout(ops.tokens, ops.tiles, a.units, num_heads, num_kv_heads, true);
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    PrefillOperands o;
    bind_workspace(a, o, w, ws);
    a.out = reinterpret_cast<float*>(ws + w.out);
    st = launch_rotate_operands(static_cast<const uint16_t*>(query_bf16), query_token_stride,
                                static_cast<const uint16_t*>(key_bf16), static_cast<const uint16_t*>(value_bf16),
                                kv_token_stride, num_heads, num_kv_heads, static_cast<const uint8_t*>(rot_k_operand),
                                static_cast<const uint8_t*>(rot_v_operand), ops, o, write, stream);
    write = nullptr;
    if (st != kOk) return st;
    int64_t wgs = 0;
    if ((st = launch_shares(a, wgs, stream)) != kOk) return st;
    if ((st = launch_output(a, wgs, rot_v_t_operand, out_bf16, stream)) != kOk) return st;
  }
  return kOk;
}

}  // namespace oscar

extern "C" int oscar_prefill_rotated(
    const void* query_bf16, int64_t query_token_stride, const void* key_bf16, const void* value_bf16,
    int64_t kv_token_stride, int32_t num_requests, const int32_t* first_tokens, const int32_t* new_tokens,
    const int64_t* cached_lens, const int32_t* table_rows, int32_t num_heads, int32_t num_kv_heads,
    int32_t head_size, const void* rot_k_operand, const void* rot_v_operand, const void* rot_v_t_operand,
    const void* k_cache, const void* v_cache, int32_t block_size, int64_t num_pages, int64_t k_stride_page,
    int64_t k_stride_token, int64_t k_stride_head, int64_t v_stride_page, int64_t v_stride_token,
    int64_t v_stride_head, const int32_t* block_table, int64_t block_table_stride, int32_t block_table_cols,
    const float* stage_k, const float* stage_v, const int64_t* stage_owner, int32_t stage_rows, float scale,
    void* out_bf16, void* workspace, size_t workspace_size, hipStream_t stream) {
  return prefill_rotated(query_bf16, query_token_stride, key_bf16, value_bf16, kv_token_stride, num_requests, first_tokens,
                         new_tokens, cached_lens, table_rows, num_heads, num_kv_heads, head_size,
                         rot_k_operand, rot_v_operand, rot_v_t_operand, k_cache, v_cache,
                         block_size, num_pages, k_stride_page, k_stride_token, k_stride_head,
                         v_stride_page, v_stride_token, v_stride_head, block_table,
                         block_table_stride, block_table_cols, stage_k, stage_v, stage_owner,
                         stage_rows, scale, out_bf16, workspace, workspace_size, nullptr, false, stream);
}
