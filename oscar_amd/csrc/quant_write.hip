// Fused rotate + sort-clip + INT2 quantize + 4-codes-per-byte pack + paged
// slot write (gfx950).
//
// Work layout of the fused entry: a workgroup of eight wavefronts takes 32
// tokens of one (kv-head, K-or-V) side.  Each wavefront computes an eighth of
// the 256x256 rotation's output features for all of them on MFMA (bf16 hi + lo
// split of R, two passes); the values change hands through LDS, after which a
// row of 16 lanes holds a vector and everything that concerns it stays in the
// row.  The pre-rotated entry, and the kernel of large writes without a window
// (prefers_ring), have one wavefront to 32 tokens, lane l holding features 128
// (l >> 5) .. +127 of token l & 31.
//
// Clip threshold (the idx-th smallest |x| of a vector, i.e. its kk-th largest
// with kk = 256 - idx) without sorting: a 64-bucket histogram of |x| keyed on
// the float bits (bucket = key(max|x|) - key(|x|), key = bits >> S, S = 18:
// 1/32 octave per bucket over two octaves) built with LDS atomics gives the
// bucket holding the answer and its rank inside that bucket; the bucket's few
// values are gathered into small LDS lists and the answer is taken exactly
// (ties counted).  Vectors whose answer lies outside the histogram's range or
// whose bucket overflows the lists use a bitwise radix select instead (exact,
// slow, rare).
//
// Quantization: the exact divide-free thresholds of int2_quant.h.
//
// With a window arena (oscar_quant_write_window) the fused kernel also does
// the window write of the step's bulk tokens from the same rotated values,
// after a seat-winner pass over the step's slots.
#include <type_traits>

#include "bulk_write.h"
#include "int2_quant.h"
#include "prefill_operands.h"
#include "step_launch.h"
#include "window_images.h"
#include "../../include/oscar_amd.h"

namespace oscar {
namespace {

constexpr int kPerLane = kHeadDim / 2;      // 128 values of one vector per lane
constexpr int kTokPerWave = 32;


// Exact value of ascending-sorted |x| at index `idx` over the 256 values held
// by this lane and its partner (l ^ 32).  Bitwise radix select on the IEEE
// bit pattern: for non-negative finite floats, float order equals bit order.
__device__ float select_abs_rank(const float (&v)[kPerLane], int idx) {
  uint32_t prefix = 0;
#pragma unroll 1
  for (int bit = 30; bit >= 0; --bit) {
    const uint32_t probe = prefix | (1u << bit);
    const float pf = __uint_as_float(probe);
    int below = 0;
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) below += (fabsf(v[i]) < pf) ? 1 : 0;
    below += __shfl_xor(below, 32, 64);
    if (idx >= below) prefix = probe;
  }
  return __uint_as_float(prefix);
}

// Per-wave LDS of the threshold search: 32 token histograms (64 buckets + one
// bucket for everything below the range; stride 65 words keeps the tokens of
// one wave on different banks) and one candidate list per lane.
constexpr int kHistBuckets = 64;
constexpr int kHistStride = kHistBuckets + 1;
constexpr int kListCap = 8;
constexpr int kListStride = kListCap + 1;          // + one slot that absorbs non-candidates
struct SelLds {
  uint32_t hist[32 * kHistStride];
  uint32_t list[64 * kListStride];
};

__device__ __forceinline__ void wave_sync_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// kk-th largest |x| (kk = 256 - idx) of the 256 values held by this lane and
// its partner, as float bits; amax_bits = bits of max |x| over both lanes.
__device__ uint32_t select_clip_bits(const float (&v)[kPerLane], int idx, uint32_t amax_bits, SelLds& L,
                                     int lane) {
  const uint32_t kk = (uint32_t)(kHeadDim - idx);
  const int t = lane & 31, g = lane >> 5;
  const int S = kk <= 40 ? 18 : 20;          // 1/32 octave per bucket (2 octaves); coarser for deep ranks
  uint4* hz = reinterpret_cast<uint4*>(L.hist);
  for (int i = lane; i < 32 * kHistStride / 4; i += 64) hz[i] = uint4{0u, 0u, 0u, 0u};
  wave_sync_lds();
  // Row t: word 0 absorbs every key below the window, word 1 + j counts key
  // kl + j (kl = kh - 63), so bucket b from the top (key kh - b) is word 64 - b.
  // The byte address of key's word is 4 key + (row + 4 - 4 kl) on the 32-bit
  // LDS address, clamped from below to the absorbing word.
  typedef __attribute__((address_space(3))) uint32_t lds_u32;
  uint32_t* H = L.hist + t * kHistStride;
  const uint32_t kh = amax_bits >> S;
  const int32_t row = (int32_t)(uint32_t)(uintptr_t)(lds_u32*)H;
  const uint32_t base = (uint32_t)(row + 4 - 4 * ((int32_t)kh - (kHistBuckets - 1)));
#pragma unroll
  for (int i = 0; i < kPerLane; ++i) {
    const uint32_t key = __builtin_amdgcn_ubfe(__float_as_uint(v[i]), S, 31 - S);
    const int32_t addr = max((int32_t)((key << 2) + base), row);
    __atomic_fetch_add((lds_u32*)(uintptr_t)(uint32_t)addr, 1u, __ATOMIC_RELAXED);
  }
  wave_sync_lds();

  // Bucket b* where the count from the top reaches kk; lane g scans buckets
  // 32g .. 32g + 31.
  uint32_t cnt[32];
#pragma unroll
  for (int i = 0; i < 32; ++i) cnt[i] = H[kHistBuckets - 32 * g - i];
  uint32_t tot = 0;
#pragma unroll
  for (int i = 0; i < 32; ++i) tot += cnt[i];
  // (the exchange runs on every lane: a shuffle reads only active lanes)
  const uint32_t tot0 = (uint32_t)__shfl((int)tot, t, 64);
  uint32_t run = g ? tot0 : 0u;
  int bf = -1;
  uint32_t above = 0;
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    if (bf < 0 && run + cnt[i] >= kk) {
      bf = 32 * g + i;
      above = run;
    }
    run += cnt[i];
  }
  const int b0 = __shfl(bf, t, 64), b1 = __shfl(bf, t + 32, 64);
  const uint32_t a0 = (uint32_t)__shfl((int)above, t, 64), a1 = (uint32_t)__shfl((int)above, t + 32, 64);
  const int bstar = b0 >= 0 ? b0 : b1;
  const uint32_t ab = b0 >= 0 ? a0 : a1;
  const uint32_t keystar = kh - (uint32_t)bstar;
  bool fb = bstar < 0 || keystar == 0;

  // Gather bucket b*'s values: every value is written at the lane's next free
  // slot, which only advances on a match (capped at the absorbing slot).
  // The raw bits are stored (sign cleared on reading them back); the match
  // |x| >> S == keystar is tested on bits << 1, which drops the sign, as one
  // wrapping subtract and compare.
  uint32_t* mine = L.list + lane * kListStride;
  uint32_t n = 0;
  const uint32_t lo2 = keystar << (S + 1), w2 = 2u << S;
#pragma unroll
  for (int i = 0; i < kPerLane; ++i) {
    const uint32_t u = __float_as_uint(v[i]);
    mine[min(n, (uint32_t)kListCap)] = u;
    n += ((u << 1) - lo2 < w2) ? 1u : 0u;
  }
  wave_sync_lds();
  const uint32_t n0 = (uint32_t)__shfl((int)n, t, 64), n1 = (uint32_t)__shfl((int)n, t + 32, 64);
  fb = fb || n0 > kListCap || n1 > kListCap;
  uint32_t c[2 * kListCap];
  const uint32_t* l0 = L.list + t * kListStride;
  const uint32_t* l1 = L.list + (t + 32) * kListStride;
#pragma unroll
  for (int i = 0; i < kListCap; ++i) {
    c[i] = (uint32_t)i < n0 ? l0[i] & 0x7FFFFFFFu : 0u;
    c[kListCap + i] = (uint32_t)i < n1 ? l1[i] & 0x7FFFFFFFu : 0u;
  }
  // j-th largest of the candidates (j = kk - above >= 1), ties counted.
  uint32_t rem = kk - ab, prev = 0xFFFFFFFFu, res = 0u;
  if (fb) rem = 0;
#pragma unroll 1
  for (int it = 0; it <= 2 * kListCap && __ballot(rem > 0); ++it) {
    uint32_t m = 0u;
#pragma unroll
    for (int i = 0; i < 2 * kListCap; ++i) m = max(m, c[i] < prev ? c[i] : 0u);
    uint32_t ce = 0u;
#pragma unroll
    for (int i = 0; i < 2 * kListCap; ++i) ce += (c[i] == m) ? 1u : 0u;
    if (rem > 0) {
      if (m == 0u) {
        fb = true;
        rem = 0;
      } else if (ce >= rem) {
        res = m;
        rem = 0;
      } else {
        rem -= ce;
        prev = m;
      }
    }
  }
  if (__ballot(fb)) {
    const uint32_t r = __float_as_uint(select_abs_rank(v, idx));
    if (fb) res = r;
  }
  return res;
}

__device__ QParams vector_params(const float (&v)[kPerLane], int clip_idx, SelLds& L, int lane) {
  float mx = v[0], mn = v[0];
#pragma unroll
  for (int i = 1; i < kPerLane; ++i) {
    mx = fmaxf(mx, v[i]);
    mn = fminf(mn, v[i]);
  }
  mx = fmaxf(mx, shfl_xor_f32(mx, 32));
  mn = fminf(mn, shfl_xor_f32(mn, 32));
  float thr = __builtin_inff();
  if (clip_idx >= 0) {
    const uint32_t amax_bits = max(__float_as_uint(mx) & 0x7FFFFFFFu, __float_as_uint(mn) & 0x7FFFFFFFu);
    thr = __uint_as_float(select_clip_bits(v, clip_idx, amax_bits, L, lane));
  }
  return make_qparams(mn, mx, thr, clip_idx >= 0);
}

// Quantize, pack and store this lane's 128 codes (32 bytes) plus, on the
// lower half lane, the 4 meta bytes of this side.
__device__ void quantize_store(const float (&v)[kPerLane], const QParams& p, int64_t slot,
                               int head, int side, int half, const CacheArgs& c) {
  uint32_t words[8];
#pragma unroll
  for (int w = 0; w < 8; ++w) {
    uint32_t acc = 0;
#pragma unroll
    for (int i = 15; i >= 0; --i) acc = (acc << 2) | int2_code(v[16 * w + i], p);
    words[w] = acc;
  }
  if (slot < 0 || slot >= c.num_slots) return;
  const int64_t page = fast_div((uint32_t)slot, c.bs_div);
  const int64_t row = slot - page * c.block_size;
  uint8_t* kslot = c.k_cache + page * c.k_page + row * c.k_tok + (int64_t)head * c.k_head;
  uint8_t* dst;
  if (side == 0) {
    dst = kslot + kKCodeOff + 32 * half;
  } else {
    dst = c.v_cache + page * c.v_page + row * c.v_tok + (int64_t)head * c.v_head + 32 * half;
  }
  u32x4* d4 = reinterpret_cast<u32x4*>(dst);
  d4[0] = u32x4{words[0], words[1], words[2], words[3]};
  d4[1] = u32x4{words[4], words[5], words[6], words[7]};
  if (half == 0) *reinterpret_cast<uint32_t*>(kslot + 4 * side) = p.meta;
}

__device__ __forceinline__ int64_t read_lane64(int64_t x, int lane) {
  return (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(x >> 32), lane) << 32) |
                   (uint32_t)__builtin_amdgcn_readlane((int)x, lane));
}

// A step's request layout on its way from the host to the device: the first
// n of the ints go to dst.
constexpr int kLayoutInts = 896;
struct HostLayout {
  int32_t* dst;
  int32_t n;
  int32_t v[kLayoutInts];
};

__global__ __launch_bounds__(256) void store_layout_kernel(HostLayout h) {
  for (int i = threadIdx.x; i < h.n; i += 256) h.dst[i] = h.v[i];
}

// (its first workgroup also stores a request layout that came with the launch)
__global__ __launch_bounds__(256) void quant_window_winner_kernel(const int64_t* __restrict__ slots, int32_t n_tokens,
                                                                   int64_t* winner, int32_t block_size, int32_t rows,
                                                                   HostLayout h) {
  __shared__ int64_t epoch;
  if (blockIdx.x == 0)
    for (int i = threadIdx.x; i < h.n; i += 256) h.dst[i] = h.v[i];
  seat_winner_pass(slots, n_tokens, winner, (int64_t)rows * block_size, block_size, rows, &epoch);
}

// ---------------------------------------------------------------------------
// Pre-rotated entry: fp32 rotated input [N, Hk, D] (token stride in elements).
// grid = (ceil(N / 128), Hk * 2), block = 256 (4 waves x 32 tokens).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void quant_write_prerotated_kernel(
    const float* __restrict__ k_rot, const float* __restrict__ v_rot, int64_t n_tokens,
    int64_t token_stride, const int64_t* __restrict__ slots, CacheArgs c, int clip_k,
    int clip_v) {
  __shared__ SelLds sel[4];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int head = blockIdx.y >> 1;
  const int side = blockIdx.y & 1;
  const int half = lane >> 5;
  const int64_t tok = (int64_t)blockIdx.x * 128 + wave * kTokPerWave + (lane & 31);
  const bool live = tok < n_tokens;
  const float* src = (side == 0 ? k_rot : v_rot) + (live ? tok : 0) * token_stride +
                     (int64_t)head * kHeadDim + half * kPerLane;
  float v[kPerLane];
#pragma unroll
  for (int i = 0; i < kPerLane; i += 4) {
    floatx4 x = live ? *reinterpret_cast<const floatx4*>(src + i) : floatx4{0.f, 0.f, 0.f, 0.f};
    v[i] = x[0];
    v[i + 1] = x[1];
    v[i + 2] = x[2];
    v[i + 3] = x[3];
  }
  const QParams p = vector_params(v, side == 0 ? clip_k : clip_v, sel[wave], lane);
  quantize_store(v, p, live ? slots[tok] : -1, head, side, half, c);
}

// ---------------------------------------------------------------------------
// Rotation on MFMA of bf16 rows.
//
// Rotation operand (prepared once per layer by oscar_rotation_operand):
//   op[m][p][T][lane][u] (bf16), m = 16-row K step, p = 0 hi / 1 lo split,
//   T = 32-feature output tile.  Entry = R[e][f] with
//     e = 128*(lane >> 5) + 8*m + u                      (input feature)
//     f = 128*((r >> 2) & 1) + 16*T + 4*(r >> 3) + (r & 3), r = lane & 31
//   so that accumulator register i of tile T in lane l is feature
//   128*(l >> 5) + 16*T + i of token (l & 31) -- the per-lane layout above.
// Two ways to multiply by it: eight waves of a workgroup take a tile T each for
// the same 32 rows and read their fragments straight from L2 (fused_write and
// rotate_operands below); or four waves take all tiles for 32 rows each
// (rotate_tile: quant_write_ring_kernel and rotate_rows_kernel, block = 256,
// two blocks per CU), the 16 K-step chunks (16 KB each) streaming through a
// 4-slot LDS ring filled with buffer_load_dwordx4 ... lds: chunk m + 3 is
// requested while chunk m is multiplied, into the slot chunk m - 1 left, and
// each K step issues the 8 tiles' hi passes, then their lo passes, so that no
// MFMA waits on the previous.
// ---------------------------------------------------------------------------
constexpr int kFusedWaves = 4;
constexpr int kChunkBytes = 2 * 8 * 64 * 16;   // one K step: 2 passes x 8 tiles x 64 lanes x 16 B
constexpr int kRing = 4;
constexpr int kSteps = 16;
// The rotation operand: the MFMA tiles (kSteps chunks, bf16 hi + lo), then R
// itself in fp32 (row-major), which short writes rotate with.
constexpr int kMfmaEntries = kSteps * kChunkBytes / 2;
constexpr size_t kMfmaOperandBytes = (size_t)kSteps * kChunkBytes;
constexpr size_t kOperandBytes = kMfmaOperandBytes + sizeof(float) * kHeadDim * kHeadDim;
constexpr size_t kRingLds = kFusedWaves * sizeof(SelLds) > kRing * kChunkBytes ? kFusedWaves * sizeof(SelLds)
                                                                               : (size_t)kRing * kChunkBytes;
constexpr int64_t kRingRound = 512;             // workgroups of the ring kernel resident at once: two per CU
constexpr int64_t kShortWriteVectors = 2048;   // at most 1024 tokens (the step write's limit)
constexpr int kDmaPerChunk = kChunkBytes / (kFusedWaves * 64 * 16);   // 2 per thread

// Workgroup barrier without a memory fence: __syncthreads() would also wait
// for every outstanding global access (vmcnt(0)) and so drain the ring's
// prefetches.  The asm memory clobber keeps the compiler from moving LDS
// accesses across it; LDS visibility comes from the vmcnt waits above it
// (direct-to-LDS loads count as complete once their data is in LDS) and
// from the LDS reads' own completion before the next overwrite.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt(0xC07F);                     // lgkmcnt(0): this wave's LDS reads done
  asm volatile("s_barrier" ::: "memory");
}

// s_waitcnt vmcnt(n) with expcnt / lgkmcnt left at their maxima (gfx9 encoding).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// DPP moves within a row of 16 lanes.
template <int kCtrl>
__device__ __forceinline__ uint32_t row_dpp(uint32_t x) {      // lanes without a source read 0
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kCtrl, 0xF, 0xF, true);
}
constexpr int kRowRor = 0x120, kRowShr = 0x110;                // + distance

template <class Op>
__device__ __forceinline__ uint32_t row_reduce(uint32_t x, Op op) {   // result in every lane of the row
  x = op(x, row_dpp<kRowRor + 8>(x));
  x = op(x, row_dpp<kRowRor + 4>(x));
  x = op(x, row_dpp<kRowRor + 2>(x));
  return op(x, row_dpp<kRowRor + 1>(x));
}

__device__ __forceinline__ uint32_t row_scan(uint32_t x) {            // inclusive sum
  x += row_dpp<kRowShr + 1>(x);
  x += row_dpp<kRowShr + 2>(x);
  x += row_dpp<kRowShr + 4>(x);
  return x + row_dpp<kRowShr + 8>(x);
}

// The bulk write's workgroup: eight waves and 32 tokens of one (kv-head, K or
// V) side.  Lane 16 i + j of a wave ends up with features 16 j .. 16 j + 15 of
// the wave's token i, so that whatever concerns a vector stays in one row of
// 16 lanes.
constexpr int kFwTokens = 32;
constexpr int kFwThreads = 512;
constexpr int kFwTokPerWave = 4;
constexpr int kFwPerLane = 16;
constexpr int kFwAhead = 3;

// LDS of the threshold search, per wave: a histogram and a candidate list per
// token, and a word per lane that absorbs what belongs in neither (one word
// per token would serialise its 16 lanes: 91 instead of 72 us for 65536
// tokens).
struct RowSelLds {
  uint32_t hist[kFwTokPerWave][kHistStride];
  uint32_t list[kFwTokPerWave][16];
  uint32_t other[64];
};

// The idx-th smallest |x| (float bits) of the 256 values a row of lanes
// holds, without sorting: select_clip_bits' histogram and candidates, a
// vector to a row.  amax_bits = bits of max |x|.
__device__ __forceinline__ uint32_t row_select(const float (&v)[kFwPerLane], int idx, uint32_t amax_bits,
                                               RowSelLds& L, int lane) {
  const uint32_t kk = (uint32_t)(kHeadDim - idx);
  const int i4 = lane >> 4, j = lane & 15;
  const int S = kk <= 40 ? 18 : 20;
  uint32_t* flat = &L.hist[0][0];
  constexpr int kWords = kFwTokPerWave * kHistStride;
#pragma unroll
  for (int i = 0; i < (kWords + 63) / 64; ++i)
    if (i * 64 + lane < kWords) flat[i * 64 + lane] = 0u;
  wave_sync_lds();
  typedef __attribute__((address_space(3))) uint32_t lds_u32;
  uint32_t* H = L.hist[i4];
  const uint32_t kh = amax_bits >> S;
  const uint32_t first = (uint32_t)(uintptr_t)(lds_u32*)H + 4u;      // bucket 63's word
  const uint32_t other = (uint32_t)(uintptr_t)(lds_u32*)&L.other[lane];
  const uint32_t low = kh - (uint32_t)(kHistBuckets - 1);
#pragma unroll
  for (int i = 0; i < kFwPerLane; ++i) {
    const uint32_t b = __builtin_amdgcn_ubfe(__float_as_uint(v[i]), S, 31 - S) - low;
    const uint32_t addr = b < (uint32_t)kHistBuckets ? first + 4u * b : other;
    __atomic_fetch_add((lds_u32*)(uintptr_t)addr, 1u, __ATOMIC_RELAXED);
  }
  wave_sync_lds();
  // Bucket b* where the count from the top reaches kk: lane j scans buckets
  // 4j .. 4j + 3 from the top (words 64 - b).
  uint32_t cnt[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) cnt[i] = H[kHistBuckets - 4 * j - i];
  const uint32_t tot = cnt[0] + cnt[1] + cnt[2] + cnt[3];
  const uint32_t upto = row_scan(tot);
  uint32_t run = upto - tot, hit = 0u;                  // hit: (bucket + 1) << 16 | count above it
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (run < kk && run + cnt[i] >= kk) hit = ((uint32_t)(4 * j + i + 1) << 16) | run;
    run += cnt[i];
  }
  auto umax = [](uint32_t a, uint32_t b) { return max(a, b); };
  hit = row_reduce(hit, umax);
  const uint32_t keystar = kh + 1u - (hit >> 16), rem = kk - (hit & 0xFFFFu);
  bool fb = hit == 0u || keystar == 0u;
  // The values of bucket b*, packed over the row.
  const uint32_t lo2 = keystar << (S + 1), w2 = 2u << S;
  uint32_t n = 0u;
#pragma unroll
  for (int i = 0; i < kFwPerLane; ++i) n += ((__float_as_uint(v[i]) << 1) - lo2 < w2) ? 1u : 0u;
  const uint32_t end = row_scan(n);
  const uint32_t total = row_reduce(end, umax);
  fb = fb || total > 16u;
  uint32_t* list = L.list[i4];
  uint32_t at = end - n;
#pragma unroll
  for (int i = 0; i < kFwPerLane; ++i) {
    const uint32_t u = __float_as_uint(v[i]);
    const bool match = (u << 1) - lo2 < w2;
    *(match && at < 16u ? list + at : &L.other[lane]) = u & 0x7FFFFFFFu;
    at += match ? 1u : 0u;
  }
  wave_sync_lds();
  // The rem-th largest of the candidates, ties counted.
  const uint32_t c = (uint32_t)j < total ? list[j] : 0u;
  uint32_t gt = 0u, ge = 1u;
  auto rank = [&](uint32_t o) {
    gt += o > c ? 1u : 0u;
    ge += o >= c ? 1u : 0u;
  };
  rank(row_dpp<kRowRor + 1>(c));
  rank(row_dpp<kRowRor + 2>(c));
  rank(row_dpp<kRowRor + 3>(c));
  rank(row_dpp<kRowRor + 4>(c));
  rank(row_dpp<kRowRor + 5>(c));
  rank(row_dpp<kRowRor + 6>(c));
  rank(row_dpp<kRowRor + 7>(c));
  rank(row_dpp<kRowRor + 8>(c));
  rank(row_dpp<kRowRor + 9>(c));
  rank(row_dpp<kRowRor + 10>(c));
  rank(row_dpp<kRowRor + 11>(c));
  rank(row_dpp<kRowRor + 12>(c));
  rank(row_dpp<kRowRor + 13>(c));
  rank(row_dpp<kRowRor + 14>(c));
  rank(row_dpp<kRowRor + 15>(c));
  uint32_t res = row_reduce(gt < rem && rem <= ge ? c : 0u, umax);
  if (__ballot(fb) != 0ull) {
    // outside the histogram, or a crowded bucket: bitwise radix select (exact)
    uint32_t prefix = 0u;
#pragma unroll 1
    for (int b = 30; b >= 0; --b) {
      const uint32_t probe = prefix | (1u << b);
      const float pf = __uint_as_float(probe);
      uint32_t below = 0u;
#pragma unroll
      for (int i = 0; i < kFwPerLane; ++i) below += fabsf(v[i]) < pf ? 1u : 0u;
      below = row_reduce(below, [](uint32_t a, uint32_t b2) { return a + b2; });
      if ((uint32_t)idx >= below) prefix = probe;
    }
    if (fb) res = prefix;
  }
  return res;
}

// The V image of the workgroup's kept tokens, from their rotated values in
// LDS (value(r, f): feature f of token r): seat_tile / seat_slot are token
// lane & 31's image tile and its slot there (-1: not kept).  Wave w stores
// features 32 w .. 32 w + 31.  An image chunk holds eight tokens of one
// feature: chunks the workgroup's tokens fill leave as 16-byte stores, the
// tokens of others go one by one.  (Two-byte stores for all of them, 256 a
// token, took 23 us.)
template <class Value>
__device__ __forceinline__ void store_v_images(const Value& value, int64_t seat_tile, int seat_slot, uint8_t* inv,
                                               _Float16* vimg, int wave, int lane) {
  const int me = lane & 31;
  uint32_t pending = (uint32_t)__ballot(seat_slot >= 0);
  uint32_t single = 0u;
  while (pending != 0u) {
    const int leader = (int)__builtin_ctz(pending);
    const int64_t tile = read_lane64(seat_tile, leader);
    const bool mine = ((pending >> me) & 1u) != 0u && seat_tile == tile;
    const uint32_t group = (uint32_t)__ballot(mine);
    pending &= ~group;
    uint32_t have = mine ? 1u << seat_slot : 0u, full = 0u;
    if (__popc(group) >= 8) {
#pragma unroll
      for (int o = 16; o >= 1; o >>= 1) have |= (uint32_t)__shfl_xor((int)have, o, 64);
#pragma unroll
      for (int g = 0; g < 4; ++g) full |= ((have >> (8 * g)) & 0xFFu) == 0xFFu ? 1u << (8 * g) : 0u;
    }
    single |= (uint32_t)__ballot(mine && ((full >> (seat_slot & 24)) & 1u) == 0u);
    if (full == 0u) continue;
    if (mine && lane < 32) inv[seat_slot] = (uint8_t)me;      // token of each slot
    wave_sync_lds();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int u = 64 * i + lane;
      const int ml = u & 15, b = (u >> 4) & 1, grp = u >> 5;
      if (((full >> (8 * grp)) & 1u) == 0u) continue;
      const int f = 32 * wave + 4 * (ml >> 1) + 2 * b + (ml & 1);
      half8 hi, lo;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int t = e == 1 ? 2 : (e == 2 ? 1 : (e == 5 ? 6 : (e == 6 ? 5 : e)));
        _Float16 x, y;
        fp16_parts(value(inv[8 * grp + t], f), x, y);
        hi[e] = x;
        lo[e] = y;
      }
      _Float16* d = vimg + tile * kVImgHalfs + vimg_offset(f, 8 * grp);
      *reinterpret_cast<half8*>(d) = hi;
      *reinterpret_cast<half8*>(d + kVPartHalfs) = lo;
    }
    wave_sync_lds();
  }
  // two tokens at a time, a feature per lane (the last token twice if odd)
  while (single != 0u) {
    const int t0 = (int)__builtin_ctz(single);
    single &= single - 1u;
    const int t1 = single != 0u ? (int)__builtin_ctz(single) : t0;
    single &= single - 1u;
    const int64_t tile0 = read_lane64(seat_tile, t0), tile1 = read_lane64(seat_tile, t1);
    const int slot0 = __builtin_amdgcn_readlane(seat_slot, t0), slot1 = __builtin_amdgcn_readlane(seat_slot, t1);
    const int f = 32 * wave + me;
    const bool first = lane < 32;
    _Float16* d = vimg + (first ? tile0 : tile1) * kVImgHalfs + vimg_offset(f, first ? slot0 : slot1);
    fp16_parts(value(first ? t0 : t1, f), d[0], d[kVPartHalfs]);
  }
}

// Rotation, clip, quantization and slot write of 32 tokens, and their window
// write.  The waves bring the tokens' rows to LDS as MFMA operands; wave t
// computes rotated features {128 h + 16 t + i} of every token, its operand
// fragments of R (bf16 high, then low part) straight from L2, kFwAhead steps
// ahead; the values then change hands through LDS (64-byte chunks, swizzled)
// so that each vector lies in one row of 16 lanes.
// Writes up to 8K tokens are bound by one workgroup's latency, larger ones by
// the products (two bf16 passes, 28 us for 65536 tokens at the rate of a
// large library product) beside the selection's vector instructions, which a
// CU's workgroups overlap: four of them (64 registers), two where the write
// shares a launch with the prefill operands (106).  With 128 tokens to a workgroup of four
// wavefronts, each with 32 tokens of its own and R through an LDS ring, 3001
// tokens took 29 us with the window (their selection 10, its image 7), 1052
// of a mixed step 36, 9256 29 and 65536 without one 71; this takes 11, 15, 20
// and 64 (a write of that size takes the ring kernel, see prefers_ring).  64
// tokens to a workgroup (half the reading of R): 17, -, 25, 68.
// 33 KB, so that four workgroups fit a CU: the operands' rows [k-step][row ^
// k-step, half] until the products are done, then the rotated values, in a
// wave's share of which its selection works once the wave has read them.
struct FusedWriteLds {
  union {
    uint16_t xs[kSteps][64][8];
    floatx4 ys[kFwTokens * kHeadDim / 4];
  };
  int64_t seat_tile[kFwTokens];
  int32_t seat_slot[kFwTokens];
  uint8_t inv[kFwThreads / 64][32];
  __device__ FusedWriteLds() {}
};
static_assert(sizeof(RowSelLds) <= kFwTokPerWave * kHeadDim * sizeof(float), "the selection fits its wave's values");

__device__ __forceinline__ void fused_write(const FusedWriteArgs& a, FusedWriteLds& S, int block) {
  auto& xs = S.xs;
  auto& ys = S.ys;
  auto& seat_tile = S.seat_tile;
  auto& seat_slot = S.seat_slot;
  auto& inv = S.inv;
  const CacheArgs& c = a.c;
  const WindowArgs& w = a.w;
  const int64_t n_tokens = a.n_tokens;
  const int64_t* slots = a.slots;
  const int by = block / a.token_blocks, bx = block - by * a.token_blocks;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int head = by >> 1;
  const int side = by & 1;
  const int half = lane >> 5;
  const int64_t tok0 = (int64_t)bx * kFwTokens;
  const u32x4* frag = reinterpret_cast<const u32x4*>(side == 0 ? a.rot_k : a.rot_v) + wave * 64 + lane;
  auto load_r = [&](int m, int p) { return __builtin_bit_cast(bf16x8, frag[(m * 16 + p * 8) * 64]); };

  // ---- rows to LDS: piece u & 31 (eight features) of token u >> 5; tokens
  // past the last read it again and store nothing ----
  u32x4 piece[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int u = (int)threadIdx.x + kFwThreads * i;
    const int64_t tok = min(tok0 + (u >> 5), n_tokens - 1);
    piece[i] = reinterpret_cast<const u32x4*>((side == 0 ? a.key : a.value) + tok * a.token_stride +
                                              (int64_t)head * kHeadDim)[u & 31];
  }
  // this lane's token from the exchange on
  const int r = kFwTokPerWave * wave + (lane >> 4), j = lane & 15;
  const int64_t tok = tok0 + r;
  const int64_t slot = tok < n_tokens ? slots[tok] : -1;
  bf16x8 f[kFwAhead][2];
#pragma unroll
  for (int m = 0; m < kFwAhead; ++m) {
    f[m][0] = load_r(m, 0);
    f[m][1] = load_r(m, 1);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int u = (int)threadIdx.x + kFwThreads * i, m = u & 15;
    *reinterpret_cast<u32x4*>(&xs[m][((u >> 5) ^ m) + 32 * ((u >> 4) & 1)][0]) = piece[i];
  }
  __syncthreads();
  floatx16 acc = floatx16{};
#pragma unroll
  for (int m = 0; m < kSteps; ++m) {
    const bf16x8 rh = f[m % kFwAhead][0], rl = f[m % kFwAhead][1];
    if (m + kFwAhead < kSteps) {
      f[m % kFwAhead][0] = load_r(m + kFwAhead, 0);
      f[m % kFwAhead][1] = load_r(m + kFwAhead, 1);
    }
    const bf16x8 x = *reinterpret_cast<const bf16x8*>(&xs[m][((lane & 31) ^ m) + (lane & 32)][0]);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(rh, x, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(rl, x, acc, 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);      // (keeps the scheduler from hoisting every step's reads)
  }

  // ---- exchange: 16-byte quarter q of token r's chunk jj (features 16 jj ..)
  // lies where 16 tokens of one chunk, and the 16 chunks of one token, fall on
  // different banks ----
  auto place = [](int rr, int jj, int q) {
    return rr * 64 + ((jj ^ (rr & 15)) * 4) + (q ^ ((rr >> 2) & 3) ^ ((jj >> 2) & 3));
  };
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 4; ++q)
    ys[place(lane & 31, 8 * half + wave, q)] = floatx4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
  __syncthreads();
  float v[kFwPerLane];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const floatx4 y = ys[place(r, j, q)];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[4 * q + e] = y[e];
  }

  // ---- quantize and store ----
  float mx = v[0], mn = v[0];
#pragma unroll
  for (int i = 1; i < kFwPerLane; ++i) {
    mx = fmaxf(mx, v[i]);
    mn = fminf(mn, v[i]);
  }
  mx = __uint_as_float(row_reduce(__float_as_uint(mx), [](uint32_t a, uint32_t b) {
    return __float_as_uint(fmaxf(__uint_as_float(a), __uint_as_float(b)));
  }));
  mn = __uint_as_float(row_reduce(__float_as_uint(mn), [](uint32_t a, uint32_t b) {
    return __float_as_uint(fminf(__uint_as_float(a), __uint_as_float(b)));
  }));
  const int clip = side == 0 ? a.clip_k : a.clip_v;
  float thr = __builtin_inff();
  if (clip >= 0) {
    const uint32_t amax_bits = max(__float_as_uint(mx) & 0x7FFFFFFFu, __float_as_uint(mn) & 0x7FFFFFFFu);
    thr = __uint_as_float(row_select(
        v, clip, amax_bits, *reinterpret_cast<RowSelLds*>(&ys[wave * kFwTokPerWave * (kHeadDim / 4)]), lane));
  }
  const QParams p = make_qparams(mn, mx, thr, clip >= 0);
  uint32_t word = 0;
#pragma unroll
  for (int i = kFwPerLane - 1; i >= 0; --i) word = (word << 2) | int2_code(v[i], p);
  if (slot >= 0 && slot < c.num_slots) {
    const int64_t page = fast_div((uint32_t)slot, c.bs_div);
    const int64_t row = slot - page * c.block_size;
    uint8_t* kslot = c.k_cache + page * c.k_page + row * c.k_tok + (int64_t)head * c.k_head;
    uint8_t* codes = side == 0 ? kslot + kKCodeOff
                               : c.v_cache + page * c.v_page + row * c.v_tok + (int64_t)head * c.v_head;
    reinterpret_cast<uint32_t*>(codes)[j] = word;
    if (j == 0) *reinterpret_cast<uint32_t*>(kslot + 4 * side) = p.meta;
  }
  if (w.rows <= 0) return;

  // ---- window (the reference's _staging_write, backend.py:439-481): the
  // token that won its seat sets the seat's owner (the K side of head 0 does)
  // to its page when it lies in the sink or recent window and to -1
  // otherwise; a kept token's unclipped rotated values go to the arena and, as
  // fp16 parts, to the operand images ----
  int64_t seat = 0, page = 0;
  bool keep = false;
  if (slot >= 0 &&
      won_seat(w.winner, (int64_t)w.rows * c.block_size, slot, tok, c.block_size, w.rows, seat, page)) {
    int lo = 0, hi = w.num_requests - 1;     // request of the token: last i with query_start[i] <= tok
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (w.query_start[mid] <= tok) lo = mid; else hi = mid - 1;
    }
    const int64_t seq = w.seq_lens[lo];
    const int64_t pos = seq - w.query_start[lo + 1] + tok;
    keep = pos >= seq - w.recent || pos < w.sink_eff;
    if (side == 0 && head == 0 && j == 0) w.owner[seat] = keep ? page : -1;
  }
  const bool v_images = side == 1 && w.kimg != nullptr;
  int64_t tile = 0;
  int tt = -1;
  if (keep) {
    floatx4* dst = reinterpret_cast<floatx4*>((side == 0 ? w.stage_k : w.stage_v) +
                                              (seat * w.num_kv_heads + head) * kHeadDim + kFwPerLane * j);
#pragma unroll
    for (int q = 0; q < 4; ++q) dst[q] = floatx4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
    if (w.kimg != nullptr) {
      const int prow = (int)(slot - page * c.block_size);
      tile = image_of(seat / c.block_size, prow, c.block_size, head, w.num_kv_heads);
      tt = prow & 31;
      if (side == 0) {
        // block m = 2 (j & 7) + b, lane tt + 32 (j >> 3), slot u: local feature 4b + (u >> 1) + 8 (u & 1)
        _Float16* img = w.kimg + tile * kKImgHalfs + (2 * (j & 7) * 64 + tt + 32 * (j >> 3)) * 8;
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          half8 h, l;
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            _Float16 x, y;
            fp16_parts(v[4 * b + (u >> 1) + 8 * (u & 1)], x, y);
            h[u] = x;
            l[u] = y;
          }
          *reinterpret_cast<half8*>(img + b * 64 * 8) = h;
          *reinterpret_cast<half8*>(img + kImgHalfs + b * 64 * 8) = l;
        }
      }
    }
  }
  if (!v_images) return;
#pragma unroll
  for (int q = 0; q < 4; ++q) ys[place(r, j, q)] = floatx4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
  if (j == 0) {
    seat_tile[r] = tile;
    seat_slot[r] = tt;
  }
  __syncthreads();
  const float* yf = reinterpret_cast<const float*>(ys);
  store_v_images([&](int rr, int ff) { return yf[4 * place(rr, ff >> 4, (ff >> 2) & 3) + (ff & 3)]; },
                 seat_tile[lane & 31], seat_slot[lane & 31], inv[wave], w.vimg, wave, lane);
}

__global__ __launch_bounds__(kFwThreads, 8) void quant_write_fused_kernel(FusedWriteArgs a) {
  __shared__ FusedWriteLds S;
  fused_write(a, S, blockIdx.x);
}

// Rows rotated on MFMA: out = in @ R for rows of D = 256 features (the
// reference's q / k / v rotations and R_v^T around its dense read,
// oscar_ascend/backend.py:392-413).  An entry for callers who rotate rows of
// their own: the prefill read here rotates in rotate_operands and
// prefill_output_kernel.  in: bf16 (an exact operand) or fp32
// (its bf16 high and low parts); R: the operand's bf16 high and low parts;
// fp32 accumulation (about 2^-16 of each product); out: fp32, or bf16
// rounded to nearest even.
// grid = ceil(rows / 128), block = 256 (4 waves x 32 rows): lane l takes row
// (l & 31) of its wave, input and output features 128 (l >> 5) .. +127, and
// the operand streams through the 4-slot LDS ring.  A bf16
// input's first half (K steps 0-7) is requested before the ring and its
// second half during step 4; an fp32 input (twice the registers) comes in
// quarters, the first before the ring and quarter q (steps 4q .. 4q + 3)
// during step 4q - 3.  kRotWait gives each step's wait: the loads issued
// after the last one the step needs (its chunk and its input).
// ---------------------------------------------------------------------------
template <bool kF32In>
struct RotSched {
  static constexpr int kParts = kF32In ? 4 : 2;                 // input parts (quarters / halves)
  static constexpr int kPartLoads = 2 * kSteps / kParts / (kF32In ? 1 : 2);   // 16-byte loads per part
  // step during which part p (> 0) is requested
  static __device__ constexpr int step_of(int p) { return kF32In ? 4 * p - 3 : 4; }
};
template <bool kF32In>
__device__ constexpr int kRotWait(int m) {
  return kF32In ? (m == 14 ? 4 : m == 15 ? 0 : ((m & 3) >= 2 ? 16 : 8))
                : ((m >= 5 && m <= 7) ? 16 : m == 14 ? 4 : m == 15 ? 0 : 8);
}

// The rotation of one wave's 32 rows: lane l's row starts at xsrc (its input
// features 128 (l >> 5) .. +127); register i of tile t is output feature 128 (l
// >> 5) + 16 t + i of row l & 31.
template <bool kF32In>
__device__ __forceinline__ void rotate_tile(const uint8_t* __restrict__ xsrc, const uint8_t* __restrict__ rop,
                                            uint8_t* ring, int wave, int lane, floatx16 (&acc)[8]) {
  using Sched = RotSched<kF32In>;
  // input of K step m: features 128 half + 8m .. +7 (one 16-byte load, or two for fp32)
  u32x4 xr[Sched::kParts * Sched::kPartLoads];
  auto load_part = [&](int p) {
#pragma unroll
    for (int i = 0; i < Sched::kPartLoads; ++i)
      xr[p * Sched::kPartLoads + i] = reinterpret_cast<const u32x4*>(xsrc)[p * Sched::kPartLoads + i];
  };
  load_part(0);
  typedef __attribute__((address_space(3))) void lds_void;
  const __amdgpu_buffer_rsrc_t rop_rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)rop, (short)0, (int)(kSteps * kChunkBytes), 0x00020000);
  auto request = [&](int chunk) {
#pragma unroll
    for (int i = 0; i < kDmaPerChunk; ++i) {
      const int blk = kDmaPerChunk * wave + i;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rop_rsrc, (lds_void*)(uintptr_t)(uint32_t)(uintptr_t)(ring + (chunk % kRing) * kChunkBytes + blk * 1024),
          16, chunk * kChunkBytes + (blk * 64 + lane) * 16, 0, 0, 0);
    }
  };
  request(0);
  request(1);
  request(2);
#pragma unroll
  for (int t = 0; t < 8; ++t) acc[t] = floatx16{};
  constexpr int kPairs = kF32In ? 24 : 16;      // (fragment, operand) products per K step
#pragma unroll
  for (int m = 0; m < kSteps; ++m) {
    {
      // (m is a constant once the loop is unrolled: one wait remains)
      const int wn = kRotWait<kF32In>(m);
      if (wn == 24) wait_vmcnt<24>();
      else if (wn == 16) wait_vmcnt<16>();
      else if (wn == 8) wait_vmcnt<8>();
      else if (wn == 4) wait_vmcnt<4>();
      else wait_vmcnt<0>();
    }
    lds_barrier();
    if (m + 3 < kSteps) request(m + 3);
    // the wait counts above assume every input load of a part after this
    // step's chunk request: keep the scheduler from hoisting one
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int p = 1; p < Sched::kParts; ++p)
      if (m == Sched::step_of(p)) load_part(p);
    bf16x8 xh, xl;
    if constexpr (kF32In) {
      const floatx4 f0 = __builtin_bit_cast(floatx4, xr[2 * m]), f1 = __builtin_bit_cast(floatx4, xr[2 * m + 1]);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float v = u < 4 ? f0[u] : f1[u - 4];
        const __bf16 h = (__bf16)v;
        xh[u] = h;
        xl[u] = (__bf16)(v - (float)h);
      }
    } else {
      xh = __builtin_bit_cast(bf16x8, xr[m]);
      xl = xh;
    }
    // pair i < 16: fragment i (8 p + t) times the high part; i >= 16 (fp32
    // input): fragment i - 16 (R's high part) times the low part
    const u32x4* a_src = reinterpret_cast<const u32x4*>(ring + (m % kRing) * kChunkBytes);
    constexpr int kAhead = 6;
    bf16x8 a[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) a[i] = __builtin_bit_cast(bf16x8, a_src[(i & 15) * 64 + lane]);
#pragma unroll
    for (int i = 0; i < kPairs; ++i) {
      const bf16x8 cur = a[i % kAhead];
      if (i + kAhead < kPairs)
        a[i % kAhead] = __builtin_bit_cast(bf16x8, a_src[((i + kAhead) & 15) * 64 + lane]);
      const bf16x8 x = i < 16 ? xh : xl;
      acc[i & 7] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur, x, acc[i & 7], 0, 0, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);
#pragma unroll
    for (int i = 0; i < kPairs; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      if (i + kAhead < kPairs) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
  }
}

// Large writes without a window: 128 tokens to a workgroup of four waves, each
// with 32 tokens of its own (lane l: features 128 (l >> 5) .. +127 of token l &
// 31), R through the LDS ring.  It reads R a quarter as often as
// quant_write_fused_kernel and needs no exchange, but a round of it takes about
// 30 us however few of its workgroups are left.  Same products in the same
// order, same bytes.  prefers_ring says when it is taken.
__global__ __launch_bounds__(256, 2) void quant_write_ring_kernel(FusedWriteArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t ring[];     // ring, then the selection buffers
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int by = (int)blockIdx.x / a.token_blocks, bx = (int)blockIdx.x - by * a.token_blocks;
  const int head = by >> 1, side = by & 1, half = lane >> 5;
  const int64_t tok = (int64_t)bx * (kFusedWaves * kTokPerWave) + wave * kTokPerWave + (lane & 31);
  const bool live = tok < a.n_tokens;       // (else token 0 is computed and nothing stored)
  floatx16 acc[8];
  rotate_tile<false>(reinterpret_cast<const uint8_t*>((side == 0 ? a.key : a.value) + (live ? tok : 0) * a.token_stride +
                                                      (int64_t)head * kHeadDim + half * kPerLane),
                     side == 0 ? a.rot_k : a.rot_v, ring, wave, lane, acc);
  __syncthreads();      // the ring becomes the waves' selection buffers
  float v[kPerLane];
#pragma unroll
  for (int t = 0; t < 8; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) v[16 * t + i] = acc[t][i];
  const QParams p =
      vector_params(v, side == 0 ? a.clip_k : a.clip_v, reinterpret_cast<SelLds*>(ring)[wave], lane);
  quantize_store(v, p, live ? a.slots[tok] : -1, head, side, half, a.c);
}

template <bool kF32In, bool kBf16Out>
__global__ __launch_bounds__(256, 2) void rotate_rows_kernel(const void* __restrict__ in, int64_t in_stride,
                                                            int64_t rows, const uint8_t* __restrict__ rop,
                                                            void* __restrict__ out, int64_t out_stride) {
  extern __shared__ __attribute__((aligned(16))) uint8_t ring[];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int half = lane >> 5;
  const int64_t row = (int64_t)blockIdx.x * (kFusedWaves * kTokPerWave) + wave * kTokPerWave + (lane & 31);
  const bool live = row < rows;
  const int64_t rr = live ? row : 0;        // a lane past the last row computes row 0 and stores nothing
  floatx16 acc[8];
  rotate_tile<kF32In>(static_cast<const uint8_t*>(in) + (rr * in_stride + kPerLane * half) * (kF32In ? 4 : 2),
                     rop, ring, wave, lane, acc);
  if (!live) return;
  // register i of tile t: output feature 128 half + 16 t + i
  if constexpr (kBf16Out) {
    __bf16* dst = static_cast<__bf16*>(out) + row * out_stride + kPerLane * half;
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        bf16x8 o;
#pragma unroll
        for (int u = 0; u < 8; ++u) o[u] = (__bf16)acc[t][8 * q + u];
        *reinterpret_cast<bf16x8*>(dst + 16 * t + 8 * q) = o;
      }
  } else {
    float* dst = static_cast<float*>(out) + row * out_stride + kPerLane * half;
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<floatx4*>(dst + 16 * t + 4 * q) =
            floatx4{acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3]};
  }
}

// Operands of the prefill read (prefill_operands.h) from the step's bf16
// query, key and value, in one launch: workgroups of 32 query rows, then of
// one 32-token key tile, then of one value tile.  The eight waves bring the
// rows to LDS as MFMA operands; then wave t computes rotated features {128 h +
// 16 t + i} of every row, its operand fragments of R (bf16 high, then low
// part) straight from L2, kOpAhead steps ahead of their use, and rounds to
// fp16 what the read rounded when it built its tiles from fp32 rows.  Queries
// and keys keep a row per lane; the values' product runs with the operands
// exchanged, so that a lane holds one feature of 16 tokens, which are its two
// 16-byte chunks of the V tile.
// Small calls are bound by one workgroup's latency, large ones by reading R
// (256 KB a workgroup) from L2.  128 rows to a workgroup with R through an LDS
// ring took 18.4 us for 3001 tokens, 12.6 for 1024, 11.0 for 77 and 41 for
// 9256 (six query heads); this takes 14.9, 7.6, 5.8 and 38.  64 rows, which
// read R half as often, took 15.2, 9.5, 7.9 and 34: only the last is better.
// (Fragments four steps ahead spill a few registers: 7.4 us for 77 tokens.)
struct RotateOperandArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  int64_t q_stride, kv_stride;
  int32_t num_heads, num_kv_heads;
  const uint8_t* rot_k;
  const uint8_t* rot_v;
  PrefillOperands o;
  int32_t q_blocks, kv_blocks;
  OperandItems items;
};
constexpr int kOpAhead = 2;

struct OperandLds {
  // [k-step][row ^ k-step, half][8]: swizzled so that the 16 k-steps of one
  // row fall on different banks
  __attribute__((aligned(16))) uint16_t xs[kSteps][64][8];
  float qs[8][32];
};

__device__ __forceinline__ void rotate_operands(const RotateOperandArgs& a, OperandLds& S, int blk) {
  auto& xs = S.xs;
  auto& qs = S.qs;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int half = lane >> 5;
  const int kind = blk < a.q_blocks ? 0 : (blk < a.q_blocks + a.kv_blocks ? 1 : 2);    // query, key, value
  blk -= kind == 0 ? 0 : (kind == 1 ? a.q_blocks : a.q_blocks + a.kv_blocks);
  const u32x4* frag = reinterpret_cast<const u32x4*>(kind == 2 ? a.rot_v : a.rot_k) + wave * 64 + lane;
  auto load_r = [&](int m, int p) { return __builtin_bit_cast(bf16x8, frag[(m * 16 + p * 8) * 64]); };
  bf16x8 f[kOpAhead][2];
#pragma unroll
  for (int m = 0; m < kOpAhead; ++m) {
    f[m][0] = load_r(m, 0);
    f[m][1] = load_r(m, 1);
  }

  // ---- rows to LDS: piece u & 31 (eight features) of row u >> 5 ----
  const int rows = a.items.tokens * a.num_heads;
  u32x4 piece[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int u = (int)threadIdx.x + 512 * i, r = u >> 5;
    const uint16_t* src;
    if (kind == 0) {
      const int rr = min(blk * 32 + r, rows - 1), ct = rr / a.num_heads, h = rr - ct * a.num_heads;
      int it = 0;
      while (it + 1 < a.items.n && a.items.it[it + 1].ctok0 <= ct) ++it;
      src = a.q + (int64_t)(a.items.it[it].tok0 + (ct - a.items.it[it].ctok0)) * a.q_stride + (int64_t)h * kHeadDim;
    } else {
      const int tile = blk / a.num_kv_heads, head = blk - tile * a.num_kv_heads;
      int n = 0;
      while (n + 1 < a.items.n && a.items.it[n + 1].tile0 <= tile) ++n;
      const OperandItem it = a.items.it[n];
      const int j = min((tile - it.tile0) * kKeyBlk + r, it.n_new - 1);
      src = (kind == 2 ? a.v : a.k) + (int64_t)(it.tok0 + j) * a.kv_stride + (int64_t)head * kHeadDim;
    }
    piece[i] = reinterpret_cast<const u32x4*>(src)[u & 31];
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int u = (int)threadIdx.x + 512 * i, r = u >> 5, m = u & 15;
    *reinterpret_cast<u32x4*>(&xs[m][(r ^ m) + 32 * ((u >> 4) & 1)][0]) = piece[i];
  }
  __syncthreads();

  floatx16 acc = floatx16{};
  auto product = [&](auto swap_tag) {
    constexpr bool kSwap = decltype(swap_tag)::value;
#pragma unroll
    for (int m = 0; m < kSteps; ++m) {
      const bf16x8 rh = f[m % kOpAhead][0], rl = f[m % kOpAhead][1];
      if (m + kOpAhead < kSteps) {
        f[m % kOpAhead][0] = load_r(m + kOpAhead, 0);
        f[m % kOpAhead][1] = load_r(m + kOpAhead, 1);
      }
      const bf16x8 x = *reinterpret_cast<const bf16x8*>(&xs[m][((lane & 31) ^ m) + (lane & 32)][0]);
      acc = kSwap ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, rh, acc, 0, 0, 0)
                  : __builtin_amdgcn_mfma_f32_32x32x16_bf16(rh, x, acc, 0, 0, 0);
      acc = kSwap ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, rl, acc, 0, 0, 0)
                  : __builtin_amdgcn_mfma_f32_32x32x16_bf16(rl, x, acc, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);      // (keeps the scheduler from hoisting every step's reads)
    }
  };
  if (kind == 2) {
    product(std::true_type{});
    const int r = lane & 31;
    const int ft = 128 * ((r >> 2) & 1) + 16 * wave + 4 * (r >> 3) + (r & 3);   // the operand's feature of this lane
    half8* dst = reinterpret_cast<half8*>(a.o.vimg + (int64_t)blk * kKeyTileHalfs);
#pragma unroll
    for (int mm = 0; mm < 2; ++mm) {
      half8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = (_Float16)acc[8 * mm + e];
      dst[ft * (kKeyBlk / 8) + v_chunk(2 * mm + half, ft)] = o;
    }
    return;
  }
  product(std::false_type{});
  const int row = blk * 32 + (lane & 31);
  half8* dst = kind == 0 ? reinterpret_cast<half8*>(a.o.q16 + (int64_t)row * kHeadDim)
                         : reinterpret_cast<half8*>(a.o.kimg + (int64_t)blk * kKeyTileHalfs) +
                               (lane & 31) * (kHeadDim / 8);
  float sum = 0.f;
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    half8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      o[e] = (_Float16)acc[k_feature(8 * g + e)];
      sum += (float)o[e];
    }
    const int c = 2 * (8 * half + wave) + g;
    if (kind == 1 || row < rows) dst[kind == 0 ? c : k_chunk(c, lane & 31)] = o;
  }
  if (kind == 1) return;
  sum += shfl_xor_f32(sum, 32);
  if (half == 0) qs[wave][lane] = sum;
  __syncthreads();
  if ((int)threadIdx.x < 32) {
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < 8; ++w) total += qs[w][threadIdx.x];
    if (row < rows) a.o.qsum[row] = total;
  }
}

__global__ __launch_bounds__(512, 4) void rotate_operands_kernel(RotateOperandArgs a) {
  __shared__ OperandLds S;
  rotate_operands(a, S, blockIdx.x);
}

// A step's bulk write and its prefill operands in one launch: neither reads
// what the other writes, and neither fills the GPU up to some thousands of
// tokens (3001: 11 + 15 us one after the other, 18.5 together; 1052 of a mixed
// step 15 + 8 and 16.4; 9256 20 + 38 and 50).  Both halves run with the
// operands' 106 registers, two workgroups a CU.
__global__ __launch_bounds__(512, 4) void write_operands_kernel(FusedWriteArgs w, RotateOperandArgs a) {
  __shared__ union Lds {
    FusedWriteLds w;
    OperandLds o;
    __device__ Lds() {}
  } S;
  const int writes = w.token_blocks * 2 * w.num_kv_heads;
  if ((int)blockIdx.x < writes)
    fused_write(w, S.w, blockIdx.x);
  else
    rotate_operands(a, S.o, (int)blockIdx.x - writes);
}

// One thread per operand element (2 x 16 x 8 x 64 x 8 = 131072 entries), then
// one per element of the fp32 copy of R that follows them (65536 entries).
__global__ void rotation_operand_kernel(const float* __restrict__ R, __bf16* __restrict__ out) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= kMfmaEntries) {
    if (idx < kMfmaEntries + kHeadDim * kHeadDim)
      reinterpret_cast<float*>(out + kMfmaEntries)[idx - kMfmaEntries] = R[idx - kMfmaEntries];
    return;
  }
  const int u = idx & 7;
  const int lane = (idx >> 3) & 63;
  const int t = (idx >> 9) & 7;
  const int p = (idx >> 12) & 1;
  const int m = idx >> 13;
  const int r = lane & 31;
  const int e = 128 * (lane >> 5) + 8 * m + u;
  const int f = 128 * ((r >> 2) & 1) + 16 * t + 4 * (r >> 3) + (r & 3);
  const float x = R[e * kHeadDim + f];
  const __bf16 hi = (__bf16)x;
  out[idx] = p == 0 ? hi : (__bf16)(x - (float)hi);
}

int check_cache_args(CacheArgs& c) {
  if (c.block_size <= 0 || c.num_slots <= 0 || c.k_cache == nullptr || c.v_cache == nullptr)
    return kErrInvalidArgument;
  if (c.num_slots >= ((int64_t)1 << 31)) return kErrUnsupportedGeometry;
  if (c.k_head < kKCodeOff + kCodeBytes || c.v_head < kCodeBytes) return kErrUnsupportedGeometry;
  const int64_t strides[6] = {c.k_page, c.k_tok, c.k_head, c.v_page, c.v_tok, c.v_head};
  for (int64_t s : strides)
    if (s <= 0 || (s & 15) != 0) return kErrUnsupportedGeometry;
  c.bs_div = make_fast_div((uint32_t)c.block_size);
  if ((reinterpret_cast<uintptr_t>(c.k_cache) & 15) || (reinterpret_cast<uintptr_t>(c.v_cache) & 15))
    return kErrUnsupportedGeometry;
  return kOk;
}

// Whether a write of that many 128-token workgroups takes the ring kernel, whose
// rounds of kRingRound cost the same however full the last one is: where that
// one is 13/16 (the first round) or 15/16 full (the second), and from 2 11/16
// rounds on, where a partial last one no longer decides.  us, ring against tile
// kernel, by rounds (one kv head): 0.5 23.9 / 23.0, 0.75 32.7 / 31.2, 0.81 32.0 /
// 33.1, 0.875 32.5 / 34.4, 0.94 33.3 / 38.2, 0.98 34.0 / 38.4, 1.02 53.6 / 40.9,
// 1.5 65.9 / 55.5, 1.75 67.4 / 60.7, 1.875 68.0 / 65.2, 1.92 68.7 / 68.0, 2.03 74.5
// / 72.5, 2.5 84.9 / 83.3, 2.75 87.8 / 91.5, 2.94 88.0 / 96.8, 3.06 95.1 / 102.3,
// 3.5 112.6 / 117.3, 5.5 169 / 180, 8 236 / 260; two heads 0.94 33.7 / 37.8, 1.875
// 64.4 / 65.4, 2.75 88.4 / 90.8; four 0.94 33.5 / 38.5, 1.875 67.3 / 64.6, 2.75 90.4
// / 90.4.  A write that can share its launch with a step's prefill operands
// (shares) does so up to those 2 11/16 rounds: a whole step of four kv heads
// without a window 240 us with the ring kernel and 227 with the shared launch at
// 0.82 rounds, 297 / 287 at 1, 815 / 810 at 2, 1427 / 1443 at 2.8; of one kv head
// 610 / 599 at 0.92.
bool prefers_ring(int64_t workgroups, bool shares) {
  const int64_t sixteenth = kRingRound / 16;
  if (workgroups >= 43 * sixteenth) return true;
  return !shares && ((workgroups >= 13 * sixteenth && workgroups <= kRingRound) ||
                     (workgroups > 31 * sixteenth && workgroups <= 2 * kRingRound));
}

std::atomic<uint64_t> g_ring_lds_set{0};   // dynamic-LDS attribute set, one bit per device
std::atomic<uint64_t> g_rot_lds_set[4] = {{0}, {0}, {0}, {0}};   // the same for the rotate_rows instances

}  // namespace

int launch_rotate_operands(const uint16_t* q, int64_t q_stride, const uint16_t* k, const uint16_t* v,
                           int64_t kv_stride, int32_t num_heads, int32_t num_kv_heads, const uint8_t* rot_k,
                           const uint8_t* rot_v, const OperandItems& items, const PrefillOperands& o,
                           const FusedWriteArgs* write, hipStream_t stream) {
  RotateOperandArgs a{q, k, v, q_stride, kv_stride, num_heads, num_kv_heads, rot_k, rot_v, o, 0, 0, items};
  const int64_t rows = (int64_t)items.tokens * num_heads, units = (int64_t)items.tiles * num_kv_heads;
  a.q_blocks = (int32_t)((rows + 31) / 32);
  a.kv_blocks = (int32_t)units;
  const unsigned blocks = (unsigned)(a.q_blocks + 2 * a.kv_blocks);
  if (write != nullptr)
    hipLaunchKernelGGL(write_operands_kernel, dim3(blocks + (unsigned)(write->token_blocks * 2 * write->num_kv_heads)),
                       dim3(512), 0, stream, *write, a);
  else
    hipLaunchKernelGGL(rotate_operands_kernel, dim3(blocks), dim3(512), 0, stream, a);
  return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}

}  // namespace oscar

using namespace oscar;

extern "C" {

size_t oscar_rotation_operand_bytes(int32_t head_size) {
  return head_size == kHeadDim ? kOperandBytes : 0;
}

int oscar_rotation_operand(const float* rotation, void* operand, int32_t head_size,
                           hipStream_t stream) {
  if (head_size != kHeadDim) return kErrUnsupportedHeadDim;
  if (rotation == nullptr || operand == nullptr) return kErrInvalidArgument;
  const int total = kMfmaEntries + kHeadDim * kHeadDim;
  hipLaunchKernelGGL(rotation_operand_kernel, dim3((total + 255) / 256), dim3(256), 0, stream,
                     rotation, static_cast<__bf16*>(operand));
  return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}

int oscar_rotate_rows(const void* in, int32_t in_f32, int64_t in_row_stride, int64_t rows, int32_t head_size,
                      const void* rot_operand, void* out, int32_t out_bf16, int64_t out_row_stride,
                      hipStream_t stream) {
  if (head_size != kHeadDim) return kErrUnsupportedHeadDim;
  if (rows < 0 || (in_f32 != 0 && in_f32 != 1) || (out_bf16 != 0 && out_bf16 != 1)) return kErrInvalidArgument;
  if (rows == 0) return kOk;
  if (!in || !rot_operand || !out || in_row_stride < kHeadDim || out_row_stride < kHeadDim)
    return kErrInvalidArgument;
  // 16-byte vector accesses: every row start 16-byte aligned
  const int64_t in_bytes = in_f32 ? 4 : 2, out_bytes = out_bf16 ? 2 : 4;
  if (((in_row_stride * in_bytes) & 15) || ((out_row_stride * out_bytes) & 15) ||
      (reinterpret_cast<uintptr_t>(in) & 15) || (reinterpret_cast<uintptr_t>(out) & 15) ||
      (reinterpret_cast<uintptr_t>(rot_operand) & 15))
    return kErrInvalidArgument;
  const int64_t per_block = kFusedWaves * kTokPerWave;
  const dim3 grid((unsigned)((rows + per_block - 1) / per_block));
  const uint8_t* rop = static_cast<const uint8_t*>(rot_operand);
  const void* k[4] = {reinterpret_cast<const void*>(rotate_rows_kernel<false, false>),
                      reinterpret_cast<const void*>(rotate_rows_kernel<false, true>),
                      reinterpret_cast<const void*>(rotate_rows_kernel<true, false>),
                      reinterpret_cast<const void*>(rotate_rows_kernel<true, true>)};
  const int which = 2 * in_f32 + out_bf16;
  constexpr int kRotLds = kRing * kChunkBytes;
  if (set_dynamic_lds(k[which], kRotLds, g_rot_lds_set[which]) != kOk) return kErrLaunch;
  if (in_f32 && out_bf16)
    hipLaunchKernelGGL((rotate_rows_kernel<true, true>), grid, dim3(256), kRotLds, stream, in, in_row_stride, rows,
                       rop, out, out_row_stride);
  else if (in_f32)
    hipLaunchKernelGGL((rotate_rows_kernel<true, false>), grid, dim3(256), kRotLds, stream, in, in_row_stride, rows,
                       rop, out, out_row_stride);
  else if (out_bf16)
    hipLaunchKernelGGL((rotate_rows_kernel<false, true>), grid, dim3(256), kRotLds, stream, in, in_row_stride, rows,
                       rop, out, out_row_stride);
  else
    hipLaunchKernelGGL((rotate_rows_kernel<false, false>), grid, dim3(256), kRotLds, stream, in, in_row_stride, rows,
                       rop, out, out_row_stride);
  return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}

int oscar_quant_write_prerotated(const float* k_rot, const float* v_rot, int64_t num_tokens,
                                 int32_t num_kv_heads, int32_t head_size, int64_t token_stride,
                                 const int64_t* slot_mapping, void* k_cache, void* v_cache,
                                 int32_t block_size, int64_t num_pages, int64_t k_stride_page,
                                 int64_t k_stride_token, int64_t k_stride_head, int64_t v_stride_page,
                                 int64_t v_stride_token, int64_t v_stride_head,
                                 int32_t clip_index_k, int32_t clip_index_v, hipStream_t stream) {
  if (head_size != kHeadDim) return kErrUnsupportedHeadDim;
  if (num_tokens < 0 || num_kv_heads <= 0 || clip_index_k >= kHeadDim || clip_index_v >= kHeadDim)
    return kErrInvalidArgument;
  if (num_tokens == 0) return kOk;
  if (k_rot == nullptr || v_rot == nullptr || slot_mapping == nullptr) return kErrInvalidArgument;
  if (token_stride < (int64_t)num_kv_heads * kHeadDim || (token_stride & 3) ||
      (reinterpret_cast<uintptr_t>(k_rot) & 15) || (reinterpret_cast<uintptr_t>(v_rot) & 15))
    return kErrInvalidArgument;
  CacheArgs c{static_cast<uint8_t*>(k_cache), static_cast<uint8_t*>(v_cache), k_stride_page,
              k_stride_token, k_stride_head, v_stride_page, v_stride_token, v_stride_head,
              block_size, num_pages * (int64_t)block_size, FastDiv{}};
  int st = check_cache_args(c);
  if (st != kOk) return st;
  dim3 grid((unsigned)((num_tokens + 127) / 128), (unsigned)(num_kv_heads * 2));
  hipLaunchKernelGGL(quant_write_prerotated_kernel, grid, dim3(256), 0, stream, k_rot, v_rot,
                     num_tokens, token_stride, slot_mapping, c, (int)clip_index_k,
                     (int)clip_index_v);
  return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}

}  // extern "C"

namespace {

// A request layout in host arrays; its device copy is the window arguments'.
struct StepLayout {
  const int32_t* query_start;
  const int32_t* seq_lens;
};

// oscar_quant_write with an optional window arena (w.rows > 0), whose request
// layout is in w's device arrays, or to be stored there from host's.  With
// `later`, a write that takes the tile kernel is left there for the caller to
// launch (waits: it was), its winner pass done.
int quant_write_impl(const void* key_bf16, const void* value_bf16, int64_t num_tokens, int32_t num_kv_heads,
                     int32_t head_size, int64_t token_stride, const void* rot_k_operand, const void* rot_v_operand,
                     const int64_t* slot_mapping, void* k_cache, void* v_cache, int32_t block_size,
                     int64_t num_pages, int64_t k_stride_page, int64_t k_stride_token, int64_t k_stride_head,
                     int64_t v_stride_page, int64_t v_stride_token, int64_t v_stride_head, int32_t clip_index_k,
                     int32_t clip_index_v, const WindowArgs& w, const StepLayout* host, FusedWriteArgs* later,
                     bool* waits, hipStream_t stream) {
  if (head_size != kHeadDim) return kErrUnsupportedHeadDim;
  if (num_tokens < 0 || num_kv_heads <= 0 || clip_index_k >= kHeadDim || clip_index_v >= kHeadDim)
    return kErrInvalidArgument;
  if (num_tokens == 0) return kOk;
  if (key_bf16 == nullptr || value_bf16 == nullptr || slot_mapping == nullptr ||
      rot_k_operand == nullptr || rot_v_operand == nullptr)
    return kErrInvalidArgument;
  if (token_stride < (int64_t)num_kv_heads * kHeadDim || (token_stride & 7) ||
      (reinterpret_cast<uintptr_t>(key_bf16) & 15) || (reinterpret_cast<uintptr_t>(value_bf16) & 15) ||
      (reinterpret_cast<uintptr_t>(rot_k_operand) & 15) ||
      (reinterpret_cast<uintptr_t>(rot_v_operand) & 15))
    return kErrInvalidArgument;
  CacheArgs c{static_cast<uint8_t*>(k_cache), static_cast<uint8_t*>(v_cache), k_stride_page,
              k_stride_token, k_stride_head, v_stride_page, v_stride_token, v_stride_head,
              block_size, num_pages * (int64_t)block_size, FastDiv{}};
  int st = check_cache_args(c);
  if (st != kOk) return st;
  // Short writes (at most kShortWriteVectors key + value vectors): the fp32
  // rotation of the short-step write (1024-thread workgroups of one to four
  // vectors, R read from the operand's fp32 copy).  (They took it when the
  // tile kernel was slower for few tokens, 19.4 against 6.2 us for four; it
  // stays because its rotation is the fp32 one, which the tiles' two bf16
  // parts only approach.)
  if (2 * num_tokens * num_kv_heads <= kShortWriteVectors) {
    const uint8_t* ok = static_cast<const uint8_t*>(rot_k_operand) + kMfmaOperandBytes;
    const uint8_t* ov = static_cast<const uint8_t*>(rot_v_operand) + kMfmaOperandBytes;
    const bool win = w.rows > 0;
    return step_write(host == nullptr, nullptr, 0, key_bf16, value_bf16, token_stride, (int32_t)num_tokens, 0, num_kv_heads,
                      head_size, reinterpret_cast<const float*>(ok), reinterpret_cast<const float*>(ov),
                      slot_mapping, win ? (host ? host->query_start : w.query_start) : nullptr,
                      win ? (host ? host->seq_lens : w.seq_lens) : nullptr,
                      win ? w.num_requests : 0, k_cache, v_cache, block_size, num_pages, k_stride_page,
                      k_stride_token, k_stride_head, v_stride_page, v_stride_token, v_stride_head,
                      clip_index_k, clip_index_v, w.stage_k, w.stage_v, w.owner, w.kimg, w.vimg, w.rows,
                      w.sink_eff, w.recent, nullptr, nullptr, nullptr, stream);
  }
  if (w.rows > 0) {
    HostLayout h{};
    if (host != nullptr) {
      // query_start, then seq_lens, in one array; the last part goes with the
      // winner pass, the others in launches of their own
      const int64_t starts = (int64_t)w.num_requests + 1, ints = starts + w.num_requests;
      for (int64_t i0 = 0; i0 < ints; i0 += kLayoutInts) {
        h.dst = const_cast<int32_t*>(w.query_start) + i0;
        h.n = (int32_t)(ints - i0 < kLayoutInts ? ints - i0 : kLayoutInts);
        for (int32_t i = 0; i < h.n; ++i)
          h.v[i] = i0 + i < starts ? host->query_start[i0 + i] : host->seq_lens[i0 + i - starts];
        if (i0 + h.n < ints) {
          hipLaunchKernelGGL(store_layout_kernel, dim3(1), dim3(256), 0, stream, h);
          if (hipGetLastError() != hipSuccess) return kErrLaunch;
        }
      }
    }
    hipLaunchKernelGGL(quant_window_winner_kernel, dim3((unsigned)((num_tokens + 255) / 256)), dim3(256), 0, stream,
                       slot_mapping, (int32_t)num_tokens, w.winner, block_size, w.rows, h);
    if (hipGetLastError() != hipSuccess) return kErrLaunch;
  }
  const FusedWriteArgs fw{static_cast<const uint16_t*>(key_bf16), static_cast<const uint16_t*>(value_bf16), num_tokens,
                          token_stride, static_cast<const uint8_t*>(rot_k_operand),
                          static_cast<const uint8_t*>(rot_v_operand), slot_mapping, c, clip_index_k, clip_index_v, w,
                          (int32_t)((num_tokens + kFwTokens - 1) / kFwTokens), num_kv_heads};
  const int64_t ring_blocks = (num_tokens + kFusedWaves * kTokPerWave - 1) / (kFusedWaves * kTokPerWave);
  const int64_t ring_wgs = ring_blocks * 2 * num_kv_heads;
  if (w.rows == 0 && prefers_ring(ring_wgs, later != nullptr)) {
    FusedWriteArgs rw = fw;
    rw.token_blocks = (int32_t)ring_blocks;
    if (ring_wgs > INT32_MAX) return kErrInvalidArgument;
    if (set_dynamic_lds(reinterpret_cast<const void*>(quant_write_ring_kernel), (int)kRingLds, g_ring_lds_set) != kOk)
      return kErrLaunch;
    hipLaunchKernelGGL(quant_write_ring_kernel, dim3((unsigned)ring_wgs), dim3(kFusedWaves * 64), kRingLds, stream,
                       rw);
    return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
  }
  if (later != nullptr) {
    *later = fw;
    *waits = true;
    return kOk;
  }
  const int64_t blocks = (int64_t)fw.token_blocks * 2 * num_kv_heads;
  if (blocks > INT32_MAX) return kErrInvalidArgument;
  hipLaunchKernelGGL(quant_write_fused_kernel, dim3((unsigned)blocks), dim3(kFwThreads), 0, stream, fw);
  return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}

}  // namespace

extern "C" {

int oscar_quant_write(const void* key_bf16, const void* value_bf16, int64_t num_tokens,
                      int32_t num_kv_heads, int32_t head_size, int64_t token_stride,
                      const void* rot_k_operand, const void* rot_v_operand,
                      const int64_t* slot_mapping, void* k_cache, void* v_cache,
                      int32_t block_size, int64_t num_pages, int64_t k_stride_page,
                      int64_t k_stride_token, int64_t k_stride_head, int64_t v_stride_page,
                      int64_t v_stride_token, int64_t v_stride_head, int32_t clip_index_k,
                      int32_t clip_index_v, hipStream_t stream) {
  return quant_write_impl(key_bf16, value_bf16, num_tokens, num_kv_heads, head_size, token_stride, rot_k_operand,
                          rot_v_operand, slot_mapping, k_cache, v_cache, block_size, num_pages, k_stride_page,
                          k_stride_token, k_stride_head, v_stride_page, v_stride_token, v_stride_head,
                          clip_index_k, clip_index_v, WindowArgs{}, nullptr, nullptr, nullptr, stream);
}

int oscar_quant_write_window(const void* key_bf16, const void* value_bf16, int64_t num_tokens,
                             int32_t num_kv_heads, int32_t head_size, int64_t token_stride,
                             const void* rot_k_operand, const void* rot_v_operand,
                             const int64_t* slot_mapping, void* k_cache, void* v_cache,
                             int32_t block_size, int64_t num_pages, int64_t k_stride_page,
                             int64_t k_stride_token, int64_t k_stride_head, int64_t v_stride_page,
                             int64_t v_stride_token, int64_t v_stride_head, int32_t clip_index_k,
                             int32_t clip_index_v, const int32_t* query_start_loc, const int32_t* seq_lens,
                             int32_t num_requests, int32_t stage_rows, int32_t sink_eff, int32_t recent,
                             float* stage_k, float* stage_v, int64_t* stage_owner, int64_t* seat_winner,
                             void* stage_k_image, void* stage_v_image, hipStream_t stream) {
  if (num_requests < 0 || stage_rows <= 0 || sink_eff < 0 || recent < 0 || num_tokens > INT32_MAX)
    return kErrInvalidArgument;
  if (num_tokens > 0 && num_requests == 0) return kErrInvalidArgument;
  if (!query_start_loc || !seq_lens || !stage_k || !stage_v || !stage_owner || !seat_winner)
    return kErrInvalidArgument;
  if ((stage_k_image == nullptr) != (stage_v_image == nullptr)) return kErrInvalidArgument;
  if (stage_k_image != nullptr && block_size % 32 != 0) return kErrUnsupportedGeometry;
  if ((reinterpret_cast<uintptr_t>(stage_k) & 15) || (reinterpret_cast<uintptr_t>(stage_v) & 15) ||
      (reinterpret_cast<uintptr_t>(stage_k_image) & 15) || (reinterpret_cast<uintptr_t>(stage_v_image) & 15))
    return kErrInvalidArgument;
  WindowArgs w{query_start_loc, seq_lens, num_requests, stage_rows, sink_eff, recent, num_kv_heads, stage_k, stage_v,
               stage_owner, seat_winner, static_cast<_Float16*>(stage_k_image),
               static_cast<_Float16*>(stage_v_image)};
  return quant_write_impl(key_bf16, value_bf16, num_tokens, num_kv_heads, head_size, token_stride, rot_k_operand,
                          rot_v_operand, slot_mapping, k_cache, v_cache, block_size, num_pages, k_stride_page,
                          k_stride_token, k_stride_head, v_stride_page, v_stride_token, v_stride_head,
                          clip_index_k, clip_index_v, w, nullptr, nullptr, nullptr, stream);
}

}  // extern "C"

namespace oscar {

int quant_write_step(const oscar_mtp_layer& L, const void* rot_k_operand, const void* rot_v_operand,
                     int64_t* seat_winner, const void* key_bf16, const void* value_bf16, int64_t kv_token_stride,
                     int32_t num_tokens, const int64_t* slot_mapping, const int32_t* query_start_loc,
                     const int32_t* seq_lens, int32_t num_requests, int32_t* layout, FusedWriteArgs* later, bool* waits,
                     hipStream_t stream) {
  WindowArgs w{};
  const StepLayout host{query_start_loc, seq_lens};
  if (L.stage_rows > 0)
    w = WindowArgs{layout, layout + num_requests + 1, num_requests, L.stage_rows, L.sink_eff, L.recent,
                   L.num_kv_heads, L.stage_k, L.stage_v, L.stage_owner, seat_winner,
                   static_cast<_Float16*>(L.stage_k_image), static_cast<_Float16*>(L.stage_v_image)};
  return quant_write_impl(key_bf16, value_bf16, num_tokens, L.num_kv_heads, L.head_size, kv_token_stride,
                          rot_k_operand, rot_v_operand, slot_mapping, L.k_cache, L.v_cache, L.block_size, L.num_pages,
                          L.k_stride_page, L.k_stride_token, L.k_stride_head, L.v_stride_page, L.v_stride_token,
                          L.v_stride_head, L.clip_index_k, L.clip_index_v, w, &host, later, waits, stream);
}

}  // namespace oscar
