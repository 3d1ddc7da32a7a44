// MFMA attention building blocks shared by the masked prefill attention and
// the grouped-query decode attention: 32x32x16 MFMAs, packing of
// probabilities, row sums with v_dot2, and the LDS layouts of K and V tiles
// (swizzles and the transpose-read addressing of V^T operands).
#pragma once
#include "common.hpp"

namespace sfl {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// Two values rounded to T and packed (v_cvt_pk_bf16_f32 / v_cvt_pk_f16_f32).
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
template <typename T> __device__ __forceinline__ uint32_t pack2(float lo, float hi);
template <> __device__ __forceinline__ uint32_t pack2<bf16_t>(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{lo, hi}), bf16x2_t));
}
template <> __device__ __forceinline__ uint32_t pack2<f16_t>(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{lo, hi}), f16x2_t));
}

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2_v __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_v __attribute__((ext_vector_type(2)));

template <typename T>
__device__ __forceinline__ f32x16 mfma32(const u32x4& a, const u32x4& b, f32x16 c);
template <>
__device__ __forceinline__ f32x16 mfma32<bf16_t>(const u32x4& a, const u32x4& b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x16 mfma32<f16_t>(const u32x4& a, const u32x4& b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// acc + lo + hi of a packed pair (v_dot2 with (1, 1)).
template <typename T> __device__ __forceinline__ float add_pair(uint32_t pk, float acc);
template <> __device__ __forceinline__ float add_pair<bf16_t>(uint32_t pk, float acc) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_v, pk), __builtin_bit_cast(bf16x2_v, 0x3f803f80u),
                                         acc, false);
}
template <> __device__ __forceinline__ float add_pair<f16_t>(uint32_t pk, float acc) {
  return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2_v, pk), __builtin_bit_cast(f16x2_v, 0x3c003c00u), acc, false);
}

// V tile layout: row-major [key][8 slots of 16 bytes]; logical slot sg (dims
// 8sg .. 8sg+7) of key row r sits at physical slot 2((sg >> 1) ^ (r & 3)) +
// (sg & 1), so the 4 rows one 16-lane transpose read touches use 4 different
// 32-byte bank groups.
__device__ __forceinline__ unsigned vt_slot(unsigned sg, unsigned r) { return 2u * ((sg >> 1) ^ (r & 3u)) + (sg & 1u); }
// Byte offset, within a tile, of lane l's 8-byte piece for key step 0, dim
// tile t, first key half: key row 4(g >> 1) + (m >> 2), dims 32t + 16(g & 1) +
// 4(m & 3) .. +3, with g = l / 16 and m = l % 16.
template <int D>
__device__ __forceinline__ unsigned vt_lane_offset(int lane, int t) {
  const unsigned g = unsigned(lane) / 16u, m = unsigned(lane) % 16u;
  const unsigned r = 4u * (g >> 1) + (m >> 2);
  const unsigned dim = 32u * unsigned(t) + 16u * (g & 1u) + 4u * (m & 3u);
  return r * (2u * D) + 16u * vt_slot(dim / 8u, r) + 2u * (dim % 8u);
}

// K tile swizzle: row r's logical 16-byte slot s sits at s ^ k_swizzle<D>(r).
// The operand reads take one logical slot of 16 consecutive rows per LDS
// cycle; rows of 128 bytes (D = 64) alternate bank halves, so (r >> 1) & 7
// separates the rest, and rows of 256 bytes (D = 128) all start at bank 0, so
// the slot itself is rotated by r & 15.
template <int D>
__device__ __forceinline__ int k_swizzle(int r) {
  return D == 64 ? (r >> 1) & 7 : r & 15;
}

typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4_t lds_i16x4_t;

constexpr float kLazyMax = 8.f;

// Workgroup -> (query tile, batch * head) of a 1-D grid, XCD-aware. Workgroups
// are dealt to the 8 XCDs round-robin and each XCD has its own 4 MB L2, so XCD
// x takes a contiguous range of the head-major tile order: the ~100
// workgroups an XCD runs at once then share the K/V of 2-3 heads (0.8 MB per
// head at 3072 x 64 bf16) instead of every XCD streaming every head's K/V.
// Query tiles run last-first, so the longest causal rows start first. When
// the XCD's range is two or more whole heads, it is dealt query-tile major
// across groups of up to kTileOrderHeads heads: the tail of each group (and
// of the range) is then the short rows of several heads, not one head's
// short rows after other heads' long ones, while the heads an XCD runs at
// once stay few enough to share their K/V in its L2 (measured: causal
// 16x16x3072 417 -> 392 us, config 5 125 -> 119 us; 4 or 6 heads per
// group gained less, 12-16 the same, all 32 at once lost the gain).
constexpr int kXcds = 8;
constexpr int kTileOrderHeads = 8;
constexpr int kXcdCus = 32;
__device__ __forceinline__ int2 attn_tile(int nqt, int nbh) {
  const int total = nqt * nbh;
  const int blk = int(blockIdx.x);
  const int x = blk % kXcds;
  int idx = blk / kXcds;
  const int base = total / kXcds, extra = total % kXcds;
  const int start = x * base + min(x, extra);
  const int len = base + (x < extra);
  // A grid of up to 4 workgroups per CU is all on the chip at once, so nothing
  // evens the CUs out later: every other round of the XCD's CUs is dealt
  // backwards, so that with the rows in descending length a CU gets a long row
  // with a short one (causal 16x16x256 at head dim 32 16.6 -> 14.7 us, 8x12x1024
  // at head dim 64 1-2% of its 34; larger grids do not gain).
  const int round0 = idx & ~(kXcdCus - 1);
  if (len <= 4 * kXcdCus && (idx & kXcdCus)) idx = round0 + min(kXcdCus, len - round0) - 1 - (idx - round0);
  if (len >= 2 * nqt && start % nqt == 0 && len % nqt == 0) {
    constexpr int G = kTileOrderHeads;
    const int heads = len / nqt;
    const int grp = idx / (G * nqt), g = min(G, heads - grp * G), r = idx - grp * G * nqt;
    return make_int2(nqt - 1 - r / g, start / nqt + grp * G + r % g);
  }
  const int t = start + idx;
  return make_int2(nqt - 1 - t % nqt, t / nqt);
}

}  // namespace sfl
