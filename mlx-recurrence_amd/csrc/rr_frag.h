// rr_frag.h — LDS row images and operand fragments of the kernels that chain MFMA
// products through accumulators (walk_bwd.hip, gdn_chunk.hip): a 32-row
// operand held as two 16-row accumulator blocks gives lane (l15, g) = (lane % 16,
// lane / 16) the rows pi(g, e) = 4 g + e (e < 4), 16 + 4 g + e - 4 (e >= 4), so every
// other operand of such a product is read with its k index in that order.
#pragma once

#include "rr_mfma.h"

namespace rr {

// Workgroup barrier ordering LDS only: loads and stores to memory stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// LDS row images of LEN columns: each 32 columns as eight 4-element pieces, piece
// p at 16-byte unit p % 4, half p / 4 (so a unit is k = pi(g, e) for g = unit),
// units permuted by row so that both the 16-byte row fragments and the
// transposing reads of 16 lanes hit distinct banks.
template <int LEN>
__device__ __forceinline__ int swz(int row) {
  return LEN == 128 ? ((row & 3) << 2) | ((row >> 2) & 3) : (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
}
template <int LEN>
__device__ __forceinline__ int piece(int row, int p) {   // element offset of columns 4 p .. 4 p + 3
  const int q = p & 7;
  return row * LEN + 8 * ((4 * (p >> 3) + (q & 3)) ^ swz<LEN>(row)) + 4 * (q >> 2);
}
template <int LEN>
__device__ __forceinline__ u16x8_t row_frag(const uint16_t* x, int row, int kk, int g) {   // X[row][32 kk + pi]
  return frag(x + row * LEN + 8 * ((4 * kk + g) ^ swz<LEN>(row)));
}
template <int LEN>
__device__ __forceinline__ u16x8_t col_frag(const uint16_t* x, int blk, int l15, int g) {   // X[pi][16 blk + l15]
  const int r0 = 4 * g + (l15 >> 2);
  const uint16_t* a = x + r0 * LEN + 8 * ((4 * (blk >> 1) + (l15 & 3)) ^ swz<LEN>(r0)) + 4 * (blk & 1);
  const u16x4_t lo = tr_read4(a), hi = tr_read4(a + 16 * LEN);
  return u16x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}
// Accumulator blocks of rows 0-15 and 16-31 -> hi and lo operand (k = pi).
__device__ __forceinline__ void split_pair(const f32x4_t& a, const f32x4_t& b, u16x8_t& hi, u16x8_t& lo) {
  const float x[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  bf_split8(x, hi, lo);
}
__device__ __forceinline__ u16x8_t join(uint2 lo, uint2 hi) {
  return __builtin_bit_cast(u16x8_t, make_uint4(lo.x, lo.y, hi.x, hi.y));
}
__device__ __forceinline__ float bf4(const uint2& v, int r) {   // element r of four packed bf16
  const uint32_t x = r < 2 ? v.x : v.y;
  return __uint_as_float(r & 1 ? x & 0xffff0000u : x << 16);
}
__device__ __forceinline__ uint2 pack4(const float (&v)[4]) {
  return make_uint2(bf_pack2(v[0], v[1]), bf_pack2(v[2], v[3]));
}

}  // namespace rr
