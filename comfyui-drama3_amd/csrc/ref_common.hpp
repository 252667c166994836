// What the kernels of the reference's own formats share: the 4-bit codes' tables, the int8 planes' ratio and sum, SiLU(gate)
// * up, and the row of the planes that a prompt's pair reads.
#pragma once
#include "common.hpp"

namespace d3 {

// W4 through tables: a 16-column group's codes all share one e4m3 scale byte, so the int8-grid values of the 16 codes at
// each of the 256 scale bytes make a 4 KB table (decode_group's own arithmetic, entry by entry), kept in LDS as bytes
// q + 128. A group then costs one 16-byte table read, and four of its codes become four bytes through two byte
// permutes and a byte mask, instead of a codebook read, a product, a rounding and a clamp per value.
constexpr int QTAB_WORDS = 256 * 4;  // qtab[4 sb + i]: bytes q + 128 of codes 4i .. 4i + 3 at scale byte sb
// cb: codebook[4 (threadIdx.x & 3) .. + 3], loaded by the caller (ahead of its weight rows); SIGNED: the bytes hold q
// itself (two's complement) instead of q + 128
template <bool SIGNED = false> D3_INLINE void build_qtab(uint32_t* qtab, f32x4 cb) {
  const float c[4] = {cb.x, cb.y, cb.z, cb.w};
  for (int i = threadIdx.x; i < QTAB_WORDS; i += blockDim.x) {  // i & 3 == threadIdx.x & 3: blockDim.x % 4 == 0
    const float sc = fp8x2_to_f32<false>((uint32_t)(i >> 2)).x;
    uint32_t word = 0u;
#pragma unroll
    for (int b = 0; b < 4; b++) {
      const float q = fminf(fmaxf(rintf(c[b] * sc), -127.0f), 127.0f);
      word |= ((uint32_t)((int)q + (SIGNED ? 0 : 128)) & 0xFFu) << (8 * b);
    }
    qtab[i] = word;
  }
}

// the table bytes (t: entries 0..15, 4 per word) at the four indices held in the low nibbles of sel's bytes
D3_INLINE uint32_t lookup16(i32x4 t, uint32_t sel) {
  const uint32_t s3 = sel & 0x07070707u;
  const uint32_t lo = __builtin_amdgcn_perm((uint32_t)t.y, (uint32_t)t.x, s3);  // entries 0..7
  const uint32_t hi = __builtin_amdgcn_perm((uint32_t)t.w, (uint32_t)t.z, s3);  // entries 8..15
  // selector byte 12 gives 0x00, 13 gives 0xFF: a byte mask of the indices >= 8
  const uint32_t m = __builtin_amdgcn_perm(0u, 0u, ((sel >> 3) & 0x01010101u) | 0x0C0C0C0Cu);
  return (hi & m) | (lo & ~m);
}

constexpr float I8_RATIO = 254.0f;  // the int8 planes' ratio

// x / 254 correctly rounded: the remainder of the first quotient by one fused step, its quotient added by another (the
// same bits as the division for every float x down to 2^-100; the divide instruction sequence takes three times as many)
D3_INLINE float over_ratio(float x) {
  constexpr float INV = 1.0f / I8_RATIO;
  const float q = x * INV;
  return fmaf(fmaf(-I8_RATIO, q, x), INV, q);
}
// SiLU(gate) * up, the product rounded by itself: left to contraction, a kernel that goes on to add it up (a rotation)
// would take it unrounded, one that stores it rounded, and a row's result would depend on which of them runs it.
D3_INLINE float silu_up(float gate, float up) {
#pragma clang fp contract(off)
  return gate / (1.0f + __expf(-gate)) * up;
}

// The planes' exact sums of one output in float32, every step rounded once: A0 + (A1 + A2 / 254) / 254. All the int8
// products end in it, so a row's result does not depend on which of them runs it.
D3_INLINE float planes_sum(int a0, int a1, int a2) {
  return (float)a0 + over_ratio((float)a1 + over_ratio((float)a2));
}

// W4: one 16-code group's int8-grid values as bytes in column order (word d: codes 4d .. 4d + 3) through the
// group's scale-byte row t of a signed table (build_qtab<true>); lo / hi: the nibble words of codes 0-7 / 8-15
// (code j's nibble at bits 4 (j & 7))
D3_INLINE i32x4 w4_group_i8(uint32_t lo, uint32_t hi, i32x4 t) {
  const uint32_t e0 = lookup16(t, lo), o0 = lookup16(t, lo >> 4);  // codes 0, 2, 4, 6 / 1, 3, 5, 7
  const uint32_t e1 = lookup16(t, hi), o1 = lookup16(t, hi >> 4);  // codes 8, 10, 12, 14 / 9, 11, 13, 15
  return i32x4{(int)__builtin_amdgcn_perm(o0, e0, 0x05010400u), (int)__builtin_amdgcn_perm(o0, e0, 0x07030602u),
               (int)__builtin_amdgcn_perm(o1, e1, 0x05010400u), (int)__builtin_amdgcn_perm(o1, e1, 0x07030602u)};
}

// The row of the planes that row p of the passes reads: p itself, or with `order` x's row order[p] / k (the rows of
// a prompt's pairs taken from its token rows, so no gathered copy is made), kept within the planes' xrows rows. (The wide
// products request all their pairs before they use one: pair_row alone.)
D3_INLINE int pair_row(int64_t pair, int k, int xrows) { return min(max((int)pair, 0) / k, xrows - 1); }
D3_INLINE size_t plane_row(const int64_t* order, int k, int xrows, int p) {
  return order ? (size_t)pair_row(order[p], k, xrows) : (size_t)p;
}

}  // namespace d3
