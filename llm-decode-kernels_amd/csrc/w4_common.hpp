// INT4 column arithmetic shared by the W4A16 GEMV kernels (see the gemv_w4a16.hip header for the derivation of the
// magic-number dequant).
#pragma once
#include "common.hpp"

namespace dk {

constexpr uint32_t kMagic = 0x64006400u;    // fp16 pair (1024, 1024): + q at mantissa bits 0..3
constexpr uint32_t kMagicHi = 0x54005400u;  // fp16 pair (64, 64): + q at mantissa bits 4..7
constexpr uint32_t kLoMask = 0x000F000Fu;
constexpr uint32_t kHiMask = 0x00F000F0u;

// The two nibble masks, held in VGPRs (vgpr_const), so that each pair costs one v_and_or_b32 (mask in the VGPR,
// the magic constant in an SGPR); the kernels build them once, ahead of their loops.
struct NibbleMasks {
  uint32_t lo, hi;
};
__device__ __forceinline__ NibbleMasks nibble_masks() { return {vgpr_const(kLoMask), vgpr_const(kHiMask)}; }
__device__ __forceinline__ f16x2 nibble_pair(uint32_t w, uint32_t mask, uint32_t magic) {
  return as_f16x2((w & mask) | magic);
}

// Sums of the x values that meet the 1024 and the 64 offsets of one column and the constant part of the column's
// result: sum (q - z) x = (d - 1024 SA - 64 SB) - z (SA + SB), so the chain d starts at base = -(1024 SA + 64 SB),
// computed once per column and shared by every row of it, and each row then needs one FMA and the scale multiply.
struct ColumnSums {
  float base, S;
};
__device__ __forceinline__ ColumnSums column_sums(const u32x4 (&xc)[4]) {
  const f16x2 one = {(f16)1.0f, (f16)1.0f};
  float SA = 0.f, SB = 0.f;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    SA = dot2(as_f16x2(xc[k].x), one, SA);
    SA = dot2(as_f16x2(xc[k].z), one, SA);
    SB = dot2(as_f16x2(xc[k].y), one, SB);
    SB = dot2(as_f16x2(xc[k].w), one, SB);
  }
  return {fmaf(-1024.f, SA, -64.f * SB), SA + SB};
}

// sum (q - z) x of one row over one column, before the scale: the packed word's 32 weights against xc.
__device__ __forceinline__ float column_row(const u32x4& w, float z, const u32x4 (&xc)[4], ColumnSums cs,
                                            NibbleMasks m) {
  float d = cs.base;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t lo = w[k], hi = lo >> 8;
    d = dot2(nibble_pair(lo, m.lo, kMagic), as_f16x2(xc[k].x), d);
    d = dot2(nibble_pair(lo, m.hi, kMagicHi), as_f16x2(xc[k].y), d);
    d = dot2(nibble_pair(hi, m.lo, kMagic), as_f16x2(xc[k].z), d);
    d = dot2(nibble_pair(hi, m.hi, kMagicHi), as_f16x2(xc[k].w), d);
  }
  return fmaf(-z, cs.S, d);
}

// 8 weights of one packed word -> fp16((q - zero) * scale), in element order, given s2 = (scale, scale), zk = (1024 +
// zero) twice and zs = (64 + zero) twice. Pairs (e0, e1) and (e4, e5) are nibbles 0 and 2 of each 16-bit half: OR-ed
// into the mantissa of fp16 1024 (step 1) they give 1024 + q; pairs (e2, e3) and (e6, e7) are nibbles 1 and 3, and
// OR-ed in place into fp16 64 (step 1/16) they give 64 + q, so one shift (by 8) serves all four pairs. Subtracting
// 1024 + zero or 64 + zero is exact, and the product with the scale rounds the exact (q - zero) * scale once.
// mlo = vgpr_const(0x000F000F), mhi = vgpr_const(0x00F000F0): one v_and_or_b32 per pair.
__device__ __forceinline__ u32x4 dequant8_sz(uint32_t word, f16x2 s2, f16x2 zk, f16x2 zs, uint32_t mlo,
                                             uint32_t mhi) {
  const uint32_t hi = word >> 8;
  const uint32_t p0 = (word & mlo) | 0x64006400u;
  const uint32_t p1 = (word & mhi) | 0x54005400u;
  const uint32_t p2 = (hi & mlo) | 0x64006400u;
  const uint32_t p3 = (hi & mhi) | 0x54005400u;
  u32x4 r;
  r[0] = as_u32((as_f16x2(p0) - zk) * s2);
  r[1] = as_u32((as_f16x2(p1) - zs) * s2);
  r[2] = as_u32((as_f16x2(p2) - zk) * s2);
  r[3] = as_u32((as_f16x2(p3) - zs) * s2);
  return r;
}

// the same from the group's packed (scale, zero) pair (1024 + zero and 64 + zero are exact: zero is an integer in
// [0, 15])
__device__ __forceinline__ u32x4 dequant8(uint32_t word, uint32_t szw, uint32_t mlo, uint32_t mhi) {
  const f16x2 sz = as_f16x2(szw);
  const f16 zk = (f16)1024.0f + sz.y, zs = (f16)64.0f + sz.y;
  return dequant8_sz(word, f16x2{sz.x, sz.x}, f16x2{zk, zk}, f16x2{zs, zs}, mlo, mhi);
}

}  // namespace dk
