// fp32 operands on the bf16 matrix cores, for the products of the compression's backward.
#pragma once
#include "common.h"

namespace {

// fp32 products on the bf16 matrix cores: a float is the exact sum of three bf16 values of 8
// significant bits each (cut off, not rounded, so hi never overflows; infinities keep zero lower
// parts and NaN stays NaN). A bf16 operand times the three parts is exact before the fp32
// accumulation; two split operands use every product but lo lo (2^-32 of the leading one). An
// operand's infinities and NaN (its exponent field all ones) enter the leading product alone: the
// others take `fin`, hi with those values 0, so that infinity never meets a zero lower part.
struct Plain {
  bf16x8 hi, fin;
};
struct Split3 {
  bf16x8 hi, mid, lo, fin;
};

__device__ __forceinline__ bf16x8 finite8(const bf16x8& v) {
  u32x4 u = __builtin_bit_cast(u32x4, v);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if ((u[q] & 0x7f80u) == 0x7f80u) u[q] &= 0xffff0000u;
    if ((u[q] & 0x7f800000u) == 0x7f800000u) u[q] &= 0xffffu;
  }
  return __builtin_bit_cast(bf16x8, u);
}

__device__ __forceinline__ Split3 split3(const float (&v)[8]) {
  u32x4 h, m, l;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    uint32_t hb[2], mb[2], lb[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float x = v[2 * q + i];
      hb[i] = __float_as_uint(x);
      const float xh = __uint_as_float(hb[i] & 0xffff0000u);
      const float r = x == xh ? 0.f : x - xh;
      mb[i] = __float_as_uint(r);
      const float rm = __uint_as_float(mb[i] & 0xffff0000u);
      lb[i] = __float_as_uint(r == rm ? 0.f : r - rm);
    }
    // the high halves of two floats side by side
    h[q] = __builtin_amdgcn_perm(hb[1], hb[0], 0x07060302);
    m[q] = __builtin_amdgcn_perm(mb[1], mb[0], 0x07060302);
    l[q] = __builtin_amdgcn_perm(lb[1], lb[0], 0x07060302);
  }
  const bf16x8 hi = __builtin_bit_cast(bf16x8, h);
  return {hi, __builtin_bit_cast(bf16x8, m), __builtin_bit_cast(bf16x8, l), finite8(hi)};
}

// hi + lo += a b, smallest products first; of two split operands only the leading products go to hi,
// so that it takes one rounding per 16 terms, as with a bf16 operand's three.
__device__ __forceinline__ void mfma_split(const Split3& a, const Plain& b, f32x16& hi, f32x16&) {
  hi = wa_mfma32(a.lo, b.fin, hi);
  hi = wa_mfma32(a.mid, b.fin, hi);
  hi = wa_mfma32(a.hi, b.hi, hi);
}
__device__ __forceinline__ void mfma_split(const Split3& a, const Split3& b, f32x16& hi, f32x16& lo) {
  lo = wa_mfma32(a.lo, b.mid, lo);
  lo = wa_mfma32(a.mid, b.lo, lo);
  lo = wa_mfma32(a.lo, b.fin, lo);
  lo = wa_mfma32(a.fin, b.lo, lo);
  lo = wa_mfma32(a.mid, b.mid, lo);
  lo = wa_mfma32(a.mid, b.fin, lo);
  lo = wa_mfma32(a.fin, b.mid, lo);
  hi = wa_mfma32(a.hi, b.hi, hi);
}

}  // namespace
