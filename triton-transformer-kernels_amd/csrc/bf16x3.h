// fp32 values as three bf16 terms, for fp32 products on the bf16 matrix cores.
//
// A float's 24 significant bits are the sum of three bf16 numbers exactly
// (8 + 8 + 8 bits; values below 2^-110 may lose their last bits).  Products of
// bf16 pairs are exact in fp32, so a product of two fp32 values is the sum of
// nine exact ones; the six with the leading terms are kept (terms 0.0, 0.1,
// 1.0, 1.1, 0.2, 2.0), the other three are below 2^-22 of the product.
// Infinities, NaN and values that round to infinity leave NaN in a sum of such
// products: callers recompute non-finite results from the fp32 operands.
#pragma once

#include "ttk_common.h"

namespace ttk {

// The three terms of eight fp32 values.
struct Split8 {
  u32x4 t[3];
};

typedef __bf16 x3bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f32x16 mfma_x3(const u32x4& a, const u32x4& b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                 0, 0);
}
__device__ __forceinline__ float high_half(float a) {
  return __uint_as_float(__float_as_uint(a) & 0xffff0000u);
}
// The upper 16 bits of (a, b) as a packed pair.
__device__ __forceinline__ unsigned pack_high(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
// The three terms of the pair (a, b), by truncation: 11 VALU operations.
// (v_dot2_f32_bf16 would subtract a term in one instruction but holds up the
// matrix pipe: beside four simple VALU operations an MFMA took 14.6 ns, beside
// four dot2 28 ns.)
__device__ __forceinline__ void split_pair(float a, float b, unsigned& t0, unsigned& t1, unsigned& t2) {
  const float a1 = a - high_half(a), b1 = b - high_half(b);
  const float a2 = a1 - high_half(a1), b2 = b1 - high_half(b1);
  t0 = pack_high(a, b);
  t1 = pack_high(a1, b1);
  t2 = pack_high(a2, b2);
  // Opaque here, so that the split stays where it is written: between the
  // MFMAs before the ones that use it.
  asm volatile("" : "+v"(t2));
}
__device__ __forceinline__ void split_pair(Split8& s, int d, float a, float b) {
  unsigned t0, t1, t2;
  split_pair(a, b, t0, t1, t2);
  s.t[0][d] = t0;
  s.t[1][d] = t1;
  s.t[2][d] = t2;
}
// The same with every term rounded to nearest: the terms' signs are then
// independent of the value's, and so are those of the products left out.
__device__ __forceinline__ void split_pair_rn(Split8& s, int d, float a, float b) {
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const x3bf16x2 r = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
    s.t[i][d] = __builtin_bit_cast(unsigned, r);
    a -= static_cast<float>(r.x);
    b -= static_cast<float>(r.y);
  }
}

}  // namespace ttk
