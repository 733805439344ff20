// fp32 values as three bf16 terms, for fp32 products on the bf16 matrix cores
// (the splitting of Henry, Tang and Heinecke, "Leveraging the bfloat16
// Artificial Intelligence Datatype For Higher-Precision Computations", ARITH
// 2019).
//
// A float's 24 significant bits are the sum of three bf16 numbers exactly
// (8 + 8 + 8 bits; values below 2^-110 may lose their last bits).  Every term
// is rounded to nearest, so the second is at most 2^-8 and the third at most
// 2^-17 of the value, both of either sign.  Products of bf16 pairs are exact in
// fp32, so a product of two fp32 values is the sum of nine exact ones; the six
// with the leading terms are kept (terms 0.0, 0.1, 1.0, 1.1, 0.2, 2.0).  The
// other three (1.2, 2.1, 2.2) come to at most 2^-24 + 2^-34 of the product, of
// random sign.  Terms cut off instead would all have the value's sign: the
// products left out come to 2^-22, and where both operands are cut off, they
// pull every sum towards zero: attention over 1024 keys with positive V had a
// mean error of -3.1e-7 (rms 5.8e-7; the fp32 MFMA's 4.7e-7), and has -3e-8
// (3.4e-7) as rounded.  Either split takes 11 VALU operations a pair; the
// conversions cost 2 - 4 % of the attention kernels, nothing of the linear ones.
// Infinities, NaN and values that round to infinity leave NaN in a sum of such
// products, and values below 2^-110 fewer bits: callers recompute results that
// are not finite, or nonzero and below 2^-80, from the fp32 operands (redo_x3).
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
// The three terms of the pair (a, b): 11 VALU operations.
// (v_dot2_f32_bf16 would subtract a term in one instruction but holds up the
// matrix pipe: beside four simple VALU operations an MFMA took 14.6 ns, beside
// four dot2 28 ns.)
__device__ __forceinline__ void split_pair(float a, float b, unsigned& t0, unsigned& t1, unsigned& t2) {
  auto round = [](float& u, float& v) __attribute__((always_inline)) -> unsigned {
    const x3bf16x2 r = {static_cast<__bf16>(u), static_cast<__bf16>(v)};
    unsigned bits = __builtin_bit_cast(unsigned, r);
    asm("" : "+v"(bits));  // one conversion of the pair, not another of its lower half
    u -= __uint_as_float(bits << 16);
    v -= high_half(__uint_as_float(bits));
    return bits;
  };
  t0 = round(a, b);
  t1 = round(a, b);
  const x3bf16x2 r = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
  t2 = __builtin_bit_cast(unsigned, r);
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
// Whether a result has to be formed again from the fp32 operands.  Bits that a
// value below 2^-110 loses are at most 2^-134 in magnitude: 2^-54 of a result
// of 2^-80 times the other operand, which keeps fp32 accuracy up to operands of
// 2^28.
constexpr float kRedoBelow = 0x1p-80f;
__device__ __forceinline__ bool redo_x3(float v) {
  return !(v * 0.0f == 0.0f) || (v != 0.0f && __builtin_fabsf(v) < kRedoBelow);
}
// The same over many results, three VALU operations each and no lane mask (33
// compares a lane kept as masks spilled up to 190 SGPRs of the attention
// kernels).  Twice the magnitude's bits less one orders zero above all others.
struct RedoWatch {
  float bad = 0.0f;              // NaN once a value was not finite
  unsigned least = 0xffffffffu;  // of the magnitudes
  __device__ __forceinline__ void see(float v) {
    bad = __builtin_fmaf(v, 0.0f, bad);
    least = min(least, (__float_as_uint(v) << 1) - 1u);
  }
  __device__ __forceinline__ bool any() const {
    return !(bad == 0.0f) || least < (__builtin_bit_cast(unsigned, kRedoBelow) << 1) - 1u;
  }
};

}  // namespace ttk
