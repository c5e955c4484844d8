// fp32 values as two f16 pieces for the matrix cores: x 2^e = p1 + p2 (+ what 23 significand bits leave), e a power of two that a
// whole row (or column) of an operand shares and that brings its largest value below 2^15.
//
// A product keeps p1 q1 + p2 q1 + p1 q2: three matrix instructions where three bf16 pieces take six.  Split error and dropped p2 q2
// are 4e-8 of a term each (root mean square), below what a fp32 sum of some 64 terms rounds; from there on the sums are more exact
// than with six partial products, because there are half as many additions.
#pragma once
#include "scan_common.h"

namespace aussm {

typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef float f2v __attribute__((ext_vector_type(2)));

constexpr float HALF_LO = 2048.0f, HALF_LO_INV = 1.0f / 2048.0f;   // second pieces kept 2^11 times larger, as exact as the first

__device__ __forceinline__ f4 xdl_half(const u4& a, const u4& b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8v, a), __builtin_bit_cast(h8v, b), c, 0, 0, 0);
}
// The exponent e that brings m (>= 0) into 2^14 .. 2^15 (at most 115, with which the smallest normal number still has two whole
// pieces and 2^(e + 11) is finite; an infinity as the largest finite value)
__device__ __forceinline__ int half_exponent(float m) {
  const int b = (int)(__float_as_uint(m) >> 23) & 255;
  return min(14 + 127 - min(b, 254), 115);
}
__device__ __forceinline__ float exp2_of(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }   // -126 .. 127

// LO: second pieces times 2^11, for an accumulator of their own
template <bool LO>
__device__ __forceinline__ void split8_half(const float (&x)[8], float scale, u4 (&out)[2]) {
  float m = LO ? -HALF_LO : -1.0f;                      // (in a register: half the code of a constant in every instruction)
  asm("" : "+s"(m));
  const float wide = LO ? scale * HALF_LO : scale;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float a = x[2 * q] * scale, b = x[2 * q + 1] * scale;
    asm("" : "+v"(a), "+v"(b));
    const h2v p = __builtin_convertvector(f2v{a, b}, h2v);
    float wa = LO ? x[2 * q] * wide : a, wb = LO ? x[2 * q + 1] * wide : b;
    asm("" : "+v"(wa), "+v"(wb));
    const h2v r = __builtin_convertvector((f2v{fmaf((float)p[0], m, wa), fmaf((float)p[1], m, wb)}), h2v);
    out[0][q] = __builtin_bit_cast(uint32_t, p);
    out[1][q] = __builtin_bit_cast(uint32_t, r);
  }
}

}  // namespace aussm
