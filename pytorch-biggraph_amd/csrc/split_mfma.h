// fp32 products on the bf16 matrix cores.
//
// An fp32 value is the exact sum of three bf16 numbers, x = h + m + l (8 + 8 + 8 significand bits; each part is the
// remainder rounded to nearest, so |m| <= 2^-9 |x| and |l| <= 2^-18 |x|), and the product of two bf16 numbers is exact in
// fp32.  A product of two fp32 values is then the sum of nine bf16 products, of which the three smallest (m l, l m, l l)
// are below 2^-26 of it -- a quarter of fp32's own rounding -- and are left out; the other six run on
// v_mfma_f32_16x16x32_bf16, smallest first, summed in fp32.
//
// Why: one such instruction does 16 times the multiply-adds of v_mfma_f32_16x16x4_f32 in the same cycles, so six of them
// are 2.7 times as fast, and -- unlike the fp32 instruction, which holds the SIMD's vector ALU for its whole length -- they
// leave the vector ALU to the other waves (measured: 8 waves, half issuing matrix and half vector instructions back to
// back, take the longer of the two times with bf16 and their sum with fp32).
// Precision, against float64 over normal, positive uniform and constant rows, k = 32 ... 1024, relative to sum |a b|: rms
// error 0.8-6.2e-8 (2.7e-7 on constant rows) where the fp32 instruction gives 1.0-7.3e-8 (9.3e-7): an instruction rounds
// once per 32 values of k here and once per value there.
//
// Not covered by the argument: |x| < 2^-110 (l falls below bf16's range; an absolute error below 2^-133), and infinite
// values and those within 2^-9 of the largest fp32 number (h is infinite), whose products come out NaN: the caller has to
// look for NaN and compute those entries otherwise.
#pragma once

#include "pbg_internal.h"

namespace pbg {

typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));

// Two values at a time: one conversion instruction per part and pair (written out, because the compiler otherwise converts
// every value on its own for the subtraction and the pair again for the result).
__device__ __forceinline__ uint32_t pack_bf16(float x, float y) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((float2v){x, y}, bf16x2));
}
__device__ __forceinline__ void split2(float x, float y, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = pack_bf16(x, y);
  const float rx = x - __uint_as_float(h << 16), ry = y - __uint_as_float(h & 0xffff0000u);
  m = pack_bf16(rx, ry);
  l = pack_bf16(rx - __uint_as_float(m << 16), ry - __uint_as_float(m & 0xffff0000u));
}
// The three parts of eight fp32 values, each in the form of a matrix instruction's operand.
struct Split8 {
  uint4 h, m, l;
};
__device__ __forceinline__ Split8 split8(const float* x) {
  Split8 s;
  split2(x[0], x[1], s.h.x, s.m.x, s.l.x);
  split2(x[2], x[3], s.h.y, s.m.y, s.l.y);
  split2(x[4], x[5], s.h.z, s.m.z, s.l.z);
  split2(x[6], x[7], s.h.w, s.m.w, s.l.w);
  return s;
}
// Eight float16 numbers held as fp32 (the conversion is exact for them).
__device__ __forceinline__ half8v pack_half8(const float* x) {
  half8v h;
#pragma unroll
  for (int i = 0; i < 8; ++i) h[i] = (_Float16)x[i];
  return h;
}

}  // namespace pbg
