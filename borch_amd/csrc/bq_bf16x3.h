// Exact products of f32 values on the bf16 MFMA: a float as the sum of three bf16 pieces.
//
// x = x1 + x2 + x3 with x1 the bf16 nearest x and x2 the bf16 nearest x - x1: x - x1 is a
// multiple of ulp_f32(x) below 2^-8 |x| (at most 16 significant bits), (x - x1) - x2 a
// multiple of it below 2^-16 |x| (at most 8), so x3 = (x - x1) - x2 is exact in bf16 and the
// split loses nothing for |x| >= 2^-109. Below that pieces fall under bf16's last bit, 2^-133 (the
// MFMA takes bf16 subnormals as they are), and a value loses up to 2^-134. Just below 2^128 x1
// may round to infinity, and an infinite x leaves NaN in x2, so either makes every sum it is part
// of NaN or infinite. Callers take sums again in plain f32 that are not finite or so small that
// such a loss matters.
#pragma once

#include "bq_common.h"

namespace bq {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef short v4s __attribute__((ext_vector_type(4)));  // four bf16 of the 16-deep MFMA
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));

// Two floats to two bf16 (round to nearest even, v_cvt_pk_bf16_f32), packed low first.
__device__ __forceinline__ uint32_t bf2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f){a, b}, v2bf));
}

// The three bf16 planes of two floats, packed low first.
__device__ __forceinline__ void split3(float a, float b, uint32_t& p1, uint32_t& p2, uint32_t& p3) {
  p1 = bf2(a, b);
  const float r0 = __fsub_rn(a, __uint_as_float(p1 << 16)), r1 = __fsub_rn(b, __uint_as_float(p1 & 0xffff0000u));
  p2 = bf2(r0, r1);
  p3 = bf2(__fsub_rn(r0, __uint_as_float(p2 << 16)), __fsub_rn(r1, __uint_as_float(p2 & 0xffff0000u)));
}

// Of eight floats: one MFMA operand fragment for each plane.
struct Split8 {
  v8bf p1, p2, p3;
};
__device__ __forceinline__ Split8 split8(float4 a, float4 b) {
  uint32_t p1[4], p2[4], p3[4];
  split3(a.x, a.y, p1[0], p2[0], p3[0]);
  split3(a.z, a.w, p1[1], p2[1], p3[1]);
  split3(b.x, b.y, p1[2], p2[2], p3[2]);
  split3(b.z, b.w, p1[3], p2[3], p3[3]);
  Split8 s;
  s.p1 = __builtin_bit_cast(v8bf, make_uint4(p1[0], p1[1], p1[2], p1[3]));
  s.p2 = __builtin_bit_cast(v8bf, make_uint4(p2[0], p2[1], p2[2], p2[3]));
  s.p3 = __builtin_bit_cast(v8bf, make_uint4(p3[0], p3[1], p3[2], p3[3]));
  return s;
}

// Four signed bytes (low first) to four bf16, exactly: f32(q) has at most 7 significant
// bits, so its bf16 is its upper half.
__device__ __forceinline__ uint2 i8x4_bf16(uint32_t w) {
  const float f0 = (float)(int)(int8_t)(w & 0xff), f1 = (float)(int)(int8_t)((w >> 8) & 0xff);
  const float f2 = (float)(int)(int8_t)((w >> 16) & 0xff), f3 = (float)(int)(int8_t)(w >> 24);
  return make_uint2(__builtin_amdgcn_perm(__float_as_uint(f1), __float_as_uint(f0), 0x07060302u),
                    __builtin_amdgcn_perm(__float_as_uint(f3), __float_as_uint(f2), 0x07060302u));
}
__device__ __forceinline__ v8bf i8x8_bf16(uint32_t lo, uint32_t hi) {
  const uint2 a = i8x4_bf16(lo), b = i8x4_bf16(hi);
  return __builtin_bit_cast(v8bf, make_uint4(a.x, a.y, b.x, b.y));
}

}  // namespace bq
