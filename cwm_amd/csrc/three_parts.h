// float32 values in products of the bfloat16 matrix instruction: three parts that hold all bits of a value, against operands that
// are bfloat16 to begin with.
#pragma once
#include "common.h"

// Eight float32 values as the operands of three bfloat16 matrix products whose sum is the product of the values: each part is
// the leading eight bits of what the parts before leave, so three hold all 24 (of values below 2^-110 the last lie among bfloat16's
// subnormals and may be lost: less than 2^-125), and with a bfloat16 second operand every single product is exact.  An infinity or
// a NaN is its first part alone; the other operand has to be finite, since a part may be zero.
__device__ __forceinline__ void three_parts(const float (&v)[8], Frag8 (&part)[3]) {
  uint32_t w[3][8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint32_t bits = __float_as_uint(v[e]);
    w[0][e] = bits;
    float rest = v[e] - __uint_as_float(bits & 0xffff0000u);
    rest = (bits & 0x7f800000u) == 0x7f800000u ? 0.f : rest;
    w[1][e] = __float_as_uint(rest);
    w[2][e] = __float_as_uint(rest - __uint_as_float(w[1][e] & 0xffff0000u));
  }
#pragma unroll
  for (int k = 0; k < 3; ++k)
    part[k].u = make_uint4(__builtin_amdgcn_perm(w[k][1], w[k][0], 0x07060302u), __builtin_amdgcn_perm(w[k][3], w[k][2], 0x07060302u),
                           __builtin_amdgcn_perm(w[k][5], w[k][4], 0x07060302u), __builtin_amdgcn_perm(w[k][7], w[k][6], 0x07060302u));
}

typedef unsigned short Halves __attribute__((ext_vector_type(2)));

// The larger magnitudes, halves apart, of two bfloat16 values a word; from 0x7f80 on an infinity or a NaN.
__device__ __forceinline__ Halves larger_magnitudes(Halves so_far, uint32_t w) {
  return __builtin_elementwise_max(so_far, __builtin_bit_cast(Halves, w & 0x7fff7fffu));
}
