// f32 activations and Q4_0 levels as bf16 operands of the matrix cores without
// a rounding: an f32 value is the sum of three bf16 (8 significant bits each,
// f32's own range), a level (-8 .. 7) is one, and a product of two bf16 is
// exact in f32.
#pragma once

#include "common.hpp"

namespace syn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// the upper halves of two words, a's in the low half
__device__ __forceinline__ uint32_t hi_halves(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(b, a, 0x07060302u);
}

// The matrix cores take bf16 subnormals as zeros.  Times 2^24 the last bit of
// every f32 value is a normal bf16; the finished sum takes it back
constexpr float kPartsUp = 16777216.0f, kPartsDown = 1.0f / 16777216.0f;

// x 2^24 = p[0] + p[1] + p[2], each part the upper half of what the ones before
// it leave.  Finite below |x| = 2^104; a sum over a block's 32 levels up to 2^8
// is, below 2^95
__device__ __forceinline__ void bf16_parts(const float (&x)[8], bf16x8 (&p)[3]) {
  uint32_t o[3][4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    uint32_t v[2], r[2], t[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const float s = x[2 * i + h] * kPartsUp;
      v[h] = __float_as_uint(s);
      const float q = s - __uint_as_float(v[h] & 0xffff0000u);
      r[h] = __float_as_uint(q);
      t[h] = __float_as_uint(q - __uint_as_float(r[h] & 0xffff0000u));
    }
    o[0][i] = hi_halves(v[0], v[1]);
    o[1][i] = hi_halves(r[0], r[1]);
    o[2][i] = hi_halves(t[0], t[1]);
  }
#pragma unroll
  for (int j = 0; j < 3; j++)
    p[j] = __builtin_bit_cast(bf16x8, u32x4{o[j][0], o[j][1], o[j][2], o[j][3]});
}

// nibble i of v, less 8, as element i
__device__ __forceinline__ bf16x8 q4_levels(uint32_t v) {
  const uint32_t lo = v & 0x0f0f0f0fu, hi = (v >> 4) & 0x0f0f0f0fu;
  uint32_t o[4];
#pragma unroll
  for (int b = 0; b < 4; b++) {
    const float e = (float)((lo >> (8 * b)) & 0xffu) - 8.0f;
    const float f = (float)((hi >> (8 * b)) & 0xffu) - 8.0f;
    o[b] = hi_halves(__float_as_uint(e), __float_as_uint(f));
  }
  return __builtin_bit_cast(bf16x8, u32x4{o[0], o[1], o[2], o[3]});
}

// the parts of chunk c (elements 8c .. 8c+7) of row m to their lane's place in
// the fragments of k_rows_gemm_parts, whose rows have B blocks
__device__ __forceinline__ void parts_put(bf16x8 *__restrict__ xf, int B, int m, int c,
                                          const float (&v)[8]) {
  bf16x8 p[3];
  bf16_parts(v, p);
  // block c / 4, half (c / 2) % 2, MFMA c % 2
  const size_t at = (((size_t)(m >> 5) * B + (c >> 2)) * 2 + (c & 1)) * 3;
  const int lane = ((c >> 1) & 1) * 32 + (m & 31);
#pragma unroll
  for (int i = 0; i < 3; i++) xf[(at + i) * 64 + lane] = p[i];
}

}  // namespace syn
