// Device side of the activation fragments of rows_gemm.hip, for kernels that
// write their output rows in that form.
#pragma once

#include "common.hpp"

namespace syn {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int kFragStep = 64;  // elements of K per step

// the power of two that puts mx in [2^14, 2^15) and its inverse; 1 for a row
// of zeros, at most 2^126.  A row with an infinity (mx; a NaN does not reach
// it) takes the scale of the largest finite values, so that those stay finite
__device__ __forceinline__ void frag_row_scale(float mx, float *up, float *down) {
  *up = *down = 1.0f;
  if (mx > 0.0f) {
    int e = 128;
    if (mx <= 3.4028235e38f) (void)frexpf(mx, &e);
    e = max(e, 15 - 126);
    *up = ldexpf(1.0f, 15 - e);
    *down = ldexpf(1.0f, e - 15);
  }
}

// chunk c (elements 8c .. 8c+7, already scaled) of row m to its lane's place.
// PERM: the nibble formats' k order 0,2,4,6,1,3,5,7; SPLIT: value and
// remainder as two f16.  An infinity or a NaN goes into the remainder alone:
// the remainder meets only the weight itself, as in a plain sum, while the
// value also meets the weight's own remainder, which is often zero
template <bool PERM, bool SPLIT>
__device__ __forceinline__ void frag_put(f16x8 *__restrict__ xf, int steps, int m, int c,
                                         const float (&v)[8]) {
  constexpr int ord[8] = {0, 2, 4, 6, 1, 3, 5, 7};
  f16x8 hi, lo;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const float s = v[PERM ? ord[i] : i];
    hi[i] = (_Float16)s;
    if constexpr (SPLIT) {
      const bool finite = fabsf(s) <= 3.4028235e38f;
      if (!finite) hi[i] = (_Float16)0.0f;
      lo[i] = (_Float16)(s - (float)hi[i]);
    }
  }
  // step c / 8, half (c / 4) % 2, group c % 4
  const size_t at = (((size_t)(m >> 5) * steps + (c >> 3)) * 4 + (c & 3)) * (SPLIT ? 2 : 1);
  const int lane = ((c >> 2) & 1) * 32 + (m & 31);
  xf[at * 64 + lane] = hi;
  if constexpr (SPLIT) xf[(at + 1) * 64 + lane] = lo;
}

}  // namespace syn
