// Device functions shared by the Mamba decode step and its prompt kernels.
#pragma once

#include "common.hpp"

namespace syn {

// softplus (ops/activation.rs:88-90); the log in double, rounded once
__device__ __forceinline__ float syn_softplus_tab(float v, const uint64_t *tab) {
  if (v > 20.0f) return v;
  const float t = 1.0f + syn_expf_tab(v, tab);
  return (float)log((double)t);
}

template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

// the scan's y over 16 states, one per lane of a 16-lane row, in
// selective_scan.zig's order: y = 0 + (((c0+c1)+c2)+c3) + (((c4+c5)+c6)+c7) + ...
__device__ __forceinline__ float row16_scan_sum(float c, int lane) {
  // each quad's ordered sum, in every lane of the quad (quad_perm broadcasts)
  const float q = ((dpp_f<0x00>(c) + dpp_f<0x55>(c)) + dpp_f<0xAA>(c)) + dpp_f<0xFF>(c);
  // the four quads of the row, in order
  const int base = lane & ~15;
  const float q0 = __shfl(q, base), q1 = __shfl(q, base + 4), q2 = __shfl(q, base + 8),
              q3 = __shfl(q, base + 12);
  return (((0.0f + q0) + q1) + q2) + q3;
}

}  // namespace syn
