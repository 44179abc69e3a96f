// Kernels of the Mamba decoder over the rows of a prompt (mamba_prefill.hip):
// every op of a layer runs over all tokens at once, and only the state
// recurrence walks them in order.  Each output is the same sequence of float
// operations as the decode step's.
#pragma once

#include "common.hpp"

namespace syn {

// conv1d + SiLU over T tokens (positions pos0 ..): proj [T, ldp] holds the
// inputs of channel i in column i, ring [di][dc] those before pos0; xc [T, di];
// with xq set also the row quantization into xq [T, ldq] and sx [T]
syn_status_t launch_mrows_conv(const float *proj, size_t ldp, const float *ring, const float *cw,
                               const float *cb, int T, int pos0, int di, int dc, float *xc,
                               int8_t *xq, size_t ldq, float *sx, hipStream_t s);
// y [T, N] = x [T, K] W^T as sequential f32 chains (W in [panel][K/4][64][4];
// rows < n8 fused); K a multiple of 4
syn_status_t launch_mrows_f32(const float *Wp, const float *x, int T, int K, int N, int n8,
                              float *y, hipStream_t s);
// dt [T, di] = softplus(dt_proj(xp[:, :dr]) + bias): INT8 W8A8 with Wdt
// (panel layout, Cdt chunks) and its scales, else f32 chains over dtwT
// [dr][di].  dr <= 64
syn_status_t launch_mrows_dt(const float *xp, int nx, int dr, const void *Wdt, int Cdt,
                             const float *wsdt, const float *dtwT, const float *dtb, int n8,
                             int T, int di, float *dt, hipStream_t s);
// selective scan over T tokens, d_state = 16: y [T, di], the state h [di][16]
// updated in place; the conv ring's slots of the last tokens are written
syn_status_t launch_mrows_scan(const float *dt, const float *xc, const float *xp, int nx, int dr,
                               const float *alc, const float *proj, size_t ldp, int T, int pos0,
                               int di, int dc, float *h, float *ring, float *y, hipStream_t s);
// gated = silu(z) * (y + D x), quantized per row into gq [T, ldq], sg [T]
syn_status_t launch_mrows_gate(const float *proj, size_t ldp, const float *y, const float *xc,
                               const float *dparam, int T, int di, int8_t *gq, size_t ldq,
                               float *sg, hipStream_t s);
// LDS row of the conv and gate kernels
constexpr int kMrowsMaxInner = 12288;

}  // namespace syn
