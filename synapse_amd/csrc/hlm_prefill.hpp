// Kernels of the hybrid decoder over the rows of a prompt (hlm_prefill.hip).
#pragma once

#include "common.hpp"
#include "rows_gemm.hpp"

namespace syn {

// the K splits of a GEMM's rows, summed in order by the kernel that reads
// them: row t, column j at p[z * zs + t * ld + j]
struct HRows {
  const float *p = nullptr;
  int kz = 1;
  size_t zs = 0;
  int ld = 0;
};

constexpr int kHrowsMaxH = 8192, kHrowsMaxF = 16384;

// x [T, H], the residual rows in the step's fixed point (or, with ids, the
// embedding rows) += add; the parts of its RMSNorm in xf
syn_status_t launch_hrows_norm(long long *x, const float *embed, const uint32_t *ids, int vocab,
                               HRows add, const float *gain, float eps, int T, int H, void *xf,
                               hipStream_t s);
// LIV conv of in_proj's [B | C | x] rows from an empty state; its parts in
// xf, the state after the last token in `state` [I][ck]
syn_status_t launch_hrows_conv(HRows p, const float *w, const float *bias, int T, int I, int ck,
                               float *state, void *xf, hipStream_t s);
// parts of silu(gate) * up from the stacked [gate | up] rows
syn_status_t launch_hrows_swiglu(HRows gu, int T, int F, void *xf, hipStream_t s);
// the last row's residual, x[T - 1] + add, in r
syn_status_t launch_hrows_last(const long long *x, HRows add, int T, int H, long long *r,
                               hipStream_t s);

}  // namespace syn
