// Quantized GEMM for a few rows (rows_gemm.hip): a batch of decoded
// sequences, a speculative verify, a short prompt.
#pragma once

#include "common.hpp"

namespace syn {

struct RowsGemm {
  int fmt = 0;
  const void *W = nullptr;       // plane layout of the format (kquant.hip, q4_0.hip)
  const uint16_t *Wd = nullptr;  // f16 block scales (Q4_0, Q8_0, Q6_K)
  int blocks = 0;                // blocks per row
  size_t n = 0, k = 0;
};

// Activations in the order the kernel's MFMA fragments take them
// ([32-row tile][64-element step][group][64 lanes][8 halfs], rows padded to
// whole tiles), each row scaled by a power of two, then the rows' inverse
// scales.
size_t rows_frag_bytes(size_t m, size_t k);
// f32 rows -> fragments in xf (rows_frag_bytes); with y0 set rows of y0 [m,
// ny] (stride ldy, whole 16-byte rows) are cleared on the way
syn_status_t launch_rows_frag(int fmt, const float *x, size_t ldx, size_t m, size_t k, void *xf,
                              float *y0, size_t ldy, size_t ny, hipStream_t s);

constexpr int kRowsMaxSplit = 8;
// K splits the launch below would use at best
int rows_gemm_splits(const RowsGemm &g, size_t m);
// y [m, n] = x W^T from fragments, in at most kz K splits (more than one adds
// into a cleared y).  Weights and activations are rounded once to f16; sums in
// f32.
syn_status_t launch_rows_gemm(const RowsGemm &g, const void *xf, size_t m, int kz, float *y,
                              size_t ldy, hipStream_t s);

// The same for Q4_0 with nothing rounded before the sums: each activation as
// three bf16 (bf16_parts.hpp) in [32-row tile][block][2][part][64 lanes][8],
// rows padded to whole tiles, k a multiple of 32.  The K splits' partial rows go
// to y + z * zs, to be added in z order; one K split is the result itself.
size_t rows_parts_bytes(size_t m, size_t k);
syn_status_t launch_rows_parts(const float *x, size_t ldx, size_t m, size_t k, void *xf,
                               hipStream_t s);
int rows_parts_splits(const RowsGemm &g, size_t m);
syn_status_t launch_rows_gemm_parts(const RowsGemm &g, const void *xf, size_t m, int kz, float *y,
                                    size_t ldy, size_t zs, hipStream_t s);
// whether the format is taken (q8_exact: every Q8_0 scale is an f16 value)
bool rows_gemm_fits(int fmt, bool q8_exact, size_t m, size_t n, size_t k);

}  // namespace syn
