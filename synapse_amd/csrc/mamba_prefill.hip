// The Mamba layer over the rows of a prompt.  The decode step spends ~22 us
// a layer and token on four dependent kernels that read 6.6 MB of weights for
// one row; here a layer is nine kernels for all rows: [norm + q8], in_proj
// GEMM, [conv + SiLU + q8], x_proj GEMM, [dt_proj + softplus], scan,
// [gate + q8], out_proj GEMM (int8_gemm.hip's whole-K form).  Every value is
// the decode step's float operations in its order, so a prompt leaves the
// same bits as the token loop.
//
// Only the scan is sequential over tokens; what it must wait for is one
// multiply and one add per token (h = ad * h + dt x B), so dt's softplus (a
// double-precision log) runs before it over all tokens in parallel, and the
// gate after it.
#include <algorithm>

#include "mamba_prefill.hpp"
#include "mamba_math.hpp"

namespace syn {

// one workgroup of kRowNT threads per token: with 256 threads a 2048-wide row
// is eight dependent rounds of loads (96 tokens: conv 16.7 us and gate 8.2;
// with 1024 threads 5.3 and 4.1)
constexpr int kRowNT = 1024;

// the A1 quantization of a row held in LDS (quantize.zig:12-47)
__device__ __forceinline__ void quantize_lds_row(const float *v, int n, float mx, float *red,
                                                 int8_t *__restrict__ q,
                                                 float *__restrict__ scale) {
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
  __syncthreads();
  mx = red[0];
#pragma unroll
  for (int i = 1; i < kRowNT / 64; i++) mx = fmaxf(mx, red[i]);
  if (mx == 0.0f) {
    for (int j = threadIdx.x; j < n; j += kRowNT) q[j] = 0;
    if (threadIdx.x == 0) *scale = 1.0f;
    return;
  }
  const float inv = 127.0f / mx;
  for (int j = threadIdx.x; j < n; j += kRowNT) q[j] = q8_level(v[j], inv);
  if (threadIdx.x == 0) *scale = mx / 127.0f;
}

// conv1d_step (int8_mamba.rs:43-56), taps oldest to newest, then SiLU.  DC:
// the taps as a constant, or 0 for any number
template <int DC>
__global__ void __launch_bounds__(kRowNT)
    k_mrows_conv(const float *__restrict__ proj, int ldp, const float *__restrict__ ring,
                 const float *__restrict__ cw, const float *__restrict__ cb, int pos0, int di,
                 int dc_arg, float *__restrict__ xc, int8_t *__restrict__ xq, int ldq,
                 float *__restrict__ sx) {
  extern __shared__ float row[];  // di
  __shared__ float red[kRowNT / 64];
  __shared__ uint64_t etab[32];
  const int dc = DC ? DC : dc_arg;
  if (threadIdx.x < 32) etab[threadIdx.x] = syn_exp2_tab[threadIdx.x];
  __syncthreads();
  const int t = blockIdx.x;
  const bool inside = t >= dc - 1;  // every tap is a token of this block
  float mx = 0.0f;
  for (int i = threadIdx.x; i < di; i += kRowNT) {
    float sum = 0.0f;
    if (DC && inside) {
      float v[DC ? DC : 1], w[DC ? DC : 1];
#pragma unroll
      for (int k = 0; k < DC; k++) {
        v[k] = proj[(size_t)(t - (DC - 1) + k) * ldp + i];
        w[k] = cw[i * DC + k];
      }
#pragma unroll
      for (int k = 0; k < DC; k++) {
        const float p = v[k] * w[k];
        sum = sum + p;
      }
    } else {
      for (int k = 0; k < dc; k++) {
        const int tt = t - (dc - 1) + k;  // token of this tap; before the prompt: the ring
        const float v = tt >= 0 ? proj[(size_t)tt * ldp + i] : ring[i * dc + (pos0 + tt + dc) % dc];
        const float p = v * cw[i * dc + k];
        sum = sum + p;
      }
    }
    const float x = syn_silu_tab(sum + cb[i], etab);
    xc[(size_t)t * di + i] = x;
    row[i] = x;
    const float a = fabsf(x);
    if (a > mx) mx = a;
  }
  if (xq) quantize_lds_row(row, di, mx, red, xq + (size_t)t * ldq, sx + t);
}

// lane = output row of a 64-row panel, a wave kF32Tok tokens: one weight load
// serves that many independent chains.  A chain is K dependent operations, so
// a panel whose rows all take the fused form runs that form alone (both forms
// and a select per element, as a panel with a tail needs: ~130 us for 96 rows
// of 2048 whatever the number of tokens up to 128; the fused form alone ~45).
constexpr int kF32Tok = 2;

template <bool MIXED>
__device__ __forceinline__ void mrows_f32_chains(const float4 *__restrict__ w,
                                                 const float *const (&xr)[kF32Tok], int K4,
                                                 bool fused, float (&acc)[kF32Tok]) {
  constexpr int U = 8;
  float4 v[U], nx[U];
  auto load = [&](float4(&d)[U], int g) {
#pragma unroll
    for (int u = 0; u < U; u++) d[u] = w[(size_t)min(g + u, K4 - 1) * 64];
  };
  auto part = [&](int g, int n) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (u < n) {
        const float wv[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
          for (int j = 0; j < kF32Tok; j++) {
            const float xv = xr[j][4 * (g + u) + c];
            const float f = __builtin_fmaf(xv, wv[c], acc[j]);
            if constexpr (MIXED) {
              const float p = xv * wv[c];
              const float q = acc[j] + p;
              acc[j] = fused ? f : q;
            } else {
              acc[j] = f;
            }
          }
      }
    }
  };
  load(v, 0);
  int g = 0;
  for (; g + U <= K4; g += U) {
    load(nx, min(g + U, K4 - 1));
    part(g, U);
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = nx[u];
  }
  part(g, K4 - g);
}

__global__ void __launch_bounds__(256)
    k_mrows_f32(const float4 *__restrict__ Wp, const float *__restrict__ x, int T, int K, int N,
                int n8, float *__restrict__ y) {
  const int lane = threadIdx.x & 63;
  const int t0 = (blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * kF32Tok;
  if (t0 >= T) return;
  const int K4 = K >> 2, row = blockIdx.x * 64 + lane;
  const float4 *w = Wp + (size_t)blockIdx.x * K4 * 64 + lane;
  const float *xr[kF32Tok];
  float acc[kF32Tok];
#pragma unroll
  for (int j = 0; j < kF32Tok; j++) {
    xr[j] = x + (size_t)min(t0 + j, T - 1) * K;
    acc[j] = 0.0f;
  }
  // rows past N are padding: a panel with all its real rows below n8 is fused
  if (min(N, (int)blockIdx.x * 64 + 64) <= n8)
    mrows_f32_chains<false>(w, xr, K4, true, acc);
  else
    mrows_f32_chains<true>(w, xr, K4, row < n8, acc);
#pragma unroll
  for (int j = 0; j < kF32Tok; j++)
    if (t0 + j < T && row < N) y[(size_t)(t0 + j) * N + row] = acc[j];
}

// thread = channel, a workgroup kDtTok tokens of 256 channels: the channel's
// dt_proj row is read once for all of them
constexpr int kDtTok = 4, kDtMax = 64;

template <bool INT8>
__global__ void __launch_bounds__(256)
    k_mrows_dt(const float *__restrict__ xp, int nx, int dr, const i32x4 *__restrict__ Wdt,
               int Cdt, const float *__restrict__ wsdt, const float *__restrict__ dtwT,
               const float *__restrict__ dtb, int n8, int T, int di, float *__restrict__ dt) {
  __shared__ float xs[kDtTok][kDtMax];
  __shared__ int xq[kDtTok][kDtMax / 4];
  __shared__ float sq[kDtTok];
  __shared__ uint64_t etab[32];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int t0 = blockIdx.y * kDtTok, c = blockIdx.x * 256 + tid, ci = min(c, di - 1);
  if (tid < 32) etab[tid] = syn_exp2_tab[tid];
  // the dt rows of x_proj's output; quantized (quantize.zig:12-47), a wave
  // a token
#pragma unroll
  for (int h = 0; h < kDtTok / 4; h++) {
    const int j = wave + 4 * h, t = min(t0 + j, T - 1);
    const float v = lane < dr ? xp[(size_t)t * nx + lane] : 0.0f;
    xs[j][lane] = v;
    if constexpr (INT8) {
      float mx = fabsf(v);
      for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
      int8_t q = 0;
      if (mx != 0.0f && lane < dr) q = q8_level(v, 127.0f / mx);
      reinterpret_cast<int8_t *>(xq[j])[lane] = q;
      if (lane == 0) sq[j] = mx == 0.0f ? 1.0f : mx / 127.0f;
    }
  }
  __syncthreads();
  float out[kDtTok];
  if constexpr (INT8) {
    int acc[kDtTok];
#pragma unroll
    for (int j = 0; j < kDtTok; j++) acc[j] = 0;
    const i32x4 *w = Wdt + (size_t)(ci >> 6) * Cdt * 64 + (ci & 63);
    for (int g = 0; g < Cdt; g++) {
      const i32x4 wv = w[g * 64];
#pragma unroll
      for (int j = 0; j < kDtTok; j++) {
        acc[j] = __builtin_amdgcn_sdot4(wv.x, xq[j][4 * g], acc[j], false);
        acc[j] = __builtin_amdgcn_sdot4(wv.y, xq[j][4 * g + 1], acc[j], false);
        acc[j] = __builtin_amdgcn_sdot4(wv.z, xq[j][4 * g + 2], acc[j], false);
        acc[j] = __builtin_amdgcn_sdot4(wv.w, xq[j][4 * g + 3], acc[j], false);
      }
    }
    const float wsc = wsdt[ci];
#pragma unroll
    for (int j = 0; j < kDtTok; j++) {
      const float f = (float)acc[j] * sq[j];
      out[j] = f * wsc;
    }
  } else {
    // f32GemvRow: fused chains for the channels below n8, plain after
    const bool fused = c < n8;
#pragma unroll
    for (int j = 0; j < kDtTok; j++) out[j] = 0.0f;
    for (int k = 0; k < dr; k++) {
      const float w = dtwT[(size_t)k * di + ci];
#pragma unroll
      for (int j = 0; j < kDtTok; j++) {
        const float f = __builtin_fmaf(xs[j][k], w, out[j]);
        const float p = xs[j][k] * w;
        const float q = out[j] + p;
        out[j] = fused ? f : q;
      }
    }
  }
  if (c >= di) return;
  const float b = dtb[c];
#pragma unroll
  for (int j = 0; j < kDtTok; j++)
    if (t0 + j < T) dt[(size_t)(t0 + j) * di + c] = syn_softplus_tab(out[j] + b, etab);
}

// 8 channels x 16 states per workgroup, kScanTok tokens at a time in three
// phases: all eight waves form exp(-dt A) and dt x B of every (token, channel,
// state) into LDS; two waves run the recurrence, a multiply and an add per
// token from LDS; 256 threads form the ordered sums over the states.  The
// expf (double precision, ~250 issue cycles a wave) is what the scan is made
// of and does not depend on the state, so it is spread over every wave of
// the CU: with the expf on the recurrence's own lanes (16 lanes a channel,
// one wave per SIMD) 96 tokens of 2048 channels took 28.6 us, now 11.2.
constexpr int kScanTok = 32, kScanCh = 8, kScanNT = 512;

__global__ void __launch_bounds__(kScanNT)
    k_mrows_scan(const float *__restrict__ dt, const float *__restrict__ xc,
                 const float *__restrict__ xp, int nx, int dr, const float *__restrict__ alc,
                 const float *__restrict__ proj, int ldp, int T, int pos0, int di, int dc,
                 float *__restrict__ h, float *__restrict__ ring, float *__restrict__ y) {
  constexpr int DS = 16, PAIRS = kScanCh * DS, TG = kScanNT / PAIRS, PER = kScanTok / TG;
  __shared__ float2 sap[kScanTok][PAIRS];  // (exp(-dt A), dt x B)
  __shared__ __align__(16) float sh[kScanTok][PAIRS + 4];  // the states after each token
  __shared__ uint64_t etab[32];
  const int tid = threadIdx.x, pair = tid % PAIRS, s = pair % DS, g = pair / DS;
  const int tg = tid / PAIRS;  // this thread's tokens of a block: tg, tg + TG, ..
  const int c0 = blockIdx.x * kScanCh, ci = min(c0 + g, di - 1);
  if (tid < 32) etab[tid] = syn_exp2_tab[tid];
  float rd[PER], rx[PER], rb[PER];
  auto load = [&](int t0) {
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const size_t t = (size_t)min(t0 + tg + TG * k, T - 1);
      rd[k] = dt[t * di + ci];
      rx[k] = xc[t * di + ci];
      rb[k] = xp[t * nx + dr + s];
    }
  };
  load(0);
  __syncthreads();  // the table
  const float e = syn_expf_tab(alc[(size_t)ci * DS + s], etab);
  float hv = h[(size_t)ci * DS + s];  // used by the recurrence's threads (tid < PAIRS)
  for (int t0 = 0; t0 < T; t0 += kScanTok) {
#pragma unroll
    for (int k = 0; k < PER; k++)
      sap[tg + TG * k][pair] = make_float2(syn_expf_tab(-rd[k] * e, etab), (rd[k] * rx[k]) * rb[k]);
    __syncthreads();
    if (t0 + kScanTok < T) load(t0 + kScanTok);
    const int n = min(kScanTok, T - t0);
    if (tid < PAIRS) {
      for (int j = 0; j < n; j++) {
        const float2 a = sap[j][pair];
        const float p1 = a.x * hv;
        hv = p1 + a.y;
        sh[j][pair] = hv;
      }
    }
    __syncthreads();
    // y of token j, channel c0 + q: groups of four states in order, then the groups
    const int j = tid / kScanCh, q = tid % kScanCh;
    if (j < n && c0 + q < di) {
      const float4 *hs = reinterpret_cast<const float4 *>(&sh[j][q * DS]);
      const float *cs = xp + (size_t)(t0 + j) * nx + dr + DS;
      float yi = 0.0f;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const float4 v = hs[k];
        yi = yi + (((cs[4 * k] * v.x + cs[4 * k + 1] * v.y) + cs[4 * k + 2] * v.z) +
                   cs[4 * k + 3] * v.w);
      }
      y[(size_t)(t0 + j) * di + c0 + q] = yi;
    }
  }
  if (tid >= PAIRS || c0 + g >= di) return;
  h[(size_t)(c0 + g) * DS + s] = hv;
  // the conv ring's slots of the last dc tokens
  for (int k = s; k < min(dc, T); k += DS) {
    const int t = T - 1 - k;
    ring[(c0 + g) * dc + (pos0 + t) % dc] = proj[(size_t)t * ldp + c0 + g];
  }
}

// int8_mamba.rs:102, then out_proj's quantizer
__global__ void __launch_bounds__(kRowNT)
    k_mrows_gate(const float *__restrict__ proj, int ldp, const float *__restrict__ y,
                 const float *__restrict__ xc, const float *__restrict__ dparam, int di,
                 int8_t *__restrict__ gq, int ldq, float *__restrict__ sg) {
  extern __shared__ float row[];  // di
  __shared__ float red[kRowNT / 64];
  __shared__ uint64_t etab[32];
  if (threadIdx.x < 32) etab[threadIdx.x] = syn_exp2_tab[threadIdx.x];
  __syncthreads();
  const size_t t = blockIdx.x;
  float mx = 0.0f;
  for (int i = threadIdx.x; i < di; i += kRowNT) {
    const float z = proj[t * ldp + di + i];
    const float v = syn_silu_tab(z, etab) * (y[t * di + i] + dparam[i] * xc[t * di + i]);
    row[i] = v;
    const float a = fabsf(v);
    if (a > mx) mx = a;
  }
  quantize_lds_row(row, di, mx, red, gq + t * ldq, sg + t);
}

syn_status_t launch_mrows_conv(const float *proj, size_t ldp, const float *ring, const float *cw,
                               const float *cb, int T, int pos0, int di, int dc, float *xc,
                               int8_t *xq, size_t ldq, float *sx, hipStream_t s) {
  const auto kern = dc == 4 ? k_mrows_conv<4> : k_mrows_conv<0>;
  hipLaunchKernelGGL(kern, dim3((unsigned)T), dim3(kRowNT), (size_t)di * 4, s, proj, (int)ldp,
                     ring, cw, cb, pos0, di, dc, xc, xq, (int)ldq, sx);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

syn_status_t launch_mrows_f32(const float *Wp, const float *x, int T, int K, int N, int n8,
                              float *y, hipStream_t s) {
  if (K % 4) return SYN_ERR_INVALID_ARG;
  const dim3 grid((unsigned)cdiv((size_t)N, 64), (unsigned)cdiv((size_t)T, 4 * kF32Tok));
  hipLaunchKernelGGL(k_mrows_f32, grid, dim3(256), 0, s, reinterpret_cast<const float4 *>(Wp), x,
                     T, K, N, n8, y);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

syn_status_t launch_mrows_dt(const float *xp, int nx, int dr, const void *Wdt, int Cdt,
                             const float *wsdt, const float *dtwT, const float *dtb, int n8,
                             int T, int di, float *dt, hipStream_t s) {
  if (dr > kDtMax || (Wdt && Cdt * 16 > kDtMax)) return SYN_ERR_INVALID_ARG;
  const dim3 grid((unsigned)cdiv((size_t)di, 256), (unsigned)cdiv((size_t)T, kDtTok));
  if (Wdt)
    hipLaunchKernelGGL(k_mrows_dt<true>, grid, dim3(256), 0, s, xp, nx, dr, (const i32x4 *)Wdt,
                       Cdt, wsdt, nullptr, dtb, n8, T, di, dt);
  else
    hipLaunchKernelGGL(k_mrows_dt<false>, grid, dim3(256), 0, s, xp, nx, dr, nullptr, 0, nullptr,
                       dtwT, dtb, n8, T, di, dt);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

syn_status_t launch_mrows_scan(const float *dt, const float *xc, const float *xp, int nx, int dr,
                               const float *alc, const float *proj, size_t ldp, int T, int pos0,
                               int di, int dc, float *h, float *ring, float *y, hipStream_t s) {
  hipLaunchKernelGGL(k_mrows_scan, dim3((unsigned)cdiv((size_t)di, kScanCh)), dim3(kScanNT), 0, s,
                     dt, xc, xp, nx, dr, alc, proj, (int)ldp, T, pos0, di, dc, h, ring, y);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

syn_status_t launch_mrows_gate(const float *proj, size_t ldp, const float *y, const float *xc,
                               const float *dparam, int T, int di, int8_t *gq, size_t ldq,
                               float *sg, hipStream_t s) {
  hipLaunchKernelGGL(k_mrows_gate, dim3((unsigned)T), dim3(kRowNT), (size_t)di * 4, s, proj,
                     (int)ldp, y, xc, dparam, di, gq, (int)ldq, sg);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

}  // namespace syn
