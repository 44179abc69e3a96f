// The hybrid (LFM2.5) layers over the rows of a prompt.  Token by token a
// prompt reads every weight and the 268 MB lm_head once per token (~0.15 ms at
// four layers); here the projections are matrix products over all tokens that
// round nothing before their f32 sums (rows_gemm.hip), and the ops between them
// are one kernel each that sums the product's K splits, computes its rows and
// writes the next product's activation parts directly.
#include "bf16_parts.hpp"
#include "hlm_prefill.hpp"

namespace syn {

namespace {

// columns 8c .. 8c+7 (offset by `off`) of row t
__device__ __forceinline__ void hrow_get(const HRows &h, int t, int off, int c, float (&v)[8]) {
  const float *p = h.p + (size_t)t * h.ld + off + 8 * c;
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = 0.0f;
  for (int z = 0; z < h.kz; z++, p += h.zs) {
    const float4 a = *reinterpret_cast<const float4 *>(p);
    const float4 b = *reinterpret_cast<const float4 *>(p + 4);
    v[0] += a.x; v[1] += a.y; v[2] += a.z; v[3] += a.w;
    v[4] += b.x; v[5] += b.y; v[6] += b.z; v[7] += b.w;
  }
}

// the same columns of each K split added to the residual row r, in the step's
// fixed point
__device__ __forceinline__ void hrow_add(const HRows &h, int t, int c, long long (&r)[8]) {
  const float *p = h.p + (size_t)t * h.ld + 8 * c;
  for (int z = 0; z < h.kz; z++, p += h.zs) {
    const float4 a = *reinterpret_cast<const float4 *>(p);
    const float4 b = *reinterpret_cast<const float4 *>(p + 4);
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int i = 0; i < 8; i++) r[i] += kqf_fix(v[i]);
  }
}

// the parts of the thread's chunks tid, tid + NT, .. (zeros for the padding
// rows of the last tile)
template <int NT, int R>
__device__ __forceinline__ void put_row(const float (&v)[R][8], int chunks, bool real, int m,
                                        bf16x8 *__restrict__ xf) {
  const float zero[8] = {};
#pragma unroll
  for (int j = 0; j < R; j++) {
    const int c = threadIdx.x + NT * j;
    if (c >= chunks) break;
    if (real) parts_put(xf, chunks >> 2, m, c, v[j]);
    else parts_put(xf, chunks >> 2, m, c, zero);
  }
}

constexpr int kNormNT = 256, kNormR = kHrowsMaxH / 8 / kNormNT;
constexpr int kGluNT = 512, kGluR = kHrowsMaxF / 8 / kGluNT;

// one workgroup per row; row values in registers between the reductions
__global__ void __launch_bounds__(kNormNT)
    k_hrows_norm(long long *__restrict__ x, const float *__restrict__ embed,
                 const uint32_t *__restrict__ ids, int vocab, HRows add,
                 const float *__restrict__ gain, float eps, int T, int H, bf16x8 *__restrict__ xf) {
  __shared__ float rss[kNormNT / 64];
  const int m = blockIdx.x, tid = threadIdx.x, chunks = H >> 3;
  const bool real = m < T;
  float v[kNormR][8];
  float ss = 0.0f;
#pragma unroll
  for (int j = 0; j < kNormR; j++) {
    const int c = tid + kNormNT * j;
    if (c >= chunks || !real) break;
    i64x2 *xr = reinterpret_cast<i64x2 *>(x + (size_t)m * H + 8 * c);
    long long r[8];
    if (ids) {  // an id outside the vocabulary is a zero row
      const uint32_t id = ids[m];
      const bool in = id < (uint32_t)vocab;
      const float *src = embed + (in ? (size_t)id * H : 0) + 8 * c;
      const float4 a = *reinterpret_cast<const float4 *>(src);
      const float4 b = *reinterpret_cast<const float4 *>(src + 4);
      const float f[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
      for (int i = 0; i < 8; i++) r[i] = in ? kqf_fix(f[i]) : 0;
    } else {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const i64x2 q = xr[i];
        r[2 * i] = q.x;
        r[2 * i + 1] = q.y;
      }
    }
    if (add.p) hrow_add(add, m, c, r);
    const float4 ga = *reinterpret_cast<const float4 *>(gain + 8 * c);
    const float4 gb = *reinterpret_cast<const float4 *>(gain + 8 * c + 4);
    const float g[8] = {ga.x, ga.y, ga.z, ga.w, gb.x, gb.y, gb.z, gb.w};
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const float s = kqf_unfix(r[i]);
      ss += s * s;
      v[j][i] = s * g[i];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) xr[i] = i64x2{r[2 * i], r[2 * i + 1]};
  }
  for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
  if ((tid & 63) == 0) rss[tid >> 6] = ss;
  __syncthreads();
  ss = 0.0f;
#pragma unroll
  for (int i = 0; i < kNormNT / 64; i++) ss += rss[i];
  const float scale = 1.0f / sqrtf(ss / (float)H + eps);
#pragma unroll
  for (int j = 0; j < kNormR; j++)
#pragma unroll
    for (int i = 0; i < 8; i++) v[j][i] *= scale;
  put_row<kNormNT>(v, chunks, real, m, xf);
}

// layer.rs:25-42, 609-627 over the prompt: taps oldest to newest, zeros before
// the first token.  A row's workgroup forms B*x of its taps itself (ck
// products a channel) rather than in a pass of their own
__global__ void __launch_bounds__(kNormNT)
    k_hrows_conv(HRows p, const float *__restrict__ w, const float *__restrict__ bias, int T,
                 int I, int ck, float *__restrict__ state, bf16x8 *__restrict__ xf) {
  const int m = blockIdx.x, tid = threadIdx.x, chunks = I >> 3;
  const bool real = m < T;
  float v[kNormR][8];
#pragma unroll
  for (int j = 0; j < kNormR; j++) {
    const int c = tid + kNormNT * j;
    if (c >= chunks || !real) break;
    float sum[8];
#pragma unroll
    for (int i = 0; i < 8; i++) sum[i] = -0.0f;
    for (int k = 0; k < ck; k++) {
      const int t = m - (ck - 1) + k;
      float bx[8] = {};
      if (t >= 0) {
        float b[8], xs[8];
        hrow_get(p, t, 0, c, b);
        hrow_get(p, t, 2 * I, c, xs);
#pragma unroll
        for (int i = 0; i < 8; i++) bx[i] = b[i] * xs[i];
      }
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const float q = bx[i] * w[(8 * c + i) * ck + k];
        sum[i] = sum[i] + q;
        if (m == T - 1) state[(size_t)(8 * c + i) * ck + k] = bx[i];
      }
    }
    float gate[8];
    hrow_get(p, m, I, c, gate);
#pragma unroll
    for (int i = 0; i < 8; i++)
      v[j][i] = gate[i] * (bias ? sum[i] + bias[8 * c + i] : sum[i]);
  }
  put_row<kNormNT>(v, chunks, real, m, xf);
}

__global__ void __launch_bounds__(kGluNT)
    k_hrows_swiglu(HRows gu, int T, int F, bf16x8 *__restrict__ xf) {
  __shared__ uint64_t etab[32];
  const int m = blockIdx.x, tid = threadIdx.x, chunks = F >> 3;
  const bool real = m < T;
  if (tid < 32) etab[tid] = syn_exp2_tab[tid];
  __syncthreads();
  float v[kGluR][8];
#pragma unroll
  for (int j = 0; j < kGluR; j++) {
    const int c = tid + kGluNT * j;
    if (c >= chunks || !real) break;
    float g[8], u[8];
    hrow_get(gu, m, 0, c, g);
    hrow_get(gu, m, F, c, u);
#pragma unroll
    for (int i = 0; i < 8; i++) v[j][i] = syn_silu_tab(g[i], etab) * u[i];
  }
  put_row<kGluNT>(v, chunks, real, m, xf);
}

__global__ void __launch_bounds__(256)
    k_hrows_last(const long long *__restrict__ x, HRows add, int T, int H,
                 long long *__restrict__ r) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (8 * c >= H) return;
  long long v[8];
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = x[(size_t)(T - 1) * H + 8 * c + i];
  hrow_add(add, T - 1, c, v);
#pragma unroll
  for (int i = 0; i < 8; i++) r[8 * c + i] = v[i];
}

}  // namespace

syn_status_t launch_hrows_norm(long long *x, const float *embed, const uint32_t *ids, int vocab,
                               HRows add, const float *gain, float eps, int T, int H, void *xf,
                               hipStream_t s) {
  if (H % 32 || H > kHrowsMaxH) return SYN_ERR_INVALID_ARG;
  hipLaunchKernelGGL(k_hrows_norm, dim3((unsigned)round_up(T, 32)), dim3(kNormNT), 0, s, x, embed,
                     ids, vocab, add, gain, eps, T, H, static_cast<bf16x8 *>(xf));
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

syn_status_t launch_hrows_conv(HRows p, const float *w, const float *bias, int T, int I, int ck,
                               float *state, void *xf, hipStream_t s) {
  if (I % 32 || I > kHrowsMaxH) return SYN_ERR_INVALID_ARG;
  hipLaunchKernelGGL(k_hrows_conv, dim3((unsigned)round_up(T, 32)), dim3(kNormNT), 0, s, p, w,
                     bias, T, I, ck, state, static_cast<bf16x8 *>(xf));
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

syn_status_t launch_hrows_swiglu(HRows gu, int T, int F, void *xf, hipStream_t s) {
  if (F % 32 || F > kHrowsMaxF) return SYN_ERR_INVALID_ARG;
  hipLaunchKernelGGL(k_hrows_swiglu, dim3((unsigned)round_up(T, 32)), dim3(kGluNT), 0, s, gu, T, F,
                     static_cast<bf16x8 *>(xf));
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

syn_status_t launch_hrows_last(const long long *x, HRows add, int T, int H, long long *r,
                               hipStream_t s) {
  if (H % 8) return SYN_ERR_INVALID_ARG;
  hipLaunchKernelGGL(k_hrows_last, dim3((unsigned)cdiv((size_t)H / 8, 256)), dim3(256), 0, s, x,
                     add, T, H, r);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

}  // namespace syn
