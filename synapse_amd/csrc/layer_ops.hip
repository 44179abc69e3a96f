// Decoder-layer kernels around the quantized GEMVs.  They are small and
// latency-bound; what matters is that each reproduces the reference's float
// operation order exactly (compiled with -ffp-contract=off; explicit
// __builtin_fmaf only where the reference uses @mulAdd), so the token stream
// matches the cpu_simd path bit for bit.
#include "layer_ops.hpp"
#include "reduce_order.hpp"

namespace syn {

// ------------------------------------------------------------------ embed
__global__ void k_embed(const float *__restrict__ embed, const uint32_t *__restrict__ ids,
                        int hidden, int vocab, float *__restrict__ x) {
  const int r = blockIdx.x;
  const uint32_t id = ids[r];
  float *xr = x + (size_t)r * hidden;
  if (id < (uint32_t)vocab) {
    const float *src = embed + (size_t)id * hidden;
    for (int j = threadIdx.x; j < hidden; j += blockDim.x) xr[j] = src[j];
  } else {
    for (int j = threadIdx.x; j < hidden; j += blockDim.x) xr[j] = 0.0f;
  }
}

syn_status_t launch_embed(const float *embed, const uint32_t *ids, int rows, int hidden,
                          int vocab, float *x, hipStream_t s) {
  hipLaunchKernelGGL(k_embed, dim3(rows), dim3(256), 0, s, embed, ids, hidden, vocab, x);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

// ------------------------------------------------------------------ residual
__global__ void k_add(float *__restrict__ x, const float *__restrict__ d, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = x[i] + d[i];
}

syn_status_t launch_add(float *x, const float *d, int n, hipStream_t s) {
  hipLaunchKernelGGL(k_add, dim3((n + 255) / 256), dim3(256), 0, s, x, d, n);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

// Sum of squares in the order of syn_vmul + syn_vreduce_sum
// (exports.zig:366-375, 503-514): lane accumulators acc[i%4] over the
// 4-aligned prefix, reduced as ((a0+a1)+a2)+a3, then the tail.  v is in LDS;
// must be called by all threads of the block (uses red[0..3] and a barrier).
__device__ float sumsq_vec4_order(const float *v, int n, float *red) {
  const int n4 = n & ~3;
  if (threadIdx.x < 4) {
    float acc = 0.0f;
    for (int i = threadIdx.x; i < n4; i += 4) {
      const float t = v[i] * v[i];
      acc = acc + t;
    }
    red[threadIdx.x] = acc;
  }
  __syncthreads();
  float s = ((red[0] + red[1]) + red[2]) + red[3];
  for (int i = n4; i < n; i++) {
    const float t = v[i] * v[i];
    s = s + t;
  }
  return s;
}

// block-wide max of non-negative values (exact in any order)
__device__ float block_max(float v, float *red) {
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  float m = red[0];
  for (int i = 1; i < nw; i++) m = fmaxf(m, red[i]);
  return m;
}

// quantize a row held in LDS (quantize.zig:12-47); all threads participate
__device__ void quantize_row_lds(const float *v, int n, int8_t *q, float *scale_out, float *red) {
  float mx = 0.0f;
  for (int j = threadIdx.x; j < n; j += blockDim.x) {
    const float a = fabsf(v[j]);
    if (a > mx) mx = a;
  }
  mx = block_max(mx, red);
  if (mx == 0.0f) {
    for (int j = threadIdx.x; j < n; j += blockDim.x) q[j] = 0;
    if (threadIdx.x == 0) *scale_out = 1.0f;
    return;
  }
  const float inv = 127.0f / mx;
  for (int j = threadIdx.x; j < n; j += blockDim.x) q[j] = q8_level(v[j], inv);
  if (threadIdx.x == 0) *scale_out = mx / 127.0f;
}

// ------------------------------------------------------------------ RMSNorm + quantize
// ops/norm.rs:8-38: out = (x*w) * (1/sqrt(sumsq/n + eps)); then A1 on out.
// One workgroup of NT threads per row.  The squares are written in the
// sumsq_chains layout, so the four reference chains run from LDS with
// 16-byte loads.  dynamic LDS: v[H] | sq[H]
template <int NT>
__global__ void __launch_bounds__(NT)
    k_rmsnorm_quant(float *__restrict__ x, const float *__restrict__ delta,
                    const float *__restrict__ w, float eps, int H, int8_t *__restrict__ xq,
                    int ldq, float *__restrict__ sx, float *__restrict__ normed) {
  extern __shared__ __align__(16) float sm[];
  __shared__ float red[64];
  float *v = sm, *sq = sm + round_up4(H);
  const int row = blockIdx.x;
  float *xr = x + (size_t)row * H;
  for (int j = threadIdx.x; j < H; j += NT) {
    float a = xr[j];
    if (delta) {
      a = a + delta[(size_t)row * H + j];
      xr[j] = a;
    }
    v[j] = a;
    sq[sq_slot(j, H)] = a * a;
  }
  __syncthreads();
  const float ss = sumsq_chains<NT>(sq, H, red);
  const float scale = 1.0f / sqrtf(ss / (float)H + eps);
  for (int j = threadIdx.x; j < H; j += NT) {
    const float t = v[j] * w[j];
    const float nv = t * scale;
    v[j] = nv;
    if (normed) normed[(size_t)row * H + j] = nv;
  }
  if (!xq) return;  // f32 path: normed rows only
  __syncthreads();
  quantize_row_lds(v, H, xq + (size_t)row * ldq, sx + row, red);
}

syn_status_t launch_rmsnorm_quant(float *x, const float *delta, const float *w, float eps,
                                  int rows, int hidden, int8_t *xq, int ldq, float *sx,
                                  float *normed, hipStream_t s) {
  const size_t shm = 2 * round_up((size_t)hidden, 4) * sizeof(float);
  if (shm > 64 * 1024) {
    set_error("rmsnorm: hidden size too large for the LDS row");
    return SYN_ERR_INVALID_ARG;
  }
  if (hidden >= 2048)
    hipLaunchKernelGGL(k_rmsnorm_quant<1024>, dim3(rows), dim3(1024), shm, s, x, delta, w, eps,
                       hidden, xq, ldq, sx, normed);
  else
    hipLaunchKernelGGL(k_rmsnorm_quant<256>, dim3(rows), dim3(256), shm, s, x, delta, w, eps,
                       hidden, xq, ldq, sx, normed);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

// ------------------------------------------------------------------ q/k norm, RoPE, KV append
// ops/attention.rs:46-66: headwise RMSNorm (norm.rs:78-93), rotate-half RoPE
// (rope.rs:13-43) at the token's position, append RoPE'd K and raw V.
// Cache row = position + cache_off: a prefill into a non-empty cache
// (cached_attention_prefill, ops/attention.rs:177-198) rotates at positions
// 0.. of the new tokens but appends after the rows already held.
// grid (n_heads + 2*n_kv, rows), one wave per head.
__global__ void __launch_bounds__(64)
    k_qk_norm_rope_kv(const float *__restrict__ qkv, int ldqkv, int nh, int nkv, int hd,
                      const float *__restrict__ qn, const float *__restrict__ kn, float eps,
                      const float *__restrict__ cosT, const float *__restrict__ sinT,
                      const int *__restrict__ d_pos, int pos_static, int cache_off,
                      float *__restrict__ q_out, float *__restrict__ kc, float *__restrict__ vc,
                      int max_seq) {
  extern __shared__ float v[];  // hd
  __shared__ float red[8];
  __shared__ float s_scale;
  const int hh = blockIdx.x, r = blockIdx.y;
  const int pos = (d_pos ? d_pos[0] : pos_static) + r;
  const int crow = pos + cache_off;
  const int qd = nh * hd, kvd = nkv * hd, half = hd / 2;
  const float *row = qkv + (size_t)r * ldqkv;
  if (hh >= nh + nkv) {  // V head: raw copy into the cache
    const int vh = hh - nh - nkv;
    for (int d = threadIdx.x; d < hd; d += 64)
      vc[kv_v_index(crow, vh, d, hd, max_seq)] = row[qd + kvd + vh * hd + d];
    return;
  }
  const bool is_q = hh < nh;
  const float *src = is_q ? row + hh * hd : row + qd + (hh - nh) * hd;
  const float *wn = is_q ? qn : kn;
  for (int d = threadIdx.x; d < hd; d += 64) v[d] = src[d];
  __syncthreads();
  if (wn) {
    const float ss = sumsq_vec4_order(v, hd, red);
    if (threadIdx.x == 0) s_scale = 1.0f / sqrtf(ss / (float)hd + eps);
    __syncthreads();
    const float scale = s_scale;
    for (int d = threadIdx.x; d < hd; d += 64) {
      const float t = v[d] * wn[d];
      v[d] = t * scale;
    }
    __syncthreads();
  }
  const float *cr = cosT + (size_t)pos * half, *sr = sinT + (size_t)pos * half;
  const int kh = hh - nh;
  for (int i = threadIdx.x; i < half; i += 64) {
    const float c = cr[i], sn = sr[i];
    const float x1 = v[i], x2 = v[half + i];
    const float a = x1 * c, b = x2 * sn;
    const float e = x2 * c, f = x1 * sn;
    if (is_q) {
      float *dst = q_out + (size_t)r * qd + hh * hd;
      dst[i] = a - b;
      dst[half + i] = e + f;
    } else {
      kc[kv_k_index(crow, kh, i, hd, max_seq)] = a - b;
      kc[kv_k_index(crow, kh, half + i, hd, max_seq)] = e + f;
    }
  }
}

syn_status_t launch_qk_norm_rope_kv(const float *qkv, int ldqkv, int rows, int n_heads,
                                    int n_kv, int head_dim, const float *q_norm,
                                    const float *k_norm, float eps, const float *rope_cos,
                                    const float *rope_sin, const int *d_pos, int pos_static,
                                    float *q_out, float *kcache, float *vcache, int max_seq,
                                    hipStream_t s, int cache_off) {
  hipLaunchKernelGGL(k_qk_norm_rope_kv, dim3(n_heads + 2 * n_kv, rows), dim3(64),
                     head_dim * sizeof(float), s, qkv, ldqkv, n_heads, n_kv, head_dim, q_norm,
                     k_norm, eps, rope_cos, rope_sin, d_pos, pos_static, cache_off, q_out, kcache,
                     vcache, max_seq);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

// ------------------------------------------------------------------ decode attention
// ops/attention.rs:24-147 without a window.  len >= 64 follows the
// gather + matmul_t / matmul_nn route, whose f32GemvRow (matmul.zig:223-347)
// uses @mulAdd chains for the 32/8-wide column blocks and plain a*b+c in the
// scalar tail; len < 64 follows the scalar loops (plain a*b+c).
__global__ void __launch_bounds__(256)
    k_attn_decode(const float *__restrict__ q, const float *__restrict__ kc,
                  const float *__restrict__ vc, const int *__restrict__ d_pos, int nh, int nkv,
                  int hd, float *__restrict__ scores, int max_seq, float *__restrict__ out) {
  extern __shared__ float qs[];  // hd
  __shared__ float red[64];
  __shared__ float s_sum;
  const int head = blockIdx.x;
  const int kvh = head / (nh / nkv);
  const int len = d_pos[0] + 1;
  const bool simd = len >= 64;
  float *e = scores + (size_t)head * max_seq;
  for (int d = threadIdx.x; d < hd; d += blockDim.x) qs[d] = q[head * hd + d];
  __syncthreads();
  const float scale = 1.0f / sqrtf((float)hd);
  const int n32 = len - len % 32;
  const int n8 = n32 + ((len - n32) / 8) * 8;
  float mx = -__builtin_inff();
  for (int sidx = threadIdx.x; sidx < len; sidx += blockDim.x) {
    float acc = 0.0f;
    if (simd && sidx < n8) {
      for (int d = 0; d < hd; d++)
        acc = __builtin_fmaf(qs[d], kc[kv_k_index(sidx, kvh, d, hd, max_seq)], acc);
    } else {
      for (int d = 0; d < hd; d++) {
        const float t = qs[d] * kc[kv_k_index(sidx, kvh, d, hd, max_seq)];
        acc = acc + t;
      }
    }
    const float sc = acc * scale;
    e[sidx] = sc;
    mx = fmaxf(mx, sc);
  }
  // softmax_slice (activation.rs:117-129)
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
  __syncthreads();
  mx = red[0];
  for (int i = 1; i < (int)(blockDim.x >> 6); i++) mx = fmaxf(mx, red[i]);
  for (int sidx = threadIdx.x; sidx < len; sidx += blockDim.x) e[sidx] = syn_expf(e[sidx] - mx);
  __syncthreads();
  if (threadIdx.x == 0) {
    float sum = 0.0f;
    for (int i = 0; i < len; i++) sum = sum + e[i];
    s_sum = sum;
  }
  __syncthreads();
  const float sum = s_sum;
  if (sum > 0.0f)
    for (int sidx = threadIdx.x; sidx < len; sidx += blockDim.x) e[sidx] = e[sidx] / sum;
  __syncthreads();
  const int d32 = hd - hd % 32;
  for (int d = threadIdx.x; d < hd; d += blockDim.x) {
    float acc = 0.0f;
    if (simd && d < d32) {
      for (int i = 0; i < len; i++)
        acc = __builtin_fmaf(e[i], vc[kv_v_index(i, kvh, d, hd, max_seq)], acc);
    } else {
      for (int i = 0; i < len; i++) {
        const float t = e[i] * vc[kv_v_index(i, kvh, d, hd, max_seq)];
        acc = acc + t;
      }
    }
    out[head * hd + d] = acc;
  }
}

syn_status_t launch_attention_decode(const float *q, const float *kcache, const float *vcache,
                                     const int *d_pos, int n_heads, int n_kv, int head_dim,
                                     float *scores, int max_seq, float *out, hipStream_t s) {
  hipLaunchKernelGGL(k_attn_decode, dim3(n_heads), dim3(256), head_dim * sizeof(float), s, q,
                     kcache, vcache, d_pos, n_heads, n_kv, head_dim, scores, max_seq, out);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

// ------------------------------------------------------------------ prefill attention
// syn_fused_attention per head (exports.zig:1364-1478): Q tiles of 32 rows;
// S = Q K^T and O = P V through sgemmTiled, whose element order is a
// sequential chain over k — @mulAdd inside full 8x8 micro-tiles (or in the
// f32GemvRow 32/8-wide blocks when a tile has <= 16 rows), plain a*b+c
// elsewhere — then scale, causal mask, online max/sum, normalise.  The
// keys and values are the t rows appended by this prefill (cache rows
// cache_off ..): attention.rs:200-244 attends among the new tokens only.
// grid (n_heads, t): one workgroup per (head, query row).
__device__ __forceinline__ bool sgemm_fused(int tqs, int il, int ncols, int j, bool gemv_trans_b) {
  if (tqs <= 16) {  // f32GemvRow per row (matmul.zig:142-155)
    const int n32 = ncols - ncols % 32;
    if (gemv_trans_b) {
      const int n8 = n32 + ((ncols - n32) / 8) * 8;
      return j < n8;
    }
    return j < n32;
  }
  // GOTO path: MC=256 > 32 rows, NC=4096
  const bool row_full = (tqs - (il / 8) * 8) >= 8;
  const int jc = (j / 4096) * 4096;
  const int nc = min(4096, ncols - jc);
  const bool col_full = (nc - ((j - jc) / 8) * 8) >= 8;
  return row_full && col_full;
}

__global__ void __launch_bounds__(256)
    k_attn_prefill(const float *__restrict__ q, const float *__restrict__ kc,
                   const float *__restrict__ vc, int t, int nh, int nkv, int hd, int max_seq,
                   int cache_off, float *__restrict__ out) {
  extern __shared__ float sm[];  // qs[hd] | e[t] | c[t]
  float *qs = sm, *e = sm + hd, *cj = sm + hd + t;
  __shared__ float s_mx, s_inv;
  __shared__ float cmax[256];
  const int head = blockIdx.x, i = blockIdx.y;
  const int kvh = head / (nh / nkv);
  const int qd = nh * hd;
  const int tq = (i / 32) * 32, tqs = min(32, t - tq), il = i - tq;
  for (int d = threadIdx.x; d < hd; d += blockDim.x) qs[d] = q[(size_t)i * qd + head * hd + d];
  __syncthreads();
  const float scale = 1.0f / sqrtf((float)hd);
  for (int j = threadIdx.x; j < t; j += blockDim.x) {
    float acc = 0.0f;
    if (sgemm_fused(tqs, il, t, j, true)) {
      for (int d = 0; d < hd; d++)
        acc = __builtin_fmaf(qs[d], kc[kv_k_index(cache_off + j, kvh, d, hd, max_seq)], acc);
    } else {
      for (int d = 0; d < hd; d++) {
        const float p = qs[d] * kc[kv_k_index(cache_off + j, kvh, d, hd, max_seq)];
        acc = acc + p;
      }
    }
    float sc = acc * scale;
    if (j > i) sc = -__builtin_inff();
    e[j] = sc;
  }
  __syncthreads();
  // Online max / sum in the reference's order: at position j the running max
  // is the max of e[0..j-1], so every exponential is known up front.  Thread
  // i takes the contiguous chunk i of the positions: chunk maxima, their
  // exclusive prefix, then per position the exponential the reference takes
  // there (exp(mx - x) at a new maximum, stored negated; else exp(x - mx)).
  // Only the dependent chain se = se * c + 1 / se + c stays on one thread.
  const int per = (t + (int)blockDim.x - 1) / (int)blockDim.x;
  const int j0 = min((int)threadIdx.x * per, t), j1 = min(j0 + per, t);
  float lm = -__builtin_inff();
  for (int j = j0; j < j1; j++) lm = fmaxf(lm, e[j]);
  cmax[threadIdx.x] = lm;
  __syncthreads();
  float run = -__builtin_inff();
  for (int i = 0; i < (int)threadIdx.x; i++) run = fmaxf(run, cmax[i]);
  for (int j = j0; j < j1; j++) {
    const float x = e[j];
    cj[j] = x > run ? -syn_expf(run - x) : syn_expf(x - run);
    run = fmaxf(run, x);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float mx = -__builtin_inff(), se = 0.0f;
    for (int i = 0; i < (int)blockDim.x; i++) mx = fmaxf(mx, cmax[i]);
    int j = 0;
    for (; j + 8 <= t; j += 8) {
      float c[8];
#pragma unroll
      for (int u = 0; u < 8; u++) c[u] = cj[j + u];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const float cu = fabsf(c[u]);
        const float p = se * cu;
        se = __builtin_signbit(c[u]) ? p + 1.0f : se + cu;
      }
    }
    for (; j < t; j++) {
      const float cu = fabsf(cj[j]);
      const float p = se * cu;
      se = __builtin_signbit(cj[j]) ? p + 1.0f : se + cu;
    }
    s_mx = mx;
    s_inv = 1.0f / se;
  }
  __syncthreads();
  const float mx = s_mx, inv = s_inv;
  for (int j = threadIdx.x; j < t; j += blockDim.x) e[j] = syn_expf(e[j] - mx) * inv;
  __syncthreads();
  for (int d = threadIdx.x; d < hd; d += blockDim.x) {
    float acc = 0.0f;
    if (sgemm_fused(tqs, il, hd, d, false)) {
      for (int p = 0; p < t; p++)
        acc = __builtin_fmaf(e[p], vc[kv_v_index(cache_off + p, kvh, d, hd, max_seq)], acc);
    } else {
      for (int p = 0; p < t; p++) {
        const float m = e[p] * vc[kv_v_index(cache_off + p, kvh, d, hd, max_seq)];
        acc = acc + m;
      }
    }
    out[(size_t)i * qd + head * hd + d] = acc;
  }
}

// Prefill attention on the matrix cores: one workgroup per (head, 16 query
// rows).  v_mfma_f32_16x16x4_f32 forms each element as four f32 fused
// multiply-adds in ascending k (checked bit for bit on gfx950 over 2M random
// elements with cancellation, subnormal sums, infinities and NaN), which is
// the chain of @mulAdd the reference's full micro-tiles run, so EXACT holds
// every bit of k_attn_prefill; the few rows and columns that the reference
// computes as plain a*b + c (its partial micro-tiles) are formed again that
// way by the vector units.
//   scores: a wave takes 16 positions; lane (g, m) = (lane / 16, lane % 16)
//     holds q[row m][4i + g] and k[position m][4i + g] for k-step i; K goes
//     from memory to registers, no staging.
//   softmax: 32 threads a row.  EXACT: the online sum's exponentials in
//     segments of 256 positions (run maxima by a scan), then the dependent
//     chain on one thread a row; masked positions add nothing to it.  Else max
//     and sum by shuffles.
//   P V: a wave takes 16 columns, k-steps run over the positions in order.  A
//     step's positions outside the block's range count as 0 * -0, the one
//     product that changes no sum's bits.  EXACT runs over the masked positions
//     too (0 * v is not always without effect).
// Both K and V are read 16 bytes a lane and brought into the lanes' layout by
// a transpose between the four 16-lane groups (4-byte loads in that layout
// took 4 cycles a 64-byte line each: 16 heads of 128, 128 tokens, 18 us
// against 13).
// What bounds it at short prompts is latency (loads, the softmax chain), at
// long ones reads of K and V, once per 16 rows.  Against VALU kernels that
// staged K and V through LDS (four or eight FMA for two to nine LDS reads):
// INT8 decoder, 16 heads of 128, 128 tokens 70.2 -> 12.9 us; tolerance form,
// 24 heads of 128, 256 tokens 76.1 -> 15.8 us.
constexpr int kPfRows = 16, kPfThreads = 512, kPfSeg = 256, kPfSegLd = kPfSeg + 4;

// stride of a row of scores: room for a start at any position of a group of
// four; 4 mod 64 puts a step's 16 rows x 4 positions in 64 different banks
__host__ __device__ __forceinline__ int pf_ld(int t) {
  const int w = (t + 6) & ~3;
  return (w + 59) / 64 * 64 + 4;
}

template <int HD, bool EXACT>
__global__ void __launch_bounds__(kPfThreads)
    k_attn_prefill_mfma(const float *__restrict__ q, const float *__restrict__ kc,
                        const float *__restrict__ vc, int t, int nh, int nkv, int max_seq,
                        int cache_off, float *__restrict__ out) {
  constexpr int NK = HD / 4, NW = kPfThreads / 64;
  extern __shared__ __align__(16) float sm[];  // e[16][ld] | cj[16][kPfSegLd] (EXACT)
  const int ld = pf_ld(t);
  float *e = sm, *cj = sm + kPfRows * ld;
  __shared__ __align__(16) float qs[kPfRows * (HD + 4)];
  __shared__ float s_inv[kPfRows];
  // the exp table in LDS: a per-lane lookup in it does not wait on memory
  __shared__ uint64_t etab[32];
  if (threadIdx.x < 32) etab[threadIdx.x] = syn_exp2_tab[threadIdx.x];
  // the last rows see the most positions: start with them
  const int head = blockIdx.x, i0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * kPfRows;
  const int kvh = head / (nh / nkv), qd = nh * HD;
  const int nrow = min(kPfRows, t - i0), nsc = i0 + nrow;  // row r sees i0 + r + 1 <= nsc
  const int npos = EXACT ? t : nsc;                        // positions of P V
  const int sh = cache_off & 3;                            // e[r][sh + j]: position j
  const int tid = threadIdx.x, wave = tid >> 6, m = tid & 15, g = (tid >> 4) & 3;
  const float scale = 1.0f / sqrtf((float)HD);
  const float ninf = -__builtin_inff();
  const int W = (sh + npos + 3) & ~3, steps = W / 4;
  // V of the first U steps of the wave's first columns: read before the scores,
  // which hide its latency
  constexpr int U = 16;
  const float *vp =
      vc + kv_v_index(cache_off & ~3, kvh, (wave % (HD / 16)) * 16 + m, HD, max_seq);
  f32x4 vb[U / 4];
  auto load_v = [&](int s0) {
#pragma unroll
    for (int u = 0; u < U / 4; u++)
      vb[u] = *reinterpret_cast<const f32x4 *>(vp + (size_t)min(s0 + 4 * u + g, steps - 1) *
                                                        (4 * HD));
  };
  // ---- scores
  {
    const int nt = (nsc + 15) / 16;
    float qa[NK];
    f32x4 kb[NK / 4];
    auto load_k = [&](int tile) {
      const int p = min(tile * 16 + m, t - 1);
      const float *kp = kc + kv_k_index(cache_off + p, kvh, 4 * g, HD, max_seq);
#pragma unroll
      for (int i = 0; i < NK / 4; i++) kb[i] = *reinterpret_cast<const f32x4 *>(kp + i * 1024);
    };
    // q by way of LDS: read as fragments from memory, 16 rows of 16 bytes a
    // load, it took longer than all of K
    f32x4 qv = {0.0f, 0.0f, 0.0f, 0.0f};
    const int qr = tid / NK, qc = tid % NK * 4;
    if (qr < kPfRows)
      qv = *reinterpret_cast<const f32x4 *>(q + (size_t)(i0 + min(qr, nrow - 1)) * qd +
                                            head * HD + qc);
    if (wave < nt) load_k(wave);
    if (wave < HD / 16) load_v(0);
    __builtin_amdgcn_sched_barrier(0);
    if (qr < kPfRows) *reinterpret_cast<f32x4 *>(qs + qr * (HD + 4) + qc) = qv;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NK; i++) qa[i] = qs[m * (HD + 4) + 4 * i + g];
    for (int tile = wave; tile < nt; tile += NW) {
      f32x4 kn[NK / 4];
#pragma unroll
      for (int i = 0; i < NK / 4; i++) kn[i] = groups_transposed(kb[i]);
      if (tile + NW < nt) load_k(tile + NW);
      f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int i = 0; i < NK; i++)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[i], kn[i / 4][i % 4], acc, 0, 0, 0);
      const int j = tile * 16 + m;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int row = 4 * g + r;
        if (j < nsc) e[row * ld + sh + j] = j <= i0 + row ? acc[r] * scale : ninf;
      }
    }
  }
  __syncthreads();
  // rows from r_plain on are the reference's partial micro-tile (plain a*b + c)
  const int tq = i0 & ~31, tqs = min(32, t - tq);
  const int r_plain =
      EXACT && tqs > 16 ? min(nrow, max(0, (tqs & ~7) - (i0 - tq))) : nrow;
  if constexpr (EXACT) {
    auto plain = [&](int r, int j) {
      const float *qr = q + (size_t)(i0 + r) * qd + head * HD;
      const float *kp = kc + kv_k_index(cache_off + j, kvh, 0, HD, max_seq);
      float acc = 0.0f;
#pragma unroll 8
      for (int d4 = 0; d4 < NK; d4++) {
        const f32x4 a = *reinterpret_cast<const f32x4 *>(qr + 4 * d4);
        const f32x4 b = *reinterpret_cast<const f32x4 *>(kp + d4 * 256);
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const float p = a[u] * b[u];
          acc = acc + p;
        }
      }
      e[r * ld + sh + j] = acc * scale;
    };
    for (int x = tid; x < (nrow - r_plain) * nsc; x += kPfThreads) {
      const int r = r_plain + x / nsc, j = x % nsc;
      if (j <= i0 + r) plain(r, j);
    }
    const int tc = t & 7;  // the last t % 8 columns
    if (nsc > t - tc)
      for (int x = tid; x < r_plain * tc; x += kPfThreads) {
        const int r = x / tc, j = t - tc + x % tc;
        if (j <= i0 + r) plain(r, j);
      }
    if (r_plain < nrow || nsc > t - tc) __syncthreads();
  }
  // ---- softmax: 32 threads a row
  {
    const int r = tid >> 5, part = tid & 31;
    const int vis = r < nrow ? i0 + r + 1 : 0;
    float *er = e + r * ld + sh;
    float mx = ninf, inv = 0.0f;
    if constexpr (EXACT) {
      // k_attn_prefill's order: at position j the running maximum is that of
      // the positions before it, so every exponential is known up front
      float se = 0.0f, *cr = cj + r * kPfSegLd;
      for (int s0 = 0; s0 < nsc; s0 += kPfSeg) {
        const int per = (min(kPfSeg, nsc - s0) + 31) / 32;
        const int j0 = min(s0 + part * per, vis), j1 = min(j0 + per, vis);
        float x[8], lm = ninf;
#pragma unroll
        for (int u = 0; u < 8; u++) {
          x[u] = u < per && j0 + u < j1 ? er[j0 + u] : ninf;
          lm = fmaxf(lm, x[u]);
        }
        for (int o = 1; o < 32; o <<= 1) {  // maxima of the parts up to this one
          const float v = __shfl_up(lm, o, 32);
          if (part >= o) lm = fmaxf(lm, v);
        }
        float run = __shfl_up(lm, 1, 32);
        run = part == 0 ? mx : fmaxf(mx, run);
        mx = fmaxf(mx, __shfl(lm, 31, 32));
#pragma unroll
        for (int u0 = 0; u0 < 8; u0 += 4)
          if (u0 < per) {
            float c[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
              const float y = x[u0 + u];
              const bool up = y > run;
              const float ex = syn_expf_sel(up ? run - y : y - run, etab);
              // (past the row's positions: 0, without effect on the chain)
              c[u] = j0 + u0 + u < j1 ? (up ? -ex : ex) : 0.0f;
              run = fmaxf(run, y);
            }
#pragma unroll
            for (int u = 0; u < 4; u++)
              if (u0 + u < per) cr[part * per + u0 + u] = c[u];
          }
        __syncthreads();
        if (part == 0) {
          const int n = min(kPfSeg, vis - s0);
          auto link = [&](float c) {
            const float cu = fabsf(c), pr = se * cu;
            se = __builtin_signbit(c) ? pr + 1.0f : se + cu;
          };
          f32x4 na = *reinterpret_cast<const f32x4 *>(cr);
          f32x4 nb = *reinterpret_cast<const f32x4 *>(cr + 4);
          for (int j = 0; j < n; j += 8) {
            const f32x4 a = na, b = nb;  // (the next eight: at most the row's padding)
            na = *reinterpret_cast<const f32x4 *>(cr + min(j + 8, kPfSegLd - 8));
            nb = *reinterpret_cast<const f32x4 *>(cr + min(j + 12, kPfSegLd - 4));
            const bool neg = __builtin_signbit(a.x) | __builtin_signbit(a.y) |
                             __builtin_signbit(a.z) | __builtin_signbit(a.w) |
                             __builtin_signbit(b.x) | __builtin_signbit(b.y) |
                             __builtin_signbit(b.z) | __builtin_signbit(b.w);
            if (neg) {
#pragma unroll
              for (int u = 0; u < 4; u++) link(a[u]);
#pragma unroll
              for (int u = 0; u < 4; u++) link(b[u]);
            } else {  // no new maximum: additions only
#pragma unroll
              for (int u = 0; u < 4; u++) se = se + a[u];
#pragma unroll
              for (int u = 0; u < 4; u++) se = se + b[u];
            }
          }
        }
        __syncthreads();
      }
      inv = 1.0f / __shfl(se, 0, 32);
      // (masked positions: 0 * inv)
      for (int j0 = part; j0 < vis; j0 += 128) {
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; u++)
          v[u] = syn_expf_sel(er[min(j0 + 32 * u, vis - 1)] - mx, etab) * inv;
#pragma unroll
        for (int u = 0; u < 4; u++)
          if (j0 + 32 * u < vis) er[j0 + 32 * u] = v[u];
      }
      if (part < sh) er[part - sh] = 0.0f;
      for (int j = vis + part; j < W - sh; j += 32)
        er[j] = r < nrow && j < npos ? 0.0f * inv : 0.0f;
    } else {
      for (int j = part; j < vis; j += 32) mx = fmaxf(mx, er[j]);
      for (int o = 1; o < 32; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
      float sum = 0.0f;
      for (int j0 = part; j0 < vis; j0 += 128) {
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = syn_expf_sel(er[min(j0 + 32 * u, vis - 1)] - mx, etab);
#pragma unroll
        for (int u = 0; u < 4; u++)
          if (j0 + 32 * u < vis) {
            er[j0 + 32 * u] = v[u];
            sum += v[u];
          }
      }
      if (part < sh) er[part - sh] = 0.0f;
      for (int j = vis + part; j < W - sh; j += 32) er[j] = 0.0f;
      for (int o = 1; o < 32; o <<= 1) sum += __shfl_xor(sum, o);
      if (part == 0) s_inv[r] = 1.0f / sum;
    }
  }
  __syncthreads();
  // ---- P V
  const int r_plain_v = EXACT && HD == 16 && tqs <= 16 ? 0 : r_plain;
  static_assert(HD / 16 <= NW, "one group of columns a wave");
  if (wave < HD / 16) {
    const int ct = wave;
    const float *ep = e + m * ld + g;
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int s0 = 0; s0 < steps; s0 += U) {
      f32x4 vn[U / 4];
#pragma unroll
      for (int u = 0; u < U / 4; u++) {
        const int j = 4 * (s0 + 4 * u + g) - sh;
        f32x4 v = vb[u];
#pragma unroll
        for (int c = 0; c < 4; c++) v[c] = j + c >= 0 && j + c < npos ? v[c] : -0.0f;
        vn[u] = groups_transposed(v);
      }
      if (s0 + U < steps) load_v(s0 + U);
      float a[U];
#pragma unroll
      for (int u = 0; u < U; u++) a[u] = ep[4 * min(s0 + u, steps - 1)];
#pragma unroll
      for (int u = 0; u < U; u++)
        if (s0 + u < steps)
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u], vn[u / 4][u % 4], acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int row = 4 * g + r;
      if (row < r_plain_v || (!EXACT && row < nrow))
        out[(size_t)(i0 + row) * qd + head * HD + ct * 16 + m] =
            EXACT ? acc[r] : acc[r] * s_inv[row];
    }
  }
  if constexpr (EXACT) {
    for (int x = tid; x < (nrow - r_plain_v) * HD; x += kPfThreads) {
      const int r = r_plain_v + x / HD, d = x % HD;
      const float *er = e + r * ld + sh;
      float acc = 0.0f;
#pragma unroll 8
      for (int j = 0; j < t; j++) {
        const float p = er[j] * vc[kv_v_index(cache_off + j, kvh, d, HD, max_seq)];
        acc = acc + p;
      }
      out[(size_t)(i0 + r) * qd + head * HD + d] = acc;
    }
  }
}

// the matrix-core kernel for head widths of 16, 32, 64 and 128 whose rows of
// scores fit LDS; *done says whether it took the call
template <bool EXACT>
static syn_status_t launch_prefill_mfma(const float *q, const float *kcache, const float *vcache,
                                        int t, int n_heads, int n_kv, int head_dim, int max_seq,
                                        int cache_off, float *out, hipStream_t s, bool *done) {
  const size_t shm =
      ((size_t)kPfRows * pf_ld(t) + (EXACT ? kPfRows * kPfSegLd : 0)) * sizeof(float);
  *done = (head_dim == 16 || head_dim == 32 || head_dim == 64 || head_dim == 128) &&
          shm <= 144 * 1024;
  if (!*done) return SYN_OK;
  static bool attr[4] = {false, false, false, false};
  auto run = [&](auto kern, int which) -> syn_status_t {
    if (!attr[which]) {  // more than the default 64 KiB of dynamic LDS
      SYN_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  144 * 1024));
      attr[which] = true;
    }
    SYN_LAUNCH(kern, dim3(n_heads, (t + kPfRows - 1) / kPfRows), dim3(kPfThreads), shm, s, q,
               kcache, vcache, t, n_heads, n_kv, max_seq, cache_off, out);
    SYN_LAUNCH_CHECK();
    return SYN_OK;
  };
  switch (head_dim) {
    case 16: return run(k_attn_prefill_mfma<16, EXACT>, 0);
    case 32: return run(k_attn_prefill_mfma<32, EXACT>, 1);
    case 64: return run(k_attn_prefill_mfma<64, EXACT>, 2);
    default: return run(k_attn_prefill_mfma<128, EXACT>, 3);
  }
}

// For the tolerance-graded decoders (K-quant, hybrid): the same causal
// attention over the prompt block (row i sees positions 0 .. i of the t new
// ones at cache_off), without the reference's serial order of the sum.
syn_status_t launch_attention_prefill_tol(const float *q, const float *kcache,
                                          const float *vcache, int t, int n_heads, int n_kv,
                                          int head_dim, int max_seq, float *out, hipStream_t s,
                                          int cache_off) {
  bool done;
  SYN_TRY(launch_prefill_mfma<false>(q, kcache, vcache, t, n_heads, n_kv, head_dim, max_seq,
                                     cache_off, out, s, &done));
  if (done) return SYN_OK;
  return launch_attention_prefill(q, kcache, vcache, t, n_heads, n_kv, head_dim, max_seq, nullptr,
                                  out, s, cache_off);
}

syn_status_t launch_attention_prefill(const float *q, const float *kcache, const float *vcache,
                                      int t, int n_heads, int n_kv, int head_dim, int max_seq,
                                      float *scores, float *out, hipStream_t s, int cache_off) {
  (void)scores;
  bool done;
  SYN_TRY(launch_prefill_mfma<true>(q, kcache, vcache, t, n_heads, n_kv, head_dim, max_seq,
                                    cache_off, out, s, &done));
  if (done) return SYN_OK;
  const size_t shm = (size_t)(head_dim + 2 * t) * sizeof(float);
  if (shm > 144 * 1024) {
    set_error("prefill attention: prompt too long for one workgroup's LDS rows");
    return SYN_ERR_INVALID_ARG;
  }
  static bool attr = false;
  if (!attr) {  // more than the default 64 KiB of dynamic LDS
    SYN_HIP(hipFuncSetAttribute((const void *)k_attn_prefill,
                                hipFuncAttributeMaxDynamicSharedMemorySize, 144 * 1024));
    attr = true;
  }
  hipLaunchKernelGGL(k_attn_prefill, dim3(n_heads, t), dim3(256), shm, s, q, kcache, vcache, t,
                     n_heads, n_kv, head_dim, max_seq, cache_off, out);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

// ------------------------------------------------------------------ SwiGLU + quantize
// one workgroup per row; a wide row takes 1024 threads (128 rows of 3072: 13.1
// us with 256, 6.4 with 1024)
__global__ void __launch_bounds__(1024)
    k_swiglu_quant(const float *__restrict__ gu, int ldgu, int inter, int8_t *__restrict__ hq,
                   int ldq, float *__restrict__ sh) {
  extern __shared__ float sm[];  // inter
  __shared__ float red[64];
  const int row = blockIdx.x;
  const float *g = gu + (size_t)row * ldgu, *u = g + inter;
  for (int j = threadIdx.x; j < inter; j += blockDim.x) {
    const float a = syn_silu(g[j]);
    sm[j] = a * u[j];
  }
  __syncthreads();
  quantize_row_lds(sm, inter, hq + (size_t)row * ldq, sh + row, red);
}

syn_status_t launch_swiglu_quant(const float *gu, int ldgu, int rows, int inter, int8_t *hq,
                                 int ldq, float *sh, hipStream_t s) {
  hipLaunchKernelGGL(k_swiglu_quant, dim3(rows), dim3(inter >= 1024 ? 1024 : 256),
                     inter * sizeof(float), s, gu, ldgu, inter, hq, ldq, sh);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

// ------------------------------------------------------------------ SwiGLU (f32 path)
// zig/src/ops/silu.zig:85-114 (syn_swiglu, used by the f32 decoder
// decoder_layer.rs:690-700): on the 4-aligned prefix sig = 1/(1+exp(-g)),
// h = (g*sig)*u; on the tail h = (g/(1+exp(-g)))*u.
__global__ void k_swiglu_f32(const float *__restrict__ gu, int ldgu, int inter,
                             float *__restrict__ h, int ldh) {
  const int row = blockIdx.y;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= inter) return;
  const float g = gu[(size_t)row * ldgu + i], u = gu[(size_t)row * ldgu + inter + i];
  const int n4 = inter - inter % 4;
  float t;
  if (i < n4) {
    const float sig = 1.0f / (1.0f + syn_expf(-g));
    t = g * sig;
  } else {
    t = g / (1.0f + syn_expf(-g));
  }
  h[(size_t)row * ldh + i] = t * u;
}

syn_status_t launch_swiglu_f32(const float *gu, int ldgu, int rows, int inter, float *h, int ldh,
                               hipStream_t s) {
  hipLaunchKernelGGL(k_swiglu_f32, dim3((inter + 255) / 256, rows), dim3(256), 0, s, gu, ldgu,
                     inter, h, ldh);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

// ------------------------------------------------------------------ argmax
struct Top2 {
  float v1;
  int i1;
  float v2;
};

__device__ __forceinline__ Top2 top2_merge(Top2 a, Top2 b) {
  // winner: larger value; on equal values the larger index (last max)
  const bool bw = (b.v1 > a.v1) || (b.v1 == a.v1 && b.i1 > a.i1);
  const Top2 w = bw ? b : a, l = bw ? a : b;
  Top2 r;
  r.v1 = w.v1;
  r.i1 = w.i1;
  r.v2 = fmaxf(w.v2, l.v1);
  return r;
}

__device__ Top2 block_top2(Top2 t, float *sv1, int *si1, float *sv2) {
  for (int o = 32; o > 0; o >>= 1) {
    Top2 u;
    u.v1 = __shfl_xor(t.v1, o);
    u.i1 = __shfl_xor(t.i1, o);
    u.v2 = __shfl_xor(t.v2, o);
    t = top2_merge(t, u);
  }
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    sv1[w] = t.v1;
    si1[w] = t.i1;
    sv2[w] = t.v2;
  }
  __syncthreads();
  Top2 r{sv1[0], si1[0], sv2[0]};
  for (int i = 1; i < nw; i++) r = top2_merge(r, Top2{sv1[i], si1[i], sv2[i]});
  return r;
}

__global__ void __launch_bounds__(256)
    k_argmax_stage1(const float *__restrict__ x, int n, float *pv, int *pi, float *pv2) {
  __shared__ float sv1[4], sv2[4];
  __shared__ int si1[4];
  Top2 t{-__builtin_inff(), -1, -__builtin_inff()};
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
    t = top2_merge(t, Top2{x[i], i, -__builtin_inff()});
  t = block_top2(t, sv1, si1, sv2);
  if (threadIdx.x == 0) {
    pv[blockIdx.x] = t.v1;
    pi[blockIdx.x] = t.i1;
    pv2[blockIdx.x] = t.v2;
  }
}

__global__ void __launch_bounds__(256)
    k_argmax_stage2(const float *pv, const int *pi, const float *pv2, int np, StepState *st,
                    uint32_t *history, float *mhist) {
  __shared__ float sv1[4], sv2[4];
  __shared__ int si1[4];
  Top2 t{-__builtin_inff(), -1, -__builtin_inff()};
  for (int i = threadIdx.x; i < np; i += 256) t = top2_merge(t, Top2{pv[i], pi[i], pv2[i]});
  t = block_top2(t, sv1, si1, sv2);
  if (threadIdx.x == 0) {
    const uint32_t tok = t.i1 < 0 ? 0u : (uint32_t)t.i1;
    st->token = tok;
    st->margin = t.v1 - t.v2;
    if (history) history[st->step] = tok;
    if (mhist) mhist[st->step] = t.v1 - t.v2;
  }
}

syn_status_t launch_argmax(const float *logits, int n, float *part_v, int *part_i,
                           float *part_v2, StepState *state, uint32_t *history,
                           float *margin_hist, hipStream_t s) {
  const int blocks = 256;
  hipLaunchKernelGGL(k_argmax_stage1, dim3(blocks), dim3(256), 0, s, logits, n, part_v, part_i,
                     part_v2);
  SYN_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_argmax_stage2, dim3(1), dim3(256), 0, s, part_v, part_i, part_v2, blocks,
                     state, history, margin_hist);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

__global__ void k_step_advance(StepState *st, int add_pos) {
  if (threadIdx.x == 0) {
    st->pos += add_pos;
    st->step += 1;
  }
}

syn_status_t launch_step_advance(StepState *state, int add_pos, hipStream_t s) {
  hipLaunchKernelGGL(k_step_advance, dim3(1), dim3(64), 0, s, state, add_pos);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

// zero K and V rows at position st->pos of `layers` consecutive layer caches
// (the draft forward's padding, causal_lm.rs:306-315); grid (layers)
__global__ void k_kv_zero_rows(float *__restrict__ kc, float *__restrict__ vc, size_t k_stride,
                               size_t v_stride, int nkv, int hd, int max_seq,
                               const StepState *__restrict__ st) {
  const int pos = st->pos;
  float *kl = kc + (size_t)blockIdx.x * k_stride, *vl = vc + (size_t)blockIdx.x * v_stride;
  for (int i = threadIdx.x; i < nkv * hd; i += blockDim.x) {
    const int g = i / hd, d = i - g * hd;
    kl[kv_k_index(pos, g, d, hd, max_seq)] = 0.0f;
    vl[kv_v_index(pos, g, d, hd, max_seq)] = 0.0f;
  }
}

syn_status_t launch_kv_zero_rows(float *kc, float *vc, size_t k_stride, size_t v_stride,
                                 int layers, int nkv, int hd, int max_seq, const StepState *st,
                                 hipStream_t s) {
  if (layers <= 0) return SYN_OK;
  hipLaunchKernelGGL(k_kv_zero_rows, dim3(layers), dim3(256), 0, s, kc, vc, k_stride, v_stride,
                     nkv, hd, max_seq, st);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

__global__ void k_state_init(StepState *st, StepState v) {
  if (threadIdx.x == 0) *st = v;
}

syn_status_t launch_state_init(StepState *state, int pos, uint32_t token, int step,
                               hipStream_t s) {
  hipLaunchKernelGGL(k_state_init, dim3(1), dim3(64), 0, s, state,
                     StepState{pos, token, step, 0.0f});
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

__global__ void k_state_set(StepState *st, int pos, int nhist) {
  if (threadIdx.x == 0) {
    if (pos >= 0) st->pos = pos;
    st->nhist = nhist;
  }
}

syn_status_t launch_state_set(StepState *state, int pos, int nhist, hipStream_t s) {
  hipLaunchKernelGGL(k_state_set, dim3(1), dim3(64), 0, s, state, pos, nhist);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

}  // namespace syn

__global__ void k_eval_expf(const float *__restrict__ x, float *__restrict__ y, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = syn_expf(x[i]);
}

extern "C" syn_status_t syn_hip_eval_expf(const float *d_x, float *d_y, size_t n, void *stream) {
  if (n == 0) return SYN_OK;
  if (!d_x || !d_y) return SYN_ERR_NULL_PTR;
  SYN_TRY(syn::ensure_init());
  hipLaunchKernelGGL(k_eval_expf, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     syn::pick_stream(stream), d_x, d_y, n);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}
