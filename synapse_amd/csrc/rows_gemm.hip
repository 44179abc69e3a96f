// Quantized GEMM for a few rows on the f16 matrix cores.
//
// With 9 to ~100 rows the product is bound by streaming the weights once and
// by latency: the tiled prompt kernels (kquant_gemm.hip) walk K through LDS
// with a barrier per 64 elements on a 128-row tile, and leave most of the
// tile and of the chip idle.  Here nothing passes through LDS inside the K
// loop and there is no barrier in it: a workgroup owns 32 or 64 columns of y,
// its eight waves take the 64-element steps of K in turn, and each wave
// brings its weights from HBM and its activations from L2 straight into
// registers, one step ahead, decodes the weights there and issues MFMAs.  The
// waves' sums meet in LDS once, at the end.
//
// Lane l of an MFMA fragment holds column (or row) l % 32; lanes l < 32 take
// the step's first 32 elements of K and the others its second 32, so a lane
// reads whole 16-byte planes of one block, and MFMA group g (0..3) covers
// elements 8g..8g+7 of both halves.  The activations are stored in that
// order by the conversion (one contiguous KiB per wave load); for the nibble
// formats a group holds the k order 0,2,4,6,1,3,5,7 (a dword's low nibbles,
// then its high ones).
#include <algorithm>

#include "bf16_parts.hpp"
#include "kquant.hpp"
#include "rows_gemm.hpp"

namespace syn {

namespace {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int RW = 8;        // waves per workgroup
constexpr int RNT = 64 * RW;
constexpr int KSTEP = 64;  // elements of K per step

constexpr bool nibble_order(int fmt) { return fmt != SYN_HIP_FMT_Q8_0; }

__device__ __forceinline__ uint32_t pick(const u32x4 &v, int i) {
  return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w;
}
__device__ __forceinline__ uint32_t pk(float a, float b) {
  return __builtin_bit_cast(uint32_t, f16x2{(_Float16)a, (_Float16)b});
}
__device__ __forceinline__ float ub(uint32_t v, int b) { return (float)((v >> (8 * b)) & 0xffu); }

// the stored bytes of one lane's 32 weights of a step
template <int FMT>
struct Raw;
template <>
struct Raw<SYN_HIP_FMT_Q4_0> {
  u32x4 q;
  uint16_t d;
};
template <>
struct Raw<SYN_HIP_FMT_Q8_0> {
  u32x4 q0, q1;
  uint16_t d;
};
template <>
struct Raw<SYN_HIP_FMT_Q4_K> {
  u32x4 sc, q;
};
template <>
struct Raw<SYN_HIP_FMT_Q6_K> {
  u32x4 q;
  uint2 h;
  uint16_t sc, d;
};

// block j32 = 2 step + lh of 32 elements of row rp of a panel (clamped to the
// row's last block: an odd block count has half a step of padding)
template <int FMT>
__device__ __forceinline__ void load_raw(Raw<FMT> &r, const u32x4 *__restrict__ W,
                                         const uint16_t *__restrict__ Wd, size_t panel, int rp,
                                         int B, int step, int lh) {
  if constexpr (FMT == SYN_HIP_FMT_Q4_0) {
    const size_t b = panel * B + min(2 * step + lh, B - 1);
    r.q = W[b * 64 + rp];
    r.d = Wd[b * 64 + rp];
  } else if constexpr (FMT == SYN_HIP_FMT_Q8_0) {
    const size_t b = panel * B + min(2 * step + lh, B - 1);
    r.q0 = W[(b * 2) * 64 + rp];
    r.q1 = W[(b * 2 + 1) * 64 + rp];
    r.d = Wd[b * 64 + rp];
  } else if constexpr (FMT == SYN_HIP_FMT_Q4_K) {
    const size_t b = panel * B + (step >> 2);
    r.sc = W[b * 9 * 64 + rp];
    r.q = W[(b * 9 + 1 + 2 * (step & 3) + lh) * 64 + rp];
  } else {
    const size_t b = panel * B + (step >> 2);
    const int st = step & 3, j = 2 * st + lh;
    const u32x4 *p = W + b * 13 * 64;
    r.q = p[j * 64 + rp];
    r.h = reinterpret_cast<const uint2 *>(p + (8 + st) * 64 + rp)[lh];
    r.sc = reinterpret_cast<const uint16_t *>(p + 12 * 64 + rp)[j];
    r.d = Wd[b * 64 + rp];
  }
}

// what a lane needs besides the quants, formed once per step
struct Scale {
  float a, b;  // Q4_K: scale and min; Q6_K: the two scales of 16
  f16x2 d;     // Q4_0, Q8_0: the block scale twice
};

template <int FMT>
__device__ __forceinline__ Scale scale_of(const Raw<FMT> &r, int B, int step, int lh) {
  Scale o;
  if constexpr (FMT == SYN_HIP_FMT_Q4_0) {  // IEEE f16 scales (QLinearQ4_0::gemm_ok)
    const _Float16 v =
        2 * step + lh < B ? __builtin_bit_cast(_Float16, r.d) : (_Float16)0.0f;
    o.d = f16x2{v, v};
  } else if constexpr (FMT == SYN_HIP_FMT_Q8_0) {  // every scale is an f16 value
    const _Float16 v = (_Float16)(2 * step + lh < B ? syn_f16_to_f32_rs_hw(r.d) : 0.0f);
    o.d = f16x2{v, v};
  } else if constexpr (FMT == SYN_HIP_FMT_Q4_K) {  // gguf.rs:383-417
    const float d = syn_f16_to_f32_rs_hw(r.sc.x & 0xffffu);
    const float dmin = syn_f16_to_f32_rs_hw(r.sc.x >> 16);
    const int sh = 8 * ((2 * (step & 3) + lh) & 3);  // sub-block % 4
    const uint32_t s0 = (r.sc.y >> sh) & 0xffu, s4 = (r.sc.z >> sh) & 0xffu,
                   s8 = (r.sc.w >> sh) & 0xffu;
    const bool low = (step & 3) < 2;  // sub-blocks 0-3
    const uint32_t sc = low ? s0 & 63u : (s4 & 15u) | ((s0 >> 6) << 4);
    const uint32_t mn = low ? (s4 >> 4) | ((s8 & 15u) << 4)
                            : ((s8 >> 4) | (((s0 >> 4) & 12u) << 4)) & 0xffu;
    o.a = d * (float)sc;
    o.b = dmin * (float)mn;
  } else {
    const float d = syn_f16_to_f32_rs_hw(r.d);
    o.a = (float)(int8_t)(r.sc & 0xffu) * d;
    o.b = (float)(int8_t)(r.sc >> 8) * d;
  }
  return o;
}

// the lane's eight weights of group g, each the dequantizer's value rounded
// once to f16
template <int FMT>
__device__ __forceinline__ f16x8 decode(const Raw<FMT> &r, const Scale &s, int g) {
  uint32_t o[4];
  if constexpr (FMT == SYN_HIP_FMT_Q4_0) {
    const f16x2 bias = f16x2{(_Float16)-1032.0f, (_Float16)-1032.0f};
    const uint32_t v = pick(r.q, g);
    const uint32_t l = v & 0x0f0f0f0fu, h = (v >> 4) & 0x0f0f0f0fu;
    const uint32_t p[4] = {__builtin_amdgcn_perm(0x64646464u, l, 0x04010400u),
                           __builtin_amdgcn_perm(0x64646464u, l, 0x04030402u),
                           __builtin_amdgcn_perm(0x64646464u, h, 0x04010400u),
                           __builtin_amdgcn_perm(0x64646464u, h, 0x04030402u)};
#pragma unroll
    for (int i = 0; i < 4; i++)
      o[i] = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(f16x2, p[i]) + bias) * s.d);
  } else if constexpr (FMT == SYN_HIP_FMT_Q8_0) {
    const f16x2 bias = f16x2{(_Float16)-1152.0f, (_Float16)-1152.0f};
#pragma unroll
    for (int w = 0; w < 2; w++) {
      const uint32_t u = pick(g < 2 ? r.q0 : r.q1, 2 * (g & 1) + w) ^ 0x80808080u;
      const uint32_t p01 = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u);
      const uint32_t p23 = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);
      o[2 * w] = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(f16x2, p01) + bias) * s.d);
      o[2 * w + 1] = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(f16x2, p23) + bias) * s.d);
    }
  } else if constexpr (FMT == SYN_HIP_FMT_Q4_K) {
    const uint32_t v = pick(r.q, g);
    const uint32_t l = v & 0x0f0f0f0fu, h = (v >> 4) & 0x0f0f0f0fu;
    auto val = [&](uint32_t x, int b) { return __builtin_fmaf(ub(x, b), s.a, -s.b); };
#pragma unroll
    for (int i = 0; i < 2; i++) {
      o[i] = pk(val(l, 2 * i), val(l, 2 * i + 1));
      o[2 + i] = pk(val(h, 2 * i), val(h, 2 * i + 1));
    }
  } else {
    const uint32_t v = pick(r.q, g);
    const uint32_t hw = g < 2 ? r.h.x : r.h.y;  // bytes 2g, 2g+1: two bits per element
    const uint32_t t = (g & 1) ? __builtin_amdgcn_perm(0u, hw, 0x03030202u)
                               : __builtin_amdgcn_perm(0u, hw, 0x01010000u);
    const uint32_t l = (v & 0x0f0f0f0fu) | ((t & 0x00030003u) << 4) | (t & 0x30003000u);
    const uint32_t h =
        ((v >> 4) & 0x0f0f0f0fu) | ((t & 0x000c000cu) << 2) | ((t & 0xc000c000u) >> 2);
    const float sc = g < 2 ? s.a : s.b, off = -32.0f * sc;
    auto val = [&](uint32_t x, int b) { return __builtin_fmaf(ub(x, b), sc, off); };
#pragma unroll
    for (int i = 0; i < 2; i++) {
      o[i] = pk(val(l, 2 * i), val(l, 2 * i + 1));
      o[2 + i] = pk(val(h, 2 * i), val(h, 2 * i + 1));
    }
  }
  return __builtin_bit_cast(f16x8, u32x4{o[0], o[1], o[2], o[3]});
}

// the eight waves' sums: the upper four through LDS into the lower four, then
// store(row, column, sum) of the tile's elements, one thread each
template <int MT, int NT, class Store>
__device__ __forceinline__ void sum_waves(f32x16 (&acc)[MT][NT],
                                          float (&red)[RW / 2][32 * MT][32 * NT + 8],
                                          Store store) {
  const int tid = threadIdx.x, l32 = tid & 31, lh = (tid >> 5) & 1;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  auto at = [&](int slot, int mt, int nt, int r) -> float & {
    return red[slot][32 * mt + 8 * (r >> 2) + 4 * lh + (r & 3)][32 * nt + l32];
  };
  auto put = [&](int slot) {
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int r = 0; r < 16; r++) at(slot, mt, nt, r) = acc[mt][nt][r];
  };
  if (wave >= RW / 2) put(wave - RW / 2);
  __syncthreads();
  if (wave < RW / 2) {
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[mt][nt][r] += at(wave, mt, nt, r);
    put(wave);
  }
  __syncthreads();
  for (int i = tid; i < 32 * MT * 32 * NT; i += RNT) {
    const int r = i / (32 * NT), c = i % (32 * NT);
    float t = red[0][r][c];
#pragma unroll
    for (int w = 1; w < RW / 2; w++) t += red[w][r][c];
    store(r, c, t);
  }
}

// grid (ceil(N / 32 NT), ceil(M / 32 MT), K splits, added into y)
template <int FMT, int MT, int NT>
__global__ void __launch_bounds__(RNT) __attribute__((amdgpu_waves_per_eu(2, 2)))
    k_rows_gemm(const u32x4 *__restrict__ W, const uint16_t *__restrict__ Wd, int N, int B,
                const f16x8 *__restrict__ xf, const float *__restrict__ rowmul, int M, int steps,
                int per, float *__restrict__ y, int ldy) {
  __shared__ float red[RW / 2][32 * MT][32 * NT + 8];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, lh = lane >> 5;
  const int n0 = blockIdx.x * 32 * NT, mt0 = blockIdx.y * MT;
  const int s0 = blockIdx.z * per, s1 = min(steps, s0 + per);
  // columns past N read the last panel's padding rows, tiles past M the last
  // tile (neither is stored)
  const int last = ((N + 63) >> 6) * 64 - 1, mlast = ((M + 31) >> 5) - 1;
  size_t panel[NT];
  int rp[NT];
#pragma unroll
  for (int nt = 0; nt < NT; nt++) {
    const int n = min(n0 + 32 * nt + l32, last);
    panel[nt] = (size_t)(n >> 6);
    rp[nt] = n & 63;
  }
  const f16x8 *xt[MT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
    xt[mt] = xf + (size_t)min(mt0 + mt, mlast) * steps * 256 + lane;
  f32x16 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[mt][nt][r] = 0.0f;
  struct Step {
    Raw<FMT> w[NT];
    f16x8 a[MT][4];
  };
  auto load = [&](Step &st, int step) {
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
      load_raw<FMT>(st.w[nt], W, Wd, panel[nt], rp[nt], B, step, lh);
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int g = 0; g < 4; g++) st.a[mt][g] = xt[mt][(size_t)step * 256 + g * 64];
  };
  auto mul = [&](const Step &st, int step) {
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
      const Scale sc = scale_of<FMT>(st.w[nt], B, step, lh);
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const f16x8 b = decode<FMT>(st.w[nt], sc, g);
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
          acc[mt][nt] =
              __builtin_amdgcn_mfma_f32_32x32x16_f16(st.a[mt][g], b, acc[mt][nt], 0, 0, 0);
      }
    }
  };
  // Two steps in flight; the loads past the last step repeat it.  Without
  // the scheduling barriers and the occupancy bound the compiler sinks a
  // step's loads to their use to save registers, and every step waits out a
  // whole load.  Three and four steps in flight measured the same or slower.
  auto hold = [] { __builtin_amdgcn_sched_barrier(0); };
  Step st0, st1;
  int step = s0 + wave;
  if (step < s1) {
    load(st0, step); hold();
    load(st1, min(step + RW, s1 - 1)); hold();
    while (true) {
      mul(st0, step);
      step += RW;
      if (step >= s1) break;
      load(st0, min(step + RW, s1 - 1)); hold();
      mul(st1, step);
      step += RW;
      if (step >= s1) break;
      load(st1, min(step + RW, s1 - 1)); hold();
    }
  }
  const bool atomic = gridDim.z > 1;
  sum_waves<MT, NT>(acc, red, [&](int r, int c, float t) {
    const int m = mt0 * 32 + r, n = n0 + c;
    if (m >= M || n >= N) return;
    const float v = t * rowmul[m];
    if (atomic) atomicAdd(&y[(size_t)m * ldy + n], v);
    else y[(size_t)m * ldy + n] = v;
  });
}

// The same from rows kept whole (bf16_parts.hpp) against Q4_0's levels: a step
// is one block, its dot six MFMAs, scaled in f32 into the sum.  Lane l < 32
// holds dwords 0 and 1 of a block's levels, the others 2 and 3, so the
// activations of MFMA j are elements 8 (2 lh + j) .. +7.  PF steps in flight.
// Bound by the activations' way from L2, six bytes an element for every tile of
// columns (1024 -> 13312, 64 rows 14.5 us, 512 rows 81), and on small grids by a
// wave's chain of loads and MFMAs (1024 -> 1024, 64 rows 6.2 us).  Operands of two
// f16, which round the activations to 22 bits, took 13.9, 71.6 and 7.0.
// grid (ceil(N / 32 NT), ceil(M / 32 MT), K splits); split z writes y + z zs
template <int MT, int NT, int PF>
__global__ void __launch_bounds__(RNT) __attribute__((amdgpu_waves_per_eu(2, 2)))
    k_rows_gemm_parts(const uint2 *__restrict__ W, const uint16_t *__restrict__ Wd, int N, int B,
                      const bf16x8 *__restrict__ xf, int M, int per, float *__restrict__ y,
                      int ldy, size_t zs) {
  __shared__ float red[RW / 2][32 * MT][32 * NT + 8];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, lh = lane >> 5;
  const int n0 = blockIdx.x * 32 * NT, mt0 = blockIdx.y * MT;
  const int s0 = blockIdx.z * per, s1 = min(B, s0 + per);
  const int last = ((N + 63) >> 6) * 64 - 1, mlast = ((M + 31) >> 5) - 1;
  size_t at[NT];
#pragma unroll
  for (int nt = 0; nt < NT; nt++) {
    const int n = min(n0 + 32 * nt + l32, last);
    at[nt] = (size_t)(n >> 6) * B * 64 + (n & 63);
  }
  const bf16x8 *xt[MT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
    xt[mt] = xf + (size_t)min(mt0 + mt, mlast) * B * 384 + lane;
  f32x16 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[mt][nt][r] = 0.0f;
  struct Step {
    uint2 q[NT];
    uint16_t d[NT];
    bf16x8 a[MT][2][3];
  };
  auto load = [&](Step &st, int b) {
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
      st.q[nt] = W[(at[nt] + (size_t)b * 64) * 2 + lh];
      st.d[nt] = Wd[at[nt] + (size_t)b * 64];
    }
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int i = 0; i < 3; i++) st.a[mt][j][i] = xt[mt][(size_t)b * 384 + (j * 3 + i) * 64];
  };
  auto mul = [&](const Step &st) {
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
      const bf16x8 w[2] = {q4_levels(st.q[nt].x), q4_levels(st.q[nt].y)};
      const float d = (float)__builtin_bit_cast(_Float16, st.d[nt]);
      f32x16 dot[MT];
#pragma unroll
      for (int mt = 0; mt < MT; mt++) dot[mt] = f32x16{};
#pragma unroll
      for (int i = 2; i >= 0; i--)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
          for (int mt = 0; mt < MT; mt++)
            dot[mt] =
                __builtin_amdgcn_mfma_f32_32x32x16_bf16(st.a[mt][j][i], w[j], dot[mt], 0, 0, 0);
#pragma unroll
      for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int r = 0; r < 16; r++)
          acc[mt][nt][r] = __builtin_fmaf(dot[mt][r], d, acc[mt][nt][r]);
    }
  };
  auto hold = [] { __builtin_amdgcn_sched_barrier(0); };
  Step st[PF];
  int b = s0 + wave;
  if (b < s1) {
#pragma unroll
    for (int u = 0; u < PF; u++) {
      // a wave of a short K has fewer steps than that (with 64 x 64 tiles it has
      // not, and the branch would cost registers)
      if (MT * NT == 4 || b + u * RW < s1) load(st[u], min(b + u * RW, s1 - 1));
      hold();
    }
    for (bool more = true; more;) {
#pragma unroll
      for (int u = 0; u < PF; u++) {
        mul(st[u]);
        b += RW;
        if (b >= s1) {
          more = false;
          break;
        }
        load(st[u], min(b + (PF - 1) * RW, s1 - 1));
        hold();
      }
    }
  }
  y += blockIdx.z * zs;
  sum_waves<MT, NT>(acc, red, [&](int r, int c, float t) {
    const int m = mt0 * 32 + r, n = n0 + c;
    if (m < M && n < N) y[(size_t)m * ldy + n] = t * kPartsDown;
  });
}

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
// PERM: the nibble formats' k order 0,2,4,6,1,3,5,7
template <bool PERM>
__device__ __forceinline__ void frag_put(f16x8 *__restrict__ xf, int steps, int m, int c,
                                         const float (&v)[8]) {
  constexpr int ord[8] = {0, 2, 4, 6, 1, 3, 5, 7};
  f16x8 h;
#pragma unroll
  for (int i = 0; i < 8; i++) h[i] = (_Float16)v[PERM ? ord[i] : i];
  // step c / 8, half (c / 4) % 2, group c % 4
  const size_t at = ((size_t)(m >> 5) * steps + (c >> 3)) * 4 + (c & 3);
  xf[at * 64 + ((c >> 2) & 1) * 32 + (m & 31)] = h;
}

// One workgroup per row (the padding rows of the last tile are zeros): the
// row scale, then chunk c of eight values to its lane's place.  A row of
// up to 16384 elements is read once, into registers.
constexpr int FNT = 512;

template <bool PERM>
__global__ void __launch_bounds__(FNT)
    k_rows_frag(const float *__restrict__ x, int ldx, int M, int K, int steps,
                f16x8 *__restrict__ xf, float *__restrict__ rowmul, float *__restrict__ y0,
                int ldy, int ny) {
  __shared__ float red[FNT / 64];
  constexpr int R = 2048 / FNT;  // chunks kept in registers per thread
  const int m = blockIdx.x, tid = threadIdx.x, chunks = K >> 3;
  if (y0 && m < M)
    for (int c = tid * 4; c < ny; c += 4 * FNT) {
      float *p = y0 + (size_t)m * ldy + c;
      if (c + 4 <= ny) *reinterpret_cast<float4 *>(p) = float4{0.0f, 0.0f, 0.0f, 0.0f};
      else
        for (int i = 0; i < ny - c; i++) p[i] = 0.0f;
    }
  const float *xr = x + (size_t)min(m, M - 1) * ldx;
  auto get = [&](int c, float(&v)[8]) {
    const float4 a = *reinterpret_cast<const float4 *>(xr + 8 * c);
    const float4 b = *reinterpret_cast<const float4 *>(xr + 8 * c + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  };
  float keep[R][8];
  float mx = 0.0f;
  auto fold = [&](const float(&v)[8]) {
#pragma unroll
    for (int i = 0; i < 8; i++) mx = fmaxf(mx, fabsf(v[i]));
  };
#pragma unroll
  for (int j = 0; j < R; j++) {
    const int c = tid + FNT * j;
    if (c < chunks) {
      get(c, keep[j]);
      fold(keep[j]);
    }
  }
  for (int c = tid + FNT * R; c < chunks; c += FNT) {
    float v[8];
    get(c, v);
    fold(v);
  }
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  if ((tid & 63) == 0) red[tid >> 6] = mx;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < FNT / 64; i++) mx = fmaxf(mx, red[i]);
  float up, down;
  frag_row_scale(mx, &up, &down);
  if (tid == 0) rowmul[m] = down;
  auto put = [&](int c, const float(&v)[8]) {
    float t[8];
#pragma unroll
    for (int i = 0; i < 8; i++) t[i] = m < M ? v[i] * up : 0.0f;
    frag_put<PERM>(xf, steps, m, c, t);
  };
#pragma unroll
  for (int j = 0; j < R; j++)
    if (tid + FNT * j < chunks) put(tid + FNT * j, keep[j]);
  for (int c = tid + FNT * R; c < chunks; c += FNT) {
    float v[8];
    get(c, v);
    put(c, v);
  }
  const float zero[8] = {};
  for (int c = chunks + tid; c < 8 * steps; c += FNT) put(c, zero);
}


// f32 rows -> parts, a thread per chunk of eight values
__global__ void __launch_bounds__(256)
    k_rows_parts(const float *__restrict__ x, int ldx, int M, int chunks,
                 bf16x8 *__restrict__ xf) {
  const int c = blockIdx.x * 256 + threadIdx.x, m = blockIdx.y;
  if (c >= chunks) return;
  float v[8] = {};
  if (m < M) {
    const float4 *p = reinterpret_cast<const float4 *>(x + (size_t)m * ldx + 8 * c);
    const float4 a = p[0], b = p[1];
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  }
  parts_put(xf, chunks >> 2, m, c, v);
}

// Columns per workgroup and K splits (at least two steps per wave) with the
// least time by this count, in steps of a 32-column wave (~0.8 us each): 256
// CUs take one workgroup at a time, a workgroup costs four steps beside its
// own, a step of 64 columns 1.75 of 32, and 250,000 atomic adds of K splits
// one.  (8192 -> 2048, Q8_0: 256 rows 24.0 us in 256 workgroups of 32 columns,
// 512 rows 36.6 in 256 of 64; 384 rows 39.0 in 384 of 32, 31.7 in 192 of 64.
// 3072 -> 3072, 384 rows: 27 us in 288 of 64, 35 in two splits of them.)  parts:
// one tile of 32 rows a workgroup while that is one round of workgroups (64 rows,
// 1024 -> 3072 6.3 us, with two tiles 9.2), and K splits down to one such step, two
// blocks, per wave (16 rows, 1024 -> 1024 4.4 us in two, 6.0 unsplit).
struct Shape {
  int mt, nt, kz, per;
};
Shape shape_of(const RowsGemm &g, size_t m, int kz_max, bool parts) {
  Shape o{};
  const int steps = (int)cdiv(g.k, KSTEP);
  o.mt = m > 32 && !(parts && cdiv(g.n, 32) * cdiv(m, 32) <= 256) ? 2 : 1;
  const int tiles_m = (int)cdiv(m, (size_t)(32 * o.mt));
  float best = 0.0f;
  for (int nt = 1; nt <= 2; nt++) {
    const size_t tiles = cdiv(g.n, (size_t)(32 * nt)) * tiles_m;
    for (int kz = 1; kz <= std::min(kz_max, std::max(1, steps / (parts ? RW : 2 * RW))); kz++) {
      const float own = (float)cdiv((size_t)steps, (size_t)(RW * kz)) * (nt == 2 ? 1.75f : 1.0f);
      const float adds = kz > 1 ? (float)m * (float)g.n * (float)kz / 250000.0f : 0.0f;
      const float cost = (float)cdiv(tiles * kz, 256) * (4.0f + own) + adds;
      if (best == 0.0f || cost < best) {
        best = cost;
        o.nt = nt;
        o.kz = kz;
      }
    }
  }
  o.per = (int)cdiv((size_t)steps, (size_t)o.kz);
  o.kz = (int)cdiv((size_t)steps, (size_t)o.per);
  return o;
}

size_t frag_halfs(size_t m, size_t k) { return round_up(m, 32) * round_up(k, KSTEP); }
float *frag_scales(void *xf, size_t m, size_t k) {
  return reinterpret_cast<float *>(static_cast<_Float16 *>(xf) + frag_halfs(m, k));
}

dim3 grid_of(const RowsGemm &g, const Shape &o, size_t m) {
  return dim3((unsigned)cdiv(g.n, (size_t)(32 * o.nt)), (unsigned)cdiv(m, (size_t)(32 * o.mt)),
              (unsigned)o.kz);
}
template <int FMT>
void go(const RowsGemm &g, const Shape &o, const void *xf, size_t m, float *y, size_t ldy,
        hipStream_t s) {
  const auto kern = o.mt == 1 ? (o.nt == 1 ? k_rows_gemm<FMT, 1, 1> : k_rows_gemm<FMT, 1, 2>)
                              : (o.nt == 1 ? k_rows_gemm<FMT, 2, 1> : k_rows_gemm<FMT, 2, 2>);
  hipLaunchKernelGGL(kern, grid_of(g, o, m), dim3(RNT), 0, s, static_cast<const u32x4 *>(g.W),
                     g.Wd, (int)g.n, g.blocks, static_cast<const f16x8 *>(xf),
                     frag_scales(const_cast<void *>(xf), m, g.k), (int)m,
                     (int)cdiv(g.k, KSTEP), o.per, y, (int)ldy);
}

}  // namespace

size_t rows_frag_bytes(size_t m, size_t k) {
  return frag_halfs(m, k) * 2 + round_up(m, 32) * sizeof(float);
}

size_t rows_parts_bytes(size_t m, size_t k) { return round_up(m, 32) * k * 6; }

// Where the line to the tiled kernels lies (whole calls, us, here against
// tiled).
//  - Up to 64 rows always: 14336 -> 4096 x 64 rows Q8_0 24 against 42; Q4_K 3072
//    -> 32000 39 against 68, Q6_K 3072 -> 128256 149 against 250.
//  - Up to 128 rows, each 64 of which decode the weights again: 4096 -> 14336 x
//    128 34 against 42, Q4_K 3072 -> 32000 67 against 69.  Not on a short K
//    where the tiled kernel's columns of 128 fill one or two rounds of 256 CUs
//    (128 rows, 1024 -> 32768 Q8_0 31 against 28, Q4_K 34 against 30, 1024 ->
//    28672 Q4_K 0.85 times as fast, 1536 -> 32768 0.94, 2048 -> 30720 0.98, 1024
//    -> 24576 and 49152, where the last round is half empty, 1.1 to 1.2; Q4_0
//    0.97 and more everywhere).
//  - To 256 rows for n <= 8192: 3072 -> 8192 30 against 34, 14336 -> 4096 52
//    against 57, 14336 -> 7168 1.07 to 1.5 times as fast (2048 -> 16384 43 against
//    31).  At n = 8192 the tiled kernel's two K splits fill 256 CUs: 14336 -> 8192 x
//    192 Q8_0 100 against 86, 256 Q4_K 114 against 100 (Q4_0 84 against 87).
//  - To 512 rows while m n <= 1.6e6: 14336 -> 4096 x 384 88 against 99, 8192 ->
//    2048 x 512 36 against 41 (14336 -> 4096 x 512 97 against 90, 3072 -> 8192 x
//    512 49 against 39).
//  - To 1024 rows while m n k <= 2.2e9: 1024 -> 2048 x 1024 20 against 27, 2048 ->
//    1024 x 1024 18 against 27 (14336 -> 1024 x 768 73 against 58); for Q8_0, whose
//    tiled kernel is the fastest, 1.5e9 at K of 4096 to 8192 (8192 -> 256 x 1024
//    40 against 36, x 768 32 against 33).
bool rows_gemm_fits(int fmt, bool q8_exact, size_t m, size_t n, size_t k) {
  if (fmt == SYN_HIP_FMT_Q8_0 && !q8_exact) return false;
  if (m <= 64) return true;
  if (m <= 128) {
    const size_t tiles = cdiv(n, 128), rounds = cdiv(tiles, 256);
    const bool full = rounds <= 2 && 8 * tiles >= 7 * 256 * rounds;
    return fmt == SYN_HIP_FMT_Q4_0 || !full || k > 1536;
  }
  if (m <= 256 && n <= 8192) return fmt == SYN_HIP_FMT_Q4_0 || n <= 7168 || k < 8192;
  if (m <= 512 && m * n <= 1600000) return true;
  const bool tiled_q8 = fmt == SYN_HIP_FMT_Q8_0 && k > 4096 && k <= 8192;
  return m <= 1024 && m * n * k <= (tiled_q8 ? 1500000000u : 2200000000u);
}

// More than two f32 adds into a cleared element depend on their order; two do
// not.  Where the tiled kernels take at most two K splits (128 tiles of 128 x
// 128), so does this one, and the bits of such a call repeat
int rows_gemm_splits(const RowsGemm &g, size_t m) {
  const bool repeats = cdiv(g.n, 128) * cdiv(m, 128) >= 128;
  return shape_of(g, m, repeats ? 2 : kRowsMaxSplit, false).kz;
}
int rows_parts_splits(const RowsGemm &g, size_t m) {
  return shape_of(g, m, kRowsMaxSplit, true).kz;
}

syn_status_t launch_rows_frag(int fmt, const float *x, size_t ldx, size_t m, size_t k, void *xf,
                              float *y0, size_t ldy, size_t ny, hipStream_t s) {
  if (ldx % 4 || k % 8) {
    set_error("GEMM activation stride must be a multiple of 4 floats and K of 8");
    return SYN_ERR_SHAPE_MISMATCH;
  }
  const auto kern = nibble_order(fmt) ? k_rows_frag<true> : k_rows_frag<false>;
  hipLaunchKernelGGL(kern, dim3((unsigned)round_up(m, 32)), dim3(FNT), 0, s, x, (int)ldx, (int)m,
                     (int)k, (int)cdiv(k, KSTEP), static_cast<f16x8 *>(xf), frag_scales(xf, m, k),
                     y0, (int)ldy, (int)ny);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

syn_status_t launch_rows_parts(const float *x, size_t ldx, size_t m, size_t k, void *xf,
                               hipStream_t s) {
  if (ldx % 4 || k % 32) {
    set_error("GEMM activation stride must be a multiple of 4 floats and K of 32");
    return SYN_ERR_SHAPE_MISMATCH;
  }
  const dim3 grid((unsigned)cdiv(k / 8, 256), (unsigned)round_up(m, 32));
  hipLaunchKernelGGL(k_rows_parts, grid, dim3(256), 0, s, x, (int)ldx, (int)m, (int)(k / 8),
                     static_cast<bf16x8 *>(xf));
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

syn_status_t launch_rows_gemm(const RowsGemm &g, const void *xf, size_t m, int kz, float *y,
                              size_t ldy, hipStream_t s) {
  const Shape o = shape_of(g, m, kz, false);
  switch (g.fmt) {
    case SYN_HIP_FMT_Q4_0: go<SYN_HIP_FMT_Q4_0>(g, o, xf, m, y, ldy, s); break;
    case SYN_HIP_FMT_Q8_0: go<SYN_HIP_FMT_Q8_0>(g, o, xf, m, y, ldy, s); break;
    case SYN_HIP_FMT_Q4_K: go<SYN_HIP_FMT_Q4_K>(g, o, xf, m, y, ldy, s); break;
    case SYN_HIP_FMT_Q6_K: go<SYN_HIP_FMT_Q6_K>(g, o, xf, m, y, ldy, s); break;
    default: return SYN_ERR_INVALID_ARG;
  }
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

syn_status_t launch_rows_gemm_parts(const RowsGemm &g, const void *xf, size_t m, int kz, float *y,
                                    size_t ldy, size_t zs, hipStream_t s) {
  if (g.fmt != SYN_HIP_FMT_Q4_0 || g.k % 32) return SYN_ERR_INVALID_ARG;
  const Shape o = shape_of(g, m, kz, true);
  const auto kern = o.mt == 1 ? (o.nt == 1 ? k_rows_gemm_parts<1, 1, 4> : k_rows_gemm_parts<1, 2, 4>)
                              : (o.nt == 1 ? k_rows_gemm_parts<2, 1, 3> : k_rows_gemm_parts<2, 2, 2>);
  hipLaunchKernelGGL(kern, grid_of(g, o, m), dim3(RNT), 0, s, static_cast<const uint2 *>(g.W),
                     g.Wd, (int)g.n, g.blocks, static_cast<const bf16x8 *>(xf), (int)m, 2 * o.per,
                     y, (int)ldy, zs);
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

}  // namespace syn
