// CombinedSampler on the device (generation/sampler.rs:152-259):
// repetition penalty -> temperature -> top-k -> top-p -> softmax + draw.
//
// Two launches.  k_sample_prep spreads what is elementwise over the chip: the
// repetition penalty, the temperature and the maximum of every 64 consecutive
// logits.  k_sample, one workgroup of 1024 threads, selects from there.  Every
// float operation is the reference's, in its order: the sums of
// softmax_inplace and top_p_filter and the categorical draw are sequential in
// index (or sorted-probability) order over the list of candidates (the finite
// logits after top-k, in index order; the other logits contribute exact
// zeros).  (One workgroup for everything read the 608 KB of 151936 logits
// five times through one CU, ~150 dependent rounds each: 380 us for top-k 50 +
// top-p 0.95, 36 now.)
//
// top-k: at least k values are >= L, the k-th largest of the 64-groups' maxima
// (found by bisection over the order of the value keys), and they sit in the
// groups whose maximum is >= L: only those are read.  Up to kSortMax
// candidates are sorted in LDS and everything after stays there.  More of
// them, NaN logits or an L of -inf take the general route: the k-th largest of
// the threads' maxima, then a bisection over all values.  top-p sorts the
// candidates by probability (descending, index ascending among equal
// probabilities): up to kSortMax of them with a bitonic sort in LDS, more
// (top-p without top-k over a large vocabulary) with a stable radix sort in
// global memory, one bit per pass over the candidates' list.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "reduce_order.hpp"
#include "sampler.hpp"

namespace syn {

constexpr int kSampNT = 1024;
constexpr int kSortMax = 4096;

// float -> unsigned key with the same order (-0 below +0)
__device__ __forceinline__ uint32_t fkey(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float fkey_inv(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// block-wide sum / max of one value per thread (every thread gets it)
__device__ int block_sum_i(int v, int *red) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  int s = 0;
  for (int i = 0; i < kSampNT / 64; i++) s += red[i];
  return s;
}

// argmax with sampler.rs:217-224's tie rule (the last maximum wins): the
// largest value, the largest index among equal values
__device__ uint32_t block_argmax(const float *w, int V, float *redf, int *redi) {
  float bv = -__builtin_inff();
  int bi = -1;
  for (int i = threadIdx.x; i < V; i += kSampNT) {
    const float x = w[i];
    if (bi < 0 || !(x < bv)) {
      bv = x;
      bi = i;
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(bv, o);
    const int oi = __shfl_xor(bi, o);
    if (oi >= 0 && (bi < 0 || ov > bv || (ov == bv && oi > bi))) {
      bv = ov;
      bi = oi;
    }
  }
  const int w_ = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    redf[w_] = bv;
    redi[w_] = bi;
  }
  __syncthreads();
  float rv = redf[0];
  int ri = redi[0];
  for (int i = 1; i < kSampNT / 64; i++) {
    const float ov = redf[i];
    const int oi = redi[i];
    if (oi >= 0 && (ri < 0 || ov > rv || (ov == rv && oi > ri))) {
      rv = ov;
      ri = oi;
    }
  }
  return ri < 0 ? 0u : (uint32_t)ri;
}

// ascending bitonic sort of n (a power of two <= kSortMax) keys in LDS
__device__ void bitonic_sort(unsigned long long *buf, int n) {
  for (int k = 2; k <= n; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = threadIdx.x; i < n; i += kSampNT) {
        const int ixj = i ^ j;
        if (ixj > i) {
          const unsigned long long a = buf[i], b = buf[ixj];
          const bool asc = (i & k) == 0;
          if ((a > b) == asc) {
            buf[i] = b;
            buf[ixj] = a;
          }
        }
      }
      __syncthreads();
    }
  }
}

// ascending order of the n different keys in buf, padded with ~0 to the n2 the
// sort network takes.  Up to one key per thread: each finds its rank among
// all (a whole call with top-k 50 and top-p: 36 us, 44 with the network's ~28
// barriers in each of the three sorts)
__device__ void sort_keys(unsigned long long *buf, int n, int n2) {
  if (n <= kSampNT) {
    const int i = threadIdx.x;
    const unsigned long long e = i < n ? buf[i] : 0;
    int r = 0;
    if (i < n)
      for (int j = 0; j < n; j++) r += buf[j] < e ? 1 : 0;
    __syncthreads();
    if (i < n) buf[r] = e;
    __syncthreads();
    return;
  }
  for (int i = n + threadIdx.x; i < n2; i += kSampNT) buf[i] = ~0ull;
  __syncthreads();
  bitonic_sort(buf, n2);
}

// Write the entries of w[0..V) that satisfy keep(value), in index order, to
// cidx/cval; returns their count (every thread).  Wave w owns the w-th
// contiguous part and reads it 64 values at a time: one pass counts, the
// second places (a contiguous part per thread reads each line 16 times).
template <class Keep>
__device__ int compact(const float *w, int V, Keep keep, uint32_t *cidx, float *cval, int *red) {
  constexpr int NW = kSampNT / 64;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int per = (((V + NW - 1) / NW) + 63) & ~63;
  const int b = min(V, wave * per), e = min(V, b + per);
  int c = 0;
#pragma unroll 8
  for (int i = b; i < e; i += 64) {
    const bool k = i + lane < e && keep(w[min(i + lane, V - 1)]);
    c += __popcll(__ballot(k));
  }
  __syncthreads();
  if (lane == 0) red[wave] = c;
  __syncthreads();
  int off = 0, total = 0;
  for (int i = 0; i < NW; i++) {
    if (i < wave) off += red[i];
    total += red[i];
  }
#pragma unroll 4
  for (int i = b; i < e; i += 64) {
    const float x = w[min(i + lane, V - 1)];
    const bool k = i + lane < e && keep(x);
    const unsigned long long m = __ballot(k);
    if (k) {
      const int at = off + __popcll(m & ((1ull << lane) - 1));
      cidx[at] = (uint32_t)(i + lane);
      cval[at] = x;
    }
    off += __popcll(m);
  }
  __syncthreads();
  return total;
}

// exclusive prefix sum of one int per thread over the block; *total gets the
// sum (every thread)
__device__ int block_excl_scan(int v, int *scan, int *total) {
  scan[threadIdx.x] = v;
  __syncthreads();
  for (int o = 1; o < kSampNT; o <<= 1) {
    const int t = threadIdx.x >= o ? scan[threadIdx.x - o] : 0;
    __syncthreads();
    scan[threadIdx.x] += t;
    __syncthreads();
  }
  *total = scan[kSampNT - 1];
  const int r = scan[threadIdx.x] - v;
  __syncthreads();
  return r;
}

// Stable ascending sort of the n (key, index) pairs in (ka, va) by the key
// bits below `bits`: one stable partition per bit (zeros before ones, each
// in their order), ping-ponging with (kb, vb).  Thread t owns a contiguous
// range, so a block scan of the zero counts places every element.  Returns
// the buffer pair that holds the result (0: ka/va, 1: kb/vb).
__device__ int radix_sort_global(uint32_t *ka, uint32_t *va, uint32_t *kb, uint32_t *vb, int n,
                                 int bits, int *scan) {
  const int chunk = (n + kSampNT - 1) / kSampNT;
  const int b = min(n, (int)threadIdx.x * chunk), e = min(n, b + chunk);
  int cur = 0;
  for (int bit = 0; bit < bits; bit++) {
    const uint32_t *ks = cur ? kb : ka, *vs = cur ? vb : va;
    uint32_t *kd = cur ? ka : kb, *vd = cur ? va : vb;
    int z = 0;
    for (int i = b; i < e; i++) z += ((ks[i] >> bit) & 1u) ? 0 : 1;
    int zeros;
    int zo = block_excl_scan(z, scan, &zeros);
    int oo = zeros + (b - zo);  // ones before this range: elements before it minus zeros
    for (int i = b; i < e; i++) {
      const uint32_t k = ks[i], v = vs[i];
      const int d = ((k >> bit) & 1u) ? oo++ : zo++;
      kd[d] = k;
      vd[d] = v;
    }
    __syncthreads();
    cur ^= 1;
  }
  return cur;
}

// Sequential sums over a list of any length: the list passes through LDS
// kStream values at a time, wave 0 adds them in order (wave_seq_sum_long)
// while the other waves bring the next ones.  get(i): value i of the list.
// With stop set the walk ends in the block of values where the running sum
// first satisfies stop(sum) and returns that index (n if none does).
constexpr int kStream = 4096;

template <class Get, class Stop>
__device__ int stream_seq(int n, Get get, Stop stop, bool stops, float *buf, float *slot, int *islot,
                          float *sum_out) {
  const int tid = threadIdx.x;
  float acc = 0.0f;  // of wave 0
  for (int i = tid; i < min(n, kStream); i += kSampNT) buf[i] = get(i);
  if (tid < 2) islot[tid] = n;  // block c writes its stop to islot[c % 2]
  __syncthreads();
  int cur = 0;
  for (int c0 = 0; c0 < n; c0 += kStream, cur ^= 1) {
    const int cnt = min(kStream, n - c0);
    const float *v = buf + cur * kStream;
    if (tid < 64) {
      const float before = acc;
      acc = wave_seq_sum_long(v, cnt, acc);
      // the sums never fall, so a block whose end does not stop the walk
      // holds no stop (a NaN at its end may follow one)
      if (stops && tid == 0 && (stop(acc) || acc != acc) && before == before) {
        float cum = before;
        for (int i = 0; i < cnt; i++) {
          cum += v[i];
          if (stop(cum)) {
            islot[cur] = c0 + i;
            break;
          }
        }
      }
    } else {
      const int c1 = c0 + kStream;
      for (int i = tid - 64; i < min(kStream, n - c1); i += kSampNT - 64)
        buf[(cur ^ 1) * kStream + i] = get(c1 + i);
    }
    __syncthreads();
    // (read here and written again two barriers later at the earliest)
    if (stops && islot[cur] < n) break;
  }
  const int at = min(islot[0], islot[1]);
  if (tid == 0) slot[0] = acc;
  __syncthreads();
  if (sum_out) *sum_out = slot[0];
  return at;
}

struct NoStop {
  __device__ bool operator()(float) const { return false; }
};

// softmax's exponentials exp(v - mx) in place (all threads), then their
// sequential sum in list order; every thread gets the sum
__device__ float exp_then_seq_sum(float *v, int n, float mx, float *buf, float *slot, int *islot) {
#pragma unroll 4
  for (int i = threadIdx.x; i < n; i += kSampNT) v[i] = syn_expf(v[i] - mx);
  __syncthreads();
  float s;
  stream_seq(n, [v](int i) { return v[i]; }, NoStop{}, false, buf, slot, islot, &s);
  return s;
}

// block-wide maximum of list values (-inf where there is none)
__device__ float block_maxf(float mx, float *redf) {
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) redf[threadIdx.x >> 6] = mx;
  __syncthreads();
  mx = redf[0];
  for (int i = 1; i < kSampNT / 64; i++) mx = fmaxf(mx, redf[i]);
  return mx;
}

constexpr int kGroup = 64, kPrepNT = 512, kPrepPer = 1024;

// w = the logits after the repetition penalty (sampler.rs:132-149: once per
// occurrence in the history, so a count is enough) and, above temperature 0,
// times its reciprocal; gmax = the maximum of each 64 values, NaN if one is
__global__ void __launch_bounds__(kPrepNT)
    k_sample_prep(const float *__restrict__ logits, int V, const uint32_t *__restrict__ hist,
                  int nh_arg, SampleArgs a, const StepState *__restrict__ st,
                  float *__restrict__ w, float *__restrict__ gmax) {
  __shared__ int cnt[kPrepPer];
  const int b0 = blockIdx.x * kPrepPer, tid = threadIdx.x;
  constexpr int R = kPrepPer / kPrepNT;
  float x[R];
#pragma unroll
  for (int j = 0; j < R; j++) x[j] = logits[min(b0 + tid + j * kPrepNT, V - 1)];
  if (a.apply_rep) {
    const int nh = st ? (st->nhist >= 0 ? st->nhist : st->step) : nh_arg;
    for (int i = tid; i < kPrepPer; i += kPrepNT) cnt[i] = 0;
    __syncthreads();
    for (int j = tid; j < nh; j += kPrepNT) {
      const uint32_t idx = hist[j];
      if (idx < (uint32_t)V && idx - (uint32_t)b0 < (uint32_t)kPrepPer) atomicAdd(&cnt[idx - b0], 1);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < R; j++)
      for (int c = cnt[tid + j * kPrepNT]; c > 0; c--) x[j] = x[j] > 0.0f ? x[j] / a.rep : x[j] * a.rep;
  }
#pragma unroll
  for (int j = 0; j < R; j++) {
    const int i = b0 + tid + j * kPrepNT;
    if (a.temperature > 0.0f) x[j] = x[j] * a.inv_t;
    if (i < V) w[i] = x[j];
    float mx = i < V ? x[j] : -__builtin_inff();
    const bool nan = __ballot(mx != mx) != 0;
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    if ((tid & 63) == 0 && i < V) gmax[i / kGroup] = nan ? __builtin_nanf("") : mx;
  }
}

// small route: candidates kept in LDS from the top-k on
struct SmallList {
  float val[kSortMax];
  uint32_t idx[kSortMax];
};

__global__ void __launch_bounds__(kSampNT)
    k_sample(int V, SampleArgs a, const float *__restrict__ u_src, float u_val, StepState *st,
             int add_pos, uint32_t *__restrict__ history, float *__restrict__ mhist,
             float *__restrict__ w, const float *__restrict__ gmax, uint32_t *__restrict__ cidx,
             float *__restrict__ cval, int *__restrict__ status, uint32_t *__restrict__ token_out,
             uint32_t *__restrict__ ka, uint32_t *__restrict__ kb, uint32_t *__restrict__ va,
             uint32_t *__restrict__ vb) {
  // sort keys, or 2 x kStream floats
  __shared__ __align__(16) unsigned long long sbuf[kSortMax];
  __shared__ __align__(16) SmallList sl;
  __shared__ int scan[kSampNT];
  __shared__ float redf[32];
  __shared__ int redi[32];
  __shared__ float bcast_f[4];
  __shared__ int bcast_i[4];
  __shared__ int s_n, s_g;
  float *buf = reinterpret_cast<float *>(sbuf);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int step = st ? st->step : 0;
  const float u = u_src ? u_src[st ? step : 0] : u_val;
  const int NG = (V + kGroup - 1) / kGroup;

  uint32_t tok = 0;
  float chosen_p = 0.0f;
  bool done = false, small = false;
  const bool greedy = a.temperature <= 0.0f || (a.top_k == 1 && a.top_k < V);  // sampler.rs:172-174
  const bool topk = !greedy && a.top_k > 1 && a.top_k < V;

  // the groups' maxima, up to four per thread in registers
  constexpr int GR = 4;
  float gm[GR];
  bool nan = false;
  float gmx = -__builtin_inff();
#pragma unroll
  for (int j = 0; j < GR; j++) {
    const int g = tid + j * kSampNT;
    gm[j] = g < NG ? gmax[g] : -__builtin_inff();
    nan |= gm[j] != gm[j];
    gmx = fmaxf(gmx, gm[j]);
  }
  const bool fits = NG <= GR * kSampNT && __syncthreads_or(nan) == 0;
  if (greedy && fits) {
    // the last maximum wins: the last group that holds it, its last value
    const float mx = block_maxf(gmx, redf);
    int g = -1;
#pragma unroll
    for (int j = 0; j < GR; j++)
      if (tid + j * kSampNT < NG && gm[j] == mx) g = tid + j * kSampNT;
    for (int o = 32; o > 0; o >>= 1) g = max(g, __shfl_xor(g, o));
    if (lane == 0) redi[wave] = g;
    __syncthreads();
    for (int i = 0; i < kSampNT / 64; i++) g = max(g, redi[i]);
    const int i = g * kGroup + lane;
    const unsigned long long m = __ballot(i < V && w[min(i, V - 1)] == mx);
    tok = (uint32_t)(g * kGroup + 63 - __clzll((long long)m));
    done = true;
  } else if (greedy) {
    tok = block_argmax(w, V, redf, redi);
    done = true;
  }

  int nc = 0;  // candidates (cidx/cval or sl, index order)
  if (!done && topk && fits && a.top_k <= NG) {
    // L: the largest key with at least k groups' maxima >= it
    uint32_t key[GR];
#pragma unroll
    for (int j = 0; j < GR; j++) key[j] = tid + j * kSampNT < NG ? fkey(gm[j]) : 0u;
    uint32_t T = 0;
    for (int bit = 31; bit >= 0; bit--) {
      const uint32_t cand = T | (1u << bit);
      int c = 0;
#pragma unroll
      for (int j = 0; j < GR; j++) c += __popcll(__ballot(key[j] >= cand));
      // counts of the bit's waves side by side, in two halves of redi so that
      // one barrier per bit is enough
      int *r = redi + (bit & 1) * 16;
      if (lane == 0) r[wave] = c;
      __syncthreads();
      int s = 0;
#pragma unroll
      for (int i = 0; i < kSampNT / 64; i++) s += r[i];
      if (s >= a.top_k) T = cand;
    }
    const float L = fkey_inv(T);
    if (tid == 0) s_n = s_g = 0;
    __syncthreads();
    if (L > -__builtin_inff()) {
      // the groups that hold candidates, then their values >= L
#pragma unroll
      for (int j = 0; j < GR; j++)
        if (tid + j * kSampNT < NG && gm[j] >= L) {
          const int at = atomicAdd(&s_g, 1);
          if (at < kSortMax) sl.idx[at] = (uint32_t)(tid + j * kSampNT);
        }
      __syncthreads();
      const int ng = min(s_g, kSortMax);
      for (int q = wave; q < ng; q += kSampNT / 64) {
        const int i = (int)sl.idx[q] * kGroup + lane;
        const float x = w[min(i, V - 1)];
        const bool k = i < V && x >= L;
        const unsigned long long m = __ballot(k);
        int base = 0;
        if (lane == 0) base = atomicAdd(&s_n, __popcll(m));
        base = __shfl(base, 0);
        const int at = base + __popcll(m & ((1ull << lane) - 1));
        if (k && at < kSortMax)
          sbuf[at] = ((unsigned long long)(~fkey(x)) << 32) | (unsigned)i;
      }
      __syncthreads();
      const int n = s_n;
      small = n <= kSortMax && s_g <= kSortMax;
      if (small) {
        // the k-th largest value is top_k_filter's threshold; the values that
        // are not below it (a prefix of the sorted ones), in index order
        int n2 = 64;
        while (n2 < n) n2 <<= 1;
        sort_keys(sbuf, n, n2);
        const float thr = fkey_inv(~(uint32_t)(sbuf[a.top_k - 1] >> 32));
        __syncthreads();
        int c = 0;
        for (int i = tid; i < n; i += kSampNT) {
          const unsigned long long e = sbuf[i];
          const bool keep = !(fkey_inv(~(uint32_t)(e >> 32)) < thr);
          c += keep ? 1 : 0;
          if (keep) sbuf[i] = (e << 32) | (uint32_t)~(e >> 32);  // (index, key)
        }
        nc = block_sum_i(c, redi);
        __syncthreads();
        sort_keys(sbuf, nc, n2);
        for (int i = tid; i < nc; i += kSampNT) {
          sl.idx[i] = (uint32_t)(sbuf[i] >> 32);
          sl.val[i] = fkey_inv((uint32_t)sbuf[i]);
        }
        __syncthreads();
      }
    }
  }
  if (!done && !small) {
    if (topk) {
      // L = the k-th largest of the threads' maxima (k <= 1024), or -inf
      float tmax = -__builtin_inff();
      for (int i = tid; i < V; i += kSampNT) tmax = fmaxf(tmax, w[i]);
      float L = -__builtin_inff();
      if (a.top_k <= kSampNT) {
        __syncthreads();
        sbuf[tid] = ((unsigned long long)(~fkey(tmax)) << 32) | (unsigned)tid;
        __syncthreads();
        bitonic_sort(sbuf, kSampNT);
        L = fkey_inv(~(uint32_t)(sbuf[a.top_k - 1] >> 32));
        __syncthreads();
      }
      nc = compact(w, V, [L](float x) { return x >= L; }, cidx, cval, redi);
      float thr;
      if (nc <= kSortMax) {
        // the k-th largest value among the candidates (top_k_filter's threshold)
        int n2 = 1;
        while (n2 < nc) n2 <<= 1;
        for (int i = tid; i < n2; i += kSampNT)
          sbuf[i] = i < nc ? ((unsigned long long)(~fkey(cval[i])) << 32) | (unsigned)i : ~0ull;
        __syncthreads();
        bitonic_sort(sbuf, n2);
        thr = fkey_inv(~(uint32_t)(sbuf[a.top_k - 1] >> 32));
        __syncthreads();
      } else {
        // the largest key T with at least k values >= T, bit by bit
        uint32_t T = 0;
        for (int bit = 31; bit >= 0; bit--) {
          const uint32_t cand = T | (1u << bit);
          int c = 0;
          for (int i = tid; i < V; i += kSampNT) c += fkey(w[i]) >= cand ? 1 : 0;
          if (block_sum_i(c, redi) >= a.top_k) T = cand;
        }
        thr = fkey_inv(T);
      }
      // top_k_filter keeps the values that are not below the threshold
      nc = compact(w, V, [thr](float x) { return !(x < thr); }, cidx, cval, redi);
    } else {
      nc = compact(w, V, [](float x) { return x > -__builtin_inff(); }, cidx, cval, redi);
    }
  }
  if (!done) {
    float *val = small ? sl.val : cval;
    const uint32_t *idx = small ? sl.idx : cidx;
    if (a.top_p > 0.0f && a.top_p < 1.0f) {  // top_p_filter (sampler.rs:279-319)
      // softmax over the candidates: max, exp, sequential sum, division
      float mx = -__builtin_inff();
      for (int i = tid; i < nc; i += kSampNT) mx = fmaxf(mx, val[i]);
      mx = block_maxf(mx, redf);
      float *pr = w;  // the probabilities, in the free working vector
      for (int i = tid; i < nc; i += kSampNT) pr[i] = val[i];
      __syncthreads();
      const float sum = exp_then_seq_sum(pr, nc, mx, buf, bcast_f, bcast_i);
      if (sum > 0.0f)
        for (int i = tid; i < nc; i += kSampNT) pr[i] = pr[i] / sum;
      __syncthreads();
      // the candidates sorted by probability descending, index ascending
      // among equal ones: rank r holds slot (LDS) or token (radix) sidx[r]
      // with the probability of key skey[r]
      const bool lds_sort = nc <= kSortMax;
      const uint32_t *sidx = va, *skey = ka;
      if (lds_sort) {
        int n2 = 1;
        while (n2 < nc) n2 <<= 1;
        for (int i = tid; i < nc; i += kSampNT)
          sbuf[i] = ((unsigned long long)(~fkey(pr[i])) << 32) | (unsigned)i;
        __syncthreads();
        sort_keys(sbuf, nc, n2);
        for (int i = tid; i < nc; i += kSampNT) {
          ka[i] = ~(uint32_t)(sbuf[i] >> 32);  // fkey of the probability
          va[i] = (uint32_t)(sbuf[i] & 0xffffffffu);
        }
        __syncthreads();
      } else {
        // probabilities are >= +0, so ~bits orders them descending; the
        // sign bit is set in every key and needs no pass
        for (int i = tid; i < nc; i += kSampNT) {
          ka[i] = ~__float_as_uint(pr[i]);
          va[i] = (uint32_t)i;
        }
        __syncthreads();
        const int in_b = radix_sort_global(ka, va, kb, vb, nc, 31, scan);
        for (int i = tid; i < nc; i += kSampNT) {  // as fkey, like the LDS route
          const uint32_t k = in_b ? kb[i] : ka[i];
          (in_b ? kb : ka)[i] = ~k | 0x80000000u;
        }
        __syncthreads();
        sidx = in_b ? vb : va;
        skey = in_b ? kb : ka;
      }
      // cumulative probability in sorted order until it reaches p; the
      // candidates after that leave
      const float p = a.top_p;
      const int at = stream_seq(nc, [skey](int i) { return fkey_inv(skey[i]); },
                                [p](float cum) { return cum >= p; }, true, buf, bcast_f, bcast_i,
                                nullptr);
      __syncthreads();
      for (int r = at + 1 + tid; r < nc; r += kSampNT) val[sidx[r]] = -__builtin_inff();
      __syncthreads();
    }

    // softmax_sample (sampler.rs:227-259) over the candidates in index order
    float mx = -__builtin_inff();
    for (int i = tid; i < nc; i += kSampNT) mx = fmaxf(mx, val[i]);
    mx = block_maxf(mx, redf);
    const float sum = exp_then_seq_sum(val, nc, mx, buf, bcast_f, bcast_i);
    if (sum > 0.0f)
      for (int i = tid; i < nc; i += kSampNT) val[i] = val[i] / sum;
    __syncthreads();
    const int at = stream_seq(nc, [val](int i) { return val[i]; },
                              [u](float cum) { return u < cum; }, true, buf, bcast_f, bcast_i,
                              nullptr);
    tok = at < nc ? idx[at] : (uint32_t)(V - 1);  // the reference's fallback: the last token
    chosen_p = at < nc ? val[at] : 0.0f;
  }

  if (tid == 0) {
    status[0] = 0;
    if (token_out) token_out[0] = tok;
    if (st) {
      st->token = tok;
      st->margin = chosen_p;
      if (history) history[step] = tok;
      if (mhist) mhist[step] = chosen_p;
      st->pos += add_pos;
      st->step = step + 1;
    }
  }
}

SampleArgs make_sample_args(const syn_hip_sampler &p) {
  SampleArgs a;
  a.temperature = p.temperature;
  a.inv_t = p.temperature > 0.0f ? 1.0f / p.temperature : 1.0f;
  a.top_k = (int)std::min<uint32_t>(p.top_k, 0x7fffffffu);
  a.top_p = p.top_p;
  a.rep = p.repetition_penalty;
  a.apply_rep = std::fabs(p.repetition_penalty - 1.0f) > 1.1920929e-07f ? 1 : 0;
  return a;
}

syn_status_t SampleScratch::ensure(size_t v) {
  if (vocab >= v && w.p) return SYN_OK;
  SYN_HIP(hipDeviceSynchronize());
  vocab = 0;
  SYN_TRY(w.alloc(v * 4));
  SYN_TRY(gmax.alloc(cdiv(v, kGroup) * 4));
  SYN_TRY(cidx.alloc(v * 4));
  SYN_TRY(cval.alloc(v * 4));
  SYN_TRY(status.alloc(64));
  SYN_TRY(ka.alloc(v * 4));
  SYN_TRY(kb.alloc(v * 4));
  SYN_TRY(va.alloc(v * 4));
  SYN_TRY(vb.alloc(v * 4));
  vocab = v;
  return SYN_OK;
}

syn_status_t launch_sample(const float *logits, int V, const uint32_t *hist, int nh,
                           const SampleArgs &a, const float *u, float u_val, StepState *st,
                           int add_pos, uint32_t *history, float *mhist, SampleScratch &scr,
                           uint32_t *token_out, hipStream_t s) {
  if (V <= 0) return SYN_ERR_INVALID_ARG;
  if (scr.vocab < (size_t)V || !scr.w.p) {
    set_error("sampler scratch not prepared for this vocabulary");
    return SYN_ERR_INTERNAL;
  }
  hipLaunchKernelGGL(k_sample_prep, dim3((unsigned)cdiv((size_t)V, kPrepPer)), dim3(kPrepNT), 0, s,
                     logits, V, hist, nh, a, st, scr.w.as<float>(), scr.gmax.as<float>());
  SYN_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_sample, dim3(1), dim3(kSampNT), 0, s, V, a, u, u_val, st, add_pos, history,
                     mhist, scr.w.as<float>(), scr.gmax.as<float>(), scr.cidx.as<uint32_t>(),
                     scr.cval.as<float>(), scr.status.as<int>(), token_out,
                     scr.ka.as<uint32_t>(), scr.kb.as<uint32_t>(), scr.va.as<uint32_t>(),
                     scr.vb.as<uint32_t>());
  SYN_LAUNCH_CHECK();
  return SYN_OK;
}

// ---------------------------------------------------------------- host RNG
static uint32_t rotl32(uint32_t x, int r) { return (x << r) | (x >> (32 - r)); }

// one ChaCha block (64-bit block counter in words 12-13, stream 0)
static void chacha_block(const uint32_t key[8], uint64_t counter, int rounds, uint32_t out[16]) {
  const uint32_t init[16] = {0x61707865u, 0x3320646eu, 0x79622d32u, 0x6b206574u,
                             key[0], key[1], key[2], key[3], key[4], key[5], key[6], key[7],
                             (uint32_t)counter, (uint32_t)(counter >> 32), 0u, 0u};
  uint32_t x[16];
  std::memcpy(x, init, sizeof(x));
  auto qr = [&](int a, int b, int c, int d) {
    x[a] += x[b]; x[d] = rotl32(x[d] ^ x[a], 16);
    x[c] += x[d]; x[b] = rotl32(x[b] ^ x[c], 12);
    x[a] += x[b]; x[d] = rotl32(x[d] ^ x[a], 8);
    x[c] += x[d]; x[b] = rotl32(x[b] ^ x[c], 7);
  };
  for (int r = 0; r < rounds; r += 2) {
    qr(0, 4, 8, 12); qr(1, 5, 9, 13); qr(2, 6, 10, 14); qr(3, 7, 11, 15);
    qr(0, 5, 10, 15); qr(1, 6, 11, 12); qr(2, 7, 8, 13); qr(3, 4, 9, 14);
  }
  for (int i = 0; i < 16; i++) out[i] = x[i] + init[i];
}

void host_stdrng_f32(uint64_t seed, size_t n, float *out) {
  // rand_core seed_from_u64: PCG32 steps (state advanced first, XSH-RR
  // output) give the eight little-endian key words
  uint32_t key[8];
  uint64_t state = seed;
  for (int i = 0; i < 8; i++) {
    state = state * 6364136223846793005ull + 11634580027462260723ull;
    const uint32_t xs = (uint32_t)(((state >> 18) ^ state) >> 27);
    const uint32_t rot = (uint32_t)(state >> 59);
    key[i] = (xs >> rot) | (xs << ((32 - rot) & 31));
  }
  // ChaCha12Rng: next_u32 walks a buffer of four consecutive blocks;
  // gen::<f32>() = (u32 >> 8) * 2^-24
  uint32_t buf[64];
  uint64_t ctr = 0;
  size_t idx = 64;
  for (size_t i = 0; i < n; i++) {
    if (idx >= 64) {
      for (int b = 0; b < 4; b++) chacha_block(key, ctr + (uint64_t)b, 12, buf + 16 * b);
      ctr += 4;
      idx = 0;
    }
    out[i] = (float)(buf[idx++] >> 8) * (1.0f / 16777216.0f);
  }
}

}  // namespace syn

using namespace syn;

namespace {
SampleScratch &standalone() {
  static SampleScratch s;
  return s;
}
}  // namespace

extern "C" syn_status_t syn_hip_sample(const float *d_logits, size_t vocab,
                                       const uint32_t *d_history, size_t n_history,
                                       const syn_hip_sampler *params, float u, uint32_t *d_token,
                                       int *d_status, void *stream) {
  if (vocab == 0) return SYN_OK;
  if (!d_logits || !params || !d_token || (n_history && !d_history)) return SYN_ERR_NULL_PTR;
  if (vocab > 0x7fffffffu || n_history > 0x7fffffffu) return SYN_ERR_INVALID_ARG;
  SYN_TRY(ensure_init());
  SampleScratch &scr = standalone();
  SYN_TRY(scr.ensure(vocab));
  hipStream_t s = pick_stream(stream);
  const SampleArgs a = make_sample_args(*params);
  SYN_TRY(launch_sample(d_logits, (int)vocab, d_history, (int)n_history, a, nullptr, u, nullptr, 0,
                        nullptr, nullptr, scr, d_token, s));
  if (d_status)
    SYN_HIP(hipMemcpyAsync(d_status, scr.status.p, 4, hipMemcpyDeviceToDevice, s));
  return SYN_OK;
}

extern "C" syn_status_t syn_hip_stdrng_f32(uint64_t seed, size_t n, float *out) {
  if (n == 0) return SYN_OK;
  if (!out) return SYN_ERR_NULL_PTR;
  host_stdrng_f32(seed, n, out);
  return SYN_OK;
}
