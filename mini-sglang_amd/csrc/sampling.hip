// Sampling kernels: greedy argmax, temperature softmax, exact top-k / top-p sampling.
//
// All three walk [rows, vocab] once or a few times with one workgroup per row; the row
// (<= 608 KB fp32) stays L2-resident between passes.  Top-k / top-p uses no sort: the k-th
// largest probability and the top-p mass cut are found by a 3-level radix select over the
// fp32 bit pattern (monotone for non-negative floats) with LDS histograms.  Every sum that
// decides a threshold or the sampled index is an INTEGER (fixed-point mass, counts), so the
// result is independent of atomic ordering: all TP ranks, which hold identical logits and
// the same Philox (seed, offset), draw the same token (reference: every rank seeds 42,
// P/engine/engine.py:37).
#include "common.h"

namespace msgl {

typedef unsigned long long u64;

// ------------------------------------------------------------------------------------------
// argmax: first index of the row maximum
// ------------------------------------------------------------------------------------------
template <int DT>
__device__ __forceinline__ float load_logit(const void* row, int64_t i) {
  if constexpr (DT == MSGL_F32) return static_cast<const float*>(row)[i];
  if constexpr (DT == MSGL_BF16) return __uint_as_float((uint32_t) static_cast<const uint16_t*>(row)[i] << 16);
  return (float)static_cast<const _Float16*>(row)[i];
}

// 8 consecutive logits starting at an 8-aligned index (16-byte loads)
template <int DT>
__device__ __forceinline__ void load_logits8(const void* row, int64_t i, float (&f)[8]) {
  if constexpr (DT == MSGL_F32) {
    const float4 a = *reinterpret_cast<const float4*>(static_cast<const float*>(row) + i);
    const float4 b = *reinterpret_cast<const float4*>(static_cast<const float*>(row) + i + 4);
    f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w; f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
  } else {
    const U4 u = ldg16(static_cast<const uint16_t*>(row) + i);
    using E = Elem<std::conditional_t<DT == MSGL_BF16, BF16, FP16>>;
    f[0] = E::lo(u.x); f[1] = E::hi(u.x); f[2] = E::lo(u.y); f[3] = E::hi(u.y);
    f[4] = E::lo(u.z); f[5] = E::hi(u.z); f[6] = E::lo(u.w); f[7] = E::hi(u.w);
  }
}

constexpr int kRowThreads = 1024;

template <int DT, bool VEC>
__global__ __launch_bounds__(kRowThreads) void argmax_kernel(int* __restrict__ out,
                                                             const char* __restrict__ logits, int64_t vocab,
                                                             int64_t row_stride_bytes) {
  __shared__ float s_val[kRowThreads / 64];
  __shared__ int s_idx[kRowThreads / 64];
  const void* row = logits + (int64_t)blockIdx.x * row_stride_bytes;
  const int tid = threadIdx.x;
  float best = -INFINITY;
  int bidx = 0x7fffffff;
  if constexpr (VEC) {
    const int64_t nvec = vocab >> 3;
    for (int64_t p = tid; p < nvec; p += kRowThreads) {
      float f[8];
      load_logits8<DT>(row, p * 8, f);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (f[e] > best) { best = f[e]; bidx = (int)(p * 8 + e); }
      }
    }
    for (int64_t i = (nvec << 3) + tid; i < vocab; i += kRowThreads) {
      const float x = load_logit<DT>(row, i);
      if (x > best) { best = x; bidx = (int)i; }
    }
  } else {
    for (int64_t i = tid; i < vocab; i += kRowThreads) {
      const float x = load_logit<DT>(row, i);
      if (x > best) { best = x; bidx = (int)i; }
    }
  }
  // (value desc, index asc) reduction
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float ov = __shfl_xor(best, off, 64);
    const int oi = __shfl_xor(bidx, off, 64);
    if (ov > best || (ov == best && oi < bidx)) { best = ov; bidx = oi; }
  }
  if ((tid & 63) == 0) { s_val[tid >> 6] = best; s_idx[tid >> 6] = bidx; }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < kRowThreads / 64; ++w) {
      if (s_val[w] > best || (s_val[w] == best && s_idx[w] < bidx)) { best = s_val[w]; bidx = s_idx[w]; }
    }
    out[blockIdx.x] = bidx == 0x7fffffff ? 0 : bidx;
  }
}

// ------------------------------------------------------------------------------------------
// probs = softmax(logits / T)
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ float block_reduce_max(float x, float* lds) {
  x = wave_max(x);
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = x;
  __syncthreads();
  float r = lds[0];
  for (int w = 1; w < kRowThreads / 64; ++w) r = fmaxf(r, lds[w]);
  __syncthreads();
  return r;
}
__device__ __forceinline__ float block_reduce_sum(float x, float* lds) {
  x = wave_sum(x);
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = x;
  __syncthreads();
  float r = 0.f;
  for (int w = 0; w < kRowThreads / 64; ++w) r += lds[w];  // fixed order: deterministic
  __syncthreads();
  return r;
}

template <int DT>
__global__ __launch_bounds__(kRowThreads) void softmax_kernel(float* __restrict__ probs,
                                                              const char* __restrict__ logits,
                                                              const float* __restrict__ temperatures,
                                                              int64_t vocab, int64_t logits_stride_bytes,
                                                              int64_t probs_stride) {
  __shared__ float lds[kRowThreads / 64];
  const void* row = logits + (int64_t)blockIdx.x * logits_stride_bytes;
  float* prow = probs + (int64_t)blockIdx.x * probs_stride;
  const float inv_t = 1.0f / temperatures[blockIdx.x];
  const int tid = threadIdx.x;
  float mx = -INFINITY;
  for (int64_t i = tid; i < vocab; i += kRowThreads) mx = fmaxf(mx, load_logit<DT>(row, i));
  mx = block_reduce_max(mx, lds);
  const float k = inv_t * 1.4426950408889634f;
  float sum = 0.f;
  for (int64_t i = tid; i < vocab; i += kRowThreads) {
    const float e = __builtin_amdgcn_exp2f((load_logit<DT>(row, i) - mx) * k);
    prow[i] = e;
    sum += e;
  }
  sum = block_reduce_sum(sum, lds);
  const float inv = 1.0f / sum;
  for (int64_t i = tid; i < vocab; i += kRowThreads) prow[i] *= inv;
}

// ------------------------------------------------------------------------------------------
// top-k / top-p sampling from probs
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ u64 fixed_mass(float p) {  // 2^-40 resolution, exact scaling
  return p > 0.f ? (u64)__float2ull_rz(p * 1099511627776.0f) : 0ull;
}

__device__ __forceinline__ u64 shfl_up_u64(u64 v, int d) {
  const uint32_t lo = __shfl_up((uint32_t)v, d, 64);
  const uint32_t hi = __shfl_up((uint32_t)(v >> 32), d, 64);
  return ((u64)hi << 32) | lo;
}
__device__ __forceinline__ u64 shfl_u64(u64 v, int src) {
  const uint32_t lo = __shfl((uint32_t)v, src, 64);
  const uint32_t hi = __shfl((uint32_t)(v >> 32), src, 64);
  return ((u64)hi << 32) | lo;
}

// inclusive prefix sum over the 1024 threads (thread order), exact integer arithmetic
__device__ __forceinline__ u64 block_prefix_incl(u64 v, u64* lds_w) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const u64 o = shfl_up_u64(v, d);
    if (lane >= d) v += o;
  }
  if (lane == 63) lds_w[w] = v;
  __syncthreads();
  u64 base = 0;
  for (int i = 0; i < w; ++i) base += lds_w[i];
  __syncthreads();
  return v + base;
}

__device__ __forceinline__ u64 block_sum_u64(u64 v, u64* lds_w) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    const uint32_t lo = __shfl_xor((uint32_t)v, d, 64);
    const uint32_t hi = __shfl_xor((uint32_t)(v >> 32), d, 64);
    v += ((u64)hi << 32) | lo;
  }
  if (lane == 0) lds_w[w] = v;
  __syncthreads();
  u64 r = 0;
  for (int i = 0; i < kRowThreads / 64; ++i) r += lds_w[i];
  __syncthreads();
  return r;
}

struct Philox {
  static __device__ __forceinline__ void round(uint32_t (&c)[4], uint32_t k0, uint32_t k1) {
    const u64 p0 = (u64)0xD2511F53u * c[0];
    const u64 p1 = (u64)0xCD9E8D57u * c[2];
    const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c[1] ^ k0;
    const uint32_t n1 = (uint32_t)p1;
    const uint32_t n2 = (uint32_t)(p0 >> 32) ^ c[3] ^ k1;
    const uint32_t n3 = (uint32_t)p0;
    c[0] = n0; c[1] = n1; c[2] = n2; c[3] = n3;
  }
  // Philox4x32-10, first output word
  static __device__ __forceinline__ uint32_t draw(u64 seed, u64 ctr) {
    uint32_t c[4] = {(uint32_t)ctr, (uint32_t)(ctr >> 32), 0u, 0u};
    uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
#pragma unroll
    for (int r = 0; r < 10; ++r) {
      round(c, k0, k1);
      k0 += 0x9E3779B9u;
      k1 += 0xBB67AE85u;
    }
    return c[0];
  }
};

constexpr int kBins = 2048;  // 11-bit digits; thread t owns bins 2047-2t and 2046-2t (descending)
constexpr uint32_t kNoDigit = 0xffffffffu;
constexpr int kStrip = 8;    // loads of a row in flight per thread: a pass is bound by their latency, not by bytes

// What a row's probabilities come from.  raw(i): the stored number; weight(x): a number in the order of the probabilities
// (the probability itself, or e = 2^((x - max) k)); prob(w): the probability of that weight.
struct ProbRow {
  static constexpr bool kSoftmax = false;
  const float* row;
  __device__ __forceinline__ float raw(int64_t i) const { return row[i]; }
  __device__ __forceinline__ float weight(float x) const { return x; }
  __device__ __forceinline__ float prob(float w) const { return w; }
};
// the same numbers softmax_kernel stores, recomputed from the logits: same maximum, same order of the sum, same rounding
template <int DT>
struct LogitRow {
  static constexpr bool kSoftmax = true;
  const void* row;
  float mx, k, inv;
  __device__ __forceinline__ float raw(int64_t i) const { return load_logit<DT>(row, i); }
  __device__ __forceinline__ float weight(float x) const { return __builtin_amdgcn_exp2f((x - mx) * k); }
  __device__ __forceinline__ float prob(float w) const { return w * inv; }
};

// Calls f(index, raw value) for the row elements tid, tid + 1024, ... in order, kStrip loads in flight; `in` is false past the end
// (the calls are uniform over the workgroup, so f may use ballots).
template <class Src, class F>
__device__ __forceinline__ void walk_row(const Src& src, int64_t vocab, F f) {
  const int tid = threadIdx.x;
  int64_t base = 0;
  for (; base + (int64_t)kStrip * kRowThreads <= vocab; base += (int64_t)kStrip * kRowThreads) {
    float x[kStrip];
#pragma unroll
    for (int u = 0; u < kStrip; ++u) x[u] = src.raw(base + u * kRowThreads + tid);
#pragma unroll
    for (int u = 0; u < kStrip; ++u) f(base + u * kRowThreads + tid, x[u], true);
  }
  for (; base < vocab; base += kRowThreads) {
    const int64_t i = base + tid;
    const bool in = i < vocab;
    f(i, in ? src.raw(i) : 0.f, in);
  }
}

// One radix-select level.  Elements taking part: bits >= floor_bits and (bits & mask) == prefix.
// BY_MASS = false: find the digit where the descending element COUNT reaches `target`;
// BY_MASS = true : where the descending fixed-point MASS reaches `target`.
// Returns the digit; `target` is reduced by what lies above it.
template <bool BY_MASS, class Src>
__device__ __forceinline__ uint32_t select_level(const Src& src, int64_t vocab, uint32_t floor_bits, uint32_t mask, uint32_t prefix,
                                                 int shift, int nbits, u64& target, uint32_t* h_cnt, u64* h_mass, u64* lds_w,
                                                 uint32_t* s_digit) {
  const int tid = threadIdx.x;
  const uint32_t dmask = (1u << nbits) - 1u;
  for (int b = tid; b < kBins; b += kRowThreads) {
    if (BY_MASS) h_mass[b] = 0ull;
    else h_cnt[b] = 0u;
  }
  if (tid == 0) *s_digit = kNoDigit;  // stays if the row holds less than `target` (fewer than k positive entries)
  __syncthreads();
  walk_row(src, vocab, [&](int64_t, float x, bool in) {
    const float p = src.prob(src.weight(x));
    const uint32_t bits = __float_as_uint(p);
    if (in && bits >= floor_bits && (bits & mask) == prefix && p > 0.f) {
      const uint32_t d = (bits >> shift) & dmask;
      if (BY_MASS) {
        const u64 m = fixed_mass(p);
        if (m) atomicAdd(&h_mass[d], m);
      } else {
        atomicAdd(&h_cnt[d], 1u);
      }
    }
  });
  __syncthreads();
  const int b_hi = kBins - 1 - 2 * tid, b_lo = b_hi - 1;  // descending ownership
  const u64 q_hi = BY_MASS ? h_mass[b_hi] : (u64)h_cnt[b_hi];
  const u64 q_lo = BY_MASS ? h_mass[b_lo] : (u64)h_cnt[b_lo];
  const u64 incl = block_prefix_incl(q_hi + q_lo, lds_w);  // quantity in bins >= b_lo
  const u64 above_hi = incl - q_hi - q_lo;                 // quantity in bins > b_hi
  const u64 above_lo = above_hi + q_hi;                    // quantity in bins > b_lo
  if (above_hi < target && target <= above_hi + q_hi) *s_digit = (uint32_t)b_hi;
  if (above_lo < target && target <= above_lo + q_lo) *s_digit = (uint32_t)b_lo;
  __syncthreads();
  const uint32_t digit = *s_digit;
  if (digit == kNoDigit) {  // uniform: every thread read the same word
    __syncthreads();
    return kNoDigit;
  }
  u64 q_above = 0;  // quantity strictly above the digit, to reduce the target
  if ((uint32_t)b_hi > digit) q_above += q_hi;
  if ((uint32_t)b_lo > digit) q_above += q_lo;
  target -= block_sum_u64(q_above, lds_w);
  return digit;
}

// bits of the value where the descending count / mass reaches `target`, or kNoDigit (no finite number has these bits)
template <bool BY_MASS, class Src>
__device__ __forceinline__ uint32_t select_bits(const Src& src, int64_t vocab, uint32_t floor_bits, u64 target, uint32_t* h_cnt, u64* h_mass,
                                                u64* lds_w, uint32_t* s_digit) {
  uint32_t prefix = 0u, mask = 0u;
#pragma unroll 1
  for (int level = 0; level < 3; ++level) {
    const int shift = level == 0 ? 21 : level == 1 ? 10 : 0, nbits = level == 2 ? 10 : 11;
    const uint32_t d = select_level<BY_MASS>(src, vocab, floor_bits, mask, prefix, shift, nbits, target, h_cnt, h_mass, lds_w, s_digit);
    if (d == kNoDigit) return kNoDigit;
    prefix |= d << shift;
    mask |= ((1u << nbits) - 1u) << shift;
  }
  return prefix;
}

// the `target`-th largest (1-based) of the workgroup's 1024 non-negative numbers, one per thread
__device__ __forceinline__ uint32_t kth_largest(uint32_t bits, int target, uint32_t* hist, uint32_t* s_two) {
  const int tid = threadIdx.x;
  uint32_t prefix = 0u, mask = 0u;
#pragma unroll 1
  for (int shift = 24; shift >= 0; shift -= 8) {
    if (tid < 256) hist[tid] = 0u;
    __syncthreads();
    if ((bits & mask) == prefix) atomicAdd(&hist[(bits >> shift) & 255u], 1u);
    __syncthreads();
    if (tid < 64) {  // lane l owns the bins 255 - 4 l ... 252 - 4 l
      int c[4], s = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) s += c[q] = (int)hist[255 - 4 * tid - q];
      int above = s;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(above, d, 64);
        if (tid >= d) above += o;
      }
      above -= s;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (above < target && target <= above + c[q]) {
          s_two[0] = (uint32_t)(255 - 4 * tid - q);
          s_two[1] = (uint32_t)above;
        }
        above += c[q];
      }
    }
    __syncthreads();
    prefix |= s_two[0] << shift;
    mask |= 255u << shift;
    target -= (int)s_two[1];
  }
  __syncthreads();
  return prefix;
}

constexpr int kList = 2048;          // candidates of a row that the short path holds (= kBins: it reuses the histograms)
constexpr int kListTopK = 1024;      // largest top-k it is tried for: one column maximum per thread bounds the k-th largest from below
// candidates asked for when only a mass is given: a list takes time with its square (512: 120 us for any row of 32000, 62 without a list), and a
// nucleus that does not fit pays for it on top (bf16 rows, top-p 0.9, one row of 151936: nucleus 8: 55 us with 64, 91 with 256, 157 with 512, 219
// without; nucleus 2127: 141, 185, 225, 217)
constexpr int kListTopP = 64;
constexpr uint32_t kTinyWeight = 0x17800000u;  // 2^-80: below it two weights apart may be one probability (denormal)

// One 1024-thread workgroup per row.
//
// Short path (any top-k up to 1024, or a top-p whose nucleus is small): thread t's largest number over the columns t, t + 1024, ...
// is known after one pass; the k-th largest of these 1024 maxima has at least k numbers at or above it, so the second pass collects
// only what reaches it -- some k numbers out of a 152 k vocabulary -- and both thresholds and the draw are integer sums over that
// list.  The general path finds the same thresholds by three radix levels over the whole row; it stays for wide nuclei, top-k above
// 1024 and rows whose largest numbers share a column.
//
// Bound: one CU walks one row (304 KB of bf16 logits) twice, an exponential and ~10 VALU operations per element in the second pass.
// 64 rows x 151936 bf16 logits, top-k and top-p: softmax_kernel + radix levels over the stored fp32 probabilities (ten passes, u64 LDS
// atomics for every element of a first level) 551 us; this kernel from the logits 49 us.
template <class Src>
__device__ __forceinline__ void sample_row(Src src, int* __restrict__ out, int64_t k, float pp, int64_t vocab, float inv_t, u64 seed, u64 offset) {
  __shared__ uint32_t h_cnt[kBins];  // histogram | candidates' probability bits
  __shared__ u64 h_mass[kBins];      // histogram | candidates' masses
  __shared__ int s_index[kList];
  __shared__ u64 lds_w[kRowThreads / 64];
  __shared__ float lds_f[kRowThreads / 64];
  __shared__ uint32_t s_digit, s_two[2];
  __shared__ int s_pick, s_n;
  const int tid = threadIdx.x;
  const int64_t r = blockIdx.x;
  const bool has_k = k >= 1 && k < vocab;
  const bool by_count = has_k && k <= kListTopK, by_mass = !has_k && pp < 1.0f;

  uint32_t thr_bits = 0u;  // keep set = { bits >= thr_bits, p > 0 }
  u64 kept_mass = 0;
  bool have_mass = false;  // kept_mass is that of the whole row
  bool done = false;       // uniform: the threshold is known and every number that reaches it is in the list
  int n = 0;

  float col = Src::kSoftmax ? -INFINITY : 0.f;
  if (Src::kSoftmax || by_count || by_mass)
    walk_row(src, vocab, [&](int64_t, float x, bool in) { col = in ? fmaxf(col, x) : col; });
  if constexpr (Src::kSoftmax) {
    src.mx = block_reduce_max(col, lds_f);
    src.k = inv_t * 1.4426950408889634f;
  }
  uint32_t floor_bits = 0u, list_bits = kNoDigit;  // list_bits: what a weight has to reach to be listed
  if (by_count || by_mass) {
    const float w = src.weight(col);
    const int want = (int)(by_count ? k : (int64_t)kListTopP);
    floor_bits = kth_largest(w > 0.f ? __float_as_uint(w) : 0u, want, h_cnt, s_two);  // NaN counts as nothing here
    // weights up to some units in the last place apart can be the same probability: the list starts a little below
    if (floor_bits > (Src::kSoftmax ? kTinyWeight : 0u)) list_bits = floor_bits - (Src::kSoftmax ? 8u : 0u);
  }
  if (tid == 0) { s_n = 0; s_pick = -1; }
  __syncthreads();
  if (Src::kSoftmax || list_bits != kNoDigit) {
    float sum = 0.f;
    walk_row(src, vocab, [&](int64_t i, float x, bool in) {
      const float w = src.weight(x);
      if (in) sum += w;
      const bool hit = in && w > 0.f && __float_as_uint(w) >= list_bits;
      const u64 votes = __ballot(hit);
      if (votes) {
        const int lane = tid & 63;
        int at = 0;
        if (lane == 0) at = atomicAdd(&s_n, __popcll(votes));
        at = __shfl(at, 0, 64) + __popcll(votes & ((1ull << lane) - 1ull));
        if (hit && at < kList) {
          s_index[at] = (int)i;
          h_cnt[at] = __float_as_uint(w);
        }
      }
    });
    if constexpr (Src::kSoftmax) src.inv = 1.0f / block_reduce_sum(sum, lds_f);
    __syncthreads();
    n = s_n;
  }
  if (list_bits != kNoDigit && n <= kList) {
    uint32_t mine[kList / kRowThreads];
    bool sure[kList / kRowThreads];  // not among the few below the floor, of whose equals some may be missing
#pragma unroll
    for (int e = 0; e < kList / kRowThreads; ++e) {
      const int c = tid + e * kRowThreads;
      sure[e] = c < n && h_cnt[c] >= floor_bits;
      const float p = c < n ? src.prob(__uint_as_float(h_cnt[c])) : 0.f;
      mine[e] = __float_as_uint(p);
      if (c < n) {
        h_cnt[c] = mine[e];
        h_mass[c] = fixed_mass(p);
      }
    }
    u64 target = 0;
    if (by_mass) {
      have_mass = true;
      u64 loc = 0;
      walk_row(src, vocab, [&](int64_t, float x, bool in) {
        const u64 m = fixed_mass(src.prob(src.weight(x)));
        loc += in ? m : 0ull;
      });
      kept_mass = block_sum_u64(loc, lds_w);
      target = (u64)((double)pp * (double)kept_mass);
      if (target < 1) target = 1;
      if (target > kept_mass) target = kept_mass;
    }
    if (tid == 0) s_digit = kNoDigit;
    __syncthreads();
    u64 m_above[kList / kRowThreads], m_same[kList / kRowThreads];
#pragma unroll
    for (int e = 0; e < kList / kRowThreads; ++e) {
      m_above[e] = m_same[e] = 0;
      if (tid + e * kRowThreads >= n) continue;
      int c_above = 0, c_same = 0;
      for (int j = 0; j < n; ++j) {
        const uint32_t b = h_cnt[j];
        const u64 m = h_mass[j];
        if (b > mine[e]) { ++c_above; m_above[e] += m; }
        else if (b == mine[e]) { ++c_same; m_same[e] += m; }
      }
      const bool here = by_count ? c_above < k && k <= c_above + c_same : m_above[e] < target && target <= m_above[e] + m_same[e];
      if (sure[e] && here) {  // equal candidates write equal words
        s_digit = mine[e];
        lds_w[0] = m_above[e] + m_same[e];
      }
    }
    __syncthreads();
    if (s_digit != kNoDigit && (by_count || kept_mass > 0)) {
      thr_bits = s_digit;
      kept_mass = lds_w[0];
      done = true;
    }
    __syncthreads();
    if (done && by_count && pp < 1.0f && kept_mass > 0) {
      target = (u64)((double)pp * (double)kept_mass);
      if (target < 1) target = 1;
      if (target > kept_mass) target = kept_mass;
#pragma unroll
      for (int e = 0; e < kList / kRowThreads; ++e)
        if (mine[e] >= thr_bits && tid + e * kRowThreads < n && m_above[e] < target && target <= m_above[e] + m_same[e]) s_digit = mine[e];
      __syncthreads();
      thr_bits = s_digit;
    }
    if (done) {  // the draw over the list, in index order
      u64 loc = 0;
#pragma unroll
      for (int e = 0; e < kList / kRowThreads; ++e)
        if (tid + e * kRowThreads < n && mine[e] >= thr_bits) loc += h_mass[tid + e * kRowThreads];
      const u64 total = block_sum_u64(loc, lds_w);
      const uint32_t x = Philox::draw(seed, offset + (u64)r);
      const u64 u = (total >> 32) * (u64)x + (((total & 0xffffffffull) * (u64)x) >> 32);
#pragma unroll
      for (int e = 0; e < kList / kRowThreads; ++e) {
        const int c = tid + e * kRowThreads;
        if (c >= n || mine[e] < thr_bits) continue;
        const int idx = s_index[c];
        u64 before = 0;
        for (int j = 0; j < n; ++j)
          if (h_cnt[j] >= thr_bits && s_index[j] < idx) before += h_mass[j];
        if (u >= before && u < before + h_mass[c]) s_pick = idx;
      }
      __syncthreads();
      if (tid == 0) out[r] = s_pick < 0 ? 0 : s_pick;
      return;
    }
  }

  if (has_k) {
    // fewer than k positive probabilities (a low temperature underflows the tail to 0): top-k keeps all of them,
    // as flashinfer does -- no threshold; ties at the k-th largest value stay in the keep set
    // (such a row comes here past its list: 64 rows x 151936 at temperature 0.02, k 1000: 100 us, 295 over stored probabilities)
    const uint32_t v = select_bits<false>(src, vocab, 0u, (u64)k, h_cnt, h_mass, lds_w, &s_digit);
    if (v != kNoDigit) thr_bits = v;
  }
  if (pp < 1.0f) {
    if (!have_mass) {
      u64 loc = 0;
      walk_row(src, vocab, [&](int64_t, float x, bool in) {
        const float p = src.prob(src.weight(x));
        if (in && __float_as_uint(p) >= thr_bits) loc += fixed_mass(p);
      });
      kept_mass = block_sum_u64(loc, lds_w);
    }
    u64 target = (u64)((double)pp * (double)kept_mass);
    if (target < 1) target = 1;
    if (target > kept_mass) target = kept_mass;
    if (kept_mass > 0) {
      const uint32_t v = select_bits<true>(src, vocab, thr_bits, target, h_cnt, h_mass, lds_w, &s_digit);
      if (v != kNoDigit) thr_bits = v > thr_bits ? v : thr_bits;  // (target <= kept_mass, so a value exists)
    }
  }

  // ---- inverse-CDF draw in index order over the keep set -------------------------------
  // wave w owns the contiguous index range [w*seg, (w+1)*seg), walked 64 indices at a time
  const int lane = tid & 63, w = tid >> 6;
  constexpr int kWaves = kRowThreads / 64;
  const int64_t seg = ((vocab + kWaves - 1) / kWaves + 63) / 64 * 64;
  const int64_t lo = (int64_t)w * seg, hi = min(vocab, lo + seg);
  auto mass_at = [&](float x) {
    const float p = src.prob(src.weight(x));
    return __float_as_uint(p) >= thr_bits ? fixed_mass(p) : 0ull;
  };
  u64 wave_mass = 0;
  int64_t at = lo + lane;
  for (; at + (kStrip - 1) * 64 < hi; at += kStrip * 64) {
    float x[kStrip];
#pragma unroll
    for (int u = 0; u < kStrip; ++u) x[u] = src.raw(at + u * 64);
#pragma unroll
    for (int u = 0; u < kStrip; ++u) wave_mass += mass_at(x[u]);
  }
  for (; at < hi; at += 64) wave_mass += mass_at(src.raw(at));
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    const uint32_t l = __shfl_xor((uint32_t)wave_mass, d, 64);
    const uint32_t h = __shfl_xor((uint32_t)(wave_mass >> 32), d, 64);
    wave_mass += ((u64)h << 32) | l;
  }
  __syncthreads();
  if (lane == 0) lds_w[w] = wave_mass;
  __syncthreads();
  u64 total = 0, before = 0;
  for (int i = 0; i < kWaves; ++i) {
    if (i < w) before += lds_w[i];
    total += lds_w[i];
  }
  const uint32_t x = Philox::draw(seed, offset + (u64)r);
  // u in [0, total): (total * x) >> 32 without 128-bit arithmetic
  const u64 u = (total >> 32) * (u64)x + (((total & 0xffffffffull) * (u64)x) >> 32);
  if (total > 0 && u >= before && u < before + wave_mass) {  // exactly one wave
    u64 run = before;
    // strips of 8 x 64 indices: their sum first, the indices one by one only in the strip that holds u
    for (int64_t base = lo; base < hi; base += kStrip * 64) {
      u64 m[kStrip], strip = 0;
#pragma unroll
      for (int e = 0; e < kStrip; ++e) {
        const int64_t i = base + e * 64 + lane;
        m[e] = i < hi ? mass_at(src.raw(i)) : 0ull;
        strip += m[e];
      }
#pragma unroll
      for (int d = 32; d > 0; d >>= 1) {
        const uint32_t l = __shfl_xor((uint32_t)strip, d, 64);
        const uint32_t h = __shfl_xor((uint32_t)(strip >> 32), d, 64);
        strip += ((u64)h << 32) | l;
      }
      if (u >= run + strip) {
        run += strip;
        continue;
      }
#pragma unroll
      for (int e = 0; e < kStrip; ++e) {
        u64 incl = m[e];
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
          const u64 o = shfl_up_u64(incl, d);
          if (lane >= d) incl += o;
        }
        if (m[e] > 0 && u >= run + incl - m[e] && u < run + incl) s_pick = (int)(base + e * 64 + lane);
        run += shfl_u64(incl, 63);
      }
      break;
    }
  }
  __syncthreads();
  if (tid == 0) out[r] = s_pick < 0 ? 0 : s_pick;  // degenerate row (all-zero mass): fall back to the first index
}

__global__ __launch_bounds__(kRowThreads) void sample_kernel(int* __restrict__ out, const float* __restrict__ probs,
                                                             const int* __restrict__ top_k, const float* __restrict__ top_p, int64_t vocab,
                                                             int64_t stride, u64 seed, u64 offset) {
  const int64_t r = blockIdx.x;
  sample_row(ProbRow{probs + r * stride}, out, top_k ? (int64_t)top_k[r] : vocab, top_p ? top_p[r] : 1.0f, vocab, 0.f, seed, offset);
}

// n numbers of type E, by one workgroup
template <class E>
__device__ __forceinline__ void copy_numbers(E* __restrict__ dst, const E* __restrict__ src, int64_t n) {
  const bool vec = ((reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(src)) & 15u) == 0;
  constexpr int kPer = 16 / sizeof(E);
  const int64_t wide = vec ? n / kPer : 0;
#pragma unroll 4
  for (int64_t i = threadIdx.x; i < wide; i += kRowThreads) reinterpret_cast<U4*>(dst)[i] = reinterpret_cast<const U4*>(src)[i];
#pragma unroll 8
  for (int64_t i = wide * kPer + threadIdx.x; i < n; i += kRowThreads) dst[i] = src[i];
}

constexpr int64_t kCopySlice = 1 << 15;  // numbers of a row that one workgroup copies

// Workgroups 0 .. rows - 1 draw; with `kept` those behind them copy the rows in slices, on compute units that the draw leaves idle (64 rows x
// 151936 bf16: 49.0 us without a copy, 51.5 with; the drawing threads storing it 59.3).
template <int DT>
__global__ __launch_bounds__(kRowThreads) void sample_filtered_logits_kernel(int* __restrict__ out, const char* __restrict__ logits,
                                                                             const float* __restrict__ temperatures,
                                                                             const int* __restrict__ top_k, const float* __restrict__ top_p,
                                                                             int64_t vocab, int64_t row_stride_bytes, u64 seed, u64 offset, int rows,
                                                                             char* __restrict__ kept, float* __restrict__ kept_t) {
  if ((int)blockIdx.x >= rows) {
    using E = std::conditional_t<DT == MSGL_F32, uint32_t, uint16_t>;
    const int slices = (int)((vocab + kCopySlice - 1) / kCopySlice), x = (int)blockIdx.x - rows;
    const int64_t r = x / slices, at = (x - r * slices) * kCopySlice;
    copy_numbers(reinterpret_cast<E*>(kept) + r * vocab + at, reinterpret_cast<const E*>(logits + r * row_stride_bytes) + at, min(kCopySlice, vocab - at));
    if (at == 0 && threadIdx.x == 0) kept_t[r] = temperatures[r];
    return;
  }
  const int64_t r = blockIdx.x;
  sample_row(LogitRow<DT>{logits + r * row_stride_bytes, 0.f, 0.f, 0.f}, out, top_k ? (int64_t)top_k[r] : vocab, top_p ? top_p[r] : 1.0f,
             vocab, 1.0f / temperatures[r], seed, offset);
}


// ------------------------------------------------------------------------------------------
// sample directly from logits (temperature only: no top-k / top-p filter)
//   index ~ softmax(logits / T).  Probabilities are never materialised: with e_i = 2^((x_i - max) k)
//   the draw is the inverse CDF over the integer masses floor(e_i 2^40) in index order, which is the
//   same distribution as normalise-then-draw up to fp32 rounding of the normalisation (and, like the
//   probs path, exact integer arithmetic from there on: identical on every TP rank).
//   Two passes over the row (max; masses per wave segment) + one wave re-walking its own segment,
//   16-byte loads throughout.  Wave w owns the contiguous index range [w seg, (w+1) seg).
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ u64 exp_mass(float x, float mx, float k) {
  return (u64)__float2ull_rz(__builtin_amdgcn_exp2f((x - mx) * k) * 1099511627776.0f);  // e in (0, 1]
}

template <int DT>
__global__ __launch_bounds__(kRowThreads) void sample_logits_kernel(int* __restrict__ out,
                                                                    const char* __restrict__ logits,
                                                                    const float* __restrict__ temperatures,
                                                                    int64_t vocab, int64_t row_stride_bytes,
                                                                    u64 seed, u64 offset) {
  __shared__ float lds_f[kRowThreads / 64];
  __shared__ u64 lds_w[kRowThreads / 64];
  __shared__ int s_pick;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t r = blockIdx.x;
  const void* row = logits + r * row_stride_bytes;
  constexpr int kWaves = kRowThreads / 64;
  constexpr int kStep = 64 * 8;  // indices per wave iteration
  const int64_t seg = ((vocab + kWaves - 1) / kWaves + kStep - 1) / kStep * kStep;
  const int64_t lo = (int64_t)w * seg, hi = min(vocab, lo + seg);

  float mx = -INFINITY;
  for (int64_t base = lo + lane * 8; base < hi; base += kStep) {
    if (base + 8 <= hi) {
      float f[8];
      load_logits8<DT>(row, base, f);
#pragma unroll
      for (int e = 0; e < 8; ++e) mx = fmaxf(mx, f[e]);
    } else {
      for (int64_t i = base; i < hi; ++i) mx = fmaxf(mx, load_logit<DT>(row, i));
    }
  }
  mx = block_reduce_max(mx, lds_f);
  const float k = 1.4426950408889634f / temperatures[r];

  auto masses8 = [&](int64_t base, u64 (&mm)[8]) {  // masses of indices base .. base+7 (0 past hi)
    if (base + 8 <= hi) {
      float f[8];
      load_logits8<DT>(row, base, f);
#pragma unroll
      for (int e = 0; e < 8; ++e) mm[e] = exp_mass(f[e], mx, k);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) mm[e] = base + e < hi ? exp_mass(load_logit<DT>(row, base + e), mx, k) : 0ull;
    }
  };
  u64 wave_mass = 0;
  for (int64_t base = lo + lane * 8; base < hi; base += kStep) {
    u64 mm[8];
    masses8(base, mm);
#pragma unroll
    for (int e = 0; e < 8; ++e) wave_mass += mm[e];
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    const uint32_t l32 = __shfl_xor((uint32_t)wave_mass, d, 64);
    const uint32_t h32 = __shfl_xor((uint32_t)(wave_mass >> 32), d, 64);
    wave_mass += ((u64)h32 << 32) | l32;
  }
  if (lane == 0) lds_w[w] = wave_mass;
  if (tid == 0) s_pick = -1;
  __syncthreads();
  u64 total = 0, before = 0;
  for (int i = 0; i < kWaves; ++i) {
    if (i < w) before += lds_w[i];
    total += lds_w[i];
  }
  const uint32_t x = Philox::draw(seed, offset + (u64)r);
  const u64 u = (total >> 32) * (u64)x + (((total & 0xffffffffull) * (u64)x) >> 32);  // [0, total)
  if (total > 0 && u >= before && u < before + wave_mass) {  // exactly one wave
    u64 run = before;
    for (int64_t base0 = lo; base0 < hi; base0 += kStep) {
      u64 mm[8];
      masses8(base0 + lane * 8, mm);
      u64 mine = 0;
#pragma unroll
      for (int e = 0; e < 8; ++e) mine += mm[e];
      u64 incl = mine;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const u64 o = shfl_up_u64(incl, d);
        if (lane >= d) incl += o;
      }
      const u64 chunk = shfl_u64(incl, 63);
      if (u < run + chunk) {
        u64 start = run + incl - mine;  // mass before this lane's 8 indices
        if (mine > 0 && u >= start && u < start + mine) {
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            if (u >= start && u < start + mm[e]) s_pick = (int)(base0 + lane * 8 + e);
            start += mm[e];
          }
        }
        break;
      }
      run += chunk;
    }
  }
  __syncthreads();
  if (tid == 0) out[r] = s_pick < 0 ? 0 : s_pick;  // degenerate row (no mass): first index
}

}  // namespace msgl

using namespace msgl;

extern "C" int msgl_argmax_rows(int32_t* out, const void* logits, int64_t rows, int64_t vocab,
                                int64_t row_stride, int logits_dtype, void* stream) {
  MSGL_REQUIRE(rows >= 0, "argmax_rows: negative rows");
  if (rows == 0) return MSGL_OK;
  MSGL_REQUIRE(out && logits, "argmax_rows: null pointer");
  MSGL_REQUIRE(vocab >= 1 && vocab < (1ll << 31) && rows < (1ll << 31), "argmax_rows: bad shape");
  const int esz = logits_dtype == MSGL_F32 ? 4 : 2;
  const bool vec = aligned16(logits) && (row_stride * esz) % 16 == 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 g((unsigned)rows), b(kRowThreads);
#define MSGL_ARGMAX(DT)                                                                                      \
  do {                                                                                                       \
    if (vec) argmax_kernel<DT, true><<<g, b, 0, s>>>(out, (const char*)logits, vocab, row_stride * esz);     \
    else argmax_kernel<DT, false><<<g, b, 0, s>>>(out, (const char*)logits, vocab, row_stride * esz);        \
  } while (0)
  if (logits_dtype == MSGL_F32) MSGL_ARGMAX(MSGL_F32);
  else if (logits_dtype == MSGL_BF16) MSGL_ARGMAX(MSGL_BF16);
  else if (logits_dtype == MSGL_FP16) MSGL_ARGMAX(MSGL_FP16);
  else {
    set_error("argmax_rows: unsupported dtype code %d", logits_dtype);
    return MSGL_EINVAL;
  }
#undef MSGL_ARGMAX
  MSGL_CHECK_LAUNCH("argmax_rows");
  return MSGL_OK;
}

extern "C" int msgl_softmax_temperature(float* probs, const void* logits, const float* temperatures,
                                        int64_t rows, int64_t vocab, int64_t logits_stride,
                                        int64_t probs_stride, int logits_dtype, void* stream) {
  MSGL_REQUIRE(rows >= 0, "softmax_temperature: negative rows");
  if (rows == 0) return MSGL_OK;
  MSGL_REQUIRE(probs && logits && temperatures, "softmax_temperature: null pointer");
  MSGL_REQUIRE(vocab >= 1 && rows < (1ll << 31), "softmax_temperature: bad shape");
  const int esz = logits_dtype == MSGL_F32 ? 4 : 2;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 g((unsigned)rows), b(kRowThreads);
  if (logits_dtype == MSGL_F32)
    softmax_kernel<MSGL_F32><<<g, b, 0, s>>>(probs, (const char*)logits, temperatures, vocab, logits_stride * esz, probs_stride);
  else if (logits_dtype == MSGL_BF16)
    softmax_kernel<MSGL_BF16><<<g, b, 0, s>>>(probs, (const char*)logits, temperatures, vocab, logits_stride * esz, probs_stride);
  else if (logits_dtype == MSGL_FP16)
    softmax_kernel<MSGL_FP16><<<g, b, 0, s>>>(probs, (const char*)logits, temperatures, vocab, logits_stride * esz, probs_stride);
  else {
    set_error("softmax_temperature: unsupported dtype code %d", logits_dtype);
    return MSGL_EINVAL;
  }
  MSGL_CHECK_LAUNCH("softmax_temperature");
  return MSGL_OK;
}

extern "C" int msgl_sample_top_k_top_p(int32_t* out, const float* probs, const int32_t* top_k,
                                       const float* top_p, int64_t rows, int64_t vocab,
                                       int64_t probs_stride, uint64_t seed, uint64_t offset, void* stream) {
  MSGL_REQUIRE(rows >= 0, "sample_top_k_top_p: negative rows");
  if (rows == 0) return MSGL_OK;
  MSGL_REQUIRE(out && probs, "sample_top_k_top_p: null pointer");
  MSGL_REQUIRE(vocab >= 1 && vocab < (1ll << 31) && rows < (1ll << 31), "sample_top_k_top_p: bad shape");
  sample_kernel<<<dim3((unsigned)rows), dim3(kRowThreads), 0, static_cast<hipStream_t>(stream)>>>(
      out, probs, top_k, top_p, vocab, probs_stride, (u64)seed, (u64)offset);
  MSGL_CHECK_LAUNCH("sample_top_k_top_p");
  return MSGL_OK;
}

// probs path's draw without the probs: same thresholds, same masses, same pick as softmax_temperature + sample_top_k_top_p
extern "C" int msgl_sample_filtered_logits_keep(int32_t* out, void* kept, float* kept_temperatures, const void* logits, const float* temperatures,
                                                const int32_t* top_k, const float* top_p, int64_t rows, int64_t vocab, int64_t logits_stride,
                                                int logits_dtype, uint64_t seed, uint64_t offset, void* stream) {
  MSGL_REQUIRE(rows >= 0, "sample_filtered_logits: negative rows");
  if (rows == 0) return MSGL_OK;
  MSGL_REQUIRE(out && logits && temperatures && !kept == !kept_temperatures, "sample_filtered_logits: null pointer");
  MSGL_REQUIRE(vocab >= 1 && vocab < (1ll << 31) && rows < (1ll << 31), "sample_filtered_logits: bad shape");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t groups = rows + (kept ? rows * ((vocab + kCopySlice - 1) / kCopySlice) : 0);
  MSGL_REQUIRE(groups < (1ll << 31), "sample_filtered_logits: too many rows");
  const dim3 g((unsigned)groups), b(kRowThreads);
#define MSGL_SAMPLE(DT, ESZ)                                                                                                       \
  sample_filtered_logits_kernel<DT><<<g, b, 0, s>>>(out, (const char*)logits, temperatures, top_k, top_p, vocab, logits_stride * ESZ, \
                                                    (u64)seed, (u64)offset, (int)rows, (char*)kept, kept_temperatures)
  if (logits_dtype == MSGL_F32) MSGL_SAMPLE(MSGL_F32, 4);
  else if (logits_dtype == MSGL_BF16) MSGL_SAMPLE(MSGL_BF16, 2);
  else if (logits_dtype == MSGL_FP16) MSGL_SAMPLE(MSGL_FP16, 2);
  else {
    set_error("sample_filtered_logits: unsupported dtype code %d", logits_dtype);
    return MSGL_EINVAL;
  }
#undef MSGL_SAMPLE
  MSGL_CHECK_LAUNCH("sample_filtered_logits");
  return MSGL_OK;
}

extern "C" int msgl_sample_filtered_logits(int32_t* out, const void* logits, const float* temperatures, const int32_t* top_k,
                                           const float* top_p, int64_t rows, int64_t vocab, int64_t logits_stride, int logits_dtype,
                                           uint64_t seed, uint64_t offset, void* stream) {
  return msgl_sample_filtered_logits_keep(out, nullptr, nullptr, logits, temperatures, top_k, top_p, rows, vocab, logits_stride, logits_dtype, seed,
                                          offset, stream);
}

extern "C" int msgl_sample_from_logits(int32_t* out, const void* logits, const float* temperatures, int64_t rows,
                                       int64_t vocab, int64_t logits_stride, int logits_dtype, uint64_t seed,
                                       uint64_t offset, void* stream) {
  MSGL_REQUIRE(rows >= 0, "sample_from_logits: negative rows");
  if (rows == 0) return MSGL_OK;
  MSGL_REQUIRE(out && logits && temperatures, "sample_from_logits: null pointer");
  MSGL_REQUIRE(vocab >= 1 && vocab < (1ll << 31) && rows < (1ll << 31), "sample_from_logits: bad shape");
  const int esz = logits_dtype == MSGL_F32 ? 4 : 2;
  MSGL_REQUIRE(aligned16(logits) && (logits_stride * esz) % 16 == 0,
               "sample_from_logits: rows must be 16-byte aligned (stride %lld elements)", (long long)logits_stride);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 g((unsigned)rows), b(kRowThreads);
  if (logits_dtype == MSGL_F32)
    sample_logits_kernel<MSGL_F32><<<g, b, 0, s>>>(out, (const char*)logits, temperatures, vocab, logits_stride * esz, (u64)seed, (u64)offset);
  else if (logits_dtype == MSGL_BF16)
    sample_logits_kernel<MSGL_BF16><<<g, b, 0, s>>>(out, (const char*)logits, temperatures, vocab, logits_stride * esz, (u64)seed, (u64)offset);
  else if (logits_dtype == MSGL_FP16)
    sample_logits_kernel<MSGL_FP16><<<g, b, 0, s>>>(out, (const char*)logits, temperatures, vocab, logits_stride * esz, (u64)seed, (u64)offset);
  else {
    set_error("sample_from_logits: unsupported dtype code %d", logits_dtype);
    return MSGL_EINVAL;
  }
  MSGL_CHECK_LAUNCH("sample_from_logits");
  return MSGL_OK;
}
