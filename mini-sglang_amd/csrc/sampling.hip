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

template <int kCtrl>
__device__ __forceinline__ u64 add_dpp_u64(u64 v) {
  const uint32_t lo = __builtin_amdgcn_mov_dpp((int)(uint32_t)v, kCtrl, 0xf, 0xf, true), hi = __builtin_amdgcn_mov_dpp((int)(uint32_t)(v >> 32), kCtrl, 0xf, 0xf, true);
  return v + ((u64)hi << 32 | lo);
}
__device__ __forceinline__ u64 wave_sum_u64(u64 v) {
  v = add_dpp_u64<kDppXor1>(v);
  v = add_dpp_u64<kDppXor2>(v);
  v = add_dpp_u64<kDppHalfMirror>(v);
  v = add_dpp_u64<kDppRowMirror>(v);
  const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)v, (uint32_t)v, false, false), hi = __builtin_amdgcn_permlane16_swap((uint32_t)(v >> 32), (uint32_t)(v >> 32), false, false);
  const uint32_t l0 = lo[0], l1 = lo[1], h0 = hi[0], h1 = hi[1];
  v = ((u64)h0 << 32 | l0) + ((u64)h1 << 32 | l1);
  const auto lo2 = __builtin_amdgcn_permlane32_swap((uint32_t)v, (uint32_t)v, false, false), hi2 = __builtin_amdgcn_permlane32_swap((uint32_t)(v >> 32), (uint32_t)(v >> 32), false, false);
  const uint32_t m0 = lo2[0], m1 = lo2[1], i0 = hi2[0], i1 = hi2[1];
  return ((u64)i0 << 32 | m0) + ((u64)i1 << 32 | m1);
}

__device__ __forceinline__ u64 block_sum_u64(u64 v, u64* lds_w) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  v = wave_sum_u64(v);
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
constexpr u64 kNoMass = ~0ull;
constexpr u64 kSure = 1ull << 63;
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

// inclusive prefix sum over a wave's lanes: within rows of 16, then row by row
__device__ __forceinline__ int wave_prefix_incl(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15 to rows 1 and 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31 to rows 2 and 3
  return x;
}

// A lower bound of the `target`-th largest of the workgroup's 1024 weights, one per thread: the lower end of the 8th of an octave that holds it,
// 0 below 2^-126.  One histogram, spread over all octaves up to weight 1: the exact one takes four, the upper ones with all 1024 in a few bins
// (64 rows x 151936: 5 us of a draw).  (With 16ths down to 2^-63 only, rows whose k-th largest number lies below went to the radix levels: at
// temperatures under 0.5 that is a distance of 20 between the logits.  256 x 151936 of deviation 10 at temperatures of 0.4 - 1: 109 us, now 42.)
__device__ __forceinline__ uint32_t kth_bound_in(uint32_t bits, int target, uint32_t* hist, uint32_t* s_one) {  // hist and *s_one are zero
  constexpr int kShift = 20;  // bins of a weight's bits; weight 1 is bin 1016
  const int tid = threadIdx.x;
  if (bits >> kShift) atomicAdd(&hist[min(bits >> kShift, 1023u)], 1u);
  __syncthreads();
  if (tid < 64) {  // lane l owns the bins 1023 - 16 l ... 1008 - 16 l
    int c[16], mine = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint4 h = *reinterpret_cast<const uint4*>(hist + 1020 - 16 * tid - 4 * q);
      c[4 * q] = (int)h.w; c[4 * q + 1] = (int)h.z; c[4 * q + 2] = (int)h.y; c[4 * q + 3] = (int)h.x;
    }
#pragma unroll
    for (int q = 0; q < 16; ++q) mine += c[q];
    int above = wave_prefix_incl(mine);
    above -= mine;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      if (above < target && target <= above + c[q]) *s_one = (uint32_t)(1023 - 16 * tid - q) << kShift;
      above += c[q];
    }
  }
  __syncthreads();
  return *s_one;
}

__device__ __forceinline__ uint32_t kth_bound(uint32_t bits, int target, uint32_t* hist, uint32_t* s_one) {
  hist[threadIdx.x] = 0u;
  if (threadIdx.x == 0) *s_one = 0u;
  __syncthreads();
  return kth_bound_in(bits, target, hist, s_one);
}

constexpr int kList = 2048;          // candidates of a row that the short path holds (= kBins: it reuses the histograms)
constexpr int kListTopK = 1024;      // largest top-k it is tried for: one column maximum per thread bounds the k-th largest from below
// candidates asked for when only a mass is given: a list takes time with its square, and a nucleus that does not fit pays for it on top (bf16 rows,
// top-p 0.9, one row of 151936, one thread a candidate: nucleus 8: 55 us with 64, 91 with 256, 157 with 512, 219 without; nucleus 2127: 141, 185,
// 225, 217)
constexpr int kListTopP = 64;

struct __attribute__((aligned(16))) RowShared {
  uint32_t h_cnt[kBins];  // histogram | candidates' probability bits
  u64 h_mass[kBins];      // histogram | candidates' masses
  int s_index[kList];
  u64 acc[kRowThreads];          // sums per candidate
  uint32_t acc_n[kRowThreads / 2];
  u64 lds_w[kRowThreads / 64];
  float lds_f[kRowThreads / 64];
  uint32_t s_digit, s_two[2];
  int s_pick, s_n;
};

__device__ __forceinline__ u64 mass_target(float pp, u64 kept_mass) {
  u64 target = (u64)((double)pp * (double)kept_mass);
  if (target < 1) target = 1;
  if (target > kept_mass) target = kept_mass;
  return target;
}

// Philox's number x, scaled to [0, total): (total * x) >> 32 without 128-bit arithmetic
__device__ __forceinline__ u64 draw_below(u64 total, uint32_t x) {
  return (total >> 32) * (u64)x + (((total & 0xffffffffull) * (u64)x) >> 32);
}

// The draw where the list (n candidates, their weights' bits in h_cnt) holds all that it needs; false where the threshold lies below the
// list.  kept_mass: set to the whole row's mass where only a mass is given.  s_pick is -1 on entry.
template <class Src>
__device__ __forceinline__ bool draw_from_list(const Src& src, RowShared& sh, int* __restrict__ out, int n, uint32_t floor_bits, bool by_count, int64_t k,
                                               float pp, int64_t vocab, u64 seed, u64 offset, int64_t r, u64& kept_mass) {
  const int tid = threadIdx.x;
  const bool by_mass = !by_count;
  const uint32_t number = Philox::draw(seed, offset + r);  // (beside the first barrier's wait)
  // Every candidate against every other one: `cp` candidates side by side, the others in `parts` portions whose sums meet in LDS.
  // 64 rows, lists of some 110: two such comparisons and the rest of the draw take 24 us with one thread a candidate, 8 so.
  constexpr int kOwn = kList / kRowThreads;
  int cp = 64;
  while (cp < n && cp < kRowThreads) cp *= 2;
  const int parts = kRowThreads / cp, part = tid / cp, c0 = tid - part * cp;
  for (int c = tid; c < n; c += kRowThreads) {
    const float p = src.prob(__uint_as_float(sh.h_cnt[c]));
    sh.h_mass[c] = fixed_mass(p) | (sh.h_cnt[c] >= floor_bits ? kSure : 0ull);  // kSure: not among the few below the floor, of whose equals some may be missing
    sh.h_cnt[c] = __float_as_uint(p);
  }
  if (tid < kRowThreads / 2) sh.acc[tid] = sh.acc[tid + kRowThreads / 2] = sh.acc_n[tid] = 0;
  u64 target = 0;
  if (by_mass) {
    u64 loc = 0;
    walk_row(src, vocab, [&](int64_t, float x, bool in) {
      const u64 m = fixed_mass(src.prob(src.weight(x)));
      loc += in ? m : 0ull;
    });
    kept_mass = block_sum_u64(loc, sh.lds_w);
    target = mass_target(pp, kept_mass);
  }
  if (tid == 0) sh.s_digit = kNoDigit;
  __syncthreads();
  u64 m_above[kOwn], m_same[kOwn];
  int c_above[kOwn], c_same[kOwn];
#pragma unroll
  for (int e = 0; e < kOwn; ++e) {
    m_above[e] = m_same[e] = 0;
    c_above[e] = c_same[e] = 0;
    const int c = c0 + e * kRowThreads;
    if (c >= n || (e > 0 && cp < kRowThreads)) continue;
    const uint32_t own = sh.h_cnt[c];
#pragma unroll 4
    for (int j = part; j < n; j += parts) {
      const uint32_t b = sh.h_cnt[j];
      const u64 m = sh.h_mass[j] & ~kSure;
      c_above[e] += b > own;
      c_same[e] += b == own;
      m_above[e] += b > own ? m : 0ull;
      m_same[e] += b == own ? m : 0ull;
    }
    if (parts > 1) {
      atomicAdd(&sh.acc[c], m_above[e]);
      atomicAdd(&sh.acc[cp + c], m_same[e]);
      atomicAdd(&sh.acc_n[c], (uint32_t)c_above[e] | (uint32_t)c_same[e] << 16);
    }
  }
  if (parts > 1) {
    __syncthreads();
    m_above[0] = sh.acc[c0];
    m_same[0] = sh.acc[cp + c0];
    c_above[0] = (int)(sh.acc_n[c0] & 0xffffu);
    c_same[0] = (int)(sh.acc_n[c0] >> 16);
  }
#pragma unroll
  for (int e = 0; e < kOwn; ++e) {
    const int c = c0 + e * kRowThreads;
    if (c >= n || (e > 0 && cp < kRowThreads)) continue;
    const bool here = by_count ? c_above[e] < k && k <= c_above[e] + c_same[e] : m_above[e] < target && target <= m_above[e] + m_same[e];
    if ((sh.h_mass[c] & kSure) && here) {  // equal candidates write equal words
      sh.s_digit = sh.h_cnt[c];
      sh.lds_w[0] = m_above[e] + m_same[e];
    }
  }
  __syncthreads();
  const uint32_t found = sh.s_digit;
  const u64 found_mass = sh.lds_w[0];
  __syncthreads();
  if (found == kNoDigit || (by_mass && kept_mass == 0)) return false;
  uint32_t thr_bits = found;
  if (by_count && pp < 1.0f && found_mass > 0) {
    target = mass_target(pp, found_mass);
#pragma unroll
    for (int e = 0; e < kOwn; ++e) {
      const int c = c0 + e * kRowThreads;
      if (c < n && (e == 0 || cp == kRowThreads) && sh.h_cnt[c] >= thr_bits && m_above[e] < target && target <= m_above[e] + m_same[e])
        sh.s_digit = sh.h_cnt[c];
    }
    __syncthreads();
    thr_bits = sh.s_digit;
  }
  // the draw over the list, in index order
  u64 loc = 0;
  for (int c = tid; c < n; c += kRowThreads) {
    const u64 m = sh.h_cnt[c] >= thr_bits ? sh.h_mass[c] & ~kSure : 0ull;  // what is left out weighs nothing from here on
    sh.h_mass[c] = m;
    loc += m;
  }
  sh.acc[tid] = 0;
  const u64 total = block_sum_u64(loc, sh.lds_w);
  const u64 u = draw_below(total, number);
#pragma unroll
  for (int e = 0; e < kOwn; ++e) {
    const int c = c0 + e * kRowThreads;
    if (c >= n || (e > 0 && cp < kRowThreads)) continue;
    const int idx = sh.s_index[c];
    u64 before = 0;
#pragma unroll 4
    for (int j = part; j < n; j += parts) before += sh.s_index[j] < idx ? sh.h_mass[j] : 0ull;
    if (parts > 1) atomicAdd(&sh.acc[c], before);
    else if (u >= before && u < before + sh.h_mass[c]) sh.s_pick = idx;
  }
  __syncthreads();
  if (parts > 1) {
    if (tid < n && u >= sh.acc[tid] && u < sh.acc[tid] + sh.h_mass[tid]) sh.s_pick = sh.s_index[tid];
    __syncthreads();
  }
  if (tid == 0) out[r] = sh.s_pick < 0 ? 0 : sh.s_pick;
  return true;
}

// The draw by three radix levels over the whole row and a walk in index order.  kept_mass: the whole row's, where it is known.
template <class Src>
__device__ __forceinline__ void draw_from_row(const Src& src, RowShared& sh, int* __restrict__ out, int64_t k, float pp, int64_t vocab, u64 seed, u64 offset,
                                              int64_t r, u64 kept_mass) {
  const int tid = threadIdx.x;
  const bool has_k = k >= 1 && k < vocab;
  uint32_t thr_bits = 0u;  // keep set = { bits >= thr_bits, p > 0 }
  if (has_k) {
    // fewer than k positive probabilities (a low temperature underflows the tail to 0): top-k keeps all of them,
    // as flashinfer does -- no threshold; ties at the k-th largest value stay in the keep set
    // (such a row comes here past its list: 64 rows x 151936 at temperature 0.02, k 1000: 100 us, 295 over stored probabilities)
    const uint32_t v = select_bits<false>(src, vocab, 0u, (u64)k, sh.h_cnt, sh.h_mass, sh.lds_w, &sh.s_digit);
    if (v != kNoDigit) thr_bits = v;
  }
  if (pp < 1.0f) {
    if (kept_mass == kNoMass) {
      u64 loc = 0;
      walk_row(src, vocab, [&](int64_t, float x, bool in) {
        const float p = src.prob(src.weight(x));
        if (in && __float_as_uint(p) >= thr_bits) loc += fixed_mass(p);
      });
      kept_mass = block_sum_u64(loc, sh.lds_w);
    }
    const u64 target = mass_target(pp, kept_mass);
    if (kept_mass > 0) {
      const uint32_t v = select_bits<true>(src, vocab, thr_bits, target, sh.h_cnt, sh.h_mass, sh.lds_w, &sh.s_digit);
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
  if (lane == 0) sh.lds_w[w] = wave_mass;
  __syncthreads();
  u64 total = 0, before = 0;
  for (int i = 0; i < kWaves; ++i) {
    if (i < w) before += sh.lds_w[i];
    total += sh.lds_w[i];
  }
  const u64 u = draw_below(total, Philox::draw(seed, offset + r));
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
        if (m[e] > 0 && u >= run + incl - m[e] && u < run + incl) sh.s_pick = (int)(base + e * 64 + lane);
        run += shfl_u64(incl, 63);
      }
      break;
    }
  }
  __syncthreads();
  if (tid == 0) out[r] = sh.s_pick < 0 ? 0 : sh.s_pick;  // degenerate row (all-zero mass): fall back to the first index
}

// One 1024-thread workgroup per row.
//
// Short path (any top-k up to 1024, or a top-p whose nucleus is small): thread t's largest number over the columns t, t + 1024, ...
// is known after one pass; the k-th largest of these 1024 maxima has at least k numbers at or above it, so the second pass collects
// only what reaches a bound just below it -- some k numbers out of a 152 k vocabulary -- and both thresholds and the draw are integer sums over that
// list.  The general path finds the same thresholds by three radix levels over the whole row; it stays for wide nuclei, top-k above
// 1024 and rows whose largest numbers share a column.
//
// Bound: one CU walks one row (304 KB of bf16 logits) twice, an exponential and ~10 VALU operations per element in the second pass.
// 64 rows x 151936 bf16 logits, top-k and top-p: softmax_kernel + radix levels over the stored fp32 probabilities (ten passes, u64 LDS
// atomics for every element of a first level) 551 us; this kernel from the logits 34 us (51 with an exact k-th maximum and one thread a candidate);
// 64 x 35186 16 us.
template <class Src>
__device__ __forceinline__ void sample_row(Src src, int* __restrict__ out, int64_t k, float pp, int64_t vocab, float inv_t, u64 seed, u64 offset) {
  __shared__ RowShared sh;
  const int tid = threadIdx.x;
  const bool has_k = k >= 1 && k < vocab;
  const bool by_count = has_k && k <= kListTopK, by_mass = !has_k && pp < 1.0f;
  int n = 0;

  float col = Src::kSoftmax ? -INFINITY : 0.f;
  if (Src::kSoftmax || by_count || by_mass)
    walk_row(src, vocab, [&](int64_t, float x, bool in) { col = in ? fmaxf(col, x) : col; });
  if constexpr (Src::kSoftmax) {
    src.mx = block_reduce_max(col, sh.lds_f);
    src.k = inv_t * 1.4426950408889634f;
  }
  uint32_t floor_bits = 0u, list_bits = kNoDigit;  // list_bits: what a weight has to reach to be listed
  if (by_count || by_mass) {
    const float w = src.weight(col);
    const int want = (int)(by_count ? k : (int64_t)kListTopP);
    floor_bits = kth_bound(w > 0.f ? __float_as_uint(w) : 0u, want, sh.h_cnt, sh.s_two);  // NaN counts as nothing here
    // weights up to some units in the last place apart can be the same probability: the list starts a little below
    if (floor_bits) list_bits = floor_bits - 8u;
  }
  if (tid == 0) { sh.s_n = 0; sh.s_pick = -1; }
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
        if (lane == 0) at = atomicAdd(&sh.s_n, __popcll(votes));
        at = __shfl(at, 0, 64) + __popcll(votes & ((1ull << lane) - 1ull));
        if (hit && at < kList) {
          sh.s_index[at] = (int)i;
          sh.h_cnt[at] = __float_as_uint(w);
        }
      }
    });
    if constexpr (Src::kSoftmax) src.inv = 1.0f / block_reduce_sum(sum, sh.lds_f);
    __syncthreads();
    n = sh.s_n;
  }
  u64 kept_mass = kNoMass;
  if (list_bits != kNoDigit && n <= kList && draw_from_list(src, sh, out, n, floor_bits, by_count, k, pp, vocab, seed, offset, blockIdx.x, kept_mass)) return;
  draw_from_row(src, sh, out, k, pp, vocab, seed, offset, blockIdx.x, kept_mass);
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

// slice x of all rows' slices: a copy of the row and, with its first slice, its temperature
template <int DT>
__device__ __forceinline__ void copy_slice(int x, const char* __restrict__ logits, const float* __restrict__ temperatures, int64_t vocab,
                                           int64_t row_stride_bytes, char* __restrict__ kept, float* __restrict__ kept_t) {
  using E = std::conditional_t<DT == MSGL_F32, uint32_t, uint16_t>;
  const int slices = (int)((vocab + kCopySlice - 1) / kCopySlice);
  const int64_t r = x / slices, at = (x - r * slices) * kCopySlice;
  copy_numbers(reinterpret_cast<E*>(kept) + r * vocab + at, reinterpret_cast<const E*>(logits + r * row_stride_bytes) + at, min(kCopySlice, vocab - at));
  if (at == 0 && threadIdx.x == 0) kept_t[r] = temperatures[r];
}

// Workgroups 0 .. rows - 1 draw; with `kept` those behind them copy the rows in slices, on compute units that the draw leaves idle (64 rows x
// 151936 bf16: 2.5 us; the drawing threads storing it 10).
template <int DT>
__global__ __launch_bounds__(kRowThreads) void sample_filtered_logits_kernel(int* __restrict__ out, const char* __restrict__ logits,
                                                                             const float* __restrict__ temperatures,
                                                                             const int* __restrict__ top_k, const float* __restrict__ top_p,
                                                                             int64_t vocab, int64_t row_stride_bytes, u64 seed, u64 offset, int rows,
                                                                             char* __restrict__ kept, float* __restrict__ kept_t) {
  if ((int)blockIdx.x >= rows) {
    copy_slice<DT>((int)blockIdx.x - rows, logits, temperatures, vocab, row_stride_bytes, kept, kept_t);
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

// ------------------------------------------------------------------------------------------
// The same draws with a row's work on several workgroups
//
// One workgroup walks a row of 151936 in two passes that wait for loads, and 64 rows leave 192 of 256 compute units idle.  Here `split`
// workgroups share a row, one launch per point where the whole row has to be known:
//   split_max    each takes a range of the row: 1024 maxima, each of some numbers of the row
//   split_sum    each takes 1024 / split of the columns i mod 1024: weights, every column's sum in the order of the rows (the sum's bits are
//                softmax_kernel's), and the candidates that reach the k-th largest maximum; or, with a mass alone, the mass per 64th of an octave
//   split_mass   each takes some of up to 1024 chunks in index order: the chunk's mass above the 64th of an octave in which the threshold
//                lies, and the candidates within (without a filter: the chunk's mass)
//   split_pick   one workgroup a row: threshold among the candidates, the draw over the list or over chunks and inside one of them; beside them
//                the copy of the rows, but for draws by a mass alone of more than 128 rows, where split_sum writes it (launch_split)
// Thresholds, masses and picks are those of one workgroup (integer sums over the same numbers); a threshold that is not among the candidates
// (ties across the bound, top-k above 1024) falls to draw_from_row, as there.
// Draws with a top-k take sample_team_kernel where a row's share fits its registers.
// Bound: the launches' ends and starts and each one's chain of a few dependent loads and barriers (5.5, 12, 10 us of 27 at 64 x 151936 with top-k, where
// the reads take 8 and the exponentials 2; it was 31 with a tile of split_sum asked for at a time, divisions and dependent scalar loads in front of the first
// load and a barrier more a tile).  us a draw, one workgroup per row -> shared: see split_of.
// ------------------------------------------------------------------------------------------
constexpr int kMaxChunks = kRowThreads;
constexpr int64_t kMostPerGroup = 1 << 17;       // numbers of a row to one workgroup
constexpr int kPart = 1024;                      // candidates that one workgroup of a row lists
constexpr int kTile = 8192;                      // numbers of a row's columns that a workgroup holds at a time
constexpr uint32_t kMassLow = 87u << 23;         // 2^-40: a smaller weight's probability has no mass
constexpr int kMassShift = 17;                   // 64 bins per octave
constexpr int kMassBins = 40 * 64 + 1;           // the last one: weight 1
constexpr int kOctaves = 41;                     // the last one: weight 1
constexpr int kMassSlots = kOctaves * 64 + 64;   // bins (the last octave's up to its 64) and, behind them, the octaves

struct SplitHead {
  float mx;
  uint32_t floor_bits;      // what a weight has to reach to be surely listed
  uint32_t cut_lo, cut_hi;  // weights' bits between which the mass threshold lies
};

struct SplitScratch {
  SplitHead* head;     // [rows]
  float* top;          // [rows][1024] maxima
  float* sum;          // [rows][1024] columns' sums
  int* count;          // [rows][split] candidates found (more than kPart: not all of them are listed)
  u64* list;           // [rows][split][kPart] candidates: weight's bits, index
  u64* chunk;          // [rows][kMaxChunks] masses
  u64* total;          // [rows][split] masses of all
  float* hist;         // [rows][split][kMassSlots]: sums of weights per 64th of an octave (the last: 1 and above), per octave
};

// lays the parts out one behind the other from `base`; returns the bytes
static inline size_t split_layout(SplitScratch* s, char* base, int64_t rows, int split, bool filtered, bool hist) {
  size_t at = 0;
  auto take = [&](size_t bytes) {
    char* p = base + at;
    at += (bytes + 255) & ~(size_t)255;
    return p;
  };
  s->head = reinterpret_cast<SplitHead*>(take(rows * sizeof(SplitHead)));
  s->top = reinterpret_cast<float*>(take(rows * kRowThreads * sizeof(float)));
  s->chunk = reinterpret_cast<u64*>(take(rows * kMaxChunks * sizeof(u64)));
  if (filtered) {
    s->sum = reinterpret_cast<float*>(take(rows * kRowThreads * sizeof(float)));
    s->count = reinterpret_cast<int*>(take(rows * split * sizeof(int)));
    s->list = reinterpret_cast<u64*>(take(rows * split * kPart * sizeof(u64)));
  }
  if (hist) {
    s->total = reinterpret_cast<u64*>(take(rows * split * sizeof(u64)));
    s->hist = reinterpret_cast<float*>(take(rows * split * kMassSlots * sizeof(float)));
  }
  return at;
}

static inline int64_t split_chunk(int64_t vocab) {
  int64_t c = 512;
  while ((vocab + c - 1) / c > kMaxChunks) c *= 2;
  return c;
}

// the eight logits of a thread in a piece of 512 per wave: consecutive ones where rows are 16-byte aligned, 64 apart otherwise
template <int DT, bool VEC>
struct Piece {
  static __device__ __forceinline__ int64_t at(int64_t base, int lane, int e) { return VEC ? base + lane * 8 + e : base + e * 64 + lane; }
  // x[e] is defined where at(base, lane, e) < hi
  static __device__ __forceinline__ void load(const void* row, int64_t base, int lane, int64_t hi, float (&x)[8]) {
    if (VEC && base + lane * 8 + 8 <= hi) {
      load_logits8<DT>(row, base + lane * 8, x);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = at(base, lane, e) < hi ? load_logit<DT>(row, at(base, lane, e)) : -INFINITY;
    }
  }
};

template <int DT, bool VEC>
__global__ __launch_bounds__(kRowThreads, 8) void split_max_kernel(SplitScratch sc, const char* __restrict__ logits, int64_t vocab,
                                                                   int64_t row_stride_bytes, int split) {
  using E = std::conditional_t<DT == MSGL_F32, uint32_t, uint16_t>;
  constexpr int kPer = 16 / sizeof(E);
  const int tid = threadIdx.x;
  const int log_split = __builtin_ctz(split);  // a power of two; divisions in front of the first load are time
  const int64_t r = blockIdx.x >> log_split;
  const int g = (int)blockIdx.x - (int)r * split;
  const char* row = logits + r * row_stride_bytes;
  const int64_t per = (((vocab + split - 1) >> log_split) + 7) & ~7ll;
  const int64_t lo = min(vocab, g * per), hi = min(vocab, lo + per);
  float mx = -INFINITY;
  if constexpr (VEC) {
    constexpr int kDeep = 4;
    const int64_t wide = lo + (hi - lo) / kPer * kPer;
    for (int64_t base = lo + tid * kPer; base < wide; base += kDeep * kRowThreads * kPer) {
      U4 raw[kDeep];
#pragma unroll
      for (int u = 0; u < kDeep; ++u) raw[u] = ldg16(reinterpret_cast<const E*>(row) + min(base + u * kRowThreads * kPer, wide - kPer));
#pragma unroll
      for (int u = 0; u < kDeep; ++u) {
        const int64_t i = base + u * kRowThreads * kPer;
        if (i >= wide) break;
        const E* e = reinterpret_cast<const E*>(&raw[u]);
#pragma unroll
        for (int q = 0; q < kPer; ++q) mx = fmaxf(mx, load_logit<DT>(e, q));
      }
    }
    if (wide + tid < hi) mx = fmaxf(mx, load_logit<DT>(row, wide + tid));
  } else {
    constexpr int kDeep = 8;
    for (int64_t base = lo + tid; base < hi; base += kDeep * kRowThreads) {
      float x[kDeep];
#pragma unroll
      for (int u = 0; u < kDeep; ++u) x[u] = load_logit<DT>(row, min(base + u * kRowThreads, hi - 1));
#pragma unroll
      for (int u = 0; u < kDeep; ++u)  // (a number counts once: the k-th largest of the maxima is to bound the k-th largest number)
        if (base + u * kRowThreads < hi) mx = fmaxf(mx, x[u]);
    }
  }
  for (int d = 1; d < split; d <<= 1) mx = fmaxf(mx, __shfl_xor(mx, d, 64));  // one maximum per `split` neighbours
  if ((tid & (split - 1)) == 0) sc.top[r * kRowThreads + g * (kRowThreads >> log_split) + (tid >> log_split)] = mx;
}

// MASS: mass per bin of the weights; else the list of candidates
template <int DT, bool VEC, bool MASS>
__global__ __launch_bounds__(kRowThreads, VEC && MASS ? 8 : 4) void split_sum_kernel(SplitScratch sc, const char* __restrict__ logits, const float* __restrict__ temperatures,
                                                                   const int* __restrict__ top_k, const float* __restrict__ top_p, int64_t vocab,
                                                                   int64_t row_stride_bytes, int split, char* __restrict__ kept, float* __restrict__ kept_t) {
  using E = std::conditional_t<DT == MSGL_F32, float, uint16_t>;
  __shared__ __attribute__((aligned(16))) float tiles[2][kTile];  // one is summed while the next is filled
  __shared__ uint32_t pool[MASS ? kOctaves * 64 : 1];  // weights per bin, each to 15 bits: no more than kMostPerGroup of them go in
  __shared__ __attribute__((aligned(16))) uint32_t hist[MASS ? 4 : kRowThreads];
  __shared__ float lds_f[kRowThreads / 64];
  __shared__ uint32_t s_bound;
  __shared__ int s_n;
  const int tid = threadIdx.x, lane = tid & 63;
  const int log_split = __builtin_ctz(split);  // a power of two; divisions in front of the first load are time
  const int64_t r = blockIdx.x >> log_split;
  const int g = (int)blockIdx.x - (int)r * split;
  const char* row = logits + r * row_stride_bytes;
  const int cols = kRowThreads >> log_split, high = kTile / kRowThreads << log_split;  // columns of this workgroup, rows of 1024 per tile
  const float top = sc.top[r * kRowThreads + tid];  // in front of the numbers: they come back in the order of the requests

  // eight numbers per thread and tile: of one row of 1024 where they can be loaded at once, else of eight rows
  const int log_cols = 10 - log_split;
  static_assert(kRowThreads == 1 << 10, "columns");
  const int at_row = tid >> (VEC ? log_cols - 3 : log_cols), at_col = VEC ? (tid & ((cols >> 3) - 1)) * 8 : tid & (cols - 1);
  auto slot = [&](int e) { return VEC ? at_row * cols + at_col + e : (at_row + e * (high / 8)) * cols + at_col; };
  // (a row has fewer than split x kMostPerGroup = 2^21 numbers at most, a step is 2^17 at most: their sums, six steps past the row included, fit 32 bits)
  const uint32_t width = (uint32_t)vocab, step = kTile * split;
  auto index = [&](uint32_t base, int e) { return base + (VEC ? at_row : at_row + e * (high / 8)) * kRowThreads + g * cols + at_col + (VEC ? e : 0); };
  // Several tiles are asked for ahead, all that a row of 151936 has on four workgroups: with one, a tile took a loaded memory's latency.
  constexpr int kDeep = !VEC ? 1 : MASS ? 2 : DT == MSGL_F32 ? 3 : 5;
  struct alignas(16) Eight {
    E e[8];
  };
  Eight raw[kDeep];
  auto load = [&](uint32_t base, Eight& x) __attribute__((always_inline)) {
    if (VEC && (base + step <= width || index(base, 0) + 8 <= width)) {
#pragma unroll
      for (int h = 0; h < (int)sizeof(Eight) / 16; ++h) reinterpret_cast<U4*>(&x)[h] = ldg16(reinterpret_cast<const char*>(reinterpret_cast<const E*>(row) + index(base, 0)) + 16 * h);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) x.e[e] = index(base, e) < width ? reinterpret_cast<const E*>(row)[index(base, e)] : (E)0;
    }
  };
#pragma unroll
  for (int u = 0; u < kDeep; ++u)
    if (u == 0 || u * step < width) load(u * step, raw[u]);
  const float pp = top_p ? top_p[r] : 1.0f, temperature = temperatures[r];
  const int64_t kk = !MASS && top_k ? (int64_t)top_k[r] : 0;

  const float mx = block_reduce_max(top, lds_f), k = 1.0f / temperature * 1.4426950408889634f;
  const bool mass = MASS && pp < 1.0f;
  uint32_t list_bits = kNoDigit;
  if constexpr (MASS) {
    if (mass)
      for (int b = tid; b < kOctaves * 64; b += kRowThreads) pool[b] = 0u;
  } else {
    const bool has_k = kk >= 1 && kk < vocab, by_count = has_k && kk <= kListTopK;
    uint32_t floor_bits = 0u;
    if (by_count || (!has_k && pp < 1.0f)) {
      const float w = __builtin_amdgcn_exp2f((top - mx) * k);
      floor_bits = kth_bound(w > 0.f ? __float_as_uint(w) : 0u, (int)(by_count ? kk : (int64_t)kListTopP), hist, &s_bound);  // NaN counts as nothing here
    }
    if (floor_bits) list_bits = floor_bits - 8u;  // see sample_row
    if (tid == 0) s_n = list_bits == kNoDigit ? kList + 1 : 0;
    if (g == 0 && tid == 0) sc.head[r].floor_bits = floor_bits;
  }
  if (g == 0 && tid == 0) {
    sc.head[r].mx = mx;
    if (MASS && kept) kept_t[r] = temperature;
  }
  __syncthreads();

  u64* list = sc.list + (r * split + g) * kPart;
  float sum = 0.f;
  int image = 0;
  auto one_tile = [&](uint32_t base, Eight& held) __attribute__((always_inline)) {
    float* tile = tiles[image];
    image ^= 1;
    float w[8], most = 0.f;
    if (MASS && kept && index(base, 0) + 8 <= width) {
#pragma unroll
      for (int h = 0; h < (int)sizeof(Eight) / 16; ++h)
        reinterpret_cast<U4*>(kept + ((int64_t)r * vocab + index(base, 0)) * sizeof(E))[h] = reinterpret_cast<const U4*>(&held)[h];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) w[e] = __builtin_amdgcn_exp2f((load_logit<DT>(held.e, e) - mx) * k);
    if (base + step > width) {  // (the row's last tile)
#pragma unroll
      for (int e = 0; e < 8; ++e) w[e] = index(base, e) < width ? w[e] : 0.f;  // a zero more leaves a sum as it is
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) most = fmaxf(most, w[e]);
    if constexpr (VEC) {
      *reinterpret_cast<float4*>(tile + slot(0)) = float4{w[0], w[1], w[2], w[3]};
      *reinterpret_cast<float4*>(tile + slot(4)) = float4{w[4], w[5], w[6], w[7]};
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) tile[slot(e)] = w[e];
    }
    if (base + kDeep * step < width) load(base + kDeep * step, held);
    if constexpr (MASS) {
      if (mass) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t b = __float_as_uint(w[e]);
          if (w[e] > 0.f && b >= kMassLow) atomicAdd(&pool[min((b - kMassLow) >> kMassShift, (uint32_t)kMassBins - 1u)], ((b & 0x7fffffu) + 0x800100u) >> 9);
        }
      }
    } else if (__any(__float_as_uint(most) >= list_bits)) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const bool hit = w[e] > 0.f && __float_as_uint(w[e]) >= list_bits;
        const u64 votes = __ballot(hit);
        if (votes) {
          int at = 0;
          if (lane == 0) at = atomicAdd(&s_n, __popcll(votes));
          at = __shfl(at, 0, 64) + __popcll(votes & ((1ull << lane) - 1ull));
          if (hit && at < kPart) list[at] = (u64)__float_as_uint(w[e]) << 32 | index(base, e);
        }
      }
    }
    __syncthreads();
    if (tid < cols) {
#pragma unroll 16
      for (int q = 0; q < high; ++q) sum += tile[q * cols + tid];
    }
  };
  for (uint32_t base = 0; base < width; base += kDeep * step) {
#pragma unroll
    for (int u = 0; u < kDeep; ++u)
      if (base + u * step < width) one_tile(base + u * step, raw[u]);
  }
  if (tid < cols) sc.sum[r * kRowThreads + g * cols + tid] = sum;
  if constexpr (MASS) {
    if (mass) {
      float* to = sc.hist + ((int64_t)r * split + g) * kMassSlots;
      for (int o = tid >> 6; o < kOctaves; o += kRowThreads / 64) {
        const float m = ldexpf((float)pool[o * 64 + lane], o - 54), all = wave_sum(m);
        to[o * 64 + lane] = m;
        if (lane == 0) to[kOctaves * 64 + o] = all;
      }
    }
  } else {
    if (tid == 0) sc.count[r * split + g] = s_n;
  }
}

// FILTER: a top-p per row (1 and above: every probability); else masses of the weights, as sample_logits_kernel's
template <int DT, bool VEC, bool FILTER>
__global__ __launch_bounds__(kRowThreads, 8) void split_mass_kernel(SplitScratch sc, const char* __restrict__ logits, const float* __restrict__ temperatures,
                                                                    const float* __restrict__ top_p, int64_t vocab, int64_t row_stride_bytes, int split,
                                                                    int64_t chunk) {
  __shared__ u64 lds_w[kRowThreads / 64];
  __shared__ float lds_f[kRowThreads / 64];
  __shared__ int s_n, s_bin[2];
  const int tid = threadIdx.x, lane = tid & 63;
  const int log_split = __builtin_ctz(split);  // a power of two; divisions in front of the first load are time
  const int64_t r = blockIdx.x >> log_split;
  const int g = (int)blockIdx.x - (int)r * split;
  const char* row = logits + r * row_stride_bytes;
  const int64_t chunks = (vocab + chunk - 1) >> __builtin_ctzll(chunk);  // a power of two
  const int64_t c0 = (int64_t)(tid >> 6) * split + g;
  float x[8];
  if constexpr (!FILTER) Piece<DT, VEC>::load(row, c0 * chunk, lane, min(vocab, (c0 + 1) * chunk), x);

  const float mx = FILTER ? sc.head[r].mx : block_reduce_max(sc.top[r * kRowThreads + tid], lds_f);
  const float inv_t = 1.0f / temperatures[r];
  const float k = FILTER ? inv_t * 1.4426950408889634f : 1.4426950408889634f / temperatures[r];  // each as the kernel whose picks these are
  const float pp = FILTER && top_p ? top_p[r] : 1.0f;
  float inv = 1.0f;
  uint32_t cut_lo = 0u, cut_hi = 0u;  // candidates: weights in [cut_lo, cut_hi); counted: those from cut_hi on
  if constexpr (FILTER) {
    inv = 1.0f / block_reduce_sum(sc.sum[r * kRowThreads + tid], lds_f);
    if (pp < 1.0f) {
      // Mass of the weights from the top, octave by octave and then inside one (a wave, lane l the l-th from the top): the sums are off from the
      // probabilities' by less than `off`.
      if (tid < 64) {
        const float* h = sc.hist + (int64_t)r * split * kMassSlots;
        auto masses = [&](int slot, bool in) {
          float m = 0.f;
          if (in)
            for (int q = 0; q < split; ++q) m += h[(int64_t)q * kMassSlots + slot];
          return m;
        };
        auto prefix = [&](float v) {
#pragma unroll
          for (int d = 1; d < 64; d <<= 1) {
            const float o = __shfl_up(v, d, 64);
            if (lane >= d) v += o;
          }
          return v;
        };
        const float oct = masses(kOctaves * 64 + kOctaves - 1 - lane, lane < kOctaves), oct_incl = prefix(oct), all = __shfl(oct_incl, 63, 64);
        const float want = pp * all, off = all * 0x1.4p-15f;
        // the first lane whose sum reaches `at`, the last one with a mass otherwise
        auto reach = [&](float m, float incl, float at) {
          const u64 there = __ballot(m > 0.f && incl >= at), some = __ballot(m > 0.f);
          return there ? __ffsll((long long)there) - 1 : some ? 63 - __clzll((long long)some) : 0;
        };
        int bin[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {  // the highest bin that may hold the threshold, the lowest one
          const float at = q ? want + off : want - off;
          const int o = reach(oct, oct_incl, at);
          const float above = o ? __shfl(oct_incl, o - 1, 64) : 0.f;
          const float m = masses((kOctaves - 1 - o) * 64 + 63 - lane, true);
          bin[q] = (kOctaves - 1 - o) * 64 + 63 - reach(m, above + prefix(m), at);
        }
        if (lane == 0) {
          s_bin[0] = bin[0];
          s_bin[1] = bin[1];
        }
      }
      __syncthreads();
      cut_lo = kMassLow + ((uint32_t)s_bin[1] << kMassShift);
      cut_hi = kMassLow + ((uint32_t)(s_bin[0] + 1) << kMassShift) + 8u;
    }
    if (g == 0 && tid == 0) {
      sc.head[r].cut_lo = cut_lo;
      sc.head[r].cut_hi = cut_hi;
    }
    if (cut_lo) cut_lo -= 8u;  // weights some units in the last place apart can be one probability
    if (tid == 0) s_n = 0;
    __syncthreads();
  }

  u64* list = FILTER ? sc.list + (r * split + g) * kPart : nullptr;
  // fixed_mass without the conversion to 64-bit integers: whole numbers below 2^53 in 64-bit floating point
  auto units = [](float p) { return fmaxf(__builtin_truncf(p * 1099511627776.0f), 0.f); };
  double total = 0;
  for (int64_t c = c0; c < chunks; c += split * (kRowThreads / 64)) {
    const int64_t hi = min(vocab, (c + 1) * chunk);
    double mass = 0;
    for (int64_t base = c * chunk; base < hi; base += 512) {
      if (FILTER || c != c0 || base != c * chunk) Piece<DT, VEC>::load(row, base, lane, hi, x);
      float w[8], most = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        w[e] = Piece<DT, VEC>::at(base, lane, e) < hi ? __builtin_amdgcn_exp2f((x[e] - mx) * k) : 0.f;
        if constexpr (!FILTER) {
          mass += units(w[e]);
        } else {
          const float m = units(w[e] * inv);
          const bool up = __float_as_uint(w[e]) >= cut_hi;
          total += m;
          mass += up ? m : 0.f;
          most = fmaxf(most, up ? 0.f : w[e]);
        }
      }
      if (FILTER && __any(__float_as_uint(most) >= cut_lo && most > 0.f)) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t b = __float_as_uint(w[e]);
          const bool hit = w[e] > 0.f && b >= cut_lo && b < cut_hi;
          const u64 votes = __ballot(hit);
          if (votes) {
            int at = 0;
            if (lane == 0) at = atomicAdd(&s_n, __popcll(votes));
            at = __shfl(at, 0, 64) + __popcll(votes & ((1ull << lane) - 1ull));
            if (hit && at < kPart) list[at] = (u64)b << 32 | (uint32_t)Piece<DT, VEC>::at(base, lane, e);
          }
        }
      }
    }
    const u64 all = wave_sum_u64((u64)mass);
    if (lane == 0) sc.chunk[r * kMaxChunks + c] = all;
  }
  if constexpr (FILTER) {
    const u64 all = block_sum_u64((u64)total, lds_w);
    if (tid == 0) {
      sc.total[r * split + g] = all;
      sc.count[r * split + g] = s_n;
    }
  }
}

// The draw over chunks (thread c: chunk c's mass) and inside the chunk that holds it.  mass_at(i): the mass of index i.
template <class M>
__device__ __forceinline__ void draw_from_chunks(RowShared& sh, int* __restrict__ out, u64 mine, int64_t vocab, int64_t chunk, u64 seed, u64 offset, M mass_at) {
  const int tid = threadIdx.x;
  const u64 incl = block_prefix_incl(mine, sh.lds_w);
  const u64 total = block_sum_u64(mine, sh.lds_w), u = draw_below(total, Philox::draw(seed, offset + blockIdx.x));
  if (tid == 0) sh.s_n = -1;
  __syncthreads();
  if (mine && u >= incl - mine && u < incl) {
    sh.s_n = tid;
    sh.h_mass[0] = incl - mine;
  }
  __syncthreads();
  const int c = sh.s_n;
  if (c < 0) {  // no mass at all: the first index
    if (tid == 0) out[blockIdx.x] = 0;
    return;
  }
  u64 run = sh.h_mass[0];
  const int64_t hi = min(vocab, (c + 1) * chunk);
  for (int64_t base = c * chunk; base < hi; base += kRowThreads) {
    const int64_t i = base + tid;
    const u64 m = i < hi ? mass_at(i) : 0ull;
    const u64 to = run + block_prefix_incl(m, sh.lds_w);
    if (m && u >= to - m && u < to) out[blockIdx.x] = (int)i;  // exactly one index
    if (tid == kRowThreads - 1) sh.h_mass[1] = to;
    __syncthreads();
    run = sh.h_mass[1];
    __syncthreads();
    if (u < run) break;
  }
}

// The lists of a row's workgroups one behind the other, in sh's indices and bits; lane g of each wave has list g's length.  false: not all candidates are listed
__device__ __forceinline__ bool gather_lists(RowShared& sh, const u64* __restrict__ list, int count, int split, int& n) {
  const int tid = threadIdx.x, lane = tid & 63;
  int upto = min(count, kPart + kList);  // (their lengths in the lanes, the places before each in `upto`)
#pragma unroll
  for (int d = 1; d < 16; d <<= 1) {
    const int o = __shfl_up(upto, d, 64);
    if (lane >= d) upto += o;
  }
  const bool listed = !__any(count > kPart) && __shfl(upto, split - 1, 64) <= kList;
  n = listed ? __shfl(upto, split - 1, 64) : 0;
  for (int c = tid; c < n; c += kRowThreads) {
    int g = 0, from = 0;
    for (int q = 0; q < split - 1; ++q) {
      const int end = __builtin_amdgcn_readlane(upto, q);
      if (c >= end) {
        g = q + 1;
        from = end;
      }
    }
    const u64 e = __hip_atomic_load(list + g * kPart + c - from, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // (sample_team_kernel's are of this launch)
    sh.s_index[c] = (int)(uint32_t)e;
    sh.h_cnt[c] = (uint32_t)(e >> 32);
  }
  return listed;
}

enum { kPickList = 0, kPickMass = 1, kPickAny = 2 };

template <int DT, int HOW>
__global__ __launch_bounds__(kRowThreads) void split_pick_kernel(SplitScratch sc, int* __restrict__ out, const char* __restrict__ logits,
                                                                 const float* __restrict__ temperatures, const int* __restrict__ top_k,
                                                                 const float* __restrict__ top_p, int64_t vocab, int64_t row_stride_bytes, int split,
                                                                 int64_t chunk, u64 seed, u64 offset, int rows, char* __restrict__ kept,
                                                                 float* __restrict__ kept_t) {
  __shared__ RowShared sh;
  const int tid = threadIdx.x;
  if (HOW != kPickAny && (int)blockIdx.x >= rows) {  // the copy, on compute units that the picks leave idle (64 rows x 151936: 3.5 us in split_max)
    copy_slice<DT>((int)blockIdx.x - rows, logits, temperatures, vocab, row_stride_bytes, kept, kept_t);
    return;
  }
  const int64_t r = blockIdx.x;
  const void* row = logits + r * row_stride_bytes;
  if constexpr (HOW == kPickAny) {
    const int64_t chunks = (vocab + chunk - 1) >> __builtin_ctzll(chunk);  // a power of two
    const u64 mine = tid < chunks ? sc.chunk[r * kMaxChunks + tid] : 0ull;
    const float mx = block_reduce_max(sc.top[r * kRowThreads + tid], sh.lds_f), k = 1.4426950408889634f / temperatures[r];
    draw_from_chunks(sh, out, mine, vocab, chunk, seed, offset, [&](int64_t i) { return exp_mass(load_logit<DT>(row, i), mx, k); });
    return;
  }
  // everything that is asked for by the row alone at once, then the list, then the sums' meeting
  const int lane = tid & 63, count = lane < split ? sc.count[r * split + lane] : 0;
  const SplitHead head = sc.head[r];
  const float sum = sc.sum[r * kRowThreads + tid], temperature = temperatures[r];
  const int64_t kk = top_k ? (int64_t)top_k[r] : vocab;
  const float pp = top_p ? top_p[r] : 1.0f;
  int n;
  const bool listed = gather_lists(sh, sc.list + r * split * kPart, count, split, n);
  LogitRow<DT> src{row, head.mx, 1.0f / temperature * 1.4426950408889634f, 1.0f};
  src.inv = 1.0f / block_reduce_sum(sum, sh.lds_f);
  if (tid == 0) sh.s_pick = -1;
  u64 kept_mass = kNoMass;
  if constexpr (HOW == kPickList) {
    const bool by_count = kk >= 1 && kk < vocab;
    __syncthreads();
    if (listed && draw_from_list(src, sh, out, n, head.floor_bits, by_count, kk, pp, vocab, seed, offset, r, kept_mass)) return;
  } else {
    const int64_t chunks = (vocab + chunk - 1) >> __builtin_ctzll(chunk);  // a power of two
    u64 mine = tid < chunks ? sc.chunk[r * kMaxChunks + tid] : 0ull;
    uint32_t thr_bits = 0u;
    bool found = !(pp < 1.0f);
    if (!found) {
      const u64 above = block_sum_u64(mine, sh.lds_w);
      kept_mass = 0;
      for (int h = 0; h < split; ++h) kept_mass += sc.total[r * split + h];
      const u64 target = mass_target(pp, kept_mass);
      // masses by 1024 equal ranges of the candidates' probabilities, then of one range, down to one value
      const uint32_t p_lo = __float_as_uint(src.prob(__uint_as_float(head.cut_lo - 8u)));
      const uint32_t p_hi = __float_as_uint(src.prob(__uint_as_float(head.cut_hi)));
      int shift = 0;
      while (p_hi > p_lo && (p_hi - p_lo) >> shift >= (uint32_t)kRowThreads) ++shift;
      u64 higher = above;
      uint32_t from = p_lo, span = ~0u;  // the threshold is among [from, from + span]
      bool in_list = listed;
#pragma unroll 1
      for (int step = shift; in_list; step = max(0, step - 10)) {  // by 1024 ranges of 2^step
        sh.h_mass[tid] = 0ull;
        if (tid == 0) sh.s_two[0] = kNoDigit;
        __syncthreads();
        for (int c = tid; c < n; c += kRowThreads) {
          const float p = src.prob(__uint_as_float(sh.h_cnt[c]));
          const uint32_t at = __float_as_uint(p) - from;
          if (__float_as_uint(p) >= from && at <= span) atomicAdd(&sh.h_mass[min(at >> step, (uint32_t)kRowThreads - 1u)], fixed_mass(p));
        }
        __syncthreads();
        const u64 m = sh.h_mass[kRowThreads - 1 - tid];  // descending
        const u64 incl = higher + block_prefix_incl(m, sh.lds_w);
        if (incl - m < target && target <= incl) {
          sh.s_two[0] = kRowThreads - 1 - tid;
          sh.h_mass[kRowThreads] = incl - m;
        }
        __syncthreads();
        const uint32_t here = sh.s_two[0];
        if (here == kNoDigit) {
          in_list = false;
        } else {
          higher = sh.h_mass[kRowThreads];
          from += here << step;
          span = (1u << step) - 1u;
        }
        __syncthreads();
        if (step == 0) break;
      }
      if (in_list) {
        if (tid == 0) sh.s_digit = kNoDigit;
        __syncthreads();
        for (int c = tid; c < n; c += kRowThreads)  // surely all of them listed: a weight from the cut's lower end on has this probability
          if (sh.h_cnt[c] >= head.cut_lo && __float_as_uint(src.prob(__uint_as_float(sh.h_cnt[c]))) == from) sh.s_digit = from;
        __syncthreads();
        found = sh.s_digit != kNoDigit && kept_mass > 0;
        thr_bits = found ? from : 0u;
      }
      if (found) {  // candidates that stay, to their chunks
        __syncthreads();
        sh.h_mass[tid] = 0ull;
        __syncthreads();
        for (int c = tid; c < n; c += kRowThreads) {
          const float p = src.prob(__uint_as_float(sh.h_cnt[c]));
          if (__float_as_uint(p) >= thr_bits) atomicAdd(&sh.h_mass[sh.s_index[c] >> __builtin_ctzll(chunk)], fixed_mass(p));
        }
        __syncthreads();
        mine += sh.h_mass[tid];
        __syncthreads();
      }
    }
    if (found) {
      draw_from_chunks(sh, out, mine, vocab, chunk, seed, offset, [&](int64_t i) {
        const float p = src.prob(src.weight(src.raw(i)));
        return __float_as_uint(p) >= thr_bits ? fixed_mass(p) : 0ull;
      });
      return;
    }
    __syncthreads();
  }
  draw_from_row(src, sh, out, kk, pp, vocab, seed, offset, r, kept_mass);
}

// ------------------------------------------------------------------------------------------
// Draws with a top-k in one launch
//
// split_max, split_sum and split_pick's work where a row's share fits a workgroup's registers: the numbers are read once, each by the thread that adds
// it to its column's sum, and the row's workgroups tell each other
//   * their maxima, as packets {value, 1}.  Whoever has waited wait_ticks for one (a workgroup that finds no place on the device beside other work)
//     looks the numbers up itself, so that no workgroup depends on another one's being resident;
//   * their columns' sums and candidates, by a count of those that are done.  Nobody waits: the last one draws, the others copy the row.
// Both are written and read at agent scope (past the L2s); the last one leaves packets and count zero, as it found them, for the next launch.
// Bound: a chain of launch, first read, packets' way, bound, weights, count's way, draw.
// 64 rows x 151936 bf16: 3.3 us to the maxima, 0.7 for the packets, 3.3 to the bound (1.5 of it the slowest wave's reads: 64 addresses of 2 bytes each), 3.4 for
// weights, candidates and sums, 0.8 for the count, 2 for lists and sums (2.9 with the lists behind their lengths), 3.7 for the draw.  us a draw with its copy, three
// launches -> one: 64 x 151936 25.4 -> 19.2, 33 x 151936 23.0 -> 17.7, 8 x 151936 19.4 -> 14.9, 1 x 151936 19.0 -> 14.3, 64 x 98304 21.6 -> 16.7, 64 x 98305
// (unaligned rows) 22.9 -> 17.3.
// Measured on the way (64 x 151936): columns by way of LDS tiles as in split_sum 24.5; the copy from the registers in front of the bound 23.7, by way of LDS
// 23.5, by the workgroups that do not draw 22.0.
// ------------------------------------------------------------------------------------------
constexpr int kTeamDeep = 40;  // numbers of a row that a thread holds,
constexpr int kTeamParts = 4;  // which are one column's in a quarter of the rows of 1024
constexpr int kTeamRows = 64;
constexpr int64_t kTeamBytes = kTeamRows * (kRowThreads * 8 + 64);  // packets, counts 64 bytes apart

// LDS is complete, stores stay under way
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int DT>
__global__ __launch_bounds__(kRowThreads, 4) void sample_team_kernel(SplitScratch sc, char* __restrict__ team, int* __restrict__ out, const char* __restrict__ logits,
                                                                     const float* __restrict__ temperatures, const int* __restrict__ top_k,
                                                                     const float* __restrict__ top_p, int64_t vocab, int64_t row_stride_bytes, int split, u64 seed,
                                                                     u64 offset, char* __restrict__ kept, float* __restrict__ kept_t, int wait_ticks) {
  using E = std::conditional_t<DT == MSGL_F32, float, uint16_t>;
  constexpr int kStep = 8;  // numbers that are looked at together
  __shared__ RowShared sh;
  __shared__ __attribute__((aligned(16))) uint32_t hist[kRowThreads];
  __shared__ float s_sum[kRowThreads / kTeamParts], s_max[kRowThreads / 64];
  __shared__ uint32_t s_bound;
  __shared__ int s_n, s_place;
  const int tid = threadIdx.x, lane = tid & 63;
  const int log_split = __builtin_ctz(split), log_cols = 10 - log_split, cols = 1 << log_cols;  // columns (i mod 1024) of this workgroup: 64, 128 or 256
  const int64_t r = blockIdx.x >> log_split;
  const int g = (int)blockIdx.x - (int)r * split;
  const char* row = logits + r * row_stride_bytes;
  u64* packets = reinterpret_cast<u64*>(team) + r * kRowThreads;
  uint32_t* left = reinterpret_cast<uint32_t*>(team + (int64_t)kTeamRows * kRowThreads * 8) + r * 16;

  // part q's rows of 1024 from first on, `here` of them; a wave is in one part (kTeamParts and more: without numbers)
  const uint32_t width = (uint32_t)vocab;
  const int rows = (int)((width + kRowThreads - 1) / kRowThreads), per = (rows + kTeamParts - 1) / kTeamParts;
  const int q = __builtin_amdgcn_readfirstlane(tid >> log_cols), first = q * per, here = q < kTeamParts ? max(0, min(per, rows - first)) : 0;
  const uint32_t column = g * cols + (tid & (cols - 1)), at0 = (uint32_t)first * kRowThreads + column;
  uint32_t bits[kTeamDeep];
#pragma unroll
  for (int i0 = 0; i0 < kTeamDeep; i0 += kStep) {
    if (i0 < here) {
#pragma unroll
      for (int i = i0; i < i0 + kStep; ++i) bits[i] = __builtin_bit_cast(std::conditional_t<DT == MSGL_F32, uint32_t, uint16_t>, reinterpret_cast<const E*>(row)[min(at0 + i * kRowThreads, width - 1)]);
    }
  }
#pragma unroll
  for (int i = 0; i < kTeamDeep; ++i) asm volatile("" : "+v"(bits[i]));  // all are asked for before one is used (converted eight at a time: 1.5 us more)
  auto number = [&](int i) {
    if constexpr (DT == MSGL_F32) return __uint_as_float(bits[i]);
    else if constexpr (DT == MSGL_BF16) return __uint_as_float(bits[i] << 16);
    else return (float)__builtin_bit_cast(_Float16, (uint16_t)bits[i]);
  };
  auto in_row = [&](int i) { return i < here && at0 + i * kRowThreads < width; };
  const float pp = top_p ? top_p[r] : 1.0f, temperature = temperatures[r];
  const int64_t kk = (int64_t)top_k[r];
  hist[tid] = 0u;
  if (tid == 0) s_bound = 0u;

  // ---- the row's 1024 maxima: of four columns' parts each ----
  float own = -INFINITY;
#pragma unroll
  for (int i0 = 0; i0 < kTeamDeep; i0 += kStep) {
    if (i0 < here) {
#pragma unroll
      for (int i = i0; i < i0 + kStep; ++i) own = fmaxf(own, in_row(i) ? number(i) : -INFINITY);
    }
  }
  own = fmaxf(own, dpp_get<kDppXor1>(own));
  own = fmaxf(own, dpp_get<kDppXor2>(own));
  if (q < kTeamParts && (tid & 3) == 0)
    __hip_atomic_store(packets + g * cols + (tid >> 2), 1ull << 32 | __float_as_uint(own), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  u64 packet = 0;
  const u64 t0 = __builtin_amdgcn_s_memrealtime();
  for (bool more = true; more;) {
    packet = __hip_atomic_load(packets + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    more = packet >> 32 == 0 && (int64_t)(__builtin_amdgcn_s_memrealtime() - t0) < wait_ticks;
  }
  float top = __uint_as_float((uint32_t)packet);
  if (packet >> 32 == 0) {
    const int from = (tid & (cols - 1)) * 4;  // the first thread of these four, in workgroup tid >> log_cols
    const uint32_t at = (uint32_t)(from >> log_cols) * per * kRowThreads + (tid >> log_cols) * cols + (from & (cols - 1));
    top = -INFINITY;
    for (int i = 0; i < min(per, rows - (from >> log_cols) * per); ++i)
      for (int c = 0; c < 4; ++c)
        if (at + i * kRowThreads + c < width) top = fmaxf(top, load_logit<DT>(row, at + i * kRowThreads + c));
  }
  {
    const float m = wave_max(top);
    if (lane == 0) s_max[tid >> 6] = m;
  }
  lds_barrier();
  float mx = s_max[0];
#pragma unroll
  for (int w = 1; w < kRowThreads / 64; ++w) mx = fmaxf(mx, s_max[w]);
  const float k = 1.0f / temperature * 1.4426950408889634f;
  const bool has_k = kk >= 1 && kk < vocab, by_count = has_k && kk <= kListTopK;
  uint32_t floor_bits = 0u, list_bits = kNoDigit;
  if (by_count || (!has_k && pp < 1.0f)) {
    const float w = __builtin_amdgcn_exp2f((top - mx) * k);
    floor_bits = kth_bound_in(w > 0.f ? __float_as_uint(w) : 0u, (int)(by_count ? kk : (int64_t)kListTopP), hist, &s_bound);  // NaN counts as nothing here
  }
  if (floor_bits) list_bits = floor_bits - 8u;  // see sample_row
  if (tid == 0) s_n = list_bits == kNoDigit ? kList + 1 : 0;
  __syncthreads();

  // ---- weights, candidates ----
  u64* list = sc.list + (r * split + g) * kPart;
  float w[kTeamDeep];
#pragma unroll
  for (int i0 = 0; i0 < kTeamDeep; i0 += kStep) {
    if (i0 < here) {
      float most = 0.f;
#pragma unroll
      for (int i = i0; i < i0 + kStep; ++i) {
        w[i] = __builtin_amdgcn_exp2f((number(i) - mx) * k);
        w[i] = in_row(i) ? w[i] : 0.f;
        most = fmaxf(most, w[i]);
      }
      if (__any(__float_as_uint(most) >= list_bits)) {
#pragma unroll
        for (int i = i0; i < i0 + kStep; ++i)
          if (w[i] > 0.f && __float_as_uint(w[i]) >= list_bits) {
            const int at = atomicAdd(&s_n, 1);
            if (at < kPart) __hip_atomic_store(list + at, (u64)__float_as_uint(w[i]) << 32 | (at0 + i * kRowThreads), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
      }
    }
  }
  // ---- the columns' sums, in the order of the rows: part after part ----
#pragma unroll
  for (int part = 0; part < kTeamParts; ++part) {
    if (q == part) {
      float sum = part ? s_sum[tid & (cols - 1)] : 0.f;
#pragma unroll
      for (int i0 = 0; i0 < kTeamDeep; i0 += kStep) {
        if (i0 < here) {
#pragma unroll
          for (int i = i0; i < i0 + kStep; ++i) sum += w[i];  // a zero more leaves a sum as it is
        }
      }
      if (part + 1 < kTeamParts) s_sum[tid & (cols - 1)] = sum;
      else __hip_atomic_store(sc.sum + r * kRowThreads + column, sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (part + 1 < kTeamParts) lds_barrier();
  }
  if (tid == 0) __hip_atomic_store(sc.count + r * split + g, s_n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // what the last one reads is out
  __syncthreads();
  if (tid == 0) s_place = (int)__hip_atomic_fetch_add(left, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const int place = __builtin_amdgcn_readfirstlane(s_place);
  if (place < split - 1) {  // the others copy the row while the last one draws
    if (kept) {
      const int64_t share = ((vocab + split - 2) / (split - 1) + 7) & ~7ll, lo = min(vocab, place * share), hi = min(vocab, lo + share);
      copy_numbers(reinterpret_cast<E*>(kept) + r * vocab + lo, reinterpret_cast<const E*>(row) + lo, hi - lo);
      if (place == 0 && tid == 0) kept_t[r] = temperature;
    }
    return;
  }

  // ---- the draw ----
  const int count = lane < split ? __hip_atomic_load(sc.count + r * split + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
  const float whole = __hip_atomic_load(sc.sum + r * kRowThreads + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const u64 ahead = __hip_atomic_load(sc.list + (r * split + q) * kPart + (tid & (cols - 1)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // list q's: most are no longer
  __hip_atomic_store(packets + tid, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (tid == 0) __hip_atomic_store(left, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  int n;
  bool listed = true;
  if (!__any(count > cols)) {
    const int upto = wave_prefix_incl(count), mine = __builtin_amdgcn_readlane(count, q), before = __builtin_amdgcn_readlane(upto, q) - mine;
    n = __builtin_amdgcn_readlane(upto, 63);
    if ((tid & (cols - 1)) < mine) {
      sh.s_index[before + (tid & (cols - 1))] = (int)(uint32_t)ahead;
      sh.h_cnt[before + (tid & (cols - 1))] = (uint32_t)(ahead >> 32);
    }
  } else {
    listed = gather_lists(sh, sc.list + r * split * kPart, count, split, n);
  }
  LogitRow<DT> src{row, mx, k, 1.0f};
  src.inv = 1.0f / block_reduce_sum(whole, sh.lds_f);
  if (tid == 0) sh.s_pick = -1;
  u64 kept_mass = kNoMass;
  __syncthreads();
  if (listed && draw_from_list(src, sh, out, n, floor_bits, has_k, kk, pp, vocab, seed, offset, r, kept_mass)) return;
  draw_from_row(src, sh, out, kk, pp, vocab, seed, offset, r, kept_mass);
}

// Workgroups per row (1: one walks the row).  One a compute unit in all: 64 rows x 151936, top-p alone, 54 us with 4 each, 58 with 8; 33 rows 51 and 54.
// Where sharing pays, us a draw, shared / one workgroup, bf16:
//   top-k      in three launches (callers without a team's memory), whose line this is: 1 x 151936 20.5 / 25.2, 33 x 151936 29.4 / 31.4, 64 x 151936 29.1 / 34.2,
//              but 8 x 65536 20.4 / 17.5, 100 x 151936 41 / 38.  sample_team_kernel is ahead of these three wherever it can be taken, and of one workgroup already
//              below the line (with top-p, in a graph): 1, 8, 64 x 80000 15.7 / 19.6, 16.3 / 20.4, 20.2 / 24.4, x 65536 15.0 / 16.5, 15.4 / 17.1, 18.7 / 19.8, but x 50304
//              14.8 / 15.3, 15.3 / 15.9, 18.3 / 17.7, x 32000 14.1 / 14.3, 14.9 / 14.9, 16.5 / 15.8, x 16384 14.4 / 10.6, 14.9 / 11.6, 16.0 / 12.0
//   no filter  64 x 65536 16.5 / 17.7, 128 x 98304 24.4 / 25.9, 100 x 151936 29 / 37, but 128 x 65536 20.4 / 18.7, 128 x 50000 18.2 / 15.3,
//              32 x 50000 14.8 / 14.8, 256 x 151936 48 / 44
//   top-p      wide nuclei (logits of deviation 2.5) and, behind them, nuclei of a few tokens in every row (deviation 10), which one workgroup
//              finds in its list of 64 candidates:
//              1 x 32000 32 / 56, 32 / 27     8 x 50304 40 / 69, 39 / 30     64 x 16384 32 / 40, 31 / 25     64 x 50304 36 / 71, 35 / 31
//              64 x 151936 51 / 161, 49 / 57     128 x 151936 72 / 175, 68 / 63     256 x 151936 108 / 195, 99 / 70
//              One wide row sets the time of a batch.  The line lies where sharing saves less on wide rows than it costs on narrow ones:
//              1 x 8200 28 / 33, 28 / 20     8 x 16384 33 / 39, 33 / 22     64 x 8200 31 / 34, 30 / 21     128 x 8200 30 / 35, 30 / 23
static inline int split_of(int64_t rows, int64_t vocab, bool filtered, bool has_k, bool has_p) {
  const bool by_mass = filtered && has_p && !has_k;
  const int64_t most = by_mass ? 256 : has_k ? 64 : 128;
  const int64_t shortest = by_mass ? (rows < 64 ? 32000 : 16384) : has_k || rows > 64 ? 98304 : 65536;
  if (rows > most || vocab < shortest) return 1;
  int split = 16;
  while (split > 2 && (rows * split > 256 || vocab / split < 2048)) split /= 2;
  return vocab / split < kMostPerGroup ? split : 1;
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

// Bytes that the draws straight from logits take to split their rows over several workgroups; 0: one workgroup a row is as good.
// filtered: through the probabilities; has_k, has_p: a top-k, a top-p per row is given.
extern "C" int64_t msgl_sample_workspace_bytes(int64_t rows, int64_t vocab, int filtered, int has_k, int has_p) {
  const int split = rows > 0 && vocab > 0 ? split_of(rows, vocab, filtered, has_k, has_p) : 1;
  SplitScratch sc{};
  return split > 1 ? (int64_t)split_layout(&sc, nullptr, rows, split, filtered, filtered && !has_k) : 0;
}

// One draw per row in three or four launches (see the comment above split_max_kernel).
template <int DT, bool VEC>
static void launch_split(const SplitScratch& sc, int32_t* out, char* kept, float* kept_t, const char* logits, const float* temperatures, const int32_t* top_k,
                         const float* top_p, bool filtered, int64_t rows, int64_t vocab, int64_t stride_bytes, int split, u64 seed, u64 offset, char* team, int wait_ticks,
                         hipStream_t s) {
  // The copy of the rows: beside the picks, on the compute units that these leave idle; where they leave few, by the sums' kernel, which has the
  // rows in registers (us: 202 x 151936, top-p alone 101 beside the picks, 92 with the sums; 105 x 120687 the same; 64 x 151936 with top-k 28, 29)
  if (team && filtered && top_k && rows <= kTeamRows && split >= kTeamParts && vocab <= (int64_t)kTeamDeep * kTeamParts * kRowThreads) {
    sample_team_kernel<DT><<<dim3((unsigned)(rows * split)), dim3(kRowThreads), 0, s>>>(sc, team, out, logits, temperatures, top_k, top_p, vocab, stride_bytes, split, seed,
                                                                                        offset, kept, kept_t, wait_ticks);
    return;
  }
  const bool here = VEC && filtered && !top_k && kept && rows > 128 && vocab % 8 == 0 && aligned16(kept);
  char* const kept_sum = here ? kept : nullptr;
  if (here) kept = nullptr;
  const int64_t copies = kept ? rows * ((vocab + kCopySlice - 1) / kCopySlice) : 0;
  const dim3 many((unsigned)(rows * split)), picks((unsigned)(rows + copies)), b(kRowThreads);
  const int64_t chunk = split_chunk(vocab);
  split_max_kernel<DT, VEC><<<many, b, 0, s>>>(sc, logits, vocab, stride_bytes, split);
  if (!filtered) {
    split_mass_kernel<DT, VEC, false><<<many, b, 0, s>>>(sc, logits, temperatures, top_p, vocab, stride_bytes, split, chunk);
    split_pick_kernel<DT, kPickAny><<<picks, b, 0, s>>>(sc, out, logits, temperatures, top_k, top_p, vocab, stride_bytes, split, chunk, seed, offset,
                                                        (int)rows, kept, kept_t);
  } else if (top_k) {
    split_sum_kernel<DT, VEC, false><<<many, b, 0, s>>>(sc, logits, temperatures, top_k, top_p, vocab, stride_bytes, split, kept_sum, kept_t);
    split_pick_kernel<DT, kPickList><<<picks, b, 0, s>>>(sc, out, logits, temperatures, top_k, top_p, vocab, stride_bytes, split, chunk, seed, offset,
                                                         (int)rows, kept, kept_t);
  } else {
    split_sum_kernel<DT, VEC, true><<<many, b, 0, s>>>(sc, logits, temperatures, top_k, top_p, vocab, stride_bytes, split, kept_sum, kept_t);
    split_mass_kernel<DT, VEC, true><<<many, b, 0, s>>>(sc, logits, temperatures, top_p, vocab, stride_bytes, split, chunk);
    split_pick_kernel<DT, kPickMass><<<picks, b, 0, s>>>(sc, out, logits, temperatures, top_k, top_p, vocab, stride_bytes, split, chunk, seed, offset,
                                                         (int)rows, kept, kept_t);
  }
}

// the workspace laid out, and one draw per row; `name` for errors
static int sample_split(const char* name, void* workspace, int64_t workspace_bytes, int32_t* out, void* kept, float* kept_t, const void* logits,
                        const float* temperatures, const int32_t* top_k, const float* top_p, bool filtered, int64_t rows, int64_t vocab, int64_t logits_stride,
                        int logits_dtype, u64 seed, u64 offset, char* team, int wait_ticks, hipStream_t s) {
  const int split = split_of(rows, vocab, filtered, top_k, top_p), esz = logits_dtype == MSGL_F32 ? 4 : 2;
  SplitScratch sc{};
  const int64_t need = (int64_t)split_layout(&sc, static_cast<char*>(workspace), rows, split, filtered, filtered && !top_k);
  MSGL_REQUIRE(aligned16(workspace) && workspace_bytes >= need, "%s: a workspace of %lld bytes, 16-byte aligned, is needed", name, (long long)need);
  const bool vec = aligned16(logits) && (logits_stride * esz) % 16 == 0;
#define MSGL_SPLIT(DT)                                                                                                                               \
  do {                                                                                                                                               \
    auto* f = vec ? &launch_split<DT, true> : &launch_split<DT, false>;                                                                              \
    f(sc, out, (char*)kept, kept_t, (const char*)logits, temperatures, top_k, top_p, filtered, rows, vocab, logits_stride * esz, split, seed, offset, team, wait_ticks, s); \
  } while (0)
  if (logits_dtype == MSGL_F32) MSGL_SPLIT(MSGL_F32);
  else if (logits_dtype == MSGL_BF16) MSGL_SPLIT(MSGL_BF16);
  else if (logits_dtype == MSGL_FP16) MSGL_SPLIT(MSGL_FP16);
  else {
    set_error("%s: unsupported dtype code %d", name, logits_dtype);
    return MSGL_EINVAL;
  }
#undef MSGL_SPLIT
  MSGL_CHECK_LAUNCH(name);
  return MSGL_OK;
}

// probs path's draw without the probs: same thresholds, same masses, same pick as softmax_temperature + sample_top_k_top_p
extern "C" int msgl_sample_filtered_logits_team(int32_t* out, void* kept, float* kept_temperatures, const void* logits, const float* temperatures,
                                                const int32_t* top_k, const float* top_p, int64_t rows, int64_t vocab, int64_t logits_stride,
                                                int logits_dtype, uint64_t seed, uint64_t offset, void* workspace, int64_t workspace_bytes, void* team,
                                                int64_t team_bytes, int wait_us, void* stream) {
  MSGL_REQUIRE(rows >= 0, "sample_filtered_logits: negative rows");
  if (rows == 0) return MSGL_OK;
  MSGL_REQUIRE(out && logits && temperatures && !kept == !kept_temperatures, "sample_filtered_logits: null pointer");
  MSGL_REQUIRE(vocab >= 1 && vocab < (1ll << 31) && rows < (1ll << 31), "sample_filtered_logits: bad shape");
  hipStream_t s = static_cast<hipStream_t>(stream);
  MSGL_REQUIRE(!team || (aligned16(team) && team_bytes >= kTeamBytes && wait_us >= 0 && wait_us <= 1000000), "sample_filtered_logits: a team of %lld bytes, 16-byte aligned, is needed",
               (long long)kTeamBytes);
  if (workspace && split_of(rows, vocab, true, top_k, top_p) > 1)
    return sample_split("sample_filtered_logits", workspace, workspace_bytes, out, kept, kept_temperatures, logits, temperatures, top_k, top_p, true, rows,
                        vocab, logits_stride, logits_dtype, seed, offset, static_cast<char*>(team), wait_us * 100, s);
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

extern "C" int64_t msgl_sample_team_bytes(void) { return kTeamBytes; }

extern "C" int msgl_sample_filtered_logits_ws(int32_t* out, void* kept, float* kept_temperatures, const void* logits, const float* temperatures,
                                              const int32_t* top_k, const float* top_p, int64_t rows, int64_t vocab, int64_t logits_stride,
                                              int logits_dtype, uint64_t seed, uint64_t offset, void* workspace, int64_t workspace_bytes, void* stream) {
  return msgl_sample_filtered_logits_team(out, kept, kept_temperatures, logits, temperatures, top_k, top_p, rows, vocab, logits_stride, logits_dtype, seed,
                                          offset, workspace, workspace_bytes, nullptr, 0, 0, stream);
}

extern "C" int msgl_sample_filtered_logits_keep(int32_t* out, void* kept, float* kept_temperatures, const void* logits, const float* temperatures,
                                                const int32_t* top_k, const float* top_p, int64_t rows, int64_t vocab, int64_t logits_stride,
                                                int logits_dtype, uint64_t seed, uint64_t offset, void* stream) {
  return msgl_sample_filtered_logits_ws(out, kept, kept_temperatures, logits, temperatures, top_k, top_p, rows, vocab, logits_stride, logits_dtype, seed,
                                        offset, nullptr, 0, stream);
}

extern "C" int msgl_sample_filtered_logits(int32_t* out, const void* logits, const float* temperatures, const int32_t* top_k,
                                           const float* top_p, int64_t rows, int64_t vocab, int64_t logits_stride, int logits_dtype,
                                           uint64_t seed, uint64_t offset, void* stream) {
  return msgl_sample_filtered_logits_keep(out, nullptr, nullptr, logits, temperatures, top_k, top_p, rows, vocab, logits_stride, logits_dtype, seed,
                                          offset, stream);
}

extern "C" int msgl_sample_from_logits_ws(int32_t* out, const void* logits, const float* temperatures, int64_t rows, int64_t vocab,
                                          int64_t logits_stride, int logits_dtype, uint64_t seed, uint64_t offset, void* workspace,
                                          int64_t workspace_bytes, void* stream) {
  MSGL_REQUIRE(rows >= 0, "sample_from_logits: negative rows");
  if (rows == 0) return MSGL_OK;
  MSGL_REQUIRE(out && logits && temperatures, "sample_from_logits: null pointer");
  MSGL_REQUIRE(vocab >= 1 && vocab < (1ll << 31) && rows < (1ll << 31), "sample_from_logits: bad shape");
  const int esz = logits_dtype == MSGL_F32 ? 4 : 2;
  MSGL_REQUIRE(aligned16(logits) && (logits_stride * esz) % 16 == 0,
               "sample_from_logits: rows must be 16-byte aligned (stride %lld elements)", (long long)logits_stride);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (workspace && split_of(rows, vocab, false, false, false) > 1)
    return sample_split("sample_from_logits", workspace, workspace_bytes, out, nullptr, nullptr, logits, temperatures, nullptr, nullptr, false, rows, vocab,
                        logits_stride, logits_dtype, seed, offset, nullptr, 0, s);
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

extern "C" int msgl_sample_from_logits(int32_t* out, const void* logits, const float* temperatures, int64_t rows, int64_t vocab, int64_t logits_stride,
                                       int logits_dtype, uint64_t seed, uint64_t offset, void* stream) {
  return msgl_sample_from_logits_ws(out, logits, temperatures, rows, vocab, logits_stride, logits_dtype, seed, offset, nullptr, 0, stream);
}
