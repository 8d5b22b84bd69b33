// Gated delta rule in blocks of 16 tokens on the fp32 matrix instructions (the token loop: delta_rule_kernel in mix_delta.hip).
//
// Per head, with S [d, dv], decays g_t per key channel (or one per head) and P_t = g_1 ... g_t from the block's start:
//   S_t = g_t S_{t-1} + k_t u_t^T,   u_t = beta_t (v_t - S_{t-1}^T (g_t k_t)),   o_t = S_t^T q_t
// Written from the block's start state S (R_{tj} = g_{j+1} ... g_t per channel):
//   (I + A) u = beta (v - (P k) S),  A_{tj} = beta_t sum_c k_tc R_{tj,c} k_jc  (j < t)
//   o = (P q) S + Q u,               Q_{tj} = sum_c q_tc R_{tj,c} k_jc         (j <= t)
//   S' = P_16 S + (R_{16,j} k_j)^T u
// delta_block_kernel computes, for all blocks at once, W = (I + A)^-1 beta (P k), U = (I + A)^-1 beta v, P q, Q, R_{16} k, P_16;
// delta_walk_kernel walks a request's blocks: u = U - W S, o = (P q) S + Q u, S = P_16 S + (R_{16} k)^T u.
//
// Everything stays fp32: v_mfma_f32_16x16x4_f32 multiplies and adds in fp32.  Ratios of decays are products of at most 15 decays, never
// quotients or exponentials of sums (an exponential of a sum of logarithms loses the digits that the sum's size takes): the pairs (t, j)
// split by the highest bit in which t and j differ, and per level both factors are running products inside a half block.
//
// What bounds it: the walk is a serial chain of blocks per (request, head), 50 fp32 MFMAs of 32 cycles a wave and block plus the meeting in
// LDS (1.4 us a block measured); the block kernel is bound by its instructions (5 waves per SIMD of them at a time) and by memory (49 d + 256 +
// 16 dv floats a block and head written, and read again by the walk).  The token loop was bound by one wave's serial walk: two passes over
// 128 registers a token, in three launches.
// 4 requests of 1500 - 2548 tokens, 16 heads, d = dv = 128, decays per channel: 4038 -> 389 us (blocks 171, walk 219); error against 64
// bits 1.9e-7 -> 1.4e-7.
#include <type_traits>

#include "mix_common.h"

namespace {

__device__ __forceinline__ float sigmoidf_(float z) { return 1.0f / (1.0f + expf(-z)); }
__device__ __forceinline__ float softplusf_(float z) { return z > 20.0f ? z : log1pf(expf(z)); }

// exp(r softplus(z)).  A 32-bit engine takes the library's functions; a 16-bit one (whose z is a bf16 sum) the hardware's exponential and
// logarithm with the parts of the arguments that fp32 drops added back: against float64 the same error (rms 8e-8 for z, r of unit size; the
// product r softplus(z) is what rounds) in a sixth of the instructions (with the library's the block kernel took 208 us, below, for 177).
__device__ __forceinline__ float exp_split(float y) {  // e^y: y log2(e) in two parts
  const float h = y * 1.4426950408889634f;
  const float l = fmaf(y, 1.4426950408889634f, -h) + y * 1.9259629911e-8f;
  const float e = __builtin_amdgcn_exp2f(h);
  return e > 0.f && e < INFINITY ? fmaf(e, l * 0.6931471805599453f, e) : e;  // past the exponents' range (an infinite gate) l is no number
}
__device__ __forceinline__ float decay_of(float r, float z, const float*) { return expf(r * softplusf_(z)); }
__device__ __forceinline__ float decay_of(float r, float z, const bf16_t*) {
  const float t = __builtin_amdgcn_exp2f(-fabsf(z) * 1.4426950408889634f);  // e^-|z| <= 1: its error counts only absolutely
  const float u = 1.0f + t, c = t - (u - 1.0f);                              // u + c = 1 + t
  const float lg = fmaf(c, __builtin_amdgcn_rcpf(u), __builtin_amdgcn_logf(u) * 0.6931471805599453f);
  return exp_split(r * (fmaxf(z, 0.f) + lg));
}

constexpr int kBT = 16;  // tokens per block

// a block's operands of one head in the scratch, in floats
struct BlockPart {
  int d, dv;
  __host__ __device__ int w() const { return 0; }                  // W        [16][d]
  __host__ __device__ int q() const { return kBT * d; }            // P q      [16][d]
  __host__ __device__ int k() const { return 2 * kBT * d; }        // R_16 k   [d][16]
  __host__ __device__ int p() const { return 3 * kBT * d; }        // P_16     [d]
  __host__ __device__ int qk() const { return 3 * kBT * d + d; }   // Q        [16][16]
  __host__ __device__ int u() const { return 3 * kBT * d + d + kBT * kBT; }  // U [16][dv]
  __host__ __device__ int size() const { return 3 * kBT * d + d + kBT * kBT + kBT * dv; }
};

// One workgroup of D threads per (block, head); thread = key channel (and value column).
template <typename T, int D, bool CHANNEL>
__global__ __launch_bounds__(D, 4) void delta_block_kernel(float* __restrict__ scratch, const float* __restrict__ qkv, const T* __restrict__ b_raw,
                                                        int64_t ld_b, const T* __restrict__ a_raw, int64_t ld_a, const float* __restrict__ rate,
                                                        const float* __restrict__ dt_bias, const int* __restrict__ cu_q, int B, int H, int G,
                                                        int dv) {
  constexpr int LD = D + 4, NWAVE = D / 64;  // rows padded so that 16 rows' 16-byte reads cover all banks
  __shared__ __attribute__((aligned(16))) float sx[48 * LD];
  __shared__ __attribute__((aligned(16))) float sa[kBT][20], sq[kBT][kBT];
  __shared__ float sbeta[kBT], sg[kBT];
  const uint32_t c = threadIdx.x;  // unsigned: a uniform row plus a 32-bit offset is one address register
  const int lane = c & 63, wave = __builtin_amdgcn_readfirstlane((int)(c >> 6)), lr = lane & 15, lg = lane >> 4;
  const int h = blockIdx.y, kvh = h / (H / G);
  int tok0 = 0;
  const int b = find_group_wave(cu_q, B, kBT, (int)blockIdx.x, &tok0);
  if (b < 0) return;
  const int t0 = __builtin_amdgcn_readfirstlane(cu_q[b]) + __builtin_amdgcn_readfirstlane(tok0);
  const int nt = min(kBT, __builtin_amdgcn_readfirstlane(cu_q[b + 1]) - t0), C = 2 * G * D + H * dv;
  auto token = [&](int t) { return (size_t)(t0 + min(t, nt - 1)); };  // rows past the portion: the last one again, selected away
  const BlockPart part{D, dv};
  float* dst = scratch + ((size_t)blockIdx.x * H + h) * part.size();
  const float r = rate[h];
  // tokens past the portion: nothing read, nothing added, nothing forgotten
  float k[kBT], q[kBT], P[kBT], S[kBT];  // P: product of the decays from the half block's start to t; S: from after t to its end
#pragma unroll
  for (int t = 0; t < kBT; ++t) {
    const float* row = qkv + token(t) * C + kvh * D;
    const float kv = row[G * D + c], qv = row[c];
    k[t] = t < nt ? kv : 0.f;
    q[t] = t < nt ? qv : 0.f;
    if (CHANNEL) sx[t * LD + c] = ld((a_raw + token(t) * ld_a + h * D) + c);
  }
  if (c < (uint32_t)kBT) {
    sbeta[c] = (int)c < nt ? sigmoidf_(ld(b_raw + (size_t)(t0 + c) * ld_b + h)) : 0.f;
    if (!CHANNEL) sg[c] = (int)c < nt ? decay_of(r, ld(a_raw + (size_t)(t0 + c) * ld_a + h) + dt_bias[h], b_raw) : 1.f;
  }
  for (uint32_t i = c; i < (uint32_t)(kBT * kBT); i += D) {
    sa[i >> 4][i & 15] = 0.f;
    sq[i >> 4][i & 15] = 0.f;
  }
  {  // the diagonal of Q: the products per channel to LDS, then PT threads a token sum its row
    constexpr int PT = D / kBT;
    float* prod = sx + kBT * LD;  // the first rows hold the decays' inputs
#pragma unroll
    for (int t = 0; t < kBT; ++t) prod[t * LD + c] = q[t] * k[t];
    __syncthreads();
    const int t = (int)c / PT, part_of = (int)c % PT;
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x4_t x = *reinterpret_cast<const f32x4_t*>(prod + t * LD + 16 * part_of + 4 * i);
      s += (x[0] + x[1]) + (x[2] + x[3]);
    }
#pragma unroll
    for (int o = PT / 2; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
    if (part_of == 0) sq[t][t] = s;
  }
  if constexpr (CHANNEL) {
    const float bias = dt_bias[h * D + c];
    // a few tokens at a time through the thread's own LDS column: sixteen at once took 223 registers, two waves per SIMD
#pragma unroll 2
    for (int t = 0; t < nt; ++t) sx[t * LD + c] = decay_of(r, sx[t * LD + c] + bias, b_raw);
#pragma unroll
    for (int t = 0; t < kBT; ++t) {
      P[t] = t < nt ? sx[t * LD + c] : 1.f;
      S[t] = 1.f;
    }
    __syncthreads();
    // two levels at a time: rows 0 - 7 of a level's image are k of the upper halves times P, rows 8 - 15 the same of q, rows 16 - 23
    // k of the lower halves times S; one product gives both kinds of pairs
#pragma unroll
    for (int round = 0; round < 2; ++round) {
      if (round) __syncthreads();
#pragma unroll
      for (int lv = 0; lv < 2; ++lv) {
        const int hb = 1 << (2 * round + lv);
        float* x = sx + lv * 24 * LD + c;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int up = i / hb * 2 * hb + hb + i % hb, low = i / hb * 2 * hb + i % hb;
          x[i * LD] = k[up] * P[up];
          x[(8 + i) * LD] = q[up] * P[up];
          x[(16 + i) * LD] = k[low] * S[low];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {  // half blocks double: lower halves go on through the upper one, upper ones start in the lower
          const int up = i / hb * 2 * hb + hb + i % hb, low = i / hb * 2 * hb + i % hb;
          S[low] *= P[i / hb * 2 * hb + 2 * hb - 1];
          (void)up;
        }
        float whole[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) whole[i] = P[i / hb * 2 * hb + hb - 1];
#pragma unroll
        for (int i = 0; i < 8; ++i) P[i / hb * 2 * hb + hb + i % hb] *= whole[i];
      }
      __syncthreads();
#pragma unroll
      for (int lv = 0; lv < 2; ++lv) {
        if (NWAVE == 2 && lv != wave) continue;
        const int hb = 1 << (2 * round + lv);
        const float* x = sx + lv * 24 * LD;
        f32x4_t acc{0.f, 0.f, 0.f, 0.f}, acc2{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kc = 0; kc < D / 16; kc += 2) {
          const f32x4_t a0 = *reinterpret_cast<const f32x4_t*>(x + lr * LD + kc * 16 + 4 * lg), b0 = *reinterpret_cast<const f32x4_t*>(x + (16 + (lr & 7)) * LD + kc * 16 + 4 * lg);
          const f32x4_t a1 = *reinterpret_cast<const f32x4_t*>(x + lr * LD + kc * 16 + 16 + 4 * lg), b1 = *reinterpret_cast<const f32x4_t*>(x + (16 + (lr & 7)) * LD + kc * 16 + 16 + 4 * lg);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[i], b0[i], acc, 0, 0, 0);
            acc2 = __builtin_amdgcn_mfma_f32_16x16x4f32(a1[i], b1[i], acc2, 0, 0, 0);
          }
          __builtin_amdgcn_sched_barrier(0);  // all operands read ahead are 128 registers
        }
        if (lr < 8) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int u = (4 * lg + i) & 7, t = u / hb * 2 * hb + hb + u % hb, j = lr / hb * 2 * hb + lr % hb;
            if (u / hb == lr / hb) {
              const float v = acc[i] + acc2[i];
              if (lg < 2) sa[t][j] = sbeta[t] * v;
              else sq[t][j] = v;
            }
          }
        }
      }
    }
  } else {
    __syncthreads();  // the diagonal's rows have been read
#pragma unroll
    for (int t = 0; t < kBT; ++t) {
      sx[t * LD + c] = k[t];
      sx[(16 + t) * LD + c] = q[t];
    }
    __syncthreads();
#pragma unroll
    for (int which = 0; which < 2; ++which) {
      if (NWAVE == 2 && which != wave) continue;
      f32x4_t acc{0.f, 0.f, 0.f, 0.f}, acc2{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kc = 0; kc < D / 16; kc += 2) {
        const f32x4_t a0 = *reinterpret_cast<const f32x4_t*>(sx + (16 * which + lr) * LD + kc * 16 + 4 * lg), b0 = *reinterpret_cast<const f32x4_t*>(sx + lr * LD + kc * 16 + 4 * lg);
        const f32x4_t a1 = *reinterpret_cast<const f32x4_t*>(sx + (16 * which + lr) * LD + kc * 16 + 16 + 4 * lg), b1 = *reinterpret_cast<const f32x4_t*>(sx + lr * LD + kc * 16 + 16 + 4 * lg);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[i], b0[i], acc, 0, 0, 0);
          acc2 = __builtin_amdgcn_mfma_f32_16x16x4f32(a1[i], b1[i], acc2, 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = 4 * lg + i, j = lr;
        if (j < t) {
          float ratio = 1.f;
          for (int s = j + 1; s <= t; ++s) ratio *= sg[s];
          const float v = (acc[i] + acc2[i]) * ratio;
          if (which == 0) sa[t][j] = sbeta[t] * v;
          else sq[t][j] = v;
        }
      }
    }
    float run = 1.f;
#pragma unroll
    for (int t = 0; t < kBT; ++t) P[t] = run *= sg[t];
    run = 1.f;
#pragma unroll
    for (int t = kBT - 1; t >= 0; --t) {
      S[t] = run;
      run *= sg[t];
    }
  }
  __syncthreads();
  // x = (I + A)^-1 x and y = (I + A)^-1 y, row after row; every thread its own columns, A's rows the same words for all.  The fences keep
  // the rows' reads apart: all of A read ahead is 144 registers, and half the waves.
  auto solve = [&](float (&x)[kBT], float (&y)[kBT]) {
#pragma unroll
    for (int t = 1; t < kBT; ++t) {
#pragma unroll
      for (int j4 = 0; j4 < t; j4 += 4) {
        const f32x4_t a = *reinterpret_cast<const f32x4_t*>(&sa[t][j4]);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (j4 + i < t) {
            x[t] = fmaf(-a[i], x[j4 + i], x[t]);
            y[t] = fmaf(-a[i], y[j4 + i], y[t]);
          }
      }
      asm volatile("" : "+v"(x[t]), "+v"(y[t]) : : "memory");
    }
  };
#pragma unroll
  for (int t = 0; t < kBT; ++t) (dst + part.q() + t * D)[c] = q[t] * P[t];
  (dst + part.p())[c] = P[kBT - 1];
#pragma unroll
  for (int t4 = 0; t4 < kBT; t4 += 4)
    *reinterpret_cast<f32x4_t*>(dst + part.k() + t4 + c * kBT) = f32x4_t{k[t4] * S[t4], k[t4 + 1] * S[t4 + 1], k[t4 + 2] * S[t4 + 2], k[t4 + 3] * S[t4 + 3]};
#pragma unroll
  for (int t = 0; t < kBT; ++t) k[t] *= sbeta[t] * P[t];
  for (uint32_t i = c; i < (uint32_t)(kBT * kBT); i += D) (dst + part.qk())[i] = sq[i >> 4][i & 15];
  __builtin_amdgcn_sched_barrier(0);
  // the key column goes along with the first value column (again with the others: dv > d is rare)
#pragma unroll 1
  for (uint32_t e = c; e < (uint32_t)max(dv, D); e += D) {
    float v[kBT], x[kBT];
#pragma unroll
    for (int t = 0; t < kBT; ++t) {
      v[t] = (qkv + token(t) * C + 2 * G * D + h * dv)[e < (uint32_t)dv ? e : 0u];
      v[t] = t < nt ? sbeta[t] * v[t] : 0.f;
      x[t] = k[t];
    }
    solve(x, v);
#pragma unroll
    for (int t = 0; t < kBT; ++t) {
      if (e < (uint32_t)dv) (dst + part.u() + t * dv)[e] = v[t];
    }
    if (e == c) {
#pragma unroll
      for (int t = 0; t < kBT; ++t) (dst + part.w() + t * D)[c] = x[t];
    }
  }
}

// One workgroup per (request, head, 32 value columns), five waves.  Waves 0 - 3: wave w holds the state rows w D / 4 ... of the 32
// columns as MFMA accumulators (lane: rows 4 lg + i, column lr), which are second operands as they stand: contraction index = state row,
// the first operands' 16-byte reads follow the same order.  W S and (P q) S are sums over all rows, so the waves' shares meet in LDS
// once a block; every wave then has u, in the layout the update takes it.  Wave 4 adds Q u and writes a block's outputs, one block
// behind: it takes everything from LDS, so that the waves which load the next blocks' operands have no stores among their loads (with
// them the compiler waited for every load in flight in front of each block: 338 us where the kernel now takes 240).
template <int D>
__global__ __launch_bounds__(320) void delta_walk_kernel(float* __restrict__ out, float* __restrict__ state, const float* __restrict__ scratch,
                                                         const int* __restrict__ cu_q, const int* __restrict__ seq_lens,
                                                         const int* __restrict__ slots, int B, int H, int dv) {
  constexpr int NT = D / 64;  // 16-row tiles of a wave
  __shared__ __attribute__((aligned(16))) f32x4_t share_u[2][4][2][64], share_o[3][4][2][64];  // [image][wave][column tile][lane]
  __shared__ __attribute__((aligned(16))) f32x4_t full_u[2][2][64], full_qk[2][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lr = lane & 15, lg = lane >> 4;
  // the column blocks of a head read the same operands: neighbours in one XCD's L2 where the heads divide by the eight of them
  const int ncb = dv / 32, groups = B * H;
  int g, cb;
  if (groups % 8 == 0) {
    const int rest = (int)blockIdx.x >> 3;
    cb = rest % ncb;
    g = rest / ncb * 8 + ((int)blockIdx.x & 7);
  } else {
    g = (int)blockIdx.x / ncb;
    cb = (int)blockIdx.x % ncb;
  }
  const int b = g / H, h = g - b * H, c0 = cb * 32;
  const int first = cu_q[b], n_new = cu_q[b + 1] - first;
  if (n_new <= 0) return;
  const int nblk = (n_new + kBT - 1) / kBT;
  if (wave == 4) {
    float* orow = out + ((size_t)first + 4 * lg) * H * dv + (size_t)h * dv + c0 + lr;
    __syncthreads();
    for (int n = 0; n < nblk; ++n, orow += (size_t)kBT * H * dv) {
      __syncthreads();
      const f32x4_t qk = full_qk[n & 1][lane];
      float zero = 0.f;
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) {
        const f32x4_t u = full_u[n & 1][ct][lane];
        f32x4_t o{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; ++e) o = __builtin_amdgcn_mfma_f32_16x16x4f32(qk[e], u[e], o, 0, 0, 0);
#pragma unroll
        for (int w = 0; w < 4; ++w) o += share_o[n % 3][w][ct][lane];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n * kBT + 4 * lg + e < n_new) orow[(size_t)e * H * dv + 16 * ct] = o[e];
        zero = fmaf(o[0], 0.f, zero);
      }
      // Q's upper triangle is zeros, so a u that is not finite spoils its column for all tokens of the block, also those before it (zero times
      // infinity), and one token's number shows it: then the outputs again, each token without the u behind it
      if (__builtin_amdgcn_ballot_w64(zero != 0.f) != 0) {
        const float* qs = reinterpret_cast<const float*>(full_qk[n & 1]);
#pragma unroll 1
        for (int x = 0; x < 8; ++x) {
          const int e = x & 3, ct = x >> 2, t = 4 * lg + e;
          const float* us = reinterpret_cast<const float*>(full_u[n & 1][ct]);
          float o = 0.f;
          for (int j = 0; j <= t; ++j) {
            const int at = (j >> 2) * 64 + (j & 3);  // a lane's four numbers are tokens 4 lg ... of row or column lr
            o = fmaf(qs[at + t * 4], us[at + lr * 4], o);
          }
          for (int w = 0; w < 4; ++w) o += reinterpret_cast<const float*>(share_o[n % 3][w][ct])[lane * 4 + e];
          if (n * kBT + t < n_new) orow[(size_t)e * H * dv + 16 * ct] = o;
        }
      }
    }
    return;
  }
  int blk = 0;  // blocks of the requests before this one
  for (int i = lane; i < b; i += 64) blk += (cu_q[i + 1] - cu_q[i] + kBT - 1) / kBT;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) blk += __shfl_xor(blk, o, 64);
  blk = __builtin_amdgcn_readfirstlane(blk);
  const int r0 = wave * (D / 4);
  const BlockPart part{D, dv};
  const size_t step = (size_t)H * part.size();
  const float* src = scratch + ((size_t)blk * H + h) * part.size();
  float* Srow = state + ((size_t)slots[b] * H + h) * D * dv + c0 + lr;
  const bool fresh = seq_lens[b] == n_new;
  f32x4_t S[NT][2];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
#pragma unroll
      for (int e = 0; e < 4; ++e) S[i][ct][e] = fresh ? 0.f : Srow[(size_t)(r0 + 16 * i + 4 * lg + e) * dv + 16 * ct];
  struct Ops {
    f32x4_t w[NT], q[NT], k[NT], p[NT], u[2], qk;
  };
  // this lane's places in a block's operands
  const uint32_t at_w = part.w() + lr * D + r0 + 4 * lg, at_q = at_w + part.q(), at_k = part.k() + (r0 + lr) * kBT + 4 * lg, at_p = part.p() + r0 + 4 * lg,
                 at_u = part.u() + 4 * lg * dv + c0 + lr, at_qk = part.qk() + lr * kBT + 4 * lg;
  auto fetch = [&](Ops& x, int n) {
    const float* at = src + (size_t)min(n, nblk - 1) * step;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      x.w[i] = *reinterpret_cast<const f32x4_t*>(at + at_w + 16 * i);
      x.q[i] = *reinterpret_cast<const f32x4_t*>(at + at_q + 16 * i);
      x.k[i] = *reinterpret_cast<const f32x4_t*>(at + at_k + 16 * i * kBT);
      x.p[i] = *reinterpret_cast<const f32x4_t*>(at + at_p + 16 * i);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) x.u[ct][e] = (at + at_u + e * dv)[16 * ct];
    x.qk = *reinterpret_cast<const f32x4_t*>(at + at_qk);
  };
  auto block = [&](const Ops& x, int n, auto tail) __attribute__((always_inline)) {
    f32x4_t pu[2], po[2];
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) pu[ct] = po[ct] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) pu[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w[i][e], S[i][ct][e], pu[ct], 0, 0, 0);
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) share_u[n & 1][wave][ct][lane] = pu[ct];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) po[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.q[i][e], S[i][ct][e], po[ct], 0, 0, 0);
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) share_o[n % 3][wave][ct][lane] = po[ct];
    __syncthreads();  // a wave is at most one block ahead of another, wave 4 one block behind: two and three images are enough
    f32x4_t u[2];
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
      u[ct] = x.u[ct];
#pragma unroll
      for (int w = 0; w < 4; ++w) u[ct] -= share_u[n & 1][w][ct][lane];
    }
    if (tail && (n + 1) * kBT > n_new) {  // rows past the portion are zero also where a value before them is infinite
#pragma unroll
      for (int ct = 0; ct < 2; ++ct)
#pragma unroll
        for (int e = 0; e < 4; ++e) u[ct][e] = n * kBT + 4 * lg + e < n_new ? u[ct][e] : 0.f;
    }
    if (wave == 0) {
      full_u[n & 1][0][lane] = u[0];
      full_u[n & 1][1][lane] = u[1];
      full_qk[n & 1][lane] = x.qk;
    }
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int ct = 0; ct < 2; ++ct) S[i][ct] *= x.p[i];
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) S[i][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[i][e], u[ct][e], S[i][ct], 0, 0, 0);
  };
  // operands are requested two blocks ahead: a block takes less than a loaded memory system's latency
  Ops x0, x1, x2;
  fetch(x0, 0);
  fetch(x1, 1);
  int n = 0;
  const std::false_type within;
  for (; n + 3 < nblk; n += 3) {
    fetch(x2, n + 2);
    block(x0, n, within);
    fetch(x0, n + 3);
    block(x1, n + 1, within);
    fetch(x1, n + 4);
    block(x2, n + 2, within);
  }
  const std::true_type tail;  // the last one to three blocks: only they look for the portion's end
  fetch(x2, n + 2);
  block(x0, n, tail);
  if (n + 1 < nblk) block(x1, n + 1, tail);
  if (n + 2 < nblk) block(x2, n + 2, tail);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
#pragma unroll
      for (int e = 0; e < 4; ++e) Srow[(size_t)(r0 + 16 * i + 4 * lg + e) * dv + 16 * ct] = S[i][ct][e];
}

}  // namespace

extern "C" {

int msgl_mix_delta_rule_block_floats(int d, int dv) {
  if ((d != 64 && d != 128) || dv < 32 || dv % 32) return 0;
  return (int)BlockPart{d, dv}.size();
}

int msgl_mix_delta_rule_blocks(float* out, const float* qkv, float* state, const void* b_raw, int64_t ld_b, const void* a_raw, int64_t ld_a,
                               int per_channel, const float* rate, const float* dt_bias, const int* cu_q, const int* seq_lens,
                               const int* slots, int batch, int total_q, int H, int G, int d, int dv, int dtype, float* scratch,
                               void* stream) {
  MIX_REQUIRE(out && qkv && state && b_raw && a_raw && rate && dt_bias && cu_q && seq_lens && slots && scratch && dtype_ok(dtype),
              "delta_rule_blocks: null pointer / dtype");
  MIX_REQUIRE(batch >= 0 && total_q >= 0 && H >= 1 && G >= 1 && H % G == 0 && (d == 64 || d == 128) && dv >= 32 && dv % 32 == 0,
              "delta_rule_blocks: bad sizes H %d G %d d %d dv %d", H, G, d, dv);
  MIX_REQUIRE(ld_b >= H && ld_a >= (per_channel ? H * d : H), "delta_rule_blocks: rows shorter than their heads");
  MIX_REQUIRE((reinterpret_cast<uintptr_t>(scratch) & 15) == 0, "delta_rule_blocks: scratch not 16-byte aligned");
  if (batch == 0 || total_q == 0) return MSGL_MIX_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid(total_q / kBT + batch, H);
#define DB_LAUNCH(D, CH)                                                                                                               \
  DISPATCH_T(dtype, hipLaunchKernelGGL((delta_block_kernel<T, D, CH>), grid, dim3(D), 0, s, scratch, qkv, cp<T>(b_raw), ld_b, cp<T>(a_raw), \
                                       ld_a, rate, dt_bias, cu_q, batch, H, G, dv);)
  if (d == 128) {
    if (per_channel) DB_LAUNCH(128, true) else DB_LAUNCH(128, false)
  } else {
    if (per_channel) DB_LAUNCH(64, true) else DB_LAUNCH(64, false)
  }
#undef DB_LAUNCH
  MIX_LAUNCHED("delta_rule_blocks");
  if (d == 128)
    hipLaunchKernelGGL((delta_walk_kernel<128>), dim3(batch * H * (dv / 32)), dim3(320), 0, s, out, state, scratch, cu_q, seq_lens, slots, batch, H, dv);
  else
    hipLaunchKernelGGL((delta_walk_kernel<64>), dim3(batch * H * (dv / 32)), dim3(320), 0, s, out, state, scratch, cu_q, seq_lens, slots, batch, H, dv);
  MIX_LAUNCHED("delta_rule_blocks (walk)");
  return MSGL_MIX_OK;
}

}  // extern "C"
