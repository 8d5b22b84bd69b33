// Gated delta rule in blocks of 16 tokens on the fp32 matrix instructions (the token loop: delta_rule_kernel in mix_delta.hip).
//
// Per head, with S [d, dv], decays g_t per key channel (or one per head) and P_t = g_1 ... g_t from the block's start:
//   S_t = g_t S_{t-1} + k_t u_t^T,   u_t = beta_t (v_t - S_{t-1}^T (g_t k_t)),   o_t = S_t^T q_t
// Written from the block's start state S (R_{tj} = g_{j+1} ... g_t per channel):
//   (I + A) u = beta (v - (P k) S),  A_{tj} = beta_t sum_c k_tc R_{tj,c} k_jc  (j < t)
//   o = (P q) S + Q u,               Q_{tj} = sum_c q_tc R_{tj,c} k_jc         (j <= t)
//   S' = P_16 S + (R_{16,j} k_j)^T u
// delta_block_kernel computes, for all blocks at once, T = (I + A)^-1 beta, W = T (P k), P q, Q, R_{16} k, P_16;
// delta_walk_kernel walks a request's blocks: u = T v - W S, o = (P q) S + Q u, S = P_16 S + (R_{16} k)^T u.
//
// Everything stays fp32: v_mfma_f32_16x16x4_f32 multiplies and adds in fp32.  Ratios of decays are products of at most 15 decays, never
// quotients or exponentials of sums (an exponential of a sum of logarithms loses the digits that the sum's size takes): the pairs (t, j)
// split by the highest bit in which t and j differ, and per level both factors are running products inside a half block.
//
// What bounds it: the walk is a serial chain of blocks per (request, head), 25 fp32 MFMAs of 32 cycles a wave and block and the meeting in
// LDS (1650 cycles a block of a chain alone, 2900 with two on a CU, whose operands, 27 KB a block and chain, come from L2 at 10 TB/s in
// all); the block kernel by memory (49 d + 512 floats a block and head written, and read again by the walk; values are read by the walk
// itself).  The token loop was bound by one wave's serial walk: two passes over 128 registers a token, in three launches.
// 4 requests of 1500 - 2548 tokens, 16 heads, d = dv = 128, decays per channel, us (blocks, walk): 4038 in the token loop; 389 (171, 219) with
// (I + A)^-1 beta v solved and stored per value column, operands in rows of d and 32 columns a workgroup; 306 (100, 207) as below, 277 (99,
// 178) with the walks in order of length.  One request of 900 tokens, 8 heads: 100 -> 62.  Error against 64 bits 1.9e-7 -> 1.4e-7 -> 1.1e-7.
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

// A block's operands of one head in the scratch, in floats: 16 x 16 tiles in the order in which the walk's lanes (lr = lane & 15, lg =
// lane >> 4) take them, 16 bytes a lane, so that a wave's load is one kilobyte in a row.  (Rows of d floats made every sixteen
// lanes of a load touch sixteen lines, and the walk waited for the address unit.)
struct BlockPart {
  int d;
  __host__ __device__ int w() const { return 0; }                           // -W    [d / 16][lane][4]: token lr, channels 4 lg ...
  __host__ __device__ int q() const { return kBT * d; }                     // P q   likewise
  __host__ __device__ int k() const { return 2 * kBT * d; }                 // R_16 k [d / 16][lane][4]: channel lr, tokens 4 lg ...
  __host__ __device__ int p() const { return 3 * kBT * d; }                 // P_16  [d]
  __host__ __device__ int qk() const { return 3 * kBT * d + d; }            // Q     [lane][4]: token lr, tokens 4 lg ...
  __host__ __device__ int t() const { return 3 * kBT * d + d + kBT * kBT; } // T     [4][lane]: token lr, token 4 lg + first index
  __host__ __device__ int size() const { return 3 * kBT * d + d + 2 * kBT * kBT; }
};

// One workgroup of D threads per (block, head); thread = key channel (and value column).
template <typename T, int D, bool CHANNEL>
__global__ __launch_bounds__(D, 4) void delta_block_kernel(float* __restrict__ scratch, const float* __restrict__ qkv, const T* __restrict__ b_raw,
                                                        int64_t ld_b, const T* __restrict__ a_raw, int64_t ld_a, const float* __restrict__ rate,
                                                        const float* __restrict__ dt_bias, const int* __restrict__ cu_q, int B, int H, int G,
                                                        int dv) {
  constexpr int LD = D + 4, NWAVE = D / 64;  // rows padded so that 16 rows' 16-byte reads cover all banks
  __shared__ __attribute__((aligned(16))) float sx[48 * LD];
  __shared__ __attribute__((aligned(16))) float sa[kBT][20], sq[kBT][20];
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
  const BlockPart part{D};
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
  // x = (I + A)^-1 x (and y = (I + A)^-1 y), row after row; every thread its own columns, A's rows the same words for all.  The fences
  // keep the rows' reads apart: all of A read ahead is 144 registers, and half the waves.
  auto solve = [&](float (&x)[kBT], float (&y)[kBT], auto both) {
#pragma unroll
    for (int t = 1; t < kBT; ++t) {
#pragma unroll
      for (int j4 = 0; j4 < t; j4 += 4) {
        const f32x4_t a = *reinterpret_cast<const f32x4_t*>(&sa[t][j4]);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (j4 + i < t) {
            x[t] = fmaf(-a[i], x[j4 + i], x[t]);
            if constexpr (both) y[t] = fmaf(-a[i], y[j4 + i], y[t]);
          }
      }
      asm volatile("" : "+v"(x[t]), "+v"(y[t]) : : "memory");
    }
  };
#pragma unroll
  for (int t = 0; t < kBT; ++t) sx[(16 + t) * LD + c] = q[t] * P[t];
  (dst + part.p())[c] = P[kBT - 1];
#pragma unroll
  for (int t4 = 0; t4 < kBT; t4 += 4)
    *reinterpret_cast<f32x4_t*>(dst + part.k() + (c >> 4) * 256 + t4 * 16 + (c & 15) * 4) =
        f32x4_t{k[t4] * S[t4], k[t4 + 1] * S[t4 + 1], k[t4 + 2] * S[t4 + 2], k[t4 + 3] * S[t4 + 3]};
#pragma unroll
  for (int t = 0; t < kBT; ++t) k[t] *= sbeta[t] * P[t];
  if (wave == 0) *reinterpret_cast<f32x4_t*>(dst + part.qk() + lane * 4) = *reinterpret_cast<const f32x4_t*>(&sq[lr][4 * lg]);
  __builtin_amdgcn_sched_barrier(0);
  // the columns of T go along with the first wave's key columns
  float y[kBT];
  if (wave == 0) {
#pragma unroll
    for (int t = 0; t < kBT; ++t) y[t] = c == (uint32_t)t ? sbeta[t] : 0.f;
    solve(k, y, std::true_type{});
    if (c < (uint32_t)kBT) {
#pragma unroll
      for (int t = 0; t < kBT; ++t) (dst + part.t())[(c & 3) * 64 + (c >> 2) * 16 + t] = y[t];
    }
  } else {
    solve(k, k, std::false_type{});
  }
#pragma unroll
  for (int t = 0; t < kBT; ++t) sx[t * LD + c] = -k[t];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < D / 16 / NWAVE; ++i) {
    const int tile = wave * (D / 16 / NWAVE) + i;
    *reinterpret_cast<f32x4_t*>(dst + part.w() + tile * 256 + lane * 4) = *reinterpret_cast<const f32x4_t*>(sx + lr * LD + 16 * tile + 4 * lg);
    *reinterpret_cast<f32x4_t*>(dst + part.q() + tile * 256 + lane * 4) = *reinterpret_cast<const f32x4_t*>(sx + (16 + lr) * LD + 16 * tile + 4 * lg);
  }
}

// The request at a place of the walks' order (`each` workgroups a request), its first token, its tokens and the blocks of the requests before it.
// A walk takes as long as its request, 0.9 us a block alone on a CU and 1.6 beside another one.  So the longest requests come first, one round of
// the CUs; those of the second round meet them in reverse, and where it is not full the longest ones stay alone; what does not fit two rounds
// follows in order, the shortest last.  Walks that each are less than a place's share of more than two rounds stay as they come: no end to wait for,
// and equal ones side by side wait for their first loads together (us of the walks, as they come -> ordered: 8 requests of 80 - 130 tokens,
// 16 heads: 29.9 -> 31.8; 8 of 300 - 1000: 134.9 -> 138.5).  Ordered: 4 of 1500 - 2548, 16 heads: 214 -> 190; 5 of 400 - 1500, 8 heads:
// 90 -> 80; 7 of 100 - 1100, 16 heads: 118 -> 104; 3 of 200 - 2600: 147.
struct WalkRequest {
  int b, first, n_new, blk;
};
__device__ __forceinline__ WalkRequest walk_request(const int* __restrict__ cu_q, int B, int each, int place) {
  const int lane = threadIdx.x & 63;
  WalkRequest r;
  if (B > 64) {
    r.b = place;
    r.first = cu_q[place];
    r.n_new = cu_q[place + 1] - r.first;
    r.blk = 0;
    for (int i = lane; i < place; i += 64) r.blk += (cu_q[i + 1] - cu_q[i] + kBT - 1) / kBT;
    r.blk = wave_total(r.blk);
    return r;
  }
  const int first = lane < B ? cu_q[lane] : 0, n = lane < B ? cu_q[lane + 1] - first : 0;
  const int round = max(1, 256 / each), met = min(round, B - round);  // requests in the second round
  const int longest = wave_fold(n, [](int x, int y) { return max(x, y); });
  const bool ordered = B <= 2 * round || (int64_t)longest * 512 >= (int64_t)wave_total(n) * each;
  r.b = place;
  if (ordered) {
    int rank = place;
    if (met > 0 && place < round) rank = place < met ? round - met + place : place - met;
    else if (met > 0 && place < 2 * round) rank = round + met - 1 - (place - round);
    int longer = 0;
    for (int i = 0; i < B; ++i) {
      const int ni = __builtin_amdgcn_readlane(n, i);
      longer += ni > n || (ni == n && i < lane);
    }
    r.b = __builtin_ctzll(__builtin_amdgcn_ballot_w64(longer == rank && lane < B));
  }
  r.first = __builtin_amdgcn_readlane(first, r.b);
  r.n_new = __builtin_amdgcn_readlane(n, r.b);
  r.blk = wave_total(lane < r.b ? (n + kBT - 1) / kBT : 0);
  return r;
}

// One workgroup per (request, head, 16 value columns), five waves.  Waves 0 - 3: wave w holds the state rows w D / 4 ... of the columns as
// MFMA accumulators (lane: rows 4 lg + i, column lr), which are second operands as they stand: contraction index = state row, the first
// operands' reads follow the same order.  u = T v - W S and (P q) S are sums over tokens and rows: wave w adds the tokens 4 g + w (one
// product) and its own rows, and the waves' shares meet in LDS once a block, behind the products of (P q) S; every wave then has u, in the
// layout the update takes it.  Wave 4 adds Q u and writes a block's outputs, one block behind: it takes everything from LDS, so that the waves
// which load the next blocks' operands have no stores among their loads (with them the compiler waited for every load in flight in front of
// each block), and no loads of its own, whose waits would be for the stores before them.
// At most 128 registers, so that two workgroups share a CU: wave 4 goes to the SIMD of wave 0, and with more the second workgroup waited for
// the first to end.  32 columns a workgroup read half as much and took 215 us for 207 (200 for 181 at 8 requests of 300 - 1000 tokens), both
// without the order of the walks: one chain's meeting is not hidden by another's products.
template <int D>
__global__ __launch_bounds__(320, 4) void delta_walk_kernel(float* __restrict__ out, float* __restrict__ state, const float* __restrict__ scratch,
                                                            const float* __restrict__ qkv, const int* __restrict__ cu_q,
                                                            const int* __restrict__ seq_lens, const int* __restrict__ slots, int B, int H, int G,
                                                            int dv) {
  constexpr int NT = D / 64;  // 16-row tiles of a wave
  __shared__ __attribute__((aligned(16))) f32x4_t share_u[2][4][64], share_o[3][4][64];  // [image][wave][lane]
  __shared__ __attribute__((aligned(16))) f32x4_t full_u[2][64], full_qk[3][64];
  __shared__ __attribute__((aligned(16))) float decays[2][4][32];  // a wave's own
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lr = lane & 15, lg = lane >> 4;
  // the column blocks of a head read the same operands: neighbours in one XCD's L2 where the heads divide by the eight of them
  const int ncb = dv / 16, groups = B * H;
  int g, cb;
  if (groups % 8 == 0) {
    const int rest = (int)blockIdx.x >> 3;
    cb = rest % ncb;
    g = rest / ncb * 8 + ((int)blockIdx.x & 7);
  } else {
    g = (int)blockIdx.x / ncb;
    cb = (int)blockIdx.x % ncb;
  }
  const int place = g / H, h = g - place * H, c0 = cb * 16;
  const WalkRequest req = walk_request(cu_q, B, H * ncb, place);
  const int b = req.b, first = req.first, n_new = req.n_new, blk = req.blk;
  if (n_new <= 0) return;
  const int nblk = (n_new + kBT - 1) / kBT;
  const BlockPart part{D};
  const uint32_t step = (uint32_t)(H * part.size());
  const float* src = scratch + ((size_t)blk * H + h) * part.size();
  const f32x4_t none{0.f, 0.f, 0.f, 0.f};
  if (wave == 4) {
    float* orow = out + ((size_t)first + 4 * lg) * H * dv + (size_t)h * dv + c0 + lr;
    __syncthreads();
    for (int n = 0; n < nblk; ++n, orow += (size_t)kBT * H * dv) {
      __syncthreads();
      const f32x4_t u = full_u[n & 1][lane], qk = full_qk[n % 3][lane];
      f32x4_t o0 = __builtin_amdgcn_mfma_f32_16x16x4f32(qk[0], u[0], none, 0, 0, 0), o1 = __builtin_amdgcn_mfma_f32_16x16x4f32(qk[1], u[1], none, 0, 0, 0);
      o0 = __builtin_amdgcn_mfma_f32_16x16x4f32(qk[2], u[2], o0, 0, 0, 0);
      o1 = __builtin_amdgcn_mfma_f32_16x16x4f32(qk[3], u[3], o1, 0, 0, 0);
      f32x4_t o = share_o[n % 3][0][lane];
#pragma unroll
      for (int w = 1; w < 4; ++w) o += share_o[n % 3][w][lane];
      o += o0 + o1;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n * kBT + 4 * lg + e < n_new) orow[(size_t)e * H * dv] = o[e];
      // Q's upper triangle is zeros, so a u that is not finite spoils its column for all tokens of the block, also those before it (zero times
      // infinity), and one token's number shows it: then the outputs again, each token without the u behind it
      if (__builtin_amdgcn_ballot_w64(fmaf(o[0], 0.f, 0.f) != 0.f) != 0) {
        const float* qs = reinterpret_cast<const float*>(full_qk[n % 3]);
        const float* us = reinterpret_cast<const float*>(full_u[n & 1]);
#pragma unroll 1
        for (int e = 0; e < 4; ++e) {
          const int t = 4 * lg + e;
          float x = 0.f;
          for (int j = 0; j <= t; ++j) {
            const int at = (j >> 2) * 64 + (j & 3);  // a lane's four numbers are tokens 4 lg ... of row or column lr
            x = fmaf(qs[at + t * 4], us[at + lr * 4], x);
          }
          for (int w = 0; w < 4; ++w) x += reinterpret_cast<const float*>(share_o[n % 3][w])[lane * 4 + e];
          if (n * kBT + t < n_new) orow[(size_t)e * H * dv] = x;
        }
      }
    }
    return;
  }
  const int r0 = wave * (D / 4);
  float* Srow = state + ((size_t)slots[b] * H + h) * D * dv + c0 + lr;
  const bool fresh = seq_lens[b] == n_new;
  f32x4_t S[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) S[i][e] = fresh ? 0.f : Srow[(size_t)(r0 + 16 * i + 4 * lg + e) * dv];
  struct Ops {
    f32x4_t w[NT], q[NT], k[NT];
    float t, v, p, qk;
  };
  // this lane's places in a block's operands; its value is of token 4 lg + wave
  const uint32_t at_w = part.w() + wave * NT * 256 + lane * 4, at_q = at_w + part.q(), at_k = at_w + part.k(), at_t = part.t() + wave * 64 + lane,
                 at_p = part.p() + r0 + (lane & (D / 4 - 1)), at_qk = part.qk() + lane * 4 + wave;
  const int C = 2 * G * D + H * dv;
  const float* vrow = qkv + (size_t)first * C + 2 * G * D + (size_t)h * dv + c0 + lr;
  // Operands are requested two blocks ahead (a block takes less than a loaded memory system's latency), each into the registers of the
  // block that has just used them: all at once they held the wave up for 500 cycles.
  auto at_block = [&](int n) { return src + (uint64_t)(uint32_t)min(n, nblk - 1) * step; };
  auto fetch_w = [&](Ops& x, int n) __attribute__((always_inline)) {
    const float* at = at_block(n);
    const int m = min(n, nblk - 1) * kBT;
    x.t = at[at_t];
    x.p = at[at_p];
    x.qk = at[at_qk];
    x.v = (vrow + (size_t)m * C)[(uint32_t)(min(4 * lg + wave, n_new - 1 - m) * C)];
#pragma unroll
    for (int i = 0; i < NT; ++i) x.w[i] = *reinterpret_cast<const f32x4_t*>(at + at_w + 256 * i);
  };
  auto fetch_q = [&](Ops& x, int n) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NT; ++i) x.q[i] = *reinterpret_cast<const f32x4_t*>(at_block(n) + at_q + 256 * i);
  };
  auto fetch_k = [&](Ops& x, int n) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NT; ++i) x.k[i] = *reinterpret_cast<const f32x4_t*>(at_block(n) + at_k + 256 * i);
  };
  auto block = [&](Ops& x, int n, auto tail) __attribute__((always_inline)) {
    float v = x.v;
    if (tail) v = n * kBT + 4 * lg + wave < n_new ? v : 0.f;
    f32x4_t pv, pu[NT], po[NT];  // T v stays out of the sums of W S until these are whole: they are the smaller numbers
    pv = __builtin_amdgcn_mfma_f32_16x16x4f32(x.t, v, none, 0, 0, 0);
    auto with_state = [&](f32x4_t (&acc)[NT], const f32x4_t (&first)[NT], int e) {
#pragma unroll
      for (int i = 0; i < NT; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(first[i][e], S[i][e], e ? acc[i] : none, 0, 0, 0);
    };
#pragma unroll
    for (int e = 0; e < 4; ++e) with_state(pu, x.w, e);
    if (__builtin_amdgcn_ballot_w64(fmaf(v, 0.f, 0.f) != 0.f) != 0) {
      // a value that is no number: the zeros of the upper triangle would carry it to the tokens before its own
#pragma unroll 1
      for (int e = 0; e < 4; ++e) {
        float sum = 0.f;
        for (int gj = 0; gj < 4; ++gj) {
          const float vj = __shfl(v, gj * 16 + lr, 64), tj = __shfl(x.t, gj * 16 + 4 * lg + e, 64);
          if (4 * gj + wave <= 4 * lg + e) sum = fmaf(tj, vj, sum);
        }
        pv[0] = e == 0 ? sum : pv[0];
        pv[1] = e == 1 ? sum : pv[1];
        pv[2] = e == 2 ? sum : pv[2];
        pv[3] = e == 3 ? sum : pv[3];
      }
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) pv += pu[i];
    share_u[n & 1][wave][lane] = pv;
    if (lane < D / 4) decays[n & 1][wave][lane] = x.p;
    reinterpret_cast<float*>(full_qk[n % 3])[lane * 4 + wave] = x.qk;
    fetch_w(x, n + 2);
#pragma unroll
    for (int e = 0; e < 4; ++e) with_state(po, x.q, e);
    fetch_q(x, n + 2);
#pragma unroll
    for (int i = 0; i < NT; ++i) S[i] *= *reinterpret_cast<const f32x4_t*>(&decays[n & 1][wave][16 * i + 4 * lg]);
#pragma unroll
    for (int i = 1; i < NT; ++i) po[0] += po[i];
    share_o[n % 3][wave][lane] = po[0];
    __syncthreads();  // a wave is at most one block ahead of another, wave 4 one block behind: two and three images are enough
    f32x4_t u = (pv + share_u[n & 1][wave ^ 1][lane]) + (share_u[n & 1][wave ^ 2][lane] + share_u[n & 1][wave ^ 3][lane]);
    if (tail && (n + 1) * kBT > n_new) {  // rows past the portion are zero also where a value before them is infinite
#pragma unroll
      for (int e = 0; e < 4; ++e) u[e] = n * kBT + 4 * lg + e < n_new ? u[e] : 0.f;
    }
    if (wave == 0) full_u[n & 1][lane] = u;
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < NT; ++i) S[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[i][e], u[e], S[i], 0, 0, 0);
    fetch_k(x, n + 2);
  };
  Ops x0, x1;
  fetch_w(x0, 0);
  fetch_q(x0, 0);
  fetch_k(x0, 0);
  fetch_w(x1, 1);
  fetch_q(x1, 1);
  fetch_k(x1, 1);
  int n = 0;
  const std::false_type within;
  for (; n + 2 < nblk; n += 2) {
    block(x0, n, within);
    block(x1, n + 1, within);
  }
  const std::true_type tail;  // the last one or two blocks: only they look for the portion's end
  block(x0, n, tail);
  if (n + 1 < nblk) block(x1, n + 1, tail);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) Srow[(size_t)(r0 + 16 * i + 4 * lg + e) * dv] = S[i][e];
}

}  // namespace

extern "C" {

int msgl_mix_delta_rule_block_floats(int d, int dv) {
  if ((d != 64 && d != 128) || dv < 32 || dv % 32) return 0;
  return (int)BlockPart{d}.size();
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
    hipLaunchKernelGGL((delta_walk_kernel<128>), dim3(batch * H * (dv / 16)), dim3(320), 0, s, out, state, scratch, qkv, cu_q, seq_lens, slots, batch, H, G, dv);
  else
    hipLaunchKernelGGL((delta_walk_kernel<64>), dim3(batch * H * (dv / 16)), dim3(320), 0, s, out, state, scratch, qkv, cu_q, seq_lens, slots, batch, H, G, dv);
  MIX_LAUNCHED("delta_rule_blocks (walk)");
  return MSGL_MIX_OK;
}

}  // extern "C"
