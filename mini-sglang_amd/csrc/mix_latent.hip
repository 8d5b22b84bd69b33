// Latent attention over bf16 caches for the usual widths (latent 512 or 256 beside 64 rotated entries): one key row per token, shared by all
// heads, whose first DV entries are the value row too.  seqmix.hip keeps the kernels for other widths and for fp32 caches; same C entry.
//
//   latent_prompt_kernel  portions of tokens: 128 query rows ((token, head) pairs) per workgroup
//   latent_decode_kernel  one 16-row group per workgroup (a decoded token's heads), its keys spread over the waves
//   latent_join_kernel    adds up the key ranges of either
//
// Both: S^T = K Q^T and O^T += V^T P^T, so that a lane ends the first product with scores of ONE query row and starts the second with
// them; the rows come to LDS by DMA (no staging registers), padded (decode: 16 bytes carried along as one more piece) so that 8 rows'
// 16-byte reads and 4 rows' transposing reads both touch all banks once.  A row's sum is of the fp32 weights.  The reference maximum
// follows every new maximum: the largest weight then is 1, exact in bf16 (letting it lag by up to 2^8 saves 2 % of the time and adds a
// tenth to the error).
#include <algorithm>
#include <type_traits>

#include "mix_common.h"

namespace {

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(1))) void glb_void_t;
typedef __attribute__((address_space(3))) void lds_void_t;

constexpr float kLn2 = 0.6931471805599453f;

constexpr int kLeastRange = 128;  // keys; a range costs a partial output's way to memory and back, as much as about 64 keys

__device__ __forceinline__ float sink_factor(const float* __restrict__ sink, int head, float m) {
  return (sink && sink[head] > m) ? expf(m - sink[head]) : 1.f;
}
__device__ __forceinline__ float sink_weight(const float* __restrict__ sink, int head, float m) {
  return sink ? (sink[head] > m ? 1.f : expf(sink[head] - m)) : 0.f;
}

// eight fp32 numbers times f as packed bf16
__device__ __forceinline__ bf16x8_t scaled8(const float* p, float f) {
  const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
  return __builtin_bit_cast(bf16x8_t, Q4{pack_bf16(a.x * f, a.y * f), pack_bf16(a.z * f, a.w * f), pack_bf16(b.x * f, b.y * f),
                                         pack_bf16(b.z * f, b.w * f)});
}

__device__ __forceinline__ float weight(float s, float sharp, float ref) { return __builtin_amdgcn_exp2f(fmaf(s, sharp, -ref)); }
// LDS accesses of one wave go in order; this keeps the compiler's order
__device__ __forceinline__ void wave_fence() { asm volatile("" ::: "memory"); }
template <int DK>
struct LatentRow {
  static constexpr int pieces = DK / 8 + 1;   // 16-byte pieces of a row in LDS, the last one padding
  static constexpr int bytes = pieces * 16;
};

// ---------------------------------------------------------------------------------------------------------------- portions
// What bounds it: both products on the matrix cores (2 (DK + DV) flops a pair and head, 2176 cycles a SIMD and tile at 512 + 64), the vector work
// beside them (O's rescaling when a maximum moves is half of it; a product of 32 cycles keeps the vector unit for 8) and the LDS reads that feed
// them: a 32 x 32 x 16 product takes 1 KB.  So a row set has to be 32 rows (with 16 the same reads feed half the products), and 32 rows x (DK of Q +
// DV of O) are 400 registers: two waves share a row set, on one SIMD.  The score wave holds Q and a quarter of O: it makes a tile's scores and weights and
// adds its quarter; the value wave, one tile behind, holds three quarters of O and takes the weights and the factor of the maximum's move from LDS.
// Each thus has registers for fragments read three products ahead, the scores meet nowhere and a weight is made once; one barrier a tile.
// (Both holding half of Q and half of O, scores meeting in LDS, two barriers a tile: fragments one product ahead, 5150 cycles a tile of 32 keys, now 3900.
// Twelve waves, one of scores and two of values a row set: 168 registers do not hold a third of O's accumulators and a second place where ways meet.)
// Value waves fetch the rows: a DMA without addresses of its own in a lane's registers, and the score waves' reads wait for nothing but themselves.
// 4 portions of 1500 - 2548 tokens, 16 heads, 512 + 64: 1535 us -> 408 -> 340 us (870 TFLOP/s), 50 us of it the rows' way to LDS, 30
// us the rescaling, some 60 us workgroups' starts and ends: four follow each other on a CU, which each fills, and the queries' and outputs' 563 MB
// (115 us at 4.9 TB/s by themselves) come and go partly beside other workgroups' tiles; the outputs
// past the L2, but for those of ranges, which the join reads (348 -> 342 on one card; 5 of 114 - 142, 256 + 64: 24.7 -> 23.1; 3 of 1720 206 -> 199; ranges' 35.4 ->
// 36.5, not so.  The queries past it: 339, but 3 of 17 - 26 13.5 -> 15.3).  2 of 2253 tokens, 8 heads 178 -> 140; 6 of 50 - 353 38 -> 32; 4 of
// 470, 256 + 64: 35 -> 31.5; 5 of 23 - 225, 8 heads 29.0 -> 28.1.  One tile and full sets cost the two roles' one after the other: 8 portions of 8 tokens, 16
// heads 12.5 -> 12.7, 40 of 17 15.9 -> 16.4, the largest loss seen.  (Two pieces of queries an LDS turn without bank conflicts, outputs several turns at a
// time, no barrier behind the last weights, sets without rows only at the barriers: 13.7, 17.2 without them; 8 of 2 tokens 13.2 -> 10.1.)
// RANGES: splits > 1 (the outputs are partial ones then)
template <int DK, int DV, bool RANGES>
__global__ __launch_bounds__(512, 2) void latent_prompt_kernel(float* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml,
                                                               const float* __restrict__ q_abs, const bf16_t* __restrict__ cache,
                                                               const int* __restrict__ table, int64_t table_stride,
                                                               const int* __restrict__ req_rows, const int* __restrict__ seq_lens,
                                                               const int* __restrict__ cu_q, int B, int H, float scale, int QT, int HB, int splits,
                                                               const float* __restrict__ sink) {
  static_assert(DK - DV == 64, "the rotated entries' image");
  constexpr int NKS = DK / 16, NA = DV / 16, KT = 32;       // 16-wide steps of the first product, those over the latent entries
  constexpr int NVS = DV / 128, NVV = 3 * NVS;               // 32-column tiles of O in a score wave (the last ones), in a value wave
  // A tile's rows in LDS: the latent entries with 48 bytes of padding (16 rows' 16-byte reads touch all banks once, and so do the 4 x 32 bytes of a
  // transposing read), and behind them the rotated entries, 128 bytes a row, a row's pieces in places changed by its number.
  constexpr int ROW = DV * 2 + 48, TAIL = KT * ROW, IMAGE = TAIL + KT * 128;
  constexpr int NL = DV == 512 ? 7 : 0, NQ = NKS - NL;  // query fragments in LDS, in registers
  // objects of their own: the compiler then knows that a tile's reads do not meet a later tile's DMA
  __shared__ __attribute__((aligned(1024))) char img0[IMAGE], img1[IMAGE], img2[IMAGE];
  __shared__ __attribute__((aligned(16))) f32x4_t s_p[2][4][2][64];  // weights [tile & 1][row set][16 keys][lane]
  __shared__ __attribute__((aligned(16))) f32x4_t s_q[4][NL ? NL : 1][64];
  __shared__ __attribute__((aligned(16))) char s_turn[NL ? 16 : 4 * 4096];
  __shared__ float s_alpha[2][4][32];
  __shared__ float2 s_ml[4][32];
  __shared__ __attribute__((aligned(16))) int s_slot[4][KT];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), hi = lane >> 5;
  const int set = wave & 3, role = wave >> 2, rows0 = set * 32;
  int tok0 = 0;
  const int b = find_group_by_keys(cu_q, seq_lens, B, QT, (int)blockIdx.x, (int)gridDim.x, &tok0);
  if (b < 0) return;
  const int h0 = blockIdx.y * HB, z = blockIdx.z;
  const int first = cu_q[b], q_len = cu_q[b + 1] - first, start = seq_lens[b] - q_len;
  const int last_tok = min(tok0 + QT, q_len) - 1;
  const int set_lo = start + tok0 + rows0 / HB;  // keys up to here are seen by every row of the set
  const int n_keys = start + last_tok + 1;
  const int per = max(((n_keys + splits - 1) / splits + KT - 1) / KT * KT, kLeastRange);
  const int k_begin = z * per, k_end = min(n_keys, k_begin + per);
  const int n_tiles = k_begin < k_end ? (k_end - k_begin + KT - 1) / KT : 0;
  const float sharp = fmaxf(fabsf(scale) * 1.4426950408889634f, 1e-30f);  // scores to log2 (times a scale's sign, which Q takes: exact)
  const int* trow = table + (size_t)req_rows[b] * table_stride;
  const char* base = reinterpret_cast<const char*>(cache);
  auto slot_at = [&](int j0) { return trow[min(j0 + (lane & 31), n_keys - 1)]; };  // past the range: some row of the sequence, weight zero
  // Value waves fetch.  Rows 8 v ... + 7: a row's latent entries are one instruction with one slot for the wave, the eight rows' rotated entries another.
  // (Rows of 73 pieces over instructions of 64 took 20 vector operations and an LDS read in front of each.)
  auto dma = [&](char* dst, int slot) __attribute__((always_inline)) {  // slot: of row 8 v + lane / 8
    int l = lane, v = wave - 4;
    asm volatile("" : "+v"(l), "+s"(v));  // the places are worked out anew each tile: kept over the loop they would spill
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const char* row = base + (uint64_t)(uint32_t)__builtin_amdgcn_readlane(slot, 8 * j) * (DK * 2);
      if (DV == 512 || lane < 32) __builtin_amdgcn_global_load_lds((glb_void_t*)(row + l * 16), (lds_void_t*)(dst + (8 * v + j) * ROW), 16, 0, 0);
    }
    const int r = 8 * v + (l >> 3);
    __builtin_amdgcn_global_load_lds((glb_void_t*)(base + (uint64_t)(uint32_t)slot * (DK * 2) + DV * 2 + ((l ^ (r >> 1)) & 7) * 16),
                                     (lds_void_t*)(dst + TAIL + v * 1024), 16, 0, 0);
  };

  // ---- queries: in whole cache lines, 8 lanes for a row's 32 columns, and by way of LDS into their fragments' order (fragments straight from memory
  // touch 64 rows' lines with every load: 60 us of 460 at 8096 tokens and 16 heads).  The two waves of a row set take 32-column pieces in turn, the
  // score wave keeps them: its own through LDS of its own, the other one's by way of two images, all at once.  (The whole way of a role, these loads
  // included, lies behind one branch: what one role alone needs must not live beside the other's.)
  constexpr int NU = DK / 64;  // a wave's pieces
  auto first_slot = [&]() { return role ? trow[min(k_begin + 8 * (wave - 4) + (lane >> 3), n_keys - 1)] : slot_at(k_begin + wave * KT); };
  auto queries = [&](auto fetch, auto keep) __attribute__((always_inline)) {
    // slots in front of the queries: the value waves' of the first tile, the next two tiles' by way of LDS
    const int slot = first_slot();
    float4 x[NU][4];
    const float sign = scale < 0.f ? -1.f : 1.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = rows0 + (lane >> 3) + 8 * i, tl = tok0 + r / HB, hh = h0 + r % HB;
      const bool valid = r < QT * HB && tl < q_len && hh < H;
      const float* qrow = q_abs + (((size_t)first + (valid ? tl : tok0)) * H + (valid ? hh : h0)) * DK + role * 32 + 4 * (lane & 7);
#pragma unroll
      for (int u = 0; u < NU; ++u) x[u][i] = *reinterpret_cast<const float4*>(qrow + 64 * u);
    }
    if (fetch) dma(img0, slot);
    else if (wave < 3 && lane < KT) s_slot[wave][lane] = slot;
    char* other = (set < 2 ? img1 : img2) + (set & 1) * (2 * NU * 1024);
    static_assert(IMAGE >= 4 * NU * 1024, "two row sets' fragments");
    // a piece to two fragments: [column / 16][column / 8 & 1][row][8 columns], four rows' places changed by the columns' number against bank conflicts
    auto put = [&](char* at, const float4(&y)[4]) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<uint2*>(at + ((lane & 7) >> 2) * 1024 + ((((lane >> 1) & 1) * 32 + (lane >> 3) + 8 * i) ^ ((lane >> 1) & 3) * 4) * 16 + (lane & 1) * 8) =
            uint2{pack_bf16(y[i].x * sign, y[i].y * sign), pack_bf16(y[i].z * sign, y[i].w * sign)};
    };
    auto place = [&](int k) { return k * 1024 + (lane ^ (2 * (k & 1) + hi) * 4) * 16; };
    if (fetch) {
#pragma unroll
      for (int u = 0; u < NU; ++u) put(other + u * 2048, x[u]);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's pieces of the first tile
    } else {
      char* turn = reinterpret_cast<char*>(s_p) + set * 4096;  // two pieces at a time
#pragma unroll
      for (int u0 = 0; u0 < NU; u0 += 2) {
#pragma unroll
        for (int u = u0; u < u0 + 2 && u < NU; ++u) put(turn + (u - u0) * 2048, x[u]);
        wave_fence();
#pragma unroll
        for (int u = u0; u < u0 + 2 && u < NU; ++u)
#pragma unroll
          for (int k = 0; k < 2; ++k) keep(4 * u + k, turn + place(2 * (u - u0) + k));
        wave_fence();
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 2 * NU; ++k) keep(k / 2 * 4 + 2 + (k & 1), other + place(k));
    __syncthreads();
  };

  // transposing read of values: a 16-lane group reads 4 keys x 16 columns and hands lane j its column's four keys
  const int v_off = (4 * hi + ((lane & 15) >> 2)) * ROW + (16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
  auto vfrag = [&](const char* p) __attribute__((always_inline)) {  // 32 columns of 16 keys
    const s16x4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)p);
    const s16x4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(p + 8 * ROW));
    return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  // a row set's outputs times f by way of LDS, `some` times 32 columns at a time, so that a row's are stored as cache lines (lanes' own 16 bytes of 64
  // rows' lines: 60 us of 460 at 8096 tokens and 16 heads); a row's 16-byte pieces change places by its number, against bank conflicts
  auto finish = [&](const f32x16_t* o, auto nvt, auto some, char* turn, int col0) __attribute__((always_inline)) {
    int l = lane;
    asm volatile("" : "+v"(l));  // the rows are worked out anew: no registers for them meanwhile
    float f = 1.f;
    if (splits == 1) {
      const int hh = min(h0 + (rows0 + (l & 31)) % HB, H - 1);
      const float2 ml = s_ml[set][l & 31];
      const float sf = sink_factor(sink, hh, ml.x);
      f = sf / (sf * ml.y + sink_weight(sink, hh, ml.x));
    }
    float* dst[4];
    bool valid[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = rows0 + (l >> 3) + 8 * i, tl = tok0 + r / HB, h = h0 + r % HB;
      valid[i] = r < QT * HB && tl < q_len && h < H && (n_tiles > 0 || splits == 1);  // without keys the partial output is not read
      const size_t row = ((size_t)first + tl) * H + h;
      dst[i] = (splits == 1 ? out + row * DV : part_o + (row * splits + z) * DV) + col0 + 4 * (l & 7);
    }
#pragma unroll
    for (int vt0 = 0; vt0 < nvt; vt0 += some) {
#pragma unroll
      for (int n = 0; n < some; ++n)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x16_t& x = o[vt0 + n];
          *reinterpret_cast<float4*>(turn + n * 4096 + (l & 31) * 128 + (((2 * g + hi) ^ l) & 7) * 16) =
              float4{x[4 * g] * f, x[4 * g + 1] * f, x[4 * g + 2] * f, x[4 * g + 3] * f};
        }
      wave_fence();
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (valid[i]) {
#pragma unroll
          for (int n = 0; n < some; ++n) {
            const f32x4_t x = *reinterpret_cast<const f32x4_t*>(turn + n * 4096 + ((l >> 3) + 8 * i) * 128 + (((l & 7) ^ (l >> 3)) & 7) * 16);
            f32x4_t* to = reinterpret_cast<f32x4_t*>(dst[i] + (vt0 + n) * 32);
            if constexpr (RANGES) *to = x;
            else __builtin_nontemporal_store(x, to);
          }
        }
      }
      wave_fence();
    }
  };

  auto fetch = [&](char* next, int t) __attribute__((always_inline)) {
    int slot = 0;
    if (wave == 7 && t + 3 < n_tiles) slot = slot_at(k_begin + (t + 3) * KT);  // in front of the DMA: waiting for it does not wait for the DMA
    if (t + 1 < n_tiles) dma(next, s_slot[(t + 1) & 3][8 * (wave - 4) + (lane >> 3)]);
    return slot;
  };
  auto arrived = [&](int slot, int t) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's pieces of tile t + 1
    if (wave == 7 && lane < KT) s_slot[(t + 3) & 3][lane] = slot;
    __syncthreads();
  };

  // ---- Iteration t: the score waves turn tile t into weights and add their columns' values, the value waves add tile t - 1's to theirs and fetch
  // tile t + 1 into the image of tile t - 2.  Both ways pass the same barriers, n_tiles of them: nothing is waited for after the last weights.
  // A set without rows: its share of the rows' way to LDS and the barriers (a scalar branch, which a wave takes or not), nothing of the LDS reads
  if (__builtin_amdgcn_readfirstlane(rows0 >= QT * HB || tok0 + rows0 / HB >= q_len) != 0) {
    if (n_tiles > 0) {
      const int slot = first_slot();
      if (role == 0) {
        if (wave < 3 && lane < KT) s_slot[wave][lane] = slot;
      } else {
        dma(img0, slot);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      __syncthreads();
      __syncthreads();
    }
    for (int t = 0; t < n_tiles; ++t) {
      if (role == 1) arrived(fetch(t % 3 == 0 ? img1 : t % 3 == 1 ? img2 : img0, t), t);
      else __syncthreads();
    }
    return;
  }
  if (role == 0) {
    const int r = rows0 + (lane & 31), tl = tok0 + r / HB;
    const int limit = r < QT * HB && tl < q_len && h0 + r % HB < H ? start + tl : -1;  // the last key position that this lane's row sees, -1: no row
    const int k_off = (lane & 31) * ROW + hi * 16;
    bf16x8_t qf[NQ];
    if (n_tiles > 0)
      queries(std::false_type{}, [&](int ks, const char* at) __attribute__((always_inline)) {
        const bf16x8_t f = *reinterpret_cast<const bf16x8_t*>(at);
        if (ks < NQ) qf[ks < NQ ? ks : 0] = f;
        else s_q[set][ks < NQ ? 0 : ks - NQ][lane] = __builtin_bit_cast(f32x4_t, f);
      });
    float m = -INFINITY, lsum = 0.f;  // reference maximum (log2), this lane's share of the row's sum
    f32x16_t o[NVS];
#pragma unroll
    for (int vt = 0; vt < NVS; ++vt)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[vt][e] = 0.f;
    auto scores = [&](const char* buf, int t) __attribute__((always_inline)) {
      constexpr int AHEAD = 3;  // fragments are read so many products before their use
      int l = lane;
      asm volatile("" : "+v"(l));
      auto kfrag = [&](int ks) __attribute__((always_inline)) {
        if (ks < NA) return *reinterpret_cast<const bf16x8_t*>(buf + k_off + ks * 32);
        return *reinterpret_cast<const bf16x8_t*>(buf + TAIL + (l & 31) * 128 + (((2 * (ks - NA) + (l >> 5)) ^ ((l & 31) >> 1)) & 7) * 16);
      };
      f32x16_t s;
      bf16x8_t kf[AHEAD + 1], ql[2];
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = 0.f;
#pragma unroll
      for (int ks = 0; ks < AHEAD; ++ks) kf[ks] = kfrag(ks);
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        if (ks + AHEAD < NKS) kf[(ks + AHEAD) % (AHEAD + 1)] = kfrag(ks + AHEAD);
        if (ks + 1 >= NQ && ks + 1 < NKS) ql[(ks + 1) & 1] = __builtin_bit_cast(bf16x8_t, s_q[set][ks + 1 >= NQ ? (ks + 1 - NQ) % (NL ? NL : 1) : 0][lane]);
        __builtin_amdgcn_sched_barrier(0);
        s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[ks % (AHEAD + 1)], ks < NQ ? qf[ks < NQ ? ks : 0] : ql[ks & 1], s, 0, 0, 0);
      }
      // a lane's keys: j0 + (e & 3) + 8 (e >> 2) + 4 hi
      const int j0 = k_begin + t * KT;
      if (j0 + KT - 1 > set_lo || j0 + KT > k_end) {
        const int last = min(limit, k_end - 1) - j0 - 4 * hi;
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if ((e & 3) + 8 * (e >> 2) > last) s[e] = -INFINITY;
      }
      float mx = -INFINITY;
#pragma unroll
      for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s[e]);
      mx = pair_max(mx) * sharp;
      const float m_new = fmaxf(m, mx);
      const float alpha = m_new == m ? 1.f : __builtin_amdgcn_exp2f(m - m_new);
      if (hi == 0) s_alpha[t & 1][set][lane] = alpha;
      if (__builtin_amdgcn_ballot_w64(m_new != m) != 0) {
#pragma unroll
        for (int vt = 0; vt < NVS; ++vt)
#pragma unroll
          for (int e = 0; e < 16; ++e) o[vt][e] *= alpha;
        lsum *= alpha;
        m = m_new;
      }
      const char* vp = buf + v_off + NVV * 64;
      bf16x8_t vf[3];
      vf[0] = vfrag(vp);
      vf[1] = vfrag(vp + 64);
      const float ref = m == -INFINITY ? 0.f : m;  // no key yet: every weight is exp2(-inf) = 0
      float sum = 0.f;  // of the fp32 weights
      uint32_t pw[8];
#pragma unroll
      for (int e = 0; e < 16; e += 2) {
        const float w0 = weight(s[e], sharp, ref), w1 = weight(s[e + 1], sharp, ref);
        sum += w0 + w1;
        pw[e >> 1] = pack_bf16(w0, w1);
      }
      lsum += sum;
      if (t + 1 == n_tiles) {
        lsum += __shfl_xor(lsum, 32, 64);
        if (hi == 0) s_ml[set][lane] = float2{m * kLn2, lsum};
      }
#pragma unroll
      for (int w = 0; w < 2; ++w)
        *reinterpret_cast<Q4*>(&s_p[t & 1][set][w][lane]) = Q4{pw[4 * w], pw[4 * w + 1], pw[4 * w + 2], pw[4 * w + 3]};
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 2 * NVS; ++i) {  // O^T += V^T P^T, 16 keys a step: a lane's eight of them are what its registers 8 step ... hold
        if (i + 2 < 2 * NVS) vf[(i + 2) % 3] = vfrag(vp + (i + 2) / NVS * 16 * ROW + (i + 2) % NVS * 64);
        __builtin_amdgcn_sched_barrier(0);
        const int w = i / NVS * 4;
        const Q4 pq{pw[w], pw[w + 1], pw[w + 2], pw[w + 3]};
        o[i % NVS] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i % 3], __builtin_bit_cast(bf16x8_t, pq), o[i % NVS], 0, 0, 0);
      }
    };
    for (int t = 0; t < n_tiles; t += 3) {
      scores(img0, t);
      if (t + 1 < n_tiles) scores(img1, t + 1);
      if (t + 2 < n_tiles) scores(img2, t + 2);
    }
    if (hi == 0 && splits > 1 && limit >= 0) {
      const size_t row = ((size_t)first + tl) * H + h0 + r % HB;
      part_ml[(row * splits + z) * 2] = m * kLn2;
      part_ml[(row * splits + z) * 2 + 1] = lsum;
    }
    finish(o, std::integral_constant<int, NVS>{}, std::integral_constant<int, 1>{}, NL ? reinterpret_cast<char*>(s_q[set]) : s_turn + set * 4096, NVV * 32);
    asm volatile("; score waves");
  } else {
    if (n_tiles > 0) queries(std::true_type{}, [](int, const char*) {});
    f32x16_t o[NVV];
#pragma unroll
    for (int vt = 0; vt < NVV; ++vt)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[vt][e] = 0.f;
    auto values = [&](const char* buf, int t) __attribute__((always_inline)) {
      constexpr int SOME = 2;  // fragments are read so many at a time, a set ahead
      const char* vp = buf + v_off;
      const float alpha = s_alpha[t & 1][set][lane & 31];
      Q4 p[2];
#pragma unroll
      for (int w = 0; w < 2; ++w) p[w] = *reinterpret_cast<const Q4*>(&s_p[t & 1][set][w][lane]);
      bf16x8_t vf[2][SOME];
#pragma unroll
      for (int n = 0; n < SOME; ++n) vf[0][n] = vfrag(vp + n * 64);
      __builtin_amdgcn_sched_barrier(0);
      if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0) {
#pragma unroll
        for (int vt = 0; vt < NVV; ++vt)
#pragma unroll
          for (int e = 0; e < 16; ++e) o[vt][e] *= alpha;
      }
#pragma unroll
      for (int i = 0; i < 2 * NVV; i += SOME) {
        if (i + SOME < 2 * NVV) {
#pragma unroll
          for (int n = 0; n < SOME; ++n) vf[(i / SOME & 1) ^ 1][n] = vfrag(vp + (i + SOME + n) / NVV * 16 * ROW + (i + SOME + n) % NVV * 64);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = 0; n < SOME; ++n)
          o[(i + n) % NVV] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i / SOME & 1][n], __builtin_bit_cast(bf16x8_t, p[(i + n) / NVV]), o[(i + n) % NVV], 0, 0, 0);
      }
    };
    auto step = [&](const char* before, char* next, int t) __attribute__((always_inline)) {
      const int slot = fetch(next, t);
      values(before, t - 1);
      if (t < n_tiles) arrived(slot, t);
    };
    if (n_tiles > 0) {
      arrived(fetch(img1, 0), 0);
      int t = 1;  // (no step of the loop is conditional: where ways met, the accumulators had two places, and hundreds were spilled)
      for (; t + 2 <= n_tiles; t += 3) {
        step(img0, img2, t);
        step(img1, img0, t + 1);
        step(img2, img1, t + 2);
      }
      if (t <= n_tiles) {
        step(img0, img2, t);
        if (t + 1 <= n_tiles) step(img1, img0, t + 1);
      }
    }
    // by way of the two images that do not hold the last tile
    static_assert(IMAGE >= 2 * NVS * 4096, "two waves' turns");
    const int free_one = (n_tiles + (set >> 1)) % 3;
    finish(o, std::integral_constant<int, NVV>{}, std::integral_constant<int, NVS>{}, (free_one == 0 ? img0 : free_one == 1 ? img1 : img2) + (set & 1) * (NVS * 4096), 0);
    asm volatile("; value waves");
  }
}

// ---------------------------------------------------------------------------------------------------------------- decoded tokens
// What bounds it: the key rows' way from memory.  A wave walks 16-key tiles of its own (every fourth of the workgroup's range) through
// two LDS images of its own, so nothing waits at a barrier until the four partial results meet at the end, and the products of a tile
// (50 short MFMAs) hide under the next one's DMA.  The table entries of the tile after next are asked for before the DMA of the next
// one: memory counters retire in order, so waiting for them does not wait for the DMA behind them.
// 32 requests, 4096 keys, 16 heads, 512 + 64: 188 -> 50 us with the join (151 MB of rows, 31 us at 4.9 TB/s).
template <int DK, int DV>
__global__ __launch_bounds__(256, 1) void latent_decode_kernel(float* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml,
                                                               const float* __restrict__ q_abs, const bf16_t* __restrict__ cache,
                                                               const int* __restrict__ table, int64_t table_stride,
                                                               const int* __restrict__ req_rows, const int* __restrict__ seq_lens,
                                                               const int* __restrict__ cu_q, int B, int H, float scale, int QT, int HB, int splits,
                                                               const float* __restrict__ sink) {
  constexpr int NKC = DK / 32, NVT = DV / 16, ROW = LatentRow<DK>::bytes, PCS = LatentRow<DK>::pieces;
  constexpr int NDMA = (16 * PCS + 63) / 64, IMAGE = NDMA * 1024;  // a tile's image, its last instruction's idle lanes included
  extern __shared__ __attribute__((aligned(1024))) char dyn[];     // [wave][2][IMAGE]; afterwards the waves' outputs
  __shared__ int s_slot[4][2][16];
  __shared__ float s_ml[4][2][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lg = lane >> 4;
  int tok0 = 0;
  const int b = find_group_by_keys(cu_q, seq_lens, B, QT, (int)blockIdx.x, (int)gridDim.x, &tok0);
  if (b < 0) return;
  const int h0 = blockIdx.y * HB, z = blockIdx.z;
  const int first = cu_q[b], q_len = cu_q[b + 1] - first, start = seq_lens[b] - q_len;
  const int tl = tok0 + lr / HB, hh = h0 + lr % HB;
  const bool valid = lr < QT * HB && tl < q_len && hh < H;
  const size_t row = ((size_t)first + (valid ? tl : tok0)) * H + (valid ? hh : h0);
  const int limit = valid ? start + tl : -1;
  const int last_tok = min(tok0 + QT, q_len) - 1, n_keys = start + last_tok + 1;
  const int per = max(((n_keys + splits - 1) / splits + 63) / 64 * 64, kLeastRange);
  if (z > 0 && z * per >= n_keys) {  // no keys left for this range: its partial output is not read
    if (tid < 16 && valid) {
      part_ml[(row * splits + z) * 2] = -INFINITY;
      part_ml[(row * splits + z) * 2 + 1] = 0.f;
    }
    return;
  }
  const int k_begin = z * per + 16 * wave, k_end = min(n_keys, z * per + per);  // this wave: tiles k_begin, k_begin + 64, ...
  const float sharp = fmaxf(fabsf(scale) * 1.4426950408889634f, 1e-30f);
  bf16x8_t qf[NKC];
  {
    const float* qrow = q_abs + row * DK + 8 * lg;
    const float f = scale < 0.f ? -1.f : 1.f;
#pragma unroll
    for (int kc = 0; kc < NKC; ++kc) qf[kc] = scaled8(qrow + 32 * kc, f);
  }
  f32x4_t o[NVT];
#pragma unroll
  for (int vt = 0; vt < NVT; ++vt) o[vt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, lsum = 0.f;
  const int* trow = table + (size_t)req_rows[b] * table_stride;
  const char* base = reinterpret_cast<const char*>(cache);
  char* mine = dyn + wave * 2 * IMAGE;
  auto slot_at = [&](int j0) { return trow[min(j0 + lr, n_keys - 1)]; };  // past the range: some row of the sequence, weight zero
  auto dma = [&](int img) {
#pragma unroll
    for (int i = 0; i < NDMA; ++i) {
      const int key = i * 64 / PCS, t = i * 64 - key * PCS + lane;
      const int next = (t >= PCS) + (t >= 2 * PCS);
      const int ch = min(t - next * PCS, PCS - 2);
      const size_t slot = (size_t)s_slot[wave][img][min(key + next, 15)];
      __builtin_amdgcn_global_load_lds((glb_void_t*)(base + slot * (DK * 2) + ch * 16), (lds_void_t*)(mine + img * IMAGE + i * 1024), 16, 0, 0);
    }
  };
  if (k_begin < k_end) {
    const int s0 = slot_at(k_begin), s1 = slot_at(k_begin + 64);
    if (lane < 16) {
      s_slot[wave][0][lr] = s0;
      s_slot[wave][1][lr] = s1;
    }
    dma(0);
  }
  int img = 0;
  for (int j0 = k_begin; j0 < k_end; j0 += 64, img ^= 1) {
    const int later = slot_at(j0 + 128);
    if (j0 + 64 < k_end) {
      dma(img ^ 1);
      static_assert(NDMA == 19 || NDMA == 11, "the counted wait below");
      if constexpr (NDMA == 19) asm volatile("s_waitcnt vmcnt(19)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(11)" ::: "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    const char* buf = mine + img * IMAGE;
    f32x4_t acc[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kc = 0; kc < NKC; ++kc) {
      const bf16x8_t kf = *reinterpret_cast<const bf16x8_t*>(buf + lr * ROW + kc * 64 + lg * 16);
      acc[kc % 3] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[kc], acc[kc % 3], 0, 0, 0);
    }
    float s[4], mx = -INFINITY;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int j = j0 + 4 * lg + c;
      s[c] = j <= limit && j < k_end ? (acc[0][c] + acc[1][c]) + acc[2][c] : -INFINITY;
      mx = fmaxf(mx, s[c]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = pair_max(mx) * sharp;
    if (__builtin_amdgcn_ballot_w64(mx > m) != 0) {
      const float m_new = fmaxf(m, mx);
      const float alpha = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - m_new);
#pragma unroll
      for (int vt = 0; vt < NVT; ++vt) o[vt] *= alpha;
      lsum *= alpha;
      m = m_new;
    }
    const float ref = m == -INFINITY ? 0.f : m;
    float w[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) w[c] = weight(s[c], sharp, ref);
    lsum += (w[0] + w[1]) + (w[2] + w[3]);
    const uint32_t p01 = pack_bf16(w[0], w[1]), p23 = pack_bf16(w[2], w[3]);
    const s16x4_t pf = __builtin_bit_cast(s16x4_t, uint2{p01, p23});
    const char* vb = buf + (4 * lg + (lr >> 2)) * ROW + 8 * (lr & 3);
#pragma unroll
    for (int vt = 0; vt < NVT; ++vt) {
      const s16x4_t vf = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(vb + vt * 32));
      o[vt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(vf, pf, o[vt], 0, 0, 0);
    }
    if (lane < 16) s_slot[wave][img][lr] = later;
  }
  lsum += __shfl_xor(lsum, 16, 64);
  lsum += __shfl_xor(lsum, 32, 64);
  if (lg == 0) {
    s_ml[wave][0][lr] = m;
    s_ml[wave][1][lr] = lsum;
  }
  __syncthreads();  // also: no wave has a DMA or a read of an image left
  float M = -INFINITY, L = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) M = fmaxf(M, s_ml[w][0][lr]);
  const float ref = M == -INFINITY ? 0.f : M;
#pragma unroll
  for (int w = 0; w < 4; ++w) L = fmaf(s_ml[w][1][lr], __builtin_amdgcn_exp2f(s_ml[w][0][lr] - ref), L);
  float f = __builtin_amdgcn_exp2f(m - ref);
  M *= kLn2;
  float* dst;
  if (splits == 1) {
    const float sf = sink_factor(sink, hh < H ? hh : h0, M);
    f *= sf / (sf * L + sink_weight(sink, hh < H ? hh : h0, M));
    dst = out + row * DV;
  } else {
    if (wave == 0 && lg == 0 && valid) {
      part_ml[(row * splits + z) * 2] = M;
      part_ml[(row * splits + z) * 2 + 1] = L;
    }
    dst = part_o + (row * splits + z) * DV;
  }
  // every wave's share of the outputs to LDS, then wave w adds up columns w NVT / 4 16 ...
  f32x4_t* so = reinterpret_cast<f32x4_t*>(dyn);  // [wave][NVT][lane]
#pragma unroll
  for (int vt = 0; vt < NVT; ++vt) so[(wave * NVT + vt) * 64 + lane] = o[vt] * f;
  __syncthreads();
  if (!valid) return;
#pragma unroll
  for (int i = 0; i < NVT / 4; ++i) {
    const int vt = wave * (NVT / 4) + i;
    f32x4_t t = so[vt * 64 + lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) t += so[(w * NVT + vt) * 64 + lane];
    *reinterpret_cast<f32x4_t*>(dst + vt * 16 + 4 * lg) = t;
  }
}

// ---------------------------------------------------------------------------------------------------------------- ranges
// A wave per row: the ranges' weights in the lanes, then the partial outputs of those that have one, four at a time (each is a line read
// that waits for memory).
template <int DV>
__global__ __launch_bounds__(256) void latent_join_kernel(float* __restrict__ out, const float* __restrict__ part_o,
                                                          const float* __restrict__ part_ml, int64_t rows, int splits,
                                                          const float* __restrict__ sink, int H) {
  constexpr int N = DV / 256;
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (row >= rows) return;
  const float* ml = part_ml + row * splits * 2;
  float M = -INFINITY, L = 0.f;
  for (int i = lane; i < splits; i += 64) M = fmaxf(M, ml[2 * i]);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) M = fmaxf(M, __shfl_xor(M, o, 64));
  const float ref = M == -INFINITY ? 0.f : M;
  for (int i = lane; i < splits; i += 64) L = fmaf(ml[2 * i + 1], expf(ml[2 * i] - ref), L);
  L = wave_sum(L);
  const float sf = sink_factor(sink, (int)(row % H), M);
  const float inv = sf / (sf * L + sink_weight(sink, (int)(row % H), M));
  f32x4_t acc[N];
#pragma unroll
  for (int n = 0; n < N; ++n) acc[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int i0 = 0; i0 < splits; i0 += 64) {
    const bool in = i0 + lane < splits;
    const float w = in && ml[2 * (i0 + lane) + 1] != 0.f ? expf(ml[2 * (i0 + lane)] - ref) : 0.f;
    uint64_t live = __builtin_amdgcn_ballot_w64(w != 0.f);
    while (live) {
      f32x4_t x[4][N];
      float f[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = live ? __builtin_ctzll(live) : 0;
        f[j] = live ? __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w), i)) * inv : 0.f;
        if (live) {
#pragma unroll
          for (int n = 0; n < N; ++n) x[j][n] = *reinterpret_cast<const f32x4_t*>(part_o + (row * splits + i0 + i) * DV + n * 256 + lane * 4);
        } else {
#pragma unroll
          for (int n = 0; n < N; ++n) x[j][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
        live &= live - 1;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int n = 0; n < N; ++n) acc[n] += x[j][n] * f[j];
    }
  }
#pragma unroll
  for (int n = 0; n < N; ++n) *reinterpret_cast<f32x4_t*>(out + row * DV + n * 256 + lane * 4) = acc[n];
}

}  // namespace

// 1: launched; 0: these sizes are not these kernels' (the caller takes the other ones); < 0: an error code.
extern "C" __attribute__((visibility("hidden"))) int mix_latent_attn_mfma(float* out, float* part_o, float* part_ml, const float* q_abs, const void* cache,
                                                                          const int* table, int64_t table_stride, const int* req_rows,
                                                                          const int* seq_lens, const int* cu_q, int batch, int total_q, int H, int dk,
                                                                          int dv, float scale, const float* sink, int splits, hipStream_t s) {
  const auto al = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if (!((dk == 576 && dv == 512) || (dk == 320 && dv == 256))) return 0;
  if (!al(cache) || !al(q_abs) || !al(out) || (part_o && !al(part_o))) return 0;  // 16-byte loads, DMA pieces and stores
  // One 16-row group per request or so: its keys over the waves; more rows: 128 a workgroup.  (One portion of 32 tokens after 1000 keys: as 32
  // groups of 16 rows every key row is read 32 times.)
  const int rows = H < 16 ? H : 16;
  const bool decode = total_q <= batch * (16 / rows);
  const int HB = decode ? rows : (H < 128 ? H : 128), QT = (decode ? 16 : 128) / HB;
  const int groups = QT == 1 ? total_q : total_q / QT + batch, heads = (H + HB - 1) / HB;
  if (heads > 65535) return 0;
  // One workgroup fills a CU's LDS: ranges past 256 workgroups would only queue, each with its own start and partial outputs (32 requests,
  // 4096 keys, 16 heads: 16 ranges 68 us, 8 ranges 50 us)
  splits = std::max(1, std::min(splits, 256 / std::max(1, groups * heads)));
  const dim3 grid(groups, heads, splits);
#define LAT_ARGS out, part_o, part_ml, q_abs, cp<bf16_t>(cache), table, table_stride, req_rows, seq_lens, cu_q, batch, H, scale, QT, HB, splits, sink
#define LAT_LAUNCH(DK, DV)                                                                                                          \
  if (decode) {                                                                                                                     \
    const size_t image = (size_t)((16 * LatentRow<DK>::pieces + 63) / 64) * 1024, join = (size_t)4 * DV * 16 * sizeof(float);       \
    const size_t lds = 8 * image > join ? 8 * image : join;                                                                         \
    MIX_REQUIRE(ensure_lds((const void*)latent_decode_kernel<DK, DV>, lds) == 0, "latent_attn: %zu bytes of LDS", lds);             \
    hipLaunchKernelGGL((latent_decode_kernel<DK, DV>), grid, dim3(256), lds, s, LAT_ARGS);                                          \
  } else if (splits > 1) {                                                                                                          \
    hipLaunchKernelGGL((latent_prompt_kernel<DK, DV, true>), grid, dim3(512), 0, s, LAT_ARGS);                                      \
  } else {                                                                                                                          \
    hipLaunchKernelGGL((latent_prompt_kernel<DK, DV, false>), grid, dim3(512), 0, s, LAT_ARGS);                                     \
  }
  if (dk == 576) {
    LAT_LAUNCH(576, 512)
  } else {
    LAT_LAUNCH(320, 256)
  }
#undef LAT_LAUNCH
#undef LAT_ARGS
  MIX_LAUNCHED("latent_attn (matrix cores)");
  if (splits > 1) {
    const int64_t n = (int64_t)total_q * H;
    if (dv == 512)
      hipLaunchKernelGGL(latent_join_kernel<512>, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, s, out, part_o, part_ml, n, splits, sink, H);
    else
      hipLaunchKernelGGL(latent_join_kernel<256>, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, s, out, part_o, part_ml, n, splits, sink, H);
    MIX_LAUNCHED("latent_attn join");
  }
  return 1;
}
