// Sliding-window attention with mixed heads on the matrix cores (bf16 caches): the form of window_attn_kernel (mix_delta.hip) for
// portions of query tokens.  Same C entry, msgl_mix_window_attn; this file holds one kernel and the function that launches it.
//
// What bounds it: per visible (query, key) pair and H heads the two products are 2 H (d + 2 dv) flops for the bf16 matrix cores, the
// mixing of the scores 2 H^2 flops in fp32 and the softmax about ten vector operations per head.  The mixing is itself a product, with the
// heads as contraction; an fp32 16 x 16 x 4 instruction holds its SIMD's vector unit for all of its 32 cycles, a bf16 one for 8 of 16 (16 x 16 x 32)
// or 8 of 32 (32 x 32 x 16, hence these where the rows are 32).  A tile of 32 keys and 16 tokens at H = 16 is 3072 matrix cycles a SIMD and about
// 3700 in which it cannot start a vector operation, of 6300 measured; 64 KB of keys and values a tile and compute unit come in at 64 bytes a cycle,
// for 20 - 40 us of the whole.
//
// 4 requests of 1500 - 2548 new tokens, 16 heads of 128 over 4 key heads, window 2048: 5182 us on the vector units, 294 us with raw scores
// exchanged through LDS, 257 us with a tile's rows free of address work, 205 us as below: raw scores stay in registers (their product's rows
// are four heads of four queries, so that its result is the mixing's first operand as it stands), rows by DMA (a register copy on its way was
// a fifth of the LDS writes), 32-row value products, a reference that lags, outputs in whole lines.  5 requests of 1053 tokens 120 -> 98; 7 decoded
// tokens of 8 heads 25 -> 21.  Of the 205, 20 are the weights' third part, 18 the start and end of a workgroup, 15 the last workgroups alone.
// Waves in opposite orders (scores first, softmax first) gain nothing: 257 against 231 at that stage.
//
// Precision: scores are bf16 x bf16 products with fp32 sums, mixed and exponentiated in fp32; a probability enters the second product
// as the sum of three bf16 numbers (its rounding, that of what is left, and the rest: 8 bits each), which is the fp32 number itself.
#include "mix_common.h"

namespace {

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(1))) void glb_void_t;
typedef __attribute__((address_space(3))) void lds_void_t;

constexpr int kWinTile = 32;           // keys per tile
constexpr int kWinKC = 4, kWinVC = 8;  // head sizes up to 128
constexpr int kWinRow = 36;            // floats of a mixed (head, query) row in LDS: 32 keys, padded so that 16 rows cover all banks
constexpr int kAllButLoads = 0x78f;    // what the compiler may still move past a mark: everything but memory loads
constexpr int kWinHead = 16 * kWinRow + 4;  // floats of a head: four of them apart, 16 heads' 16-byte writes cover all banks

// Workgroup = 16 query tokens of one request x all NH heads (x one of `splits` key ranges), NH / 2 waves of two heads each, which share
// a key / value head.  Two phases per tile t of 32 keys, a barrier behind each:
//   the waves share the tile's (query, key) pairs: 4 queries x 16 keys of a wave (twice as many at 8 heads): raw scores of tile t + 1 as
//   Q K^T with rows (head of four, query of four), mixed scores as their product with the table over the heads
//   mixed scores to LDS; the waves share the heads, 32 rows (two heads of 16 queries): mask, online softmax, O^T += V^T P^T (a lane reads
//   four consecutive keys of its row, the layout the product takes; V through transposing LDS reads).  Meanwhile the next rows arrive.
// FULL: key heads of 128
template <int NH, int G, bool FULL>
__global__ __launch_bounds__(NH * 32, 2) void window_attn_mfma_kernel(bf16_t* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml,
                                                                  const bf16_t* __restrict__ src, int64_t ld_src, int g_off,
                                                                  const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
                                                                  const int* __restrict__ table, int64_t table_stride,
                                                                  const int* __restrict__ req_rows, const int* __restrict__ seq_lens,
                                                                  const int* __restrict__ cu_q, int B, int total_q, int d, int dv,
                                                                  int window, float scale, const float* __restrict__ talk, int splits) {
  constexpr int HPW = 2, NT = NH * 32, NW = NH / 2, KC = kWinKC, VC = kWinVC, NJ = NH / 4, KSW = 8 / NW;
  constexpr int RS = G * KC * 32;  // a row of keys or values in LDS
  // objects of their own: the compiler then knows which reads do not meet a DMA under way
  __shared__ __attribute__((aligned(16))) float mixed[NH * kWinHead];  // [NH][16 queries][kWinRow], a head's rows kWinHead floats
  __shared__ __attribute__((aligned(1024))) uint16_t sk[kWinTile * RS], sv0[kWinTile * RS], sv1[kWinTile * RS];
  __shared__ int s_slot[4][kWinTile];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lr = lane & 15, lg = lane >> 4, hi = lane >> 5;
  int tok0 = 0;
  const int b = find_group_by_keys(cu_q, seq_lens, B, 16, (int)blockIdx.x, (int)gridDim.x, &tok0);
  if (b < 0) return;
  const int q_len = cu_q[b + 1] - cu_q[b], start = seq_lens[b] - q_len;
  const int last_tok = min(tok0 + 16, q_len) - 1;
  const bool valid = tok0 + lr < q_len;
  const size_t tok = (size_t)cu_q[b] + (valid ? tok0 + lr : tok0);
  const int limit = valid ? start + tok0 + lr : -1;
  const int lo_row = window > 0 ? max(0, limit - window + 1) : 0;
  const int n_keys = start + last_tok + 1, lo_blk = window > 0 ? max(0, start + tok0 - window + 1) : 0;
  const int per = ((n_keys - lo_blk + splits - 1) / splits + kWinTile - 1) / kWinTile * kWinTile;
  const int k_begin = lo_blk + (int)blockIdx.y * per, k_end = min(n_keys, k_begin + per);
  const int all_hi = start + tok0, all_lo = window > 0 ? max(0, start + last_tok - window + 1) : 0;  // keys that every row sees
  constexpr int TW = kWinTile;
  const int* trow = table + (size_t)req_rows[b] * table_stride;
  const int last_key = max(k_end - 1, 0);
  const int in_tile = (int)threadIdx.x & (kWinTile - 1);
  auto slot_at = [&](int j0) { return trow[min(j0 + in_tile, last_key)]; };
  auto put_slot = [&](int slot, int buf) {
    if (threadIdx.x < kWinTile) s_slot[buf][threadIdx.x] = slot;
  };
  // the first tiles' slots, in front of the queries; later ones a tile before they go to LDS: there the whole workgroup waited for the table
  const int slot0 = slot_at(k_begin), slot1 = slot_at(k_begin + TW), slot2 = slot_at(k_begin + 2 * TW);
  int next_slot = slot_at(k_begin + 3 * TW);
  const int h0 = wave * HPW, rep = NH / G, grp = h0 / rep;
  const float scale2 = scale * 1.4426950408889634f;
  // the table as second operand: column = mixed head, contraction index 4 j + lg = raw head
  const int quad = NH == 16 ? wave & 3 : wave, ks0 = NH == 16 ? wave >> 2 : 0;
  float tk[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) tk[j] = lr < NH ? talk[lr * NH + 4 * j + lg] * scale2 : 0.f;
  bf16x8_t qf[NJ][KC];  // row 4 (head of four) + (query of four); a row that is none takes the first one's queries, its sums go nowhere
  {
    const int t = tok0 + 4 * quad + (lr & 3);
    const bf16_t* qrow = src + (size_t)(cu_q[b] + (t < q_len ? t : tok0)) * (size_t)ld_src + (size_t)(lr >> 2) * d;
    // 16 bytes from where they lie, whatever the rows' stride: global memory takes any alignment (12 tokens, unaligned: 16.6 us, number by number
    // 31.5).  Past the head its last piece for now: a lane's condition on a load would be a wait for it.
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        const int k = kc * 32 + lg * 8;
        qf[j][kc] = bf16x8_t{};
        if (FULL || kc * 32 < d) __builtin_memcpy(&qf[j][kc], qrow + 4 * j * d + (FULL ? k : min(k, d - 8)), 16);
      }
  }
  // this lane's row of the second product: head h0 + (lane >> 4 & 1), query lr
  f32x16_t o[VC / 2];
#pragma unroll
  for (int nb = 0; nb < VC / 2; ++nb)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[nb][e] = 0.f;
  float m = -INFINITY, lsum = 0.f;
  const uint32_t nk = (uint32_t)(G * d), nv = (uint32_t)(G * dv);
  // 16-byte pieces of a tile's key and value rows (both 128 wide per head in LDS).  A row's pieces divide the workgroup
  // (both are powers of two), so a thread has one column of the rows key0, key0 + ROWS, ...: its offsets are known once (a division and four
  // 32-bit products a piece and tile, at a quarter of the rate, were a tenth of the kernel).
  static_assert(KC * 4 == VC * 2, "keys and values share the piece map");
  constexpr int PCS = G * VC * 2, ROWS = NT / PCS, NP = kWinTile / ROWS;
  const int key0 = (int)threadIdx.x / PCS, piece = (int)threadIdx.x & (VC * 2 - 1), hv = (int)threadIdx.x % PCS / (VC * 2);
  // Rows come by DMA, their pieces in places changed by the row's number: 16 rows' reads of keys and 4 rows' transposing reads of values touch all
  // banks once.  (Rows 8 apart: odd ones' keys the other half.)
  constexpr int FLIP = ROWS & 8;
  const int ck0 = (piece ^ key0) & 15, ck1 = ck0 ^ FLIP, cv = piece ^ ((key0 & 3) << 2);
  const uint32_t k_at0 = hv * d + 8 * ck0, k_at1 = hv * d + 8 * ck1, v_at = hv * dv + min(8 * cv, dv - 8);
  // a tile's slots of this thread's rows, read together ahead of their use: a read in front of each request waited for all LDS reads before it
  struct Slots {
    int of[NP];
  };
  auto slots_of = [&](int buf) __attribute__((always_inline)) {
    Slots x;
#pragma unroll
    for (int u = 0; u < NP; ++u) x.of[u] = s_slot[buf][key0 + u * ROWS];
    return x;
  };
  auto row_at = [&](const bf16_t* cache, int slot, uint32_t ld_row) __attribute__((always_inline)) {
    if (PCS >= 64) slot = __builtin_amdgcn_readfirstlane(slot);  // a wave's pieces are one row's
    return cache + (uint64_t)(uint32_t)slot * ld_row;
  };
  auto request_k = [&](uint16_t* img, const Slots& slots, int u) __attribute__((always_inline)) {
    if (u < NP && (FULL || 8 * (u & 1 ? ck1 : ck0) < d))
      __builtin_amdgcn_global_load_lds((glb_void_t*)(row_at(k_cache, slots.of[u < NP ? u : 0], nk) + (u & 1 ? k_at1 : k_at0)),
                                       (lds_void_t*)(img + (u * NT + wave * 64) * 8), 16, 0, 0);
    __builtin_amdgcn_sched_barrier(kAllButLoads);
  };
  auto request_v = [&](uint16_t* img, const Slots& slots, int u) __attribute__((always_inline)) {
    if (u < NP)
      __builtin_amdgcn_global_load_lds((glb_void_t*)(row_at(v_cache, slots.of[u < NP ? u : 0], nv) + v_at),
                                       (lds_void_t*)(img + (u * NT + wave * 64) * 8), 16, 0, 0);
    __builtin_amdgcn_sched_barrier(kAllButLoads);
  };
  // this wave's pieces are there; values of rows past the last key become zeros: a row that sees an infinite last one would add zero times infinity
  auto arrived = [&](uint16_t* img, int j0) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (j0 < k_end && j0 + kWinTile > k_end) {
      for (int key = key0; key < kWinTile; key += ROWS)
        if (j0 + key >= k_end) *reinterpret_cast<Q4*>(img + (key * PCS + (int)threadIdx.x % PCS) * 8) = Q4{0u, 0u, 0u, 0u};
    }
  };
  // Zeros past the heads of keys, where no DMA goes.  (Past the values' heads lies their last piece again: those columns of O are not stored.)
  if (!FULL) {
#pragma unroll
    for (int u = 0; u < NP; ++u) {
      const int at = (u * NT + (int)threadIdx.x) * 8;
      if (8 * (u & 1 ? ck1 : ck0) >= d) *reinterpret_cast<Q4*>(sk + at) = *reinterpret_cast<Q4*>(sv1 + at) = Q4{0u, 0u, 0u, 0u};
    }
  }
  // mixed scores of an image's tile
  f32x4_t mx[KSW][4];
  auto scores = [&](const uint16_t* img) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < KSW; ++u) {
      const int ks = ks0 + u;
      f32x4_t sc[NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        sc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        const uint16_t* at = img + (ks * 16 + lr) * RS + 4 * j / rep * KC * 32;
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) sc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qf[j][kc], *reinterpret_cast<const bf16x8_t*>(at + ((4 * kc + lg) ^ lr) * 8), sc[j], 0, 0, 0);
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) mx[u][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int c = 0; c < 4; ++c) mx[u][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(sc[j][c], tk[j], mx[u][c], 0, 0, 0);
    }
  };
  auto put_scores = [&]() __attribute__((always_inline)) {
    if (NH == 16 || lr < NH) {
#pragma unroll
      for (int u = 0; u < KSW; ++u)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          *reinterpret_cast<f32x4_t*>(mixed + lr * kWinHead + (4 * quad + c) * kWinRow + (ks0 + u) * 16 + 4 * lg) = mx[u][c];
    }
  };
  put_slot(slot0, 0);
  put_slot(slot1, 1);
  put_slot(slot2, 2);
  __syncthreads();
  Slots slots_v = slots_of(0), slots_k = slots_of(1);
#pragma unroll
  for (int u = 0; u < NP; ++u) request_k(sv1, slots_v, u);  // the first tile's keys in the second one's values' place
#pragma unroll
  for (int u = 0; u < NP; ++u) request_k(sk, slots_k, u);
#pragma unroll
  for (int u = 0; u < NP; ++u) request_v(sv0, slots_v, u);
  arrived(sv0, k_begin);
  if (!FULL) {  // zeros past the head
#pragma unroll
    for (int kc = 0; kc < KC; ++kc)
      if (kc * 32 + lg * 8 >= d) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) qf[j][kc] = bf16x8_t{};
      }
  }
  __syncthreads();
  scores(sv1);
  put_scores();
  __syncthreads();
  // tile t: the next one's keys are there, its values and the keys of the one after it are asked for
  auto tile = [&](uint16_t* cur, uint16_t* next, int t) __attribute__((always_inline)) {
    const int j0 = k_begin + t * TW, nj = j0 + TW, buf = t & 3;
    f32x4_t s[4];  // keys 8 g + 4 hi + c
#pragma unroll
    for (int g = 0; g < 4; ++g) s[g] = *reinterpret_cast<const f32x4_t*>(mixed + (h0 + (lane >> 4 & 1)) * kWinHead + lr * kWinRow + 8 * g + 4 * hi);
    slots_v = slots_of((buf + 1) & 3);
    slots_k = slots_of((buf + 2) & 3);
    put_slot(next_slot, (buf + 3) & 3);
    scores(sk);  // of tile t + 1
    __syncthreads();
    put_scores();
    // The next tile's values and the keys of the one after it (past the range: its last row), a few at a time: a wave waits where it asks for more
    // than the address unit takes
    auto request_keys = [&](int u0) __attribute__((always_inline)) {
#pragma unroll
      for (int u = u0; u < u0 + 2; ++u) request_k(sk, slots_k, u);
    };
    request_keys(0);
    if (wave == 0) next_slot = slot_at(j0 + 4 * TW);
    const bool whole = nj <= k_end && nj - 1 <= all_hi && j0 >= all_lo;
    if (!whole) {
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int j = j0 + 8 * g + 4 * hi + c;
          s[g][c] = ((j <= limit) & (j >= lo_row) & (j < k_end)) ? s[g][c] : -INFINITY;
        }
    }
    float tmax = -INFINITY;
#pragma unroll
    for (int g = 0; g < 4; ++g) tmax = fmaxf(tmax, fmaxf(fmaxf(s[g][0], s[g][1]), fmaxf(s[g][2], s[g][3])));
    tmax = pair_max(tmax);
    request_keys(2);
    // The reference maximum may lag by 2^8: the weights' three parts have their 24 bits wherever these lie (rescaling O at every new maximum was
    // a quarter of the vector work).  A row's moves for its own scores only: its bits do not depend on the wave's other rows.
    if (__builtin_amdgcn_ballot_w64(tmax > m + 8.f) != 0) {
      const float m_new = tmax > m + 8.f ? tmax : m;
      const float alpha = m_new == m ? 1.f : __builtin_amdgcn_exp2f(m - m_new);
#pragma unroll
      for (int nb = 0; nb < VC / 2; ++nb)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[nb][e] *= alpha;
      lsum *= alpha;
      m = m_new;
    }
    const float ref = m == -INFINITY ? 0.f : m;  // no visible key yet: every weight below is exp2(-inf) = 0
    uint32_t part[3][8];                          // a weight's three bf16 parts, the largest first
    float psum = 0.f;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float p[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        p[c] = __builtin_amdgcn_exp2f(s[g][c] - ref);
        psum += p[c];
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const uint32_t x = part[i][2 * g] = pack_bf16(p[0], p[1]), y = part[i][2 * g + 1] = pack_bf16(p[2], p[3]);
        p[0] -= __uint_as_float(x << 16);
        p[1] -= __uint_as_float(x & 0xffff0000u);
        p[2] -= __uint_as_float(y << 16);
        p[3] -= __uint_as_float(y & 0xffff0000u);
      }
    }
    lsum += psum;
    // transposing read: a 16-lane group reads 4 keys x 16 columns and hands lane j its column's four keys
    const uint16_t* vbase = cur + (4 * hi + (lr >> 2)) * RS + grp * VC * 16 + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    auto vfrag = [&](int i) {  // 32 columns i % 4, 16 keys i / 4
      const uint16_t* at = vbase + (i >> 2) * 16 * RS + ((i ^ (lr >> 2)) & 3) * 32;
      const s16x4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)at);
      const s16x4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(at + 8 * RS));
      return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    // two fragments' products at a time, on accumulators in turn; the next two are read meanwhile
    bf16x8_t vf[2][2];
    vf[0][0] = vfrag(0);
    vf[0][1] = vfrag(1);
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      if (i + 2 < 8) {
        vf[(i >> 1 & 1) ^ 1][0] = vfrag(i + 2);
        vf[(i >> 1 & 1) ^ 1][1] = vfrag(i + 3);
      }
      request_v(next, slots_v, i >> 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 2; x >= 0; --x)
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          const uint32_t* w = part[x] + (i >> 2) * 4;
          o[(i + n) & 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i >> 1 & 1][n], __builtin_bit_cast(bf16x8_t, Q4{w[0], w[1], w[2], w[3]}), o[(i + n) & 3], 0, 0, 0);
        }
    }
    arrived(next, nj);
    __syncthreads();
  };
  const int n_tiles = k_begin < k_end ? (k_end - k_begin + TW - 1) / TW : 0;
  for (int t = 0; t < n_tiles; t += 2) {
    tile(sv0, sv1, t);
    if (t + 1 < n_tiles) tile(sv1, sv0, t + 1);
  }
  const float l = lsum + __shfl_xor(lsum, 32, 64);
  const int h = h0 + (lane >> 4 & 1);
  // this lane's columns: 32 nb + 8 g + 4 hi ...
  if (splits == 1) {
    const float gz = ld(src + tok * (size_t)ld_src + g_off + h);
    const float f = 1.0f / (l * (1.0f + __expf(-gz)));
    // 64 columns at a time through LDS, so that a row's leave as one cache line (lanes' own 8 bytes of 32 rows: 4.4 us a workgroup instead of 1.7)
    char* turn = reinterpret_cast<char*>(mixed) + wave * 4096;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const int nb = 2 * half + (c >> 2), g = c & 3;
        *reinterpret_cast<uint2*>(turn + (lane & 31) * 128 + ((c ^ (lane & 7)) << 4) + 8 * hi) =
            uint2{pack_bf16(o[nb][4 * g] * f, o[nb][4 * g + 1] * f), pack_bf16(o[nb][4 * g + 2] * f, o[nb][4 * g + 3] * f)};
      }
      asm volatile("" ::: "memory");  // a wave's LDS accesses go in order; this keeps the compiler's
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 8 * i + (lane >> 3), query = tok0 + (row & 15), col = 64 * half + 8 * (lane & 7);
        const Q4 x = *reinterpret_cast<const Q4*>(turn + row * 128 + (((lane ^ row) & 7) << 4));
        if (query < q_len && col < dv)  // past the L2 (4 portions of 1500 - 2548 tokens, 16 heads: 205.5 -> 203.8 us)
          __builtin_nontemporal_store(__builtin_bit_cast(f32x4_t, x), reinterpret_cast<f32x4_t*>(out + ((size_t)(cu_q[b] + query) * NH + h0 + (row >> 4)) * dv + col));
      }
      asm volatile("" ::: "memory");
    }
  } else if (valid) {
    const size_t row = ((size_t)blockIdx.y * total_q + tok) * NH + h;
#pragma unroll
    for (int nb = 0; nb < VC / 2; ++nb)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int e = 32 * nb + 8 * g + 4 * hi;
        if (e < dv) *reinterpret_cast<f32x4_t*>(part_o + row * dv + e) = f32x4_t{o[nb][4 * g], o[nb][4 * g + 1], o[nb][4 * g + 2], o[nb][4 * g + 3]};
      }
    if (hi == 0) {
      part_ml[row * 2] = m * 0.6931471805599453f;  // the maxima leave in natural units
      part_ml[row * 2 + 1] = l;
    }
  }
}

}  // namespace

// heads of 8 | 16 so that a wave's heads share a value head; rows that 16-byte loads and 8-byte stores may walk
extern "C" int msgl_mix_window_attn_on_matrix_cores(int H, int G, int d, int dv, int dtype) {
  return dtype == MSGL_MIX_BF16 && (H == 8 || H == 16) && G >= 1 && G <= H / 4 && (H / 2) % G == 0 && d >= 1 && d <= 128 && dv >= 1 && dv <= 128 &&
         d % 8 == 0 && dv % 8 == 0;
}

// 1: launched; 0: these sizes are not this kernel's (the caller takes the other one); < 0: an error code.
extern "C" __attribute__((visibility("hidden"))) int mix_window_attn_mfma(
    void* out, float* part_o, float* part_ml, const void* src, int64_t ld_src, int g_off, const void* k_cache, const void* v_cache, const int* table,
    int64_t table_stride, const int* req_rows, const int* seq_lens, const int* cu_q, int batch, int total_q, int H, int G, int d, int dv, int window,
    float scale, const float* talk, int splits, hipStream_t s) {
  const auto al = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if (!msgl_mix_window_attn_on_matrix_cores(H, G, d, dv, MSGL_MIX_BF16)) return 0;
  if (!al(k_cache) || !al(v_cache) || !al(out) || (part_o && !al(part_o))) return 0;
  const dim3 grid(total_q / 16 + batch, splits);
#define WIN_KERNEL(NH, G) (d == 128 ? window_attn_mfma_kernel<NH, G, true> : window_attn_mfma_kernel<NH, G, false>)
  const auto kernel = H == 16 ? (G == 4 ? WIN_KERNEL(16, 4) : G == 2 ? WIN_KERNEL(16, 2) : WIN_KERNEL(16, 1)) : G == 2 ? WIN_KERNEL(8, 2) : WIN_KERNEL(8, 1);
#undef WIN_KERNEL
  hipLaunchKernelGGL(kernel, grid, dim3(H * 32), 0, s, mp<bf16_t>(out), part_o, part_ml, cp<bf16_t>(src), ld_src, g_off, cp<bf16_t>(k_cache),
                     cp<bf16_t>(v_cache), table, table_stride, req_rows, seq_lens, cu_q, batch, total_q, d, dv, window, scale, talk, splits);
  MIX_LAUNCHED("window_attn");
  return 1;
}
