// Sliding-window attention with mixed heads on the matrix cores (bf16 caches): the form of window_attn_kernel (mix_delta.hip) for
// portions of query tokens.  Same C entry, msgl_mix_window_attn; this file holds one kernel and the function that launches it.
//
// What bounds it: per visible (query, key) pair and H heads the two products are 2 H (d + 2 dv) flops for the bf16 matrix cores, the
// mixing of the scores 2 H^2 flops in fp32 and the softmax about fifteen vector operations per head; at H = 16, d = dv = 128 each of the
// three takes about the same time, so they have to run beside each other.  The mixing is itself a product, table x scores with the heads
// as contraction: it goes to the fp32 matrix instructions (on vector FMAs it was 256 of them a pair, and every wave read every head's
// scores back from LDS).
//
// 4 requests of 1500 - 2548 new tokens, 16 heads of 128 over 4 key heads, window 2048: 5182 us on the vector units, 453 us with both
// products on the matrix cores and the mixing on vector FMAs in step with them, 294 us with all three as below, 257 us with the rows' addresses
// known once instead of a division and four products per piece and tile, loads without conditions, the table entries a tile ahead and the raw
// scores' writes over all banks (3 requests of 700 - 1700 tokens after 333, 8 heads, window 512: 63 -> 49; 20 decoded tokens 35 -> 33).  The
// softmax and the LDS round trip of the scores are what is left, a wave's vector and matrix work one after the other; 20 us are the
// weights' third part.  Sixteen waves of one head each need 23 registers more than they have.
//
// Precision: scores are bf16 x bf16 products with fp32 sums, mixed and exponentiated in fp32; a probability enters the second product
// as the sum of three bf16 numbers (its rounding, that of what is left, and the rest: 8 bits each), which is the fp32 number itself.
#include "mix_common.h"

namespace {

constexpr int kWinTile = 32;           // keys per tile
constexpr int kWinKC = 4, kWinVC = 8;  // head sizes up to 128
constexpr int kWinRow = 36;            // floats of a mixed (head, query) row in LDS: 32 keys, padded so that 16 rows cover all banks
template <int NH>
constexpr int kWinRaw = kWinTile * NH + 4;  // floats of a query's raw scores in LDS: [32 keys][NH], padded the same way

// Workgroup = 16 query tokens of one request x all NH heads (x one of `splits` key ranges), NH / 2 waves of two heads each, which share
// a key / value head.  Two phases per tile of 32 keys, a barrier behind each:
//   C(t)  the waves share the tile's keys: mixed scores = talk x raw, a product over the heads per key; the next tile's K rows and this
//         tile's V rows, requested a phase before, go to LDS
//   D(t)  the waves share the heads: S^T = K Q^T of tile t + 1 (Q held in registers) -> raw scores to LDS, which the vector work of
//         tile t covers: mask, online softmax, O^T += V^T P^T (a lane reads four consecutive keys of its query, the layout the product
//         takes; V through transposing LDS reads)
template <int NH>
__global__ __launch_bounds__(NH * 32, 2) void window_attn_mfma_kernel(bf16_t* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml,
                                                                  const bf16_t* __restrict__ src, int64_t ld_src, int g_off,
                                                                  const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
                                                                  const int* __restrict__ table, int64_t table_stride,
                                                                  const int* __restrict__ req_rows, const int* __restrict__ seq_lens,
                                                                  const int* __restrict__ cu_q, int B, int total_q, int G, int d, int dv,
                                                                  int window, float scale, const float* __restrict__ talk, int splits, int qvec) {
  constexpr int HPW = 2, NT = NH * 32, NW = NH / 2, KC = kWinKC, VC = kWinVC, KS = kWinTile / 16, GS = NH / 4, RAW = kWinRaw<NH>;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int VS = G * VC * 16 + 8, KSR = G * KC * 32 + 8;
  float* raw = smem;                                                      // [16 queries][32 keys][NH]
  float* mixed = raw + 16 * RAW;                                          // [NH][16 queries][kWinRow]
  uint16_t* sv = reinterpret_cast<uint16_t*>(mixed + NH * 16 * kWinRow);  // [32][VS]
  uint16_t* sk = sv + kWinTile * VS;                                      // [32][KSR]
  __shared__ int s_slot[4][kWinTile];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lr = lane & 15, lg = lane >> 4;
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
  const int h0 = wave * HPW, rep = NH / G, grp = h0 / rep;
  const float scale2 = scale * 1.4426950408889634f;
  // A wave's raw scores go to LDS two heads a key, 16 keys apart for lane groups that are written together: with 16 heads, the pairs of four
  // heads change places in every other four keys, which all are one wave's in phase C, and the writes cover all banks.
  auto swap_of = [](int four_keys) { return NH == 16 ? 2 * (four_keys & 1) : 0; };
  // the table as first operand: row = head, contraction index 4 steps (NH = 16) of g = GS lg + step, which is what a lane reads at once
  float tk[GS];
#pragma unroll
  for (int u = 0; u < GS; ++u) tk[u] = lr < NH ? talk[lr * NH + GS * lg + (u ^ (swap_of(wave)))] * scale2 : 0.f;
  bf16x8_t qf[HPW][KC];
  f32x4_t o[HPW][VC];
  float m[HPW], lsum[HPW];
#pragma unroll
  for (int hh = 0; hh < HPW; ++hh) {
    const bf16_t* qrow = src + tok * (size_t)ld_src + (size_t)(h0 + hh) * d;
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) {
      const int k = kc * 32 + lg * 8;
      Q4 f{0u, 0u, 0u, 0u};
      if (valid && k < d) f = load8(qrow + k, d - k, qvec != 0);
      qf[hh][kc] = __builtin_bit_cast(bf16x8_t, f);
    }
#pragma unroll
    for (int vt = 0; vt < VC; ++vt) o[hh][vt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    m[hh] = -INFINITY;
    lsum[hh] = 0.f;
  }
  const int* trow = table + (size_t)req_rows[b] * table_stride;
  const uint32_t nk = (uint32_t)(G * d), nv = (uint32_t)(G * dv);
  // 16-byte pieces of a tile's key and value rows (both 128 wide per head in LDS, zeros past the head); at most NH / 4 key heads.  A row's
  // pieces divide the workgroup (both are powers of two), so a thread has one column of the rows key0, key0 + rows, ...: its offsets are
  // known once (a division and four 32-bit products a piece and tile, at a quarter of the rate, were a tenth of the kernel).
  static_assert(KC * 4 == VC * 2, "keys and values share the piece map");
  const int chunks = G * VC * 2, rows = NT / chunks, key0 = (int)threadIdx.x / chunks, col = ((int)threadIdx.x - key0 * chunks) * 8;
  const int hv = col / (VC * 16), in_head = col - hv * (VC * 16);
  const bool has_k = in_head < d, has_v = in_head < dv;
  const bf16_t *k_at = k_cache + (size_t)hv * d + (has_k ? in_head : 0), *v_at = v_cache + (size_t)hv * dv + (has_v ? in_head : 0);
  constexpr int NP = kWinTile * (NH / 4) * VC * 2 / NT;  // pieces per thread; with fewer key heads rows come more than once
  typedef uint32_t Piece __attribute__((ext_vector_type(4)));  // (as a struct the registers became memory)
  Piece pre_k[NP], pre_v[NP];
  // the rows of a tile (its slots in s_slot[buf]) into registers, and from there to LDS; a tile's rows past the last key are that key's again
  // (their values become zeros in LDS).
  // No condition on a load or a store (columns past the head go to the row's padding): where one was skipped, the loaded registers were
  // copied, and the wave waited for the loads at once (464 - 533 us).
  const int to_k = has_k ? col : G * KC * 32, to_v = has_v ? col : G * VC * 16;
  auto key_of = [&](int u) { return (key0 + u * rows) & (kWinTile - 1); };
  auto request = [&](Piece (&pre)[NP], const bf16_t* at, uint32_t ld_row, int buf) {
#pragma unroll
    for (int u = 0; u < NP; ++u) pre[u] = *reinterpret_cast<const Piece*>(at + (uint64_t)(uint32_t)s_slot[buf][key_of(u)] * ld_row);
  };
  auto stage = [&](const Piece (&pre)[NP], uint16_t* dst, int ld_row) {
#pragma unroll
    for (int u = 0; u < NP; ++u) *reinterpret_cast<Piece*>(dst + key_of(u) * ld_row) = pre[u];
  };
  const int last_key = max(k_end - 1, 0);
  const int in_tile = (int)threadIdx.x & (kWinTile - 1);
  auto slot_at = [&](int j0) { return trow[min(j0 + in_tile, last_key)]; };
  auto put_slot = [&](int slot, int buf) {
    if (threadIdx.x < kWinTile) s_slot[buf][threadIdx.x] = slot;
  };
  if (!has_k || !has_v) {
    for (int key = key0; key < kWinTile; key += rows) {
      if (!has_k) *reinterpret_cast<Q4*>(sk + key * KSR + col) = Q4{0u, 0u, 0u, 0u};
      if (!has_v) *reinterpret_cast<Q4*>(sv + key * VS + col) = Q4{0u, 0u, 0u, 0u};
    }
  }
  f32x4_t sc[HPW][KS];
  auto scores = [&]() {  // raw scores of the tile in sk
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
      for (int hh = 0; hh < HPW; ++hh) sc[hh][ks] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        const bf16x8_t kf = *reinterpret_cast<const bf16x8_t*>(&sk[(ks * 16 + lr) * KSR + grp * KC * 32 + kc * 32 + lg * 8]);
#pragma unroll
        for (int hh = 0; hh < HPW; ++hh) sc[hh][ks] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[hh][kc], sc[hh][ks], 0, 0, 0);
      }
    }
  };
  auto store_raw = [&]() {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        *reinterpret_cast<float2*>(raw + lr * RAW + (ks * 16 + 4 * lg + c) * NH + (h0 ^ swap_of(lg))) = float2{sc[0][ks][c], sc[1][ks][c]};
  };
  constexpr int TW = kWinTile;
  int next_slot = slot_at(k_begin + 3 * TW);  // asked for a tile before it goes to LDS: there the whole workgroup waited for the table
  put_slot(slot_at(k_begin), 0);
  put_slot(slot_at(k_begin + TW), 1);
  put_slot(slot_at(k_begin + 2 * TW), 2);
  __syncthreads();
  request(pre_k, k_at, nk, 0);
  stage(pre_k, sk + to_k, KSR);
  request(pre_v, v_at, nv, 0);
  request(pre_k, k_at, nk, 1);
  __syncthreads();
  scores();
  store_raw();
  __syncthreads();
  int buf = 0;
  for (int j0 = k_begin; j0 < k_end; j0 += TW, buf = (buf + 1) & 3) {
    const int nj = j0 + TW;
    // ---- C(t)
    {
      constexpr int KPW = kWinTile / NW;  // keys of this wave
#pragma unroll
      for (int k0 = 0; k0 < KPW; k0 += 4) {
        f32x4_t mx[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float* x = raw + lr * RAW + (wave * KPW + k0 + i) * NH + GS * lg;
          mx[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int u = 0; u < GS; ++u) mx[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(tk[u], x[u], mx[i], 0, 0, 0);
        }
        if (4 * lg < NH) {
#pragma unroll
          for (int c = 0; c < 4; ++c)
            *reinterpret_cast<f32x4_t*>(mixed + ((4 * lg + c) * 16 + lr) * kWinRow + wave * KPW + k0) = f32x4_t{mx[0][c], mx[1][c], mx[2][c], mx[3][c]};
        }
      }
    }
    stage(pre_v, sv + to_v, VS);
    if (nj > k_end) {  // values past the last key: a row that sees an infinite last one would add zero times infinity
      for (int key = key0; key < kWinTile; key += rows)
        if (j0 + key >= k_end) *reinterpret_cast<Piece*>(sv + to_v + key * VS) = Piece{0u, 0u, 0u, 0u};
    }
    stage(pre_k, sk + to_k, KSR);
    put_slot(next_slot, (buf + 3) & 3);
    __syncthreads();
    // ---- D(t)
    request(pre_v, v_at, nv, (buf + 1) & 3);
    request(pre_k, k_at, nk, (buf + 2) & 3);
    if (wave == 0) next_slot = slot_at(j0 + 4 * TW);
    __builtin_amdgcn_sched_barrier(0);  // every load ahead of the products
    scores();  // of tile t + 1
    f32x4_t s[HPW][KS];
#pragma unroll
    for (int hh = 0; hh < HPW; ++hh)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s[hh][ks] = *reinterpret_cast<const f32x4_t*>(mixed + ((h0 + hh) * 16 + lr) * kWinRow + ks * 16 + 4 * lg);
    const bool whole = nj <= k_end && nj - 1 <= all_hi && j0 >= all_lo;
    uint2 part[3][HPW][KS];  // a weight's three bf16 parts, the largest first
#pragma unroll
    for (int hh = 0; hh < HPW; ++hh) {
      float tmax = -INFINITY;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (!whole) {
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const int j = j0 + ks * 16 + 4 * lg + c;
            if (!(j <= limit && j >= lo_row && j < k_end)) s[hh][ks][c] = -INFINITY;
          }
        }
        tmax = fmaxf(tmax, fmaxf(fmaxf(s[hh][ks][0], s[hh][ks][1]), fmaxf(s[hh][ks][2], s[hh][ks][3])));
      }
      tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
      tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
      const float m_new = fmaxf(m[hh], tmax);
      const float base = m_new == -INFINITY ? 0.f : m_new;  // no visible key yet: every weight below is exp2(-inf) = 0
      const float alpha = __builtin_amdgcn_exp2f(m[hh] - base);
      float psum = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        float p[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          p[c] = __builtin_amdgcn_exp2f(s[hh][ks][c] - base);
          psum += p[c];
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const uint2 x = part[i][hh][ks] = uint2{pack_bf16(p[0], p[1]), pack_bf16(p[2], p[3])};
          p[0] -= __uint_as_float(x.x << 16);
          p[1] -= __uint_as_float(x.x & 0xffff0000u);
          p[2] -= __uint_as_float(x.y << 16);
          p[3] -= __uint_as_float(x.y & 0xffff0000u);
        }
      }
      lsum[hh] = fmaf(lsum[hh], alpha, psum);
      if (__builtin_amdgcn_ballot_w64(m_new > m[hh]) != 0) {
#pragma unroll
        for (int vt = 0; vt < VC; ++vt)
#pragma unroll
          for (int c = 0; c < 4; ++c) o[hh][vt][c] *= alpha;
      }
      m[hh] = m_new;
    }
    store_raw();
    const uint16_t* vbase = &sv[(4 * lg + (lr >> 2)) * VS + grp * VC * 16 + 4 * (lr & 3)];
#pragma unroll
    for (int kp = 0; kp < KS / 2; ++kp) {
      if (j0 + kp * 32 >= k_end) break;
#pragma unroll
      for (int vt = 0; vt < VC; ++vt) {
        const s16x4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(vbase + kp * 32 * VS + vt * 16));
        const s16x4_t v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(vbase + (kp * 32 + 16) * VS + vt * 16));
        const bf16x8_t vf = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
        for (int hh = 0; hh < HPW; ++hh) {
#pragma unroll
          for (int i = 2; i >= 0; --i) {
            const uint2 a = part[i][hh][2 * kp], b = part[i][hh][2 * kp + 1];
            o[hh][vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, __builtin_bit_cast(bf16x8_t, Q4{a.x, a.y, b.x, b.y}), o[hh][vt], 0, 0, 0);
          }
        }
      }
    }
    __syncthreads();
  }
  if (!valid) return;
#pragma unroll
  for (int hh = 0; hh < HPW; ++hh) {
    float l = lsum[hh];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    const int h = h0 + hh;
    if (splits == 1) {
      const float gz = ld(src + tok * (size_t)ld_src + g_off + h);
      const float f = 1.0f / (l * (1.0f + __expf(-gz)));
#pragma unroll
      for (int vt = 0; vt < VC; ++vt) {
        const int e = vt * 16 + 4 * lg;
        if (e < dv)
          *reinterpret_cast<uint2*>(out + tok * (size_t)(NH * dv) + (size_t)h * dv + e) =
              uint2{pack_bf16(o[hh][vt][0] * f, o[hh][vt][1] * f), pack_bf16(o[hh][vt][2] * f, o[hh][vt][3] * f)};
      }
    } else {
      const size_t row = ((size_t)blockIdx.y * total_q + tok) * NH + h;
#pragma unroll
      for (int vt = 0; vt < VC; ++vt) {
        const int e = vt * 16 + 4 * lg;
        if (e < dv) *reinterpret_cast<f32x4_t*>(part_o + row * dv + e) = o[hh][vt];
      }
      if (lg == 0) {
        part_ml[row * 2] = m[hh] * 0.6931471805599453f;  // the maxima leave in natural units
        part_ml[row * 2 + 1] = l;
      }
    }
  }
}

template <int NH>
size_t window_lds(int G) {
  return (size_t)(NH * 16 * kWinRow + 16 * kWinRaw<NH>) * sizeof(float) + (size_t)kWinTile * (G * (kWinVC * 16 + kWinKC * 32) + 16) * sizeof(uint16_t);
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
  const int qvec = al(src) && ld_src % 8 == 0;
  const dim3 grid(total_q / 16 + batch, splits);
#define WIN_LAUNCH(NH)                                                                                                                        \
  {                                                                                                                                           \
    const size_t lds = window_lds<NH>(G);                                                                                                     \
    MIX_REQUIRE(ensure_lds((const void*)window_attn_mfma_kernel<NH>, lds) == 0, "window_attn: %zu bytes of LDS", lds);                        \
    hipLaunchKernelGGL((window_attn_mfma_kernel<NH>), grid, dim3(NH * 32), lds, s, mp<bf16_t>(out), part_o, part_ml, cp<bf16_t>(src), ld_src,     \
                       g_off, cp<bf16_t>(k_cache), cp<bf16_t>(v_cache), table, table_stride, req_rows, seq_lens, cu_q, batch, total_q, G, d,  \
                       dv, window, scale, talk, splits, qvec);                                                                                \
  }
  if (H == 16) WIN_LAUNCH(16) else WIN_LAUNCH(8)
#undef WIN_LAUNCH
  MIX_LAUNCHED("window_attn");
  return 1;
}
