// The difference of two softmax maps over the values of a whole head (keys 64 wide per map, values 128), bf16 caches, portions of prompts.
// mix_scan.hip keeps the kernels for decoded tokens, other widths and fp32 caches; same C entry, same partial results of key ranges.
#include "mix_common.h"

namespace {

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(1))) void glb_void_t;
typedef __attribute__((address_space(3))) void lds_void_t;

// What bounds it: a 32 x 32 block of a wave is 24 MFMAs of 32 cycles (scores of both maps, then their weights times the same values) and 32
// scores per lane to turn into weights, about 28 cycles each with the exponential's 16, on the vector units: both kinds of work must run
// beside each other.  Hence 32-row waves (a fragment of keys or values serves 32 rows: 64 KB of LDS reads in 768 cycles a CU, half of what
// LDS gives), two workgroups of 128 rows per CU, 64-key tiles by DMA into two LDS images, one barrier a tile.
//   S^T[32 keys x 32 rows] = K Q^T, O^T[32 columns x 32 rows] += V^T P^T: a lane has 16 scores of one row, which are the second product's
//   operand; V^T by transposing LDS reads.  A row's 16-byte pieces change places by its number when they are fetched: no bank twice.
// 4 portions of 1500 - 2548 tokens, 16 heads on 4: 325 us (16-row waves, tiles through registers) -> 183 us -> 151 us (order of the
// workgroups), of which about 30 us are the outputs' rescaling when a maximum moves.
// RANGES: several key ranges per group, partial results
template <bool RANGES>
__global__ __launch_bounds__(256, 2) void maps_prompt_kernel(bf16_t* __restrict__ out, int64_t ld_out, float* __restrict__ part_o,
                                                             float* __restrict__ part_ml, const float* __restrict__ q,
                                                             const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
                                                             const int* __restrict__ table, int64_t table_stride,
                                                             const int* __restrict__ req_rows, const int* __restrict__ seq_lens,
                                                             const int* __restrict__ cu_q, int B, int total_q, int H, int G, float scale, int window,
                                                             int keep, const float* __restrict__ lam, const bf16_t* __restrict__ gate,
                                                             int64_t ld_gate, float post, float eps, int hb_log2, int splits) {
  constexpr int D = 64, DV = 128, KT = 64, PART = KT * 256;  // PART: bytes of a tile's keys, and of its values
  __shared__ __attribute__((aligned(1024))) char img0[2 * PART], img1[2 * PART];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), hi = lane >> 5;
  const int HB = 1 << hb_log2, QT = 128 >> hb_log2;
  int tok0 = 0;
  // The longest groups first, all of a group's heads before the next group: what starts last is short.  (A head's groups after another's: the
  // last head's longest groups start when half the work is done, and end long after the rest.  182 -> 151 us; window 1024,
  // 8 heads on 4: 84 -> 78; 3 portions of 1500, 16 heads on 4: 100 -> 83.  Of 408 sizes of 1 - 8 portions, 8 and 16 heads on 2 and 4, 65 to 1000
  // workgroups, 5 % faster on average; eight are 4 - 13 % slower, of 513 - 780 workgroups behind long prefixes, mostly with two heads' groups to an
  // index: 5 of 850 after 650, 16 on 2: 109 -> 126.)  With key ranges, a few tens of groups and no rest to wait for, it is the other way round: 1
  // portion of 300 after 2000, 8 heads on 4: 39.1 us, a group's heads together 42.3; 2 of 300 after 650 37.0 and 40.8.
  const int rep = H / G, hblocks = (rep + HB - 1) >> hb_log2, n_heads = G * hblocks, n_groups = (int)gridDim.x / n_heads;
  const int index = RANGES ? (int)blockIdx.x % n_groups : (int)blockIdx.x / n_heads;
  const int hy = RANGES ? (int)blockIdx.x / n_groups : (int)blockIdx.x - index * n_heads;
  const int b = find_group_by_keys(cu_q, seq_lens, B, QT, index, n_groups, &tok0);
  if (b < 0) return;
  const int kvh = hy / hblocks, h0 = kvh * rep + (hy - kvh * hblocks) * HB, h_end = (kvh + 1) * rep, z = blockIdx.z;
  const int first = cu_q[b], q_len = cu_q[b + 1] - first, start = seq_lens[b] - q_len;
  const int last_tok = min(tok0 + QT, q_len) - 1, n_keys = start + last_tok + 1;
  // the visible keys in a row: the kept ones in front of the window's first, then the window's
  const int lo_blk = window > 0 ? max(0, start + tok0 - window + 1) : 0;
  const int keep_eff = min(keep, lo_blk), shift = lo_blk - keep_eff, n_vis = n_keys - shift;
  const int per = max(((n_vis + splits - 1) / splits + KT - 1) / KT * KT, splits > 1 ? 256 : 0);  // short sequences leave the later ranges empty
  const int k_begin = z * per, k_end = min(n_vis, k_begin + per);
  auto key_at = [&](int v) { return v < keep_eff ? v : v + shift; };
  const int r_own = wave * 32 + (lane & 31);
  const int tl = tok0 + (r_own >> hb_log2), hh = h0 + (r_own & (HB - 1));
  const int limit = tl < q_len && hh < h_end ? start + tl : -1;
  if (RANGES && k_begin >= k_end) {  // no keys left for this range: its partial outputs are not read
    if (hi == 0 && limit >= 0) {
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const size_t row = (((size_t)z * total_q + first + tl) * H + hh) * 2 + a;
        part_ml[row * 2] = -INFINITY;
        part_ml[row * 2 + 1] = 0.f;
      }
    }
    return;
  }
  const int lo_row = window > 0 ? max(0, limit - window + 1) : 0;
  // this wave's rows: the first and the last token's position, the last one's first key
  const int w_min = start + tok0 + ((wave * 32) >> hb_log2), w_max = min(start + last_tok, w_min + ((31 + HB) >> hb_log2) - 1);
  const int w_lo = window > 0 ? max(0, w_max - window + 1) : 0;

  // ---- tiles: instruction i of this wave fills rows 16 i + 4 wave + lane / 16
  const int* trow = table + (size_t)req_rows[b] * table_stride;
  const int st_row = 4 * wave + (lane >> 4);
  const uint32_t row_bytes = (uint32_t)G * 256;
  const char* k_lane = reinterpret_cast<const char*>(k_cache) + (size_t)kvh * 256 + ((lane & 15) ^ st_row) * 16;
  const char* v_lane = reinterpret_cast<const char*>(v_cache) + (size_t)kvh * 256 + ((lane & 15) ^ ((st_row & 3) << 2)) * 16;
  int slot[4];
  auto load_slots = [&](int t) __attribute__((always_inline)) {  // past the range: some row of it, weight zero
#pragma unroll
    for (int i = 0; i < 4; ++i) slot[i] = trow[key_at(min(k_begin + t * KT + st_row + 16 * i, k_end - 1))];
  };
  auto dma = [&](char* img) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint64_t off = (uint64_t)(uint32_t)slot[i] * row_bytes;
      __builtin_amdgcn_global_load_lds((glb_void_t*)(k_lane + off), (lds_void_t*)(img + (4 * i + wave) * 1024), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((glb_void_t*)(v_lane + off), (lds_void_t*)(img + PART + (4 * i + wave) * 1024), 16, 0, 0);
    }
  };
  const int n_tiles = k_begin < k_end ? (k_end - k_begin + KT - 1) / KT : 0;
  if (n_tiles > 0) {
    load_slots(0);
    dma(img0);
    if (n_tiles > 1) load_slots(1);
  }

  // ---- queries: 32 lanes for a row's 512 bytes, then their fragments' order by way of the second image (free until the first tile's barrier)
  bf16x8_t qf[2][4];
  {
    char* turn = img1 + wave * 8192;
    const float scale2 = scale * 1.4426950408889634f;  // weights are exp2 of what the first product gives
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int rr = 2 * i + hi, r = wave * 32 + rr, t = tok0 + (r >> hb_log2), h = h0 + (r & (HB - 1));
      const bool ok = t < q_len && h < h_end;
      const float4 x = *reinterpret_cast<const float4*>(q + ((size_t)(first + (ok ? t : tok0)) * H + (ok ? h : h0)) * (2 * D) + 4 * (lane & 31));
      *reinterpret_cast<uint2*>(turn + rr * 256 + ((((lane & 31) >> 1) ^ (rr & 15)) << 4) + (lane & 1) * 8) =
          uint2{pack_bf16(x.x * scale2, x.y * scale2), pack_bf16(x.z * scale2, x.w * scale2)};
    }
    asm volatile("" ::: "memory");
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        qf[a][ks] = *reinterpret_cast<const bf16x8_t*>(turn + (lane & 31) * 256 + (((8 * a + 2 * ks + hi) ^ (lane & 15)) << 4));
  }
  f32x16_t o[2][4];
  float m[2], lsum[2];  // the row's reference maximum (log2), this lane's share of the row's sum
#pragma unroll
  for (int a = 0; a < 2; ++a) {
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[a][nb][e] = 0.f;
    m[a] = -INFINITY;
    lsum[a] = 0.f;
  }
  // map 0's fragments; map 1's are 128 bytes on, or back where the exchange of places turns that over (a sum, not ^ 128: through that the
  // compiler loses sight of the image and waits for the other one's DMA before each read)
  int k_off[4], v_off[4];
  const int flip = lane & 8 ? -128 : 128;
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) k_off[ks] = (lane & 31) * 256 + (((2 * ks + hi) ^ (lane & 15)) << 4);
#pragma unroll
  for (int nb = 0; nb < 4; ++nb)
    v_off[nb] = PART + hi * 1024 + ((lane & 15) >> 2) * 256 + ((nb ^ ((lane & 15) >> 2)) << 6) + (16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
  auto block = [&](const char* img, int j0, int kb) __attribute__((always_inline)) {  // 32 keys
    const int v0 = j0 + kb * 32;
    if (v0 >= k_end || key_at(v0) > w_max) return;
    f32x16_t s[2];
    uint32_t pw[2][8];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int e = 0; e < 16; ++e) s[a][e] = 0.f;
    constexpr int AHEAD = 2;  // fragments are read so many products (of values: pairs of products) before their use
    bf16x8_t kf[AHEAD + 1];
    auto kfrag = [&](int i) { return *reinterpret_cast<const bf16x8_t*>(img + kb * 8192 + k_off[i >> 1] + (i & 1) * flip); };
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) kf[i] = kfrag(i);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (i + AHEAD < 8) kf[(i + AHEAD) % (AHEAD + 1)] = kfrag(i + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
      s[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[i % (AHEAD + 1)], qf[i & 1][i >> 1], s[i & 1], 0, 0, 0);
    }
    bf16x8_t vf[AHEAD + 1];
    auto vfrag = [&](int i) {  // 32 columns i % 4, keys of step i / 4
      const char* p = img + v_off[i & 3] + (kb * 8 + (i >> 2) * 4) * 1024;
      const s16x4_t x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)p);
      const s16x4_t x1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(p + 2048));
      return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7));
    };
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) vf[i] = vfrag(i);  // on their way during the softmax
    __builtin_amdgcn_sched_barrier(0);
    const int last = key_at(v0 + 31);
    if (!(v0 + 32 <= k_end && last <= w_min && (key_at(v0) >= w_lo || last < keep))) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int v = v0 + (e & 3) + 8 * (e >> 2) + 4 * hi, j = key_at(v);
        const bool seen = (j <= limit) & ((j >= lo_row) | (j < keep)) & (v < k_end);
        s[0][e] = seen ? s[0][e] : -INFINITY;
        s[1][e] = seen ? s[1][e] : -INFINITY;
      }
    }
    float mx[2] = {-INFINITY, -INFINITY};
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      mx[0] = fmaxf(mx[0], s[0][e]);
      mx[1] = fmaxf(mx[1], s[1][e]);
    }
    mx[0] = pair_max(mx[0]);
    mx[1] = pair_max(mx[1]);
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      if (__builtin_amdgcn_ballot_w64(mx[a] > m[a]) != 0) {
        const float m_new = fmaxf(m[a], mx[a]);
        const float alpha = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m[a] - m_new);
#pragma unroll
        for (int nb = 0; nb < 4; ++nb)
#pragma unroll
          for (int e = 0; e < 16; ++e) o[a][nb][e] *= alpha;
        lsum[a] *= alpha;
        m[a] = m_new;
      }
    }
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const float ref = m[a] == -INFINITY ? 0.f : m[a];  // no key yet: every weight is exp2(-inf) = 0
      float sum = 0.f;  // of the fp32 weights
#pragma unroll
      for (int e = 0; e < 16; e += 2) {
        const float w0 = __builtin_amdgcn_exp2f(s[a][e] - ref), w1 = __builtin_amdgcn_exp2f(s[a][e + 1] - ref);
        sum += w0 + w1;
        pw[a][e >> 1] = pack_bf16(w0, w1);
      }
      lsum[a] += sum;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (i + AHEAD < 8) vf[(i + AHEAD) % (AHEAD + 1)] = vfrag(i + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const int w = (i >> 2) * 4;
        const Q4 p{pw[a][w], pw[a][w + 1], pw[a][w + 2], pw[a][w + 3]};
        o[a][i & 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i % (AHEAD + 1)], __builtin_bit_cast(bf16x8_t, p), o[a][i & 3], 0, 0, 0);
      }
    }
  };
  auto tile = [&](char* img, char* other, int t) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's pieces of tile t and the slots of tile t + 1
    __syncthreads();                                  // everybody's; everybody done with the other image
    if (t + 1 < n_tiles) {
      dma(other);
      if (t + 2 < n_tiles) load_slots(t + 2);
    }
    block(img, k_begin + t * KT, 0);
    block(img, k_begin + t * KT, 1);
  };
  for (int t = 0; t < n_tiles; t += 2) {
    tile(img0, img1, t);
    if (t + 1 < n_tiles) tile(img1, img0, t + 1);
  }
  __syncthreads();  // the images are free

  // ---- results: a lane has 64 columns of its row (32 nb + 8 g + 4 hi ...); through LDS to whole rows
  char* turn = (wave < 2 ? img0 : img1) + (wave & 1) * 16384;
  auto to_lds = [&](const f32x16_t* x) __attribute__((always_inline)) {
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<float4*>(turn + (lane & 31) * 512 + (((8 * nb + 2 * g + hi) ^ (lane & 31)) << 4)) =
            float4{x[nb][4 * g], x[nb][4 * g + 1], x[nb][4 * g + 2], x[nb][4 * g + 3]};
    asm volatile("" ::: "memory");
  };
  auto from_lds = [&](int rr, int chunk) { return *reinterpret_cast<const float4*>(turn + rr * 512 + ((chunk ^ rr) << 4)); };
  auto row_of = [&](int rr, size_t* tok, int* head) {  // row rr of this wave
    const int r = wave * 32 + rr, t = tok0 + (r >> hb_log2), h = h0 + (r & (HB - 1));
    *tok = (size_t)first + t;
    *head = h;
    return t < q_len && h < h_end;
  };
#pragma unroll
  for (int a = 0; a < 2; ++a) lsum[a] += __shfl_xor(lsum[a], 32, 64);
  if constexpr (!RANGES) {
    const float f0 = 1.0f / lsum[0], f1 = lam[0] / lsum[1];  // a row that is none has no sum and is not stored
    float ss = 0.f;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        o[0][nb][e] = o[0][nb][e] * f0 - o[1][nb][e] * f1;
        ss = fmaf(o[0][nb][e], o[0][nb][e], ss);
      }
    ss += __shfl_xor(ss, 32, 64);
    const float f = post / sqrtf(ss / (float)DV + eps);
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[0][nb][e] *= f;
    to_lds(o[0]);
#pragma unroll 2
    for (int i = 0; i < 8; ++i) {
      const int rr = 4 * i + (lane >> 4), c = 8 * (lane & 15);
      size_t tok;
      int head;
      if (!row_of(rr, &tok, &head)) continue;
      const float4 x = from_lds(rr, c / 4), y = from_lds(rr, c / 4 + 1);
      float v[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
      if (gate) {
        const Q4 gq = *reinterpret_cast<const Q4*>(gate + tok * ld_gate + (size_t)head * DV + c);
        const uint32_t gw[4] = {gq.x, gq.y, gq.z, gq.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] *= 1.0f / (1.0f + __expf(-__builtin_bit_cast(float, e & 1 ? gw[e >> 1] & 0xffff0000u : gw[e >> 1] << 16)));
      }
      // past the L2 (4 portions of 1500 - 2548 tokens, 16 heads on 4: 149.5 -> 146.5 us; the queries' loads too: 148.3)
      const Q4 packed{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7])};
      __builtin_nontemporal_store(__builtin_bit_cast(f32x4_t, packed), reinterpret_cast<f32x4_t*>(out + tok * ld_out + (size_t)head * DV + c));
    }
    return;
  }
#pragma unroll
  for (int a = 0; RANGES && a < 2; ++a) {
    to_lds(o[a]);
#pragma unroll 2
    for (int i = 0; i < 16; ++i) {
      const int rr = 2 * i + hi;
      size_t tok;
      int head;
      if (row_of(rr, &tok, &head))
        *reinterpret_cast<float4*>(part_o + ((((size_t)z * total_q + tok) * H + head) * 2 + a) * DV + 4 * (lane & 31)) = from_lds(rr, lane & 31);
    }
    asm volatile("" ::: "memory");
    if (hi == 0 && limit >= 0) {
      const size_t row = (((size_t)z * total_q + first + tl) * H + hh) * 2 + a;
      part_ml[row * 2] = m[a] * 0.6931471805599453f;  // in natural units
      part_ml[row * 2 + 1] = lsum[a];
    }
  }
}

}  // namespace

// 1: launched (with splits > 1 the caller joins the ranges); 0: not this kernel's sizes; < 0: an error code.
extern "C" __attribute__((visibility("hidden"))) int mix_maps_prompt(void* out, int64_t ld_out, float* part_o, float* part_ml, const float* q,
                                                                     const void* k_cache, const void* v_cache, const int* table, int64_t table_stride,
                                                                     const int* req_rows, const int* seq_lens, const int* cu_q, int batch, int total_q,
                                                                     int H, int G, int d, int dv, float scale, int window, int keep, const float* lam,
                                                                     const void* gate, int64_t ld_gate, float post, float eps, int splits,
                                                                     hipStream_t s) {
  const auto al = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if (d != 64 || dv != 128) return 0;
  // 16-byte loads, DMA pieces and stores
  if (!al(q) || !al(k_cache) || !al(v_cache) || !al(out) || ld_out % 8 || (gate && (!al(gate) || ld_gate % 8)) || (part_o && !al(part_o))) return 0;
  const int rep = H / G;
  int hb_log2 = 0;
  while ((2 << hb_log2) <= rep && hb_log2 < 5) ++hb_log2;
  const int HB = 1 << hb_log2, QT = 128 >> hb_log2, hblocks = (rep + HB - 1) >> hb_log2;
  const int64_t blocks = (int64_t)(total_q / QT + batch) * G * hblocks;
  if (blocks >= 1 << 24) return 0;  // a launch has fewer than 2^32 threads
  const auto kernel = splits > 1 ? maps_prompt_kernel<true> : maps_prompt_kernel<false>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks, 1, splits), dim3(256), 0, s, mp<bf16_t>(out), ld_out, part_o, part_ml, q,
                     cp<bf16_t>(k_cache), cp<bf16_t>(v_cache), table, table_stride, req_rows, seq_lens, cu_q, batch, total_q, H, G, scale, window, keep,
                     lam, cp<bf16_t>(gate), ld_gate, post, eps, hb_log2, splits);
  MIX_LAUNCHED("diff_attn (portions)");
  return 1;
}
