// Decode attention of a small batch in two launches: the new tokens' per-head RMSNorm, RoPE and K / V store inside the attention
// kernel, then the join of its key ranges.
//
// At a handful of requests a decode layer's attention is latency: 0.3 - 4 MB of keys and values, read in 1 - 2 us, behind a chain of
// launches and of dependent loads.  qk_norm_rope_store, the planned kernel of attn_decode.hip (plan -> piece -> request -> table
// -> rows) and its merge took 11.8 us a layer of Qwen3-0.6B's heads at 533 tokens, this 9.1 (both in a captured chain; a decode step
// 983 -> 849 us; other sizes at HipAttnBackend.small_decode).  Here there is no plan: workgroup (range, kv head, request)
// finds its tiles from the length alone, so that the longest chain is length -> table entry -> rows, and each workgroup
// normalises and rotates the G query heads of its kv head itself while its first rows are on their way.
//   * eight waves, each with its own 16-token tiles: tile i of a request goes to wave i % (8 R) of R workgroups, R = min(ranges of
//     the launch, ceil(tiles / 8)) -- ranges without a tile leave at once, so the grid can be fixed at capture;
//   * K rows come straight into the first product's operand (lane = token, 16 bytes of 32 dims), V rows through the wave's 4-KB
//     LDS image and transposing reads, as in attn_decode.hip; the next tile is requested before the present one is used;
//   * the queries are the second operand: column j < G is query head j, and column G carries the NEW KEY through the same norm and
//     rotation.  The wave that owns the last tile puts that key into the tile's operand, reads the new value row where the
//     projection left it, and stores both in the cache.  Nobody uses what the cache row holds that is being written: its value is
//     never read, its key is by the owner (put aside for the new one), by lanes past the end of the last tile (their scores are
//     masked) and by waves without a tile (which multiply nothing);
//   * the eight waves' sums meet in LDS; a request of one range is finished there.
// Same arithmetic as msgl_qk_norm_rope_store for the stored rows (same bits); fp32 partial sums as before.
#include "attn_decode_tile.h"

namespace msgl {

constexpr int kSmallWaves = 8;
constexpr int kSmallMaxRanges = 64;  // the join reads one (m, l) pair per lane

struct SmallDecodeParams {
  const uint16_t *q, *k, *v;  // the projection's rows [batch, heads * 128]
  const uint16_t *qw, *kw;    // per-head norm weights, or nullptr
  const int* positions;
  const float* cos_sin;  // [positions][64 cos | 64 sin], or nullptr: rows are taken as they are
  uint16_t *kc, *vc;
  const int *out_loc, *page_table, *req_rows, *seq_lens;
  uint16_t* out;
  float *part_o, *part_ml;
  int64_t pt_stride, q_stride, k_stride, v_stride, kv_stride_tok, kv_stride_head, out_stride;
  int hq, hkv, ranges;
  float eps, scale_log2;
};

__device__ __forceinline__ int small_ranges(int tiles, int ranges) { return min(ranges, (tiles + kSmallWaves - 1) / kSmallWaves); }

template <typename T>
__global__ __launch_bounds__(64 * kSmallWaves, 2) void attn_decode_small_kernel(const SmallDecodeParams p) {
  constexpr int D = 128;
  __shared__ __attribute__((aligned(16))) char lds[kSmallWaves * 4096];  // V images; then the waves' sums [wave][head][D]
  __shared__ float2 stat[kSmallWaves][8];                                // (m, l) of (wave, head)
  const int lane = threadIdx.x & 63, tok = lane & 15, qd = lane >> 4;
  const int wv = sgpr((int)(threadIdx.x >> 6));
  const int range = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int G = p.hq / p.hkv, hq0 = h * G;
  const int S = p.seq_lens[b];
  const int row = p.req_rows ? p.req_rows[b] : b;
  const int nt = (S + 15) >> 4;
  const int active = small_ranges(nt, p.ranges);
  if (range >= active) return;  // the whole workgroup
  const int step = active * kSmallWaves;
  const int first = range * kSmallWaves + wv;
  const int* pt = p.page_table + (int64_t)row * p.pt_stride;
  const int last = S - 1;  // the new token

  // slot of this lane's token of tile ti (tokens past the end: the last one's)
  auto slot_of = [&](int ti) { return pt[min(ti * 16 + tok, last)]; };
  struct Tile {
    V4 k[4], v[4];
  };
  const uint16_t* v_new = p.v + (int64_t)b * p.v_stride + (int64_t)h * D + qd * 8;
  auto load_tile = [&](Tile& t, int ti, int slot) {
    const int64_t off = (int64_t)slot * p.kv_stride_tok + (int64_t)h * p.kv_stride_head + qd * 8;
    const uint16_t* ka = p.kc + off;
    const uint16_t* va = ti * 16 + tok >= last ? v_new : p.vc + off;  // (past the end: a finite row for the masked lanes)
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) t.k[kk] = *reinterpret_cast<const V4*>(ka + kk * 32);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) t.v[kk] = *reinterpret_cast<const V4*>(va + kk * 32);
  };
  const int slot0 = slot_of(min(first, nt - 1));

  // ---- columns 0 .. G - 1: the query heads, column G: the new key; lane (column, qd) holds dims 32 kk + 8 qd .. + 7 ----
  const bool is_k = tok == G;
  V4 qf[4];
  {
    const uint16_t* src = is_k ? p.k + (int64_t)b * p.k_stride + (int64_t)h * D
                               : p.q + (int64_t)b * p.q_stride + (int64_t)(hq0 + (tok < G ? tok : 0)) * D;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) qf[kk] = *reinterpret_cast<const V4*>(src + kk * 32 + qd * 8);
  }
  V4 wq[4];
  if (p.qw) {
    const uint16_t* w = is_k ? p.kw : p.qw;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) wq[kk] = *reinterpret_cast<const V4*>(w + kk * 32 + qd * 8);
  }
  float cs[2][8], sn[2][8];
  if (p.cos_sin) {
    const float* c = p.cos_sin + (int64_t)p.positions[b] * D + qd * 8;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        *reinterpret_cast<float4*>(&cs[kk][e]) = *reinterpret_cast<const float4*>(c + kk * 32 + e);
        *reinterpret_cast<float4*>(&sn[kk][e]) = *reinterpret_cast<const float4*>(c + 64 + kk * 32 + e);
      }
    }
  }
  Tile cur;
  load_tile(cur, first, slot0);
  int slot1 = first + step < nt ? slot_of(first + step) : slot0;

  // The rounding points are msgl_qk_norm_rope_store's: the normed value passes through the 16-bit type (as packed words, so that
  // the rotation multiplies 16-bit operands in both kernels and rounds to fp16 once, in the multiply-add itself, in both)
  if (p.qw) {
    float x[4][8], ss[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {  // the order of row16_sum over the head's sixteen pieces (piece 4 kk + qd)
      unpack8<T>(__builtin_bit_cast(U4, qf[kk]), x[kk]);
      float t = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) t = fmaf(x[kk][e], x[kk][e], t);
      ss[kk] = sum_over_rows(t);
    }
    const float inv = rsqrtf(((ss[0] + ss[1]) + (ss[2] + ss[3])) / (float)D + p.eps);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      float w[8], y[8];
      unpack8<T>(__builtin_bit_cast(U4, wq[kk]), w);
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = __fmul_rn(__fmul_rn(x[kk][e], inv), w[e]);
      qf[kk] = __builtin_bit_cast(V4, pack8<T>(y));
    }
  }
  if (p.cos_sin) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      float lo[8], hi[8], y0[8], y1[8];
      unpack8<T>(__builtin_bit_cast(U4, qf[kk]), lo);
      unpack8<T>(__builtin_bit_cast(U4, qf[kk + 2]), hi);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        y0[e] = fmaf(lo[e], cs[kk][e], -__fmul_rn(hi[e], sn[kk][e]));
        y1[e] = fmaf(hi[e], cs[kk][e], __fmul_rn(lo[e], sn[kk][e]));
      }
      qf[kk] = __builtin_bit_cast(V4, pack8<T>(y0));
      qf[kk + 2] = __builtin_bit_cast(V4, pack8<T>(y1));
    }
  }

  float m = kNegBig, l = 0.f;
  f32x4 o[8];
#pragma unroll
  for (int db = 0; db < 8; ++db) o[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  dlds_char* img = (dlds_char*)lds + wv * 4096;

  for (int ti = first; ti < nt; ti += step) {
    Tile t = cur;
    if (ti + step < nt) {
      load_tile(cur, ti + step, slot1);
      if (ti + 2 * step < nt) slot1 = slot_of(ti + 2 * step);
    }
    if (ti == nt - 1) {  // the new token's tile: its key from column G, both rows into the cache
      const int lt = last & 15;
      const int64_t dst = (int64_t)p.out_loc[b] * p.kv_stride_tok + (int64_t)h * p.kv_stride_head + qd * 8;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        V4 nk;
#pragma unroll
        for (int e = 0; e < 4; ++e) nk[e] = (uint32_t)__shfl((int)qf[kk][e], (lane & 48) | G, 64);
        if (tok == lt) {
          t.k[kk] = nk;
          *reinterpret_cast<V4*>(p.kc + dst + kk * 32) = nk;
          *reinterpret_cast<V4*>(p.vc + dst + kk * 32) = t.v[kk];
        }
      }
    }
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
      *reinterpret_cast<__attribute__((address_space(3))) V4*>(img + vimg_off(tok, kk * 64 + qd * 16)) = t.v[kk];
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) s = mfma_k32<T>(t.k[kk], qf[kk], s);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (ti * 16 + 4 * qd + i > last) s[i] = -INFINITY;
    const float mx = max_over_rows(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))) * p.scale_log2;
    const float mn = fmaxf(m, mx);
    const float alpha = __builtin_amdgcn_exp2f(m - mn);
    m = mn;
    float pe[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) pe[i] = __builtin_amdgcn_exp2f(fmaf(s[i], p.scale_log2, -m));
    l = fmaf(l, alpha, (pe[0] + pe[1]) + (pe[2] + pe[3]));
    uint2 pf;
    pf.x = Elem<T>::pack(pe[0], pe[1]);
    pf.y = Elem<T>::pack(pe[2], pe[3]);
#pragma unroll
    for (int db = 0; db < 8; ++db) {
#pragma unroll
      for (int i = 0; i < 4; ++i) o[db][i] *= alpha;
      const ds16x4 vt = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_ds16x4*)(img + vimg_off(4 * qd + (tok >> 2), db * 32 + (tok & 3) * 8)));
      o[db] = mfma_k16<T>(__builtin_bit_cast(uint2, vt), pf, o[db]);
    }
  }

  // ---- the eight waves' sums ----
  l = sum_over_rows(l);
  __syncthreads();  // every wave is done with its V image
  float* sums = reinterpret_cast<float*>(lds);
  if (tok < G) {
    float* so = sums + (wv * G + tok) * D + 4 * qd;
#pragma unroll
    for (int db = 0; db < 8; ++db) *reinterpret_cast<f32x4*>(so + db * 16) = o[db];
    if (qd == 0) stat[wv][tok] = make_float2(m, l);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < G * (D / 2); i += 64 * kSmallWaves) {
    const int g = i >> 6, d = (i & 63) * 2;
    float mx = kNegBig;
#pragma unroll
    for (int w = 0; w < kSmallWaves; ++w) mx = fmaxf(mx, stat[w][g].x);
    float a0 = 0.f, a1 = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < kSmallWaves; ++w) {  // (a wave without a tile: weight 0 or 1, sums 0)
      const float2 ml = stat[w][g];
      const float wgt = __builtin_amdgcn_exp2f(ml.x - mx);
      const float2 ov = *reinterpret_cast<const float2*>(sums + (w * G + g) * D + d);
      a0 = fmaf(wgt, ov.x, a0);
      a1 = fmaf(wgt, ov.y, a1);
      den = fmaf(wgt, ml.y, den);
    }
    if (active == 1) {
      const float inv = 1.0f / den;
      *reinterpret_cast<uint32_t*>(p.out + (int64_t)b * p.out_stride + (int64_t)(hq0 + g) * D + d) = Elem<T>::pack(a0 * inv, a1 * inv);
    } else {
      const int64_t at = ((int64_t)b * p.ranges + range) * p.hq + hq0 + g;
      *reinterpret_cast<float2*>(p.part_o + at * D + d) = make_float2(a0, a1);
      if (d == 0) *reinterpret_cast<float2*>(p.part_ml + at * 2) = make_float2(mx, den);
    }
  }
}

// the ranges of one (request, query head): wave w adds ranges w, w + 4, ..., all of a wave's loads in flight together
template <typename T>
__global__ __launch_bounds__(256) void attn_decode_small_join_kernel(const SmallDecodeParams p) {
  constexpr int D = 128;
  __shared__ float2 sums[4][64];
  const int lane = threadIdx.x & 63, wv = sgpr((int)(threadIdx.x >> 6));
  const int hq = blockIdx.x, b = blockIdx.y;
  const int n = small_ranges((p.seq_lens[b] + 15) >> 4, p.ranges);
  if (n <= 1) return;
  const int64_t at = (int64_t)b * p.ranges * p.hq + hq;
  const float* po = p.part_o + at * D + lane * 2;
  constexpr int kEach = kSmallMaxRanges / 4;
  float2 ml = make_float2(kNegBig, 0.f);
  if (lane < n) ml = *reinterpret_cast<const float2*>(p.part_ml + (at + (int64_t)lane * p.hq) * 2);
  float2 ov[kEach];
#pragma unroll
  for (int u = 0; u < kEach; ++u)
    if (wv + 4 * u < n) ov[u] = *reinterpret_cast<const float2*>(po + (int64_t)(wv + 4 * u) * p.hq * D);
  const float wl = __builtin_amdgcn_exp2f(ml.x - wave_max(ml.x));
  const float den = wave_sum(wl * ml.y);
  float a0 = 0.f, a1 = 0.f;
#pragma unroll
  for (int u = 0; u < kEach; ++u) {
    if (wv + 4 * u < n) {
      const float wgt = __shfl(wl, wv + 4 * u, 64);
      a0 = fmaf(wgt, ov[u].x, a0);
      a1 = fmaf(wgt, ov[u].y, a1);
    }
  }
  sums[wv][lane] = make_float2(a0, a1);
  __syncthreads();
  if (wv == 0) {
#pragma unroll
    for (int w = 1; w < 4; ++w) {
      a0 += sums[w][lane].x;
      a1 += sums[w][lane].y;
    }
    const float inv = 1.0f / den;
    reinterpret_cast<uint32_t*>(p.out + (int64_t)b * p.out_stride + (int64_t)hq * D)[lane] = Elem<T>::pack(a0 * inv, a1 * inv);
  }
}

template <typename T>
static void launch_small(const SmallDecodeParams& p, int batch, hipStream_t s) {
  attn_decode_small_kernel<T><<<dim3((unsigned)p.ranges, (unsigned)p.hkv, (unsigned)batch), dim3(64 * kSmallWaves), 0, s>>>(p);
  if (p.ranges > 1) attn_decode_small_join_kernel<T><<<dim3((unsigned)p.hq, (unsigned)batch), dim3(256), 0, s>>>(p);
}

}  // namespace msgl

using namespace msgl;

// Ranges a launch cuts every request into: enough workgroups for two per CU at full length, no more than a request of max_seq_len
// tokens has 128-token pieces, at most 64.
extern "C" int msgl_attn_decode_small_ranges(int batch, int num_kv_heads, int64_t max_seq_len) {
  if (batch < 1 || num_kv_heads < 1 || max_seq_len < 1) return MSGL_EINVAL;
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  int64_t r = (2ll * cus + (int64_t)batch * num_kv_heads - 1) / ((int64_t)batch * num_kv_heads);
  const int64_t pieces = (max_seq_len + 16 * kSmallWaves - 1) / (16 * kSmallWaves);
  if (r > pieces) r = pieces;
  if (r > kSmallMaxRanges) r = kSmallMaxRanges;
  return r < 1 ? 1 : (int)r;
}

extern "C" int64_t msgl_attn_decode_small_workspace_bytes(int batch, int ranges, int num_q_heads) {
  if (batch < 1 || ranges < 1 || num_q_heads < 1) return MSGL_EINVAL;
  return (int64_t)batch * ranges * num_q_heads * (128 + 2) * (int64_t)sizeof(float);
}

extern "C" int msgl_attn_decode_small(void* out, const void* q, const void* k, const void* v, const void* q_norm_w, const void* k_norm_w,
                                      float eps, const int32_t* positions, const float* cos_sin, void* k_cache, void* v_cache,
                                      const int32_t* out_loc, const int32_t* page_table, int64_t pt_stride, const int32_t* req_rows,
                                      const int32_t* seq_lens, void* workspace, int64_t workspace_bytes, int batch, int ranges,
                                      int num_q_heads, int num_kv_heads, int head_dim, int64_t q_stride, int64_t k_stride, int64_t v_stride,
                                      int64_t kv_stride_tok, int64_t kv_stride_head, int64_t out_stride, float sm_scale, int dtype,
                                      void* stream) {
  MSGL_REQUIRE(out && q && k && v && k_cache && v_cache && out_loc && page_table && seq_lens && workspace, "attn_decode_small: null pointer");
  MSGL_REQUIRE((q_norm_w == nullptr) == (k_norm_w == nullptr) && (cos_sin == nullptr) == (positions == nullptr),
               "attn_decode_small: both norm weights or neither, a rotation table with positions or neither");
  MSGL_REQUIRE(head_dim == 128, "attn_decode_small: head_dim %d unsupported (128 only)", head_dim);
  MSGL_REQUIRE(num_kv_heads >= 1 && num_kv_heads < 65536 && num_q_heads % num_kv_heads == 0 && num_q_heads / num_kv_heads >= 1 &&
                   num_q_heads / num_kv_heads <= 8,
               "attn_decode_small: %d q heads / %d kv heads", num_q_heads, num_kv_heads);
  MSGL_REQUIRE(batch >= 1 && batch < 65536 && ranges >= 1 && ranges <= kSmallMaxRanges, "attn_decode_small: batch %d, %d ranges", batch, ranges);
  MSGL_REQUIRE(workspace_bytes >= msgl_attn_decode_small_workspace_bytes(batch, ranges, num_q_heads), "attn_decode_small: workspace of %lld bytes",
               (long long)workspace_bytes);
  MSGL_REQUIRE(q_stride % 8 == 0 && k_stride % 8 == 0 && v_stride % 8 == 0 && kv_stride_tok % 8 == 0 && kv_stride_head % 8 == 0 && out_stride % 8 == 0,
               "attn_decode_small: strides must be multiples of 8 elements");
  MSGL_REQUIRE(aligned16(out) && aligned16(q) && aligned16(k) && aligned16(v) && aligned16(k_cache) && aligned16(v_cache) && aligned16(workspace) &&
                   aligned16(q_norm_w) && aligned16(k_norm_w) && aligned16(cos_sin),
               "attn_decode_small: pointers must be 16-byte aligned");
  MSGL_REQUIRE(dtype == MSGL_BF16 || dtype == MSGL_FP16, "attn_decode_small: unsupported dtype code %d", dtype);
  SmallDecodeParams p{};
  p.q = (const uint16_t*)q; p.k = (const uint16_t*)k; p.v = (const uint16_t*)v;
  p.qw = (const uint16_t*)q_norm_w; p.kw = (const uint16_t*)k_norm_w;
  p.positions = positions; p.cos_sin = cos_sin;
  p.kc = (uint16_t*)k_cache; p.vc = (uint16_t*)v_cache;
  p.out_loc = out_loc; p.page_table = page_table; p.req_rows = req_rows; p.seq_lens = seq_lens;
  p.out = (uint16_t*)out;
  p.part_o = (float*)workspace;
  p.part_ml = p.part_o + (int64_t)batch * ranges * num_q_heads * 128;
  p.pt_stride = pt_stride; p.q_stride = q_stride; p.k_stride = k_stride; p.v_stride = v_stride;
  p.kv_stride_tok = kv_stride_tok; p.kv_stride_head = kv_stride_head; p.out_stride = out_stride;
  p.hq = num_q_heads; p.hkv = num_kv_heads; p.ranges = ranges;
  p.eps = eps;
  p.scale_log2 = sm_scale * 1.4426950408889634f;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == MSGL_BF16) launch_small<BF16>(p, batch, s);
  else launch_small<FP16>(p, batch, s);
  MSGL_CHECK_LAUNCH("attn_decode_small");
  return MSGL_OK;
}
