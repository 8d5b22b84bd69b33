// Paged varlen causal prefill attention for gfx950 (MFMA 32x32x16, fp32 accumulate).
//
// Two kernels with the same math per query row, bit-identical to each other (impl codes in include/msgl_hip.h): the default DMA-staged one
// (attn_prefill_dma_kernel, impl 4 = 0; 6 = two heads a workgroup) and its register-staged predecessor (attn_prefill_tr_kernel, impl 2), kept as the A/B
// partner and cross-check.  One workgroup = 4 waves = one 128-row query tile of one (request, q head), with impl 6 8 waves = the same tile of two heads of a
// kv head; each wave owns 32 query rows of a head.  K/V are gathered through the reference's token-granular page table in 64-key tiles one tile ahead of
// the MFMAs: global -> registers -> LDS (impl 2), global -> LDS by DMA (global_load_lds_dwordx4; impl 4, 6).  Launches that leave compute units empty cut a
// job's keys into ranges, whose sums attn_prefill_join_kernel puts together.  Ablation variants (ABL != 0: timing only, WRONG results) are compiled only with
// -DMSGL_PREFILL_DIAG (MSGL_PREFILL_DIAG=1 python mini-sglang_amd/build.py): a stray impl code cannot select one in a production build.
//
// Data flow per 64-key tile and wave (all in registers except the K/V tile):
//   S^T = K . Q^T   ("swapped" QK^T: A = K rows from LDS (XOR-swizzled, conflict-free
//                    ds_read_b128), B = the wave's Q fragments held in VGPRs)
//        => lane l owns query row (l & 31): its 32 scores are in-lane (+ lane l^32), so the
//           online softmax needs one cross-lane exchange per row statistic, no LDS;
//   O^T += V^T . P^T (A = V^T fragments read from a transposed, swizzled LDS image of V with
//                    two ds_read_b64; B = P packed to 16-bit straight from the score registers:
//                    the contraction index is permuted so each lane uses its OWN 8 keys -- no
//                    cross-lane movement of P)
//        => every O accumulator of lane l belongs to query row (l & 31): rescale and the final
//           1/l are lane-local.
// Causal mask is bottom-right aligned (query j of q_len sees keys t <= k_len - q_len + j),
// applied only on tiles that cross the diagonal; tiles fully above it are skipped.
#include <stdlib.h>

#include <type_traits>

#include "common.h"

namespace msgl {

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;

constexpr int kQTile = MSGL_PREFILL_QTILE;  // 128 query rows per workgroup
constexpr int kKTile = 64;                  // keys per tile
constexpr int kD = 128;
constexpr float kNegBigP = -3.0e38f;
typedef float f32x4p __attribute__((ext_vector_type(4)));

template <typename T>
__device__ __forceinline__ f32x16 mfma32(const U4& a, const U4& b, f32x16 c) {
  if constexpr (std::is_same_v<T, BF16>) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                   c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c,
                                                  0, 0, 0);
  }
}

struct PrefillParams {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const int* page_table;
  const int* req_rows;
  const int* seq_lens;
  const int* cu_q;
  const int* tile_cu;
  const int* tile_order;  // optional [total_tiles]: launch order of the q tiles (heaviest first); tr kernel only
  uint16_t* out;
  int64_t pt_stride, q_stride, kv_stride_tok, kv_stride_head, out_stride;
  int batch, hq, group;
  int share_log2, per;  // XCDs that share their kv heads, kv heads of each
  int stretch;     // workgroups of an XCD where each takes a stretch of the list, or 0
  int few;         // q tiles of fewer rows load and store by lanes' own pieces
  int idle;        // waves without rows make no products (one head a workgroup)
  int ranges, run;  // key ranges, and tiles of each (the last one: what is left)
  const uint16_t *k_new, *v_new;  // FRESH: the rows of all requests' keys and values as they come, and where they are to be stored
  uint16_t *k_pool, *v_pool;
  const int* out_loc;
  int64_t new_stride;
  float *part_o, *part_ml;
  float scale_log2;
};

// Workgroup -> (kv head, q tile, query head).  XCD x = blockIdx % 8 keeps to `per` kv heads, so that their rows stay in its L2; the 8 / gcd(8,
// kv heads) XCDs with the same ones take turns down one list, the tiles in the order given (most keys first) with all their heads: every XCD
// gets long tiles and short ones, and what starts last is short.  (Cut into eight stretches instead, the first XCDs of a list had all the long
// tiles, or one kv head's short tiles came before the next one's long ones.  8 requests of 300 - 1300 tokens, 16 heads on 2: 69 -> 47 us; 4000
// tokens, 10 on 2: 106 -> 88; 20 requests of 100 - 1024, 9 on 3: 56 -> 47, 24 on 12: 129 -> 126, 32 on 16: 156 -> 152.  8 kv heads: as before.
// Many requests of like length lose where an XCD's list has several kv heads, whose rows then pass through its L2 together: 20 of 90 - 170 tokens,
// 24 on 12: 28 -> 30, after 3000 200 -> 213; 9 on 3: 14.8 -> 16.0.)
// A launch of one workgroup per CU or less starts all of them at once: stretches of the list, which leave an XCD fewer requests' keys (6 requests of
// 100 - 400 after 2500, 16 on 2: 63 us, in turns 65).
struct PrefillJob {
  int kvh, hq, tile;  // tile < 0: none left
};
__device__ __forceinline__ PrefillJob prefill_job(const PrefillParams& p, int total_tiles) {
  const int xcd = (int)(blockIdx.x & 7), list = xcd >> p.share_log2, seat = xcd - (list << p.share_log2), n = (int)(blockIdx.x >> 3);
  const int u = p.stretch ? seat * p.stretch + n : (n << p.share_log2) + seat;
  const int each = p.group * p.per, ti = u / each, r = u - ti * each, sub = r / p.group;
  PrefillJob j;
  j.kvh = list * p.per + sub;
  j.hq = j.kvh * p.group + (r - sub * p.group);
  j.tile = ti >= total_tiles ? -1 : p.tile_order ? p.tile_order[ti] : ti;
  return j;
}

// element offset of a pool slot: slot and the token stride are both < 2^32 (checked at launch), so ONE v_mad_u64_u32
// does it; the int64 x int64 product the types ask for costs two quarter-rate 32-bit multiplies and a carry chain more
__device__ __forceinline__ int64_t slot_offset(int slot, int64_t stride_tok) {
  return (int64_t)((uint64_t)(uint32_t)slot * (uint64_t)(uint32_t)stride_tok);
}

// The request a q tile belongs to and its scalars, in ONE memory latency for batches up to 64 requests (the bisection over
// tile_cu followed by the four scalar loads paid log2(B) + 1 dependent ones: ~2.5 us of a workgroup that computes for
// ~5 us on the benchmark's prefill chunks).  Lane i of a 64-request block loads request i's tile_cu, cu_q, cu_q[+1],
// seq_len and table row together; b = the last request with tile_cu[b] <= tile is counted with a ballot and its values are
// taken from that lane.
struct TileRequest {
  int b, q_begin, q_end, k_len, row, tile_first;
};
__device__ __forceinline__ TileRequest find_request(const PrefillParams& p, int tile, int lane) {
  TileRequest r;
  int base = 0;
  for (;;) {
    const int idx = min(base + lane, p.batch - 1);
    const int tc = base + lane < p.batch ? p.tile_cu[idx] : 0x7fffffff;
    const int cq0 = p.cu_q[idx], cq1 = p.cu_q[idx + 1], kl = p.seq_lens[idx];
    const int rr = p.req_rows ? p.req_rows[idx] : idx;
    const int cnt = __popcll(__ballot(tc <= tile));
    if (cnt > 0 && (cnt < 64 || base + 64 >= p.batch)) {
      const int l = cnt - 1;
      r.b = base + l;
      r.tile_first = __builtin_amdgcn_readlane(tc, l);
      r.q_begin = __builtin_amdgcn_readlane(cq0, l);
      r.q_end = __builtin_amdgcn_readlane(cq1, l);
      r.k_len = __builtin_amdgcn_readlane(kl, l);
      r.row = __builtin_amdgcn_readlane(rr, l);
      return r;
    }
    if (cnt == 0) {  // the last request of the previous block (more than 64 requests only)
      r.b = base - 1;
      r.tile_first = p.tile_cu[r.b];
      r.q_begin = p.cu_q[r.b];
      r.q_end = p.cu_q[r.b + 1];
      r.k_len = p.seq_lens[r.b];
      r.row = p.req_rows ? p.req_rows[r.b] : r.b;
      return r;
    }
    base += 64;
  }
}

// swizzles (see header comment): K image [64 keys][256 B], V^T image [128 d][128 B = 64 keys]
__device__ __forceinline__ int k_off(int key, int byte_in_row) { return key * 256 + (byte_in_row ^ ((key & 15) << 4)); }
__device__ __forceinline__ int vt_g(int d) { return ((d >> 1) & 15) ^ ((d >> 5) & 3); }
__device__ __forceinline__ int vt_off(int d, int unit) { return d * 128 + ((unit ^ vt_g(d)) << 3); }

// ------------------------------------------------------------------------------------------------
// Second-generation kernel (impl 2; the default until the DMA-staged impl 4 below): same math and fragment ownership as above, but
//   * V is staged ROW-major ([64 keys][256 B], like K: four ds_write_b128 per thread and tile instead of
//     thirty-two 2-byte transposing stores) and the V^T MFMA fragments come out of LDS through the gfx950
//     transposing read ds_read_b64_tr_b16: a 16-lane group reads one [4 keys][16 d] block (lane j passes the
//     address of row j>>2, columns 4(j&3)..+3) and lane j receives column j of it = its 4 consecutive keys.
//     64-B XOR swizzle on the key's low two bits => the 32 lanes of a read hit 64 distinct banks;
//   * K/V tiles are double-buffered in LDS (64 KB per workgroup): ONE barrier per 64-key tile; loads for tile
//     t+1 are issued before tile t's MFMAs and written to LDS after them; page-table slots run one more
//     tile ahead so the gather never waits for its own indices;
//   * <= 256 registers: two workgroups (8 waves) per CU, so one workgroup's softmax overlaps the other's MFMAs;
//   * 1-D grid remapped so that each XCD owns a contiguous range of (kv head, q tile, q head of the group):
//     the G query heads that share a K/V tile run back to back on ONE XCD's L2 (at Hkv = 8: kv head == XCD);
//     q tiles are taken in the caller's order (heaviest first) so the tail is made of light tiles;
//   * the O rescale is skipped (exactly) on tiles where no row's running max moved.
// ------------------------------------------------------------------------------------------------
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) char lds_char;

__device__ __forceinline__ int v_off(int key, int byte_in_row) { return key * 256 + (byte_in_row ^ ((key & 3) << 6)); }

__device__ __forceinline__ uint2 tr_read_b64(const char* lds_ptr) {
  const s16x4 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(lds_char*)lds_ptr);
  return __builtin_bit_cast(uint2, r);
}

// This lane's number and lane ^ 32's, without LDS: a swap of halves between two copies leaves both numbers in every lane.
__device__ __forceinline__ float2 both_halves(float x) {
  const auto y = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const uint32_t y0 = y[0], y1 = y[1];  // (a bit cast of the vector's element itself takes element 0 both times)
  return float2{__uint_as_float(y0), __uint_as_float(y1)};
}
__device__ __forceinline__ float pair_max(float x) {
  const float2 y = both_halves(x);
  return fmaxf(y.x, y.y);
}
__device__ __forceinline__ float pair_sum(float x) {
  const float2 y = both_halves(x);
  return y.x + y.y;
}

// 16 bytes that nobody reads in this launch
__device__ __forceinline__ void store_past(uint16_t* to, const char* from) {
  typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
  __builtin_nontemporal_store(*reinterpret_cast<const u32x4_t*>(from), reinterpret_cast<u32x4_t*>(to));
}

constexpr int kTileBytes = kKTile * kD * 2;  // 16 KB: one K (or V) tile image

// ABL (diagnosis only, wrong results): 1 = K/V tiles loaded once (no HBM/L2 stream, no LDS writes after the first tile),
// 2 = no QK^T MFMAs, 4 = no softmax arithmetic, 8 = no PV MFMAs, 16 = no barrier after the first tile
template <typename T, bool kFold = true, int ABL = 0>
__global__ __launch_bounds__(256, 2) void attn_prefill_tr_kernel(const PrefillParams p, int total_tiles) {
  __shared__ __attribute__((aligned(16))) char lds[4 * kTileBytes];  // [buf][K | V]

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: the diagonal tests below are scalar branches
  const int hi = lane >> 5;

  const PrefillJob job = prefill_job(p, total_tiles);
  if (job.tile < 0) return;
  const int kvh = job.kvh, hq = job.hq, tile = job.tile;

  int lo = 0, hi_b = p.batch;  // find b with tile_cu[b] <= tile < tile_cu[b+1]
  while (hi_b - lo > 1) {
    const int mid = (lo + hi_b) >> 1;
    if (p.tile_cu[mid] <= tile) lo = mid; else hi_b = mid;
  }
  const int b = lo;
  const int q_begin = p.cu_q[b];
  const int q_len = p.cu_q[b + 1] - q_begin;
  const int k_len = p.seq_lens[b];
  const int q0 = (tile - p.tile_cu[b]) * kQTile;
  const int row = p.req_rows ? p.req_rows[b] : b;
  const int* pt = p.page_table + (int64_t)row * p.pt_stride;
  const int diag = k_len - q_len;
  const int kend = min(k_len, diag + min(q0 + kQTile, q_len));
  const int ntiles = (kend + kKTile - 1) / kKTile;

  // ---- Q fragments ------------------------------------------------------------------------------
  const int my_q = q0 + wave * 32 + (lane & 31);
  const bool q_valid = my_q < q_len;
  const int64_t q_tok = q_begin + (q_valid ? my_q : q_len - 1);
  U4 qf[8];
  {
    const uint16_t* qp = p.q + q_tok * p.q_stride + (int64_t)hq * kD + hi * 8;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qf[ks] = ldg16(qp + ks * 16);
  }
  const int my_qpos = diag + my_q;
  const int wave_min_qpos = diag + q0 + wave * 32;

  f32x16 o[4];
#pragma unroll
  for (int nb = 0; nb < 4; ++nb)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[nb][r] = 0.f;
  float m_run = kNegBigP, l_run = 0.f;

  // ---- staging: thread owns 16-byte pieces c = tid + 256 i (key = c >> 4, piece = c & 15) -----------
  const int st_key = tid >> 4, st_piece = tid & 15;  // key of piece i = st_key + 16 i
  const int64_t head_off = (int64_t)kvh * p.kv_stride_head + st_piece * 8;
  int sl[4];
  U4 kreg[4], vreg[4];
  auto load_slots = [&](int kt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) sl[i] = pt[min(kt * kKTile + st_key + 16 * i, k_len - 1)];  // never past the sequence
  };
  auto issue_loads = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t off = slot_offset(sl[i], p.kv_stride_tok) + head_off;
      kreg[i] = ldg16(p.k + off);
      vreg[i] = ldg16(p.v + off);
    }
  };
  auto write_lds = [&](char* buf) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = st_key + 16 * i;
      *reinterpret_cast<U4*>(buf + k_off(key, st_piece * 16)) = kreg[i];
      *reinterpret_cast<U4*>(buf + kTileBytes + v_off(key, st_piece * 16)) = vreg[i];
    }
  };
  // V^T fragment addressing: lane = 16 g4 + j; the lane's share of a [4 keys][16 d] block is row j >> 2,
  // columns 16 (g4 & 1) + 4 (j & 3) .. +3 of d block nb; the swizzle term depends on the lane's row only
  int voff[4];
  {
    const int j = lane & 15;
    const int r4 = j >> 2;  // lane j of a 16-lane tr-read group passes row j >> 2, 8-byte chunk j & 3
    const int ch = j & 3;   // (layout confirmed on hardware by tools/tr_probe.hip, pattern 1)
    const int w = (16 * ((lane >> 4) & 1) + 4 * ch) * 2;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) voff[nb] = kTileBytes + hi * 1024 + r4 * 256 + (((nb ^ r4) & 3) << 6) + w;
  }

  if (ntiles > 0) {
    load_slots(0);
    issue_loads();
    if (ntiles > 1) load_slots(1);
  }
  for (int kt = 0; kt < ntiles; ++kt) {
    char* buf = lds + ((ABL & 1) ? 0 : (kt & 1)) * (2 * kTileBytes);
    if (!(ABL & 1) || kt == 0) write_lds(buf);  // tile kt (its loads were issued one tile ago); the buffer was last read at tile kt-2
    if (kt + 1 < ntiles && !(ABL & 1)) {
      issue_loads();  // tile kt+1: in flight during this tile's MFMAs
      if (kt + 2 < ntiles) load_slots(kt + 2);
    }
    if (!(ABL & 16) || kt == 0) __syncthreads();

    const int key0 = kt * kKTile;
    if (key0 > diag + q0 + wave * 32 + 31) continue;  // whole tile above this wave's diagonal

    // ---- S^T = K . Q^T -----------------------------------------------------------------
    f32x16 s[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[kb][r] = 0.f;
      const int key = kb * 32 + (lane & 31);
      if (!(ABL & 2)) {
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
          const U4 a = *reinterpret_cast<const U4*>(buf + k_off(key, ks * 32 + hi * 16));
          s[kb] = mfma32<T>(a, qf[ks], s[kb]);
        }
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[kb][r] = __uint_as_float(qf[r & 7].x) * 1e-30f + (float)kt;
      }
    }
    // ---- mask, online softmax (lane-local row); kFold: the softmax scale folded into the exponent's fma
    if constexpr (ABL & 4) {  // diagnosis: no softmax arithmetic (p = s as it is)
      m_run = 0.f;
      l_run += s[0][0] + s[1][15];
    } else {
      float tmax = kNegBigP;
      float m_new, alpha, rsum = 0.f;
      const bool need_mask = key0 + kKTile - 1 > wave_min_qpos;
      if constexpr (!kFold) {
  #pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
  #pragma unroll
          for (int r = 0; r < 16; ++r) {
            float x = s[kb][r] * p.scale_log2;
            if (need_mask) {
              const int key = key0 + kb * 32 + (r & 3) + 8 * (r >> 2) + 4 * hi;
              if (key > my_qpos) x = -INFINITY;
            }
            s[kb][r] = x;
            tmax = fmaxf(tmax, x);
          }
        }
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
        m_new = fmaxf(m_run, tmax);
        alpha = __builtin_amdgcn_exp2f(m_run - m_new);
  #pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
  #pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float e = __builtin_amdgcn_exp2f(s[kb][r] - m_new);
            s[kb][r] = e;
            rsum += e;
          }
        }
      } else {
  #pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
  #pragma unroll
          for (int r = 0; r < 16; ++r) {
            float x = s[kb][r];
            if (need_mask) {
              const int key = key0 + kb * 32 + (r & 3) + 8 * (r >> 2) + 4 * hi;
              if (key > my_qpos) x = -INFINITY;
              s[kb][r] = x;
            }
            tmax = fmaxf(tmax, x);
          }
        }
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64)) * p.scale_log2;  // scale > 0: max commutes with it
        m_new = fmaxf(m_run, tmax);
        alpha = __builtin_amdgcn_exp2f(m_run - m_new);
  #pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
  #pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float e = __builtin_amdgcn_exp2f(fmaf(s[kb][r], p.scale_log2, -m_new));
            s[kb][r] = e;
            rsum += e;
          }
        }
      }
      rsum += __shfl_xor(rsum, 32, 64);
      l_run = fmaf(l_run, alpha, rsum);
      if (!__all(m_new == m_run)) {  // alpha == 1 on every row otherwise: the rescale would be the identity
  #pragma unroll
        for (int nb = 0; nb < 4; ++nb)
  #pragma unroll
          for (int r = 0; r < 16; ++r) o[nb][r] *= alpha;
      }
      m_run = m_new;
    }

    if constexpr (!(ABL & 8)) {
    // ---- O^T += V^T . P^T ------------------------------------------------------------------
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        U4 pf;
        pf.x = Elem<T>::pack(s[kb][8 * half + 0], s[kb][8 * half + 1]);
        pf.y = Elem<T>::pack(s[kb][8 * half + 2], s[kb][8 * half + 3]);
        pf.z = Elem<T>::pack(s[kb][8 * half + 4], s[kb][8 * half + 5]);
        pf.w = Elem<T>::pack(s[kb][8 * half + 6], s[kb][8 * half + 7]);
        // lane's keys: 4-key unit u1 = kb 8 + half 4 + hi (k slots 0..3) and unit u1 + 2 (k slots 4..7);
        // unit u = rows 4u..4u+3 = 1 KB of the image (hi is folded into voff)
        constexpr int kUnitBytes = 4 * 256;
        const int ub = (kb * 8 + half * 4) * kUnitBytes;
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
          const uint2 v1 = tr_read_b64(buf + voff[nb] + ub);
          const uint2 v2 = tr_read_b64(buf + voff[nb] + ub + 2 * kUnitBytes);
          U4 vf;
          vf.x = v1.x; vf.y = v1.y; vf.z = v2.x; vf.w = v2.y;
          o[nb] = mfma32<T>(vf, pf, o[nb]);
        }
      }
    }
    } else {
      o[0][0] += s[0][3] + s[1][7];
    }
  }

  // ---- epilogue: O[q row][d] = O^T / l ---------------------------------------------------------
  if (q_valid) {
    const float inv = 1.0f / l_run;
    uint16_t* op = p.out + (int64_t)(q_begin + my_q) * p.out_stride + (int64_t)hq * kD;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        const int d = nb * 32 + 8 * rg + 4 * hi;
        uint2 w;
        w.x = Elem<T>::pack(o[nb][4 * rg + 0] * inv, o[nb][4 * rg + 1] * inv);
        w.y = Elem<T>::pack(o[nb][4 * rg + 2] * inv, o[nb][4 * rg + 3] * inv);
        *reinterpret_cast<uint2*>(op + d) = w;
      }
    }
  }
}


// ------------------------------------------------------------------------------------------------
// Third-generation kernel (impl 4, the default): the math, fragment ownership and LDS images of the tr-read kernel, with
//   * K/V tiles moved global -> LDS by the DMA path (global_load_lds_dwordx4): no staging registers, no ds_write, no
//     LDS-write bandwidth.  A wave instruction fills 1 KB = 4 key rows lane-linearly, so the XOR swizzles of the images
//     are applied on the SOURCE side: the lane that lands on 16-byte slot c of row r fetches piece c ^ swz(r);
//   * the tile loop unrolled by two: every LDS address is (a per-lane register computed once) + an immediate;
//   * the causal mask hoisted out of the per-element path (one uniform branch per tile; compare against inline constants);
//   * one barrier per tile as before: wait own DMA of tile t, barrier, issue the DMA of tile t+1 into the buffer
//     everyone has just finished reading, compute tile t;
//   * LDS reads issued >= 4 MFMAs ahead of their use (pinned with sched_barrier); beside a DMA under way the compiler waits for ALL of a
//     wave's reads at the first use of any, so the V^T fragments are asked for after the second key block's have come;
//   * nothing of the softmax crosses LDS: the halves' maximum and their shares of a tile's sum by lane swaps.
// What bounds it: power, where the launch is long (1.8 GHz; inputs of zeros 5330 -> 4020 us), and the copies.  64 heads, 8192 tokens after 16384, us
// with a part left out (one head a workgroup, 5290 with all): all copies but the first 4330, no exponentials 5025, no rescale 5200, none of exponentials,
// rescale and mask 4930; the scores of the next tile in the same wave beside a tile's weights: 5290.  A wave's tile is 1024 cycles of the matrix cores and
// about as many of the vector units (32 scores a lane, the exponential 16 cycles each).  5240 us with a row's offset found once, 4960 with two heads a
// workgroup (1110 TFLOP/s).  40 heads on 8, 29 requests of 100 - 1024 tokens, with store_kv_kernel (23): 238 -> 234 us with a row's offset found once, 226
// with Q and the outputs in whole rows by way of LDS, 220 without products for rows that are none; starts and outputs are half of such a launch (in us
// before those two: empty workgroups 14, requests and outputs 41, the first tile 48, the second 17, each of the others 19).  60 requests of 128 - 256
// tokens 125 -> 109.  (Sums of the rounded weights, one instruction a pair: 0.5 % faster, and 2^-9 of a row's weight off.)
// HEADS = 2: eight waves, two heads of a kv head beside each other over the same tiles: half the copies.  One workgroup a CU then, so nothing runs
// under its start, and the last round is coarser: for many long chains of tiles (the rule and its other side: ops.prefill_pairs).
// RANGES: workgroup (.., z) takes the tiles z * run .. of the job's keys; sums of more than one range go to attn_prefill_join_kernel in fp32, in
// the order of the lanes.  For launches that leave compute units empty, where the longest chain of tiles (1.26 us each) is the time: 16 heads on
// 8, 100 tokens after 2000: 45.1 -> 13.7 us, 1000 after 3000: 81.7 -> 53.2; 5 on 1, 2000 tokens: 43.0 -> 20.5 (both launches, in a captured chain;
// the rule and its other side: ops.prefill_ranges)
// FRESH: nothing is cached, so keys and values are read from the rows as they come, without the page table, and stored to the pool from the two tiles that a
// workgroup's query rows are the keys of, which lie in LDS at its end (by the first head of a kv head).  Prompts longer than
// ops.FRESH_TOKENS take the store and the other launch.  us, store_kv_kernel and launch -> this, inputs in cache, 40 heads on 8: 29
// requests of 100 - 1024 tokens 214 -> 192 (not in cache 221 -> 208), 60 of 128 - 256 99 -> 85, 8 of 600 - 1000 91 -> 85, 6 of 1500 184 -> 176; 16 on 8: 60 of 128 -
// 256 54.5 -> 43.9; 64 on 8 155 -> 140.  Beyond, 40 on 8: 4 of 2048 210 -> 202, one of 8192 706 -> 692.  (The pool's rows by way of the L2 212 where 206; each of a kv head's heads a
// share of them: slower, each waits for its slots.)
// ABL (diagnosis, wrong results): 1 = tiles DMA'd once, 2 = no QK^T, 4 = no softmax, 8 = no PV.
// ------------------------------------------------------------------------------------------------
typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) const void glb_void_t;

// lane I's number of every 16 lanes
template <int I>
__device__ __forceinline__ uint64_t row_lane(uint64_t x) {
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)x, 0x150 + I, 0xf, 0xf, true);  // row_newbcast
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(x >> 32), 0x150 + I, 0xf, 0xf, true);
  return (uint64_t)hi << 32 | lo;
}

template <typename T, int ABL = 0, bool RANGES = false, int HEADS = 1, bool FRESH = false>
__global__ __launch_bounds__(256 * HEADS, 2) void attn_prefill_dma_kernel(const PrefillParams p, int total_tiles) {
  // two distinct LDS objects, not one array: the compiler then knows a tile's fragment reads cannot alias the DMA writes
  // of the next tile (other object) and does not wait for them (vmcnt) before the reads
  __shared__ __attribute__((aligned(1024))) char lds_a[2 * kTileBytes];  // tiles 0, 2, ..: [K | V]
  __shared__ __attribute__((aligned(1024))) char lds_b[2 * kTileBytes];  // tiles 1, 3, ..

  // ABL bit 16: MFMA blocks at s_setprio 1, bit 32: the softmax at priority 1 instead.  Neither moves the kernel outside
  // run-to-run noise once the variants are timed interleaved (tools/prefill_ablate.py), so the default sets no priority
  constexpr bool kPrioMatrix = (ABL & 16) != 0;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), rows = wave & 3;  // rows 32 rows .. + 31 of the q tile
  const int hi = lane >> 5;

  const PrefillJob job = prefill_job(p, total_tiles);
  if (job.tile < 0) return;
  const int kvh = job.kvh, hq = job.hq * HEADS + (wave >> 2), tile = job.tile;

  const TileRequest rq = find_request(p, tile, lane);
  const int q_begin = rq.q_begin;
  const int q_len = rq.q_end - q_begin;
  const int k_len = rq.k_len;
  const int q0 = (tile - rq.tile_first) * kQTile;
  const int* pt = p.page_table + (int64_t)rq.row * p.pt_stride;
  const int diag = k_len - q_len;
  const int kend = min(k_len, diag + min(q0 + kQTile, q_len));
  const int all_tiles = (kend + kKTile - 1) / kKTile;
  const int t0 = RANGES ? (int)blockIdx.y * p.run : 0;
  const int ntiles = RANGES && blockIdx.y + 1 < gridDim.y ? min(all_tiles, t0 + p.run) : all_tiles;  // past this workgroup's last
  if (RANGES && t0 > 0 && t0 >= ntiles) return;

  const int my_q = q0 + rows * 32 + (lane & 31);
  const bool q_valid = my_q < q_len;
  U4 qf[8];
  const bool own_pieces = HEADS == 2 || q_len - q0 < p.few;  // a lane loads and stores its own pieces of its row
  if (own_pieces) {
    const uint16_t* qp = p.q + (int64_t)(q_begin + (q_valid ? my_q : q_len - 1)) * p.q_stride + (int64_t)hq * kD + hi * 8;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qf[ks] = ldg16(qp + ks * 16);
  }
  const int my_qpos = diag + my_q;
  const int left = q_len - (q0 + rows * 32);  // this wave's rows, 32 of them at most
  const int wave_min_qpos = HEADS == 2 || left > 0 || !p.idle ? diag + q0 + rows * 32 : -kKTile;  // scalar; no row: no tile

  f32x16 o[4];
#pragma unroll
  for (int nb = 0; nb < 4; ++nb)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[nb][r] = 0.f;
  float m_run = kNegBigP, l_run = 0.f;

  // ---- staging: DMA instruction i of this wave fills rows kApart i + 4 wave .. + 3 of the image; lane -> row st_row + kApart i,
  //      16-byte slot (lane & 15)
  constexpr int kApart = 16 * HEADS, kTurns = 4 / HEADS;
  const int st_row = tid >> 4;
  const int64_t head_at = FRESH ? (int64_t)q_begin * p.new_stride + kvh * kD : (int64_t)kvh * p.kv_stride_head;
  const char* k_lane = reinterpret_cast<const char*>((FRESH ? p.k_new : p.k) + head_at + (((lane & 15) ^ (st_row & 15)) << 3));
  const char* v_lane = reinterpret_cast<const char*>((FRESH ? p.v_new : p.v) + head_at + (((lane & 15) ^ ((st_row & 3) << 2)) << 3));
  // A row's slot and offset are found once: lane i of the 16 that copy rows st_row, st_row + kApart, .. has row st_row + kApart i's, and the sixteen
  // take it from there as the address is added up (every lane for its own four rows, HEADS = 1: three more quarter-rate multiplies and three more
  // loads a tile; 64 heads, 8192 tokens after 16384: 5285 -> 5210 us, 29 requests of 100 - 1024, 40 heads on 8: 236 -> 234)
  const uint32_t row_of = st_row + kApart * (lane & (kTurns - 1));
  int sl;
  auto load_slots = [&](int kt) {
    const uint32_t key = min((uint32_t)(kt * kKTile) + row_of, (uint32_t)(k_len - 1));
    sl = FRESH ? (int)key : pt[key];
  };
  auto issue_dma = [&](char* buf) {
    const uint64_t off = (uint64_t)slot_offset(sl, FRESH ? p.new_stride : p.kv_stride_tok) * 2;
    auto four_rows = [&](auto I) __attribute__((always_inline)) {
      constexpr int i = decltype(I)::value;
      const uint64_t o = row_lane<i>(off);
      __builtin_amdgcn_global_load_lds((glb_void_t*)(k_lane + o), (lds_void_t*)(buf + (kApart / 4 * i + wave) * 1024), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((glb_void_t*)(v_lane + o), (lds_void_t*)(buf + kTileBytes + (kApart / 4 * i + wave) * 1024), 16, 0, 0);
    };
    four_rows(std::integral_constant<int, 0>{});
    four_rows(std::integral_constant<int, 1>{});
    if constexpr (kTurns == 4) {
      four_rows(std::integral_constant<int, 2>{});
      four_rows(std::integral_constant<int, 3>{});
    }
  };
  // per-lane LDS addresses (buffer 0): K fragment of k-step ks, V^T fragment of d block nb
  int koff[8], voff[4];
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) koff[ks] = k_off(lane & 31, ks * 32 + hi * 16);
  {
    const int j = lane & 15;
    const int r4 = j >> 2;
    const int ch = j & 3;
    const int w = (16 * ((lane >> 4) & 1) + 4 * ch) * 2;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) voff[nb] = kTileBytes + hi * 1024 + r4 * 256 + (((nb ^ r4) & 3) << 6) + w;
  }

  auto tile_body = [&](auto BUFC, const int kt) {
    constexpr int BUF = decltype(BUFC)::value;
    char* buf = BUF ? lds_b : lds_a;
    char* nxt = BUF ? lds_a : lds_b;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's pieces of tile kt (and the slots of tile kt + 1/2)
    __syncthreads();                                  // everyone's pieces; everyone done with the other buffer
    if (!(ABL & 1) && kt + 1 < ntiles) {
      issue_dma(nxt);
      if (kt + 2 < ntiles) load_slots(kt + 2);
    }
    const int key0 = kt * kKTile;
    if (key0 > wave_min_qpos + 31) return;  // whole tile above this wave's diagonal

    // ---- S^T = K . Q^T.  Issue order is pinned (sched_barrier): the 8 fragments of key block 0 first, then one
    //      MFMA per further LDS read -- key block 1's fragments under block 0's chain, the V^T fragments of the first
    //      half of P.V (they do not depend on the softmax) under block 1's chain: no MFMA waits on a read issued just
    //      before it
    f32x16 s[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[kb][r] = 0.f;
    if constexpr (kPrioMatrix) __builtin_amdgcn_s_setprio(1);
    if constexpr (ABL & 32) __builtin_amdgcn_s_setprio(0);
    U4 vfa[8];  // V^T fragments of keys 0..31: [half][nb]
    constexpr int kUnitBytes = 4 * 256;
    auto read_vf = [&](int kb, int half, int nb) {
      const int ub = (kb * 8 + half * 4) * kUnitBytes;
      const uint2 v1 = tr_read_b64(buf + voff[nb] + ub);
      const uint2 v2 = tr_read_b64(buf + voff[nb] + ub + 2 * kUnitBytes);
      U4 vf;
      vf.x = v1.x; vf.y = v1.y; vf.z = v2.x; vf.w = v2.y;
      return vf;
    };
    if constexpr (!(ABL & 2)) {
      U4 kf0[8], kf1[8];
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) kf0[ks] = *reinterpret_cast<const U4*>(buf + koff[ks]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {  // every read is issued >= 4 MFMAs (128 cycles) ahead of its use
        s[0] = mfma32<T>(kf0[ks], qf[ks], s[0]);
        if (ks < 4) {
          kf1[2 * ks] = *reinterpret_cast<const U4*>(buf + koff[2 * ks] + 8192);
          kf1[2 * ks + 1] = *reinterpret_cast<const U4*>(buf + koff[2 * ks + 1] + 8192);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
        s[1] = mfma32<T>(kf1[ks], qf[ks], s[1]);
        if constexpr (!(ABL & 8)) vfa[ks] = read_vf(0, ks >> 2, ks & 3);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) s[kb][r] = __uint_as_float(qf[r & 7].x) * 1e-30f + (float)kt;
      if constexpr (!(ABL & 8)) {
#pragma unroll
        for (int j = 0; j < 8; ++j) vfa[j] = read_vf(0, j >> 2, j & 3);
      }
    }
    if constexpr (kPrioMatrix) __builtin_amdgcn_s_setprio(0);
    if constexpr (ABL & 32) __builtin_amdgcn_s_setprio(1);
    uint32_t pw[2][8];  // the weights, packed in pairs
    if constexpr (ABL & 4) {
      m_run = 0.f;
      l_run += s[0][0] + s[1][15];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; r += 2) pw[kb][r >> 1] = Elem<T>::pack(s[kb][r], s[kb][r + 1]);
    } else {
      // ---- causal mask (tiles crossing this wave's diagonal only): key0 + c + 4 hi > my_qpos  <=>  c > thr
      if (key0 + kKTile - 1 > wave_min_qpos) {
        const int thr = my_qpos - key0 - 4 * hi;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (kb * 32 + (r & 3) + 8 * (r >> 2) > thr) s[kb][r] = -INFINITY;
      }
      // ---- online softmax, lane-local row (+ lane ^ 32); the scale is folded into the exponent's fma
      float tmax = kNegBigP;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, s[kb][r]);
      tmax = pair_max(tmax) * p.scale_log2;
      float alpha = 1.f;
      if (!__all(tmax <= m_run)) {
        const float m_new = fmaxf(m_run, tmax);
        alpha = __builtin_amdgcn_exp2f(m_run - m_new);
#pragma unroll
        for (int nb = 0; nb < 4; ++nb)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[nb][r] *= alpha;
        m_run = m_new;
      }
      // the row's sum is of the fp32 weights, tile by tile: its order is part of the result (the other instances' bits)
      float rsum = 0.f;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
          const float e0 = __builtin_amdgcn_exp2f(fmaf(s[kb][r], p.scale_log2, -m_run));
          const float e1 = __builtin_amdgcn_exp2f(fmaf(s[kb][r + 1], p.scale_log2, -m_run));
          rsum += e0;
          rsum += e1;
          pw[kb][r >> 1] = Elem<T>::pack(e0, e1);
        }
      l_run = fmaf(l_run, alpha, pair_sum(rsum));
    }
    // ---- O^T += V^T . P^T: keys 0..31 on the fragments read during QK^T, the fragments of keys 32..63 read under them
    if constexpr (!(ABL & 8)) {
      auto pack_p = [&](int kb, int half) {
        U4 pf;
        pf.x = pw[kb][4 * half];
        pf.y = pw[kb][4 * half + 1];
        pf.z = pw[kb][4 * half + 2];
        pf.w = pw[kb][4 * half + 3];
        return pf;
      };
      U4 vfb[8];
      const U4 p00 = pack_p(0, 0), p01 = pack_p(0, 1);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (kPrioMatrix) __builtin_amdgcn_s_setprio(1);
      if constexpr (ABL & 32) __builtin_amdgcn_s_setprio(0);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        o[j & 3] = mfma32<T>(vfa[j], (j >> 2) ? p01 : p00, o[j & 3]);
        if (j < 4) {
          vfb[2 * j] = read_vf(1, (2 * j) >> 2, (2 * j) & 3);
          vfb[2 * j + 1] = read_vf(1, (2 * j + 1) >> 2, (2 * j + 1) & 3);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      const U4 p10 = pack_p(1, 0), p11 = pack_p(1, 1);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j & 3] = mfma32<T>(vfb[j], (j >> 2) ? p11 : p10, o[j & 3]);
      if constexpr (kPrioMatrix) __builtin_amdgcn_s_setprio(0);
    } else {
      o[0][0] += s[0][3] + s[1][7];
    }
  };

  if (t0 < ntiles) {
    load_slots(t0);
    issue_dma(lds_a);
    if (own_pieces && t0 + 1 < ntiles) load_slots(t0 + 1);
  }
  if (!own_pieces) {
    // Q's rows by the DMA path too, into the image that is free until the first tile's barrier, a wave's own 32: whole rows, where a load of a
    // lane's own pieces touches 32 rows.  (With two heads the image would hold half of them.)  Tiles of few rows have few to touch, and the way
    // through LDS and back is 0.4 us of a workgroup: not where it is all of a launch's time.
    char* mine = lds_b + wave * 8192;
    if (left > 0) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int r = 4 * i + (lane >> 4), q_row = min(q0 + rows * 32 + r, q_len - 1);
        __builtin_amdgcn_global_load_lds((glb_void_t*)(p.q + (int64_t)(q_begin + q_row) * p.q_stride + (int64_t)hq * kD + (((lane & 15) ^ (r & 15)) << 3)),
                                         (lds_void_t*)(mine + i * 1024), 16, 0, 0);
      }
    }
    if (t0 + 1 < ntiles) load_slots(t0 + 1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qf[ks] = *reinterpret_cast<const U4*>(mine + (lane & 31) * 256 + (((2 * ks + hi) ^ (lane & 15)) << 4));
  }
  constexpr int kSlots = FRESH ? kQTile / kApart : 1;
  const bool stores = FRESH && job.hq % p.group == 0;  // a kv head's first head
  int slot[kSlots];
  if (stores) {
#pragma unroll
    for (int i = 0; i < kSlots; ++i) slot[i] = p.out_loc[q_begin + min(q0 + st_row + kApart * i, q_len - 1)];
  }
  for (int kt = t0; kt < ntiles; kt += 2) {
    tile_body(std::integral_constant<int, 0>{}, kt);
    if (kt + 1 < ntiles) tile_body(std::integral_constant<int, 1>{}, kt + 1);
  }

  if (stores) {  // q0 is a multiple of two tiles: its first one is in lds_a
    uint16_t *k_to = p.k_pool + (int64_t)kvh * p.kv_stride_head + (lane & 15) * 8, *v_to = p.v_pool + (int64_t)kvh * p.kv_stride_head + (lane & 15) * 8;
#pragma unroll
    for (int i = 0; i < kSlots; ++i) {
      const int r = st_row + kApart * (i & (kTurns - 1));  // of the image
      const char* img = (i < kTurns ? lds_a : lds_b) + r * 256;
      if (q0 + st_row + kApart * i < q_len) {
        const int64_t at = slot_offset(slot[i], p.kv_stride_tok);
        store_past(k_to + at, img + (((lane & 15) ^ (r & 15)) << 4));
        store_past(v_to + at, img + kTileBytes + (((lane & 15) ^ ((r & 3) << 2)) << 4));
      }
    }
    __syncthreads();  // the images are read
  }
  if (RANGES && all_tiles > p.run) {
    const int64_t at = ((int64_t)blockIdx.y * total_tiles * p.hq + (int64_t)tile * p.hq + hq) * 4 + rows;
    f32x4p* po = reinterpret_cast<f32x4p*>(p.part_o) + at * 1024 + lane;  // [16 pieces][64 lanes]
#pragma unroll
    for (int i = 0; i < 16; ++i)
      po[i * 64] = f32x4p{o[i >> 2][4 * (i & 3)], o[i >> 2][4 * (i & 3) + 1], o[i >> 2][4 * (i & 3) + 2], o[i >> 2][4 * (i & 3) + 3]};
    *reinterpret_cast<float2*>(p.part_ml + (at * 64 + lane) * 2) = make_float2(m_run, l_run);
    return;
  }
  const float inv = 1.0f / l_run;
  auto piece = [&](int nb, int rg) __attribute__((always_inline)) {  // columns 32 nb + 8 rg + 4 hi .. + 3 of the lane's row
    return uint2{Elem<T>::pack(o[nb][4 * rg] * inv, o[nb][4 * rg + 1] * inv), Elem<T>::pack(o[nb][4 * rg + 2] * inv, o[nb][4 * rg + 3] * inv)};
  };
  if (HEADS == 1 && left <= 0) return;
  if (!own_pieces) {
    // Outputs by way of the image that does not hold the last tile (everyone is done with it), a wave's rows in its own part: whole rows of 256
    // bytes leave it, where a lane's own pieces are 16 bytes of 32 rows a store.  16-byte pieces change places by the row's number.  Nobody reads them in this
    // launch: past the L2, which keeps keys and values (40 heads on 8, with store_kv_kernel: 29 requests of 100 - 1024 217 -> 214 us, 60 of 128 - 256
    // 111 -> 99; 64 on 8 332 -> 328 and 160 -> 155; one of 8192 the same.  Q's copies past it too: 99 -> 105).
    char* turn = (((ntiles - t0) & 1) ? lds_b : lds_a) + wave * 8192;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg)
        *reinterpret_cast<uint2*>(turn + (lane & 31) * 256 + (((nb * 4 + rg) ^ (lane & 15)) << 4) + 8 * hi) = piece(nb, rg);
    asm volatile("" ::: "memory");  // a wave's own part: its LDS operations keep their order
    uint16_t* op = p.out + (int64_t)(q_begin + q0 + rows * 32) * p.out_stride + (int64_t)hq * kD + (lane & 31) * 4;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = 2 * i + hi;
      const uint2 w = *reinterpret_cast<const uint2*>(turn + r * 256 + ((((lane & 31) >> 1) ^ (r & 15)) << 4) + 8 * (lane & 1));
      if (r < left) __builtin_nontemporal_store(__builtin_bit_cast(uint64_t, w), reinterpret_cast<uint64_t*>(op + (int64_t)r * p.out_stride));
    }
  } else if (q_valid) {
    uint16_t* op = p.out + (int64_t)(q_begin + my_q) * p.out_stride + (int64_t)hq * kD;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) *reinterpret_cast<uint2*>(op + nb * 32 + 8 * rg + 4 * hi) = piece(nb, rg);
  }
}

// The ranges of a job: one wave for 32 rows and 32 columns (piece group nb) of one wave of the kernel above, all loads coalesced.
template <typename T>
__global__ __launch_bounds__(64) void attn_prefill_join_kernel(const PrefillParams p, int total_tiles) {
  const int lane = threadIdx.x & 63, hi = lane >> 5;
  const PrefillJob job = prefill_job(p, total_tiles);
  if (job.tile < 0) return;
  const TileRequest rq = find_request(p, job.tile, lane);
  const int q_len = rq.q_end - rq.q_begin, q0 = (job.tile - rq.tile_first) * kQTile;
  const int kend = min(rq.k_len, rq.k_len - q_len + min(q0 + kQTile, q_len));
  const int n = min(((kend + kKTile - 1) / kKTile + p.run - 1) / p.run, p.ranges);
  if (n <= 1) return;
  const int wave = (int)blockIdx.y >> 2, nb = (int)blockIdx.y & 3;
  const int64_t step = (int64_t)total_tiles * p.hq * 4, at0 = ((int64_t)job.tile * p.hq + job.hq) * 4 + wave;
  float m = kNegBigP, l = 0.f;
  f32x4p acc[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) acc[r] = f32x4p{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int z = 0; z < n; ++z) {  // a range without a visible key for the row: weight 0
    const int64_t at = at0 + z * step;
    const float2 st = *reinterpret_cast<const float2*>(p.part_ml + (at * 64 + lane) * 2);
    const f32x4p* po = reinterpret_cast<const f32x4p*>(p.part_o) + at * 1024 + nb * 256 + lane;
    f32x4p x[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = po[r * 64];
    const float mn = fmaxf(m, st.x), w0 = __builtin_amdgcn_exp2f(m - mn), w1 = __builtin_amdgcn_exp2f(st.x - mn);
    m = mn;
    l = fmaf(l, w0, st.y * w1);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[r][e] = fmaf(acc[r][e], w0, x[r][e] * w1);
  }
  const int my_q = q0 + wave * 32 + (lane & 31);
  if (my_q >= q_len) return;
  const float inv = 1.0f / l;
  uint16_t* op = p.out + (int64_t)(rq.q_begin + my_q) * p.out_stride + (int64_t)job.hq * kD + nb * 32 + 4 * hi;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    uint2 w;
    w.x = Elem<T>::pack(acc[r][0] * inv, acc[r][1] * inv);
    w.y = Elem<T>::pack(acc[r][2] * inv, acc[r][3] * inv);
    *reinterpret_cast<uint2*>(op + 8 * r) = w;
  }
}


}  // namespace msgl

using namespace msgl;

extern "C" int msgl_attn_prefill_q_tile(int /*impl*/) { return kQTile; }

// the new rows of a launch that stores them (FRESH)
struct PrefillFresh {
  const void *k, *v;
  int64_t stride;
  const int32_t* out_loc;
};

// ranges > 1: impl 0 with that many key ranges at most, `run` tiles each; fresh: not with ranges
static int prefill(void* out, const void* q, const void* k_cache, const void* v_cache,
                                 const int32_t* page_table, int64_t pt_stride, const int32_t* req_rows,
                                 const int32_t* seq_lens, const int32_t* cu_seqlens_q, const int32_t* tile_cu,
                                 int batch, int total_tiles, int num_q_heads, int num_kv_heads, int head_dim,
                                 int64_t q_stride_tok, int64_t kv_stride_tok, int64_t kv_stride_head,
                                 int64_t out_stride_tok, float sm_scale, int dtype, const int32_t* tile_order,
                                 int impl, int ranges, int run, float* workspace, const PrefillFresh* fresh, void* stream) {
  MSGL_REQUIRE(batch >= 0 && total_tiles >= 0, "attn_prefill: negative sizes");
#ifdef MSGL_PREFILL_DIAG
  MSGL_REQUIRE(impl == 0 || impl == 2 || impl == 4 || impl == 6 || (impl >= 16 && impl < 48) || (impl >= 64 && impl < 128),
               "attn_prefill: impl %d (0 = 4 DMA-staged, 6 with two heads a workgroup, 2 register-staged; diagnostic build: 16 + bits / 64 + bits = ablations)", impl);
#else
  MSGL_REQUIRE(impl == 0 || impl == 2 || impl == 4 || impl == 6,
               "attn_prefill: impl %d (0 = 4 the DMA-staged kernel, 6 with two heads a workgroup, 2 the register-staged kernel; ablation codes need a "
               "-DMSGL_PREFILL_DIAG build)", impl);
#endif
  if (batch == 0 || total_tiles == 0) return MSGL_OK;
  MSGL_REQUIRE(out && q && k_cache && v_cache && page_table && seq_lens && cu_seqlens_q && tile_cu,
               "attn_prefill: null pointer");
  MSGL_REQUIRE(head_dim == 128, "attn_prefill: head_dim %d unsupported (128 only)", head_dim);
  MSGL_REQUIRE(num_kv_heads >= 1 && num_q_heads % num_kv_heads == 0 && num_q_heads <= 65535,
               "attn_prefill: %d q heads / %d kv heads", num_q_heads, num_kv_heads);
  MSGL_REQUIRE(impl != 6 || num_q_heads / num_kv_heads % 2 == 0, "attn_prefill: heads in pairs, %d q heads / %d kv heads", num_q_heads, num_kv_heads);
  MSGL_REQUIRE(kv_stride_tok > 0 && kv_stride_tok < (1ll << 32), "attn_prefill: kv token stride %lld", (long long)kv_stride_tok);
  MSGL_REQUIRE(q_stride_tok % 8 == 0 && kv_stride_tok % 8 == 0 && kv_stride_head % 8 == 0 &&
                   out_stride_tok % 4 == 0,
               "attn_prefill: strides must be multiples of 8 elements");
  MSGL_REQUIRE(aligned16(q) && aligned16(k_cache) && aligned16(v_cache) &&
                   (reinterpret_cast<uintptr_t>(out) & 7u) == 0,
               "attn_prefill: pointers must be 16-byte aligned");
  PrefillParams p{};
  p.q = (const uint16_t*)q;
  p.k = (const uint16_t*)k_cache;
  p.v = (const uint16_t*)v_cache;
  p.page_table = page_table;
  p.req_rows = req_rows;
  p.seq_lens = seq_lens;
  p.cu_q = cu_seqlens_q;
  p.tile_cu = tile_cu;
  p.tile_order = tile_order;
  p.out = (uint16_t*)out;
  p.pt_stride = pt_stride;
  p.q_stride = q_stride_tok;
  p.kv_stride_tok = kv_stride_tok;
  p.kv_stride_head = kv_stride_head;
  p.out_stride = out_stride_tok;
  if (fresh) {
    MSGL_REQUIRE(fresh->k && fresh->v && fresh->out_loc && aligned16(fresh->k) && aligned16(fresh->v) && fresh->stride > 0 && fresh->stride < (1ll << 32) && fresh->stride % 8 == 0,
                 "attn_prefill_fresh: new rows must be 16-byte aligned, stride %lld", (long long)fresh->stride);
    p.k_new = (const uint16_t*)fresh->k;
    p.v_new = (const uint16_t*)fresh->v;
    p.k_pool = (uint16_t*)const_cast<void*>(k_cache);
    p.v_pool = (uint16_t*)const_cast<void*>(v_cache);
    p.out_loc = fresh->out_loc;
    p.new_stride = fresh->stride;
  }
  p.batch = batch;
  p.hq = num_q_heads;
  const int heads = impl == 6 ? 2 : 1;  // of a workgroup
  p.group = num_q_heads / num_kv_heads / heads;
  p.per = num_kv_heads;
  p.share_log2 = 3;
  while (p.share_log2 > 0 && p.per % 2 == 0) {
    p.per /= 2;
    --p.share_log2;
  }
  p.scale_log2 = sm_scale * 1.4426950408889634f;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype != MSGL_BF16 && dtype != MSGL_FP16) {
    set_error("attn_prefill: unsupported dtype code %d", dtype);
    return MSGL_EINVAL;
  }
  if (impl == 0) impl = 4;  // the DMA-staged kernel; impl 2 keeps its predecessor callable (A/B timing, cross-check in tests)
  const int64_t total = (int64_t)total_tiles * (num_q_heads / heads);
  MSGL_REQUIRE(total < (1ll << 30), "attn_prefill: %lld workgroups", (long long)total);
  const int even = (int)(((int64_t)total_tiles * p.group * p.per + (1 << p.share_log2) - 1) >> p.share_log2);
  p.stretch = ranges == 1 && total <= 256 ? even : 0;
  // Waves without rows leave the matrix cores to the others (40 heads on 8, 14 requests of 14 - 41 tokens after 300: 25.7 -> 23.7 us; 64 on 8, 20 of 65 -
  // 187 after 2000 287 -> 259; 29 of 100 - 1024 on 40 heads 229 -> 225).  Not in one and a half rounds: who then ends early takes two of the last
  // workgroups onto one CU (768: 8 of 93 - 218 after 2000 120 -> 132; 740: 83 -> 90; above, none of 100 sizes more than 2.5 % slower).
  const int64_t wanted = total * ranges;
  p.idle = wanted <= 512 || wanted > 768;
  // Where all workgroups start at once the time is one workgroup's, and only full tiles go in whole rows by way of LDS; else from about half a tile on.
  // us, 8 requests of n tokens, own pieces / whole rows: 16 heads on 8 (128 workgroups) of 32 7.5 / 8.3, 64 8.8 / 9.0, 100 10.9 / 11.4, 128 11.8 /
  // 11.9; 40 requests, 40 on 8 (1600): of 20 20.5 / 22.5, 40 26.4 / 27.4, 64 30.8 / 29.9, 100 42.3 / 40.3, 128 48.8 / 43.7; where all four waves stay, 61
  // rows behind full tiles (640) 23.1 / 22.1
  p.few = wanted <= 512 ? kQTile : p.idle ? kQTile / 2 : 48;
  const unsigned blocks = (unsigned)even * 8;
  if (ranges > 1) {
    p.ranges = ranges;
    p.run = run;
    p.part_o = workspace;
    p.part_ml = workspace + total * ranges * kQTile * kD;
    const dim3 grid(blocks, (unsigned)ranges), joins(blocks, 16);
    if (dtype == MSGL_BF16) {
      attn_prefill_dma_kernel<BF16, 0, true><<<grid, dim3(256), 0, s>>>(p, total_tiles);
      attn_prefill_join_kernel<BF16><<<joins, dim3(64), 0, s>>>(p, total_tiles);
    } else {
      attn_prefill_dma_kernel<FP16, 0, true><<<grid, dim3(256), 0, s>>>(p, total_tiles);
      attn_prefill_join_kernel<FP16><<<joins, dim3(64), 0, s>>>(p, total_tiles);
    }
  } else if (fresh) {
    if (dtype == MSGL_BF16) attn_prefill_dma_kernel<BF16, 0, false, 1, true><<<dim3(blocks), dim3(256), 0, s>>>(p, total_tiles);
    else attn_prefill_dma_kernel<FP16, 0, false, 1, true><<<dim3(blocks), dim3(256), 0, s>>>(p, total_tiles);
  } else if (impl == 4) {
    if (dtype == MSGL_BF16) attn_prefill_dma_kernel<BF16><<<dim3(blocks), dim3(256), 0, s>>>(p, total_tiles);
    else attn_prefill_dma_kernel<FP16><<<dim3(blocks), dim3(256), 0, s>>>(p, total_tiles);
  } else if (impl == 6) {
    if (dtype == MSGL_BF16) attn_prefill_dma_kernel<BF16, 0, false, 2><<<dim3(blocks), dim3(512), 0, s>>>(p, total_tiles);
    else attn_prefill_dma_kernel<FP16, 0, false, 2><<<dim3(blocks), dim3(512), 0, s>>>(p, total_tiles);
  } else if (impl == 2) {
    if (dtype == MSGL_BF16) attn_prefill_tr_kernel<BF16><<<dim3(blocks), dim3(256), 0, s>>>(p, total_tiles);
    else attn_prefill_tr_kernel<FP16><<<dim3(blocks), dim3(256), 0, s>>>(p, total_tiles);
  }
#ifdef MSGL_PREFILL_DIAG
  else if (impl >= 64) {  // DMA-staged kernel, ablation bits = impl - 64 (timing only: WRONG results)
    MSGL_REQUIRE(dtype == MSGL_BF16, "attn_prefill: ablations are bf16 only");
#define MSGL_PF_DMA(A) case A: attn_prefill_dma_kernel<BF16, A><<<dim3(blocks), dim3(256), 0, s>>>(p, total_tiles); break
    switch (impl - 64) {
      MSGL_PF_DMA(1); MSGL_PF_DMA(2); MSGL_PF_DMA(4); MSGL_PF_DMA(8); MSGL_PF_DMA(6); MSGL_PF_DMA(12);
      MSGL_PF_DMA(10); MSGL_PF_DMA(14); MSGL_PF_DMA(15); MSGL_PF_DMA(16); MSGL_PF_DMA(32);
      default: set_error("attn_prefill: unknown ablation %d", impl - 64); return MSGL_EINVAL;
    }
#undef MSGL_PF_DMA
  } else {  // register-staged kernel, ablation bits = impl - 16
    MSGL_REQUIRE(dtype == MSGL_BF16, "attn_prefill: ablations are bf16 only");
#define MSGL_PF_ABL(A) case A: attn_prefill_tr_kernel<BF16, true, A><<<dim3(blocks), dim3(256), 0, s>>>(p, total_tiles); break
    switch (impl - 16) {
      MSGL_PF_ABL(1); MSGL_PF_ABL(2); MSGL_PF_ABL(4); MSGL_PF_ABL(8); MSGL_PF_ABL(6); MSGL_PF_ABL(10); MSGL_PF_ABL(12);
      MSGL_PF_ABL(14); MSGL_PF_ABL(15); MSGL_PF_ABL(17); MSGL_PF_ABL(31); MSGL_PF_ABL(16);
      default: set_error("attn_prefill: unknown ablation %d", impl - 16); return MSGL_EINVAL;
    }
#undef MSGL_PF_ABL
  }
#endif
  MSGL_CHECK_LAUNCH("attn_prefill");
  return MSGL_OK;
}

extern "C" int msgl_attn_prefill(void* out, const void* q, const void* k_cache, const void* v_cache, const int32_t* page_table, int64_t pt_stride,
                                       const int32_t* req_rows, const int32_t* seq_lens, const int32_t* cu_seqlens_q, const int32_t* tile_cu,
                                       int batch, int total_tiles, int num_q_heads, int num_kv_heads, int head_dim, int64_t q_stride_tok,
                                       int64_t kv_stride_tok, int64_t kv_stride_head, int64_t out_stride_tok, float sm_scale, int dtype,
                                       const int32_t* tile_order, int impl, void* stream) {
  return prefill(out, q, k_cache, v_cache, page_table, pt_stride, req_rows, seq_lens, cu_seqlens_q, tile_cu, batch, total_tiles, num_q_heads,
                 num_kv_heads, head_dim, q_stride_tok, kv_stride_tok, kv_stride_head, out_stride_tok, sm_scale, dtype, tile_order, impl, 1, 0, nullptr, nullptr, stream);
}

extern "C" int64_t msgl_attn_prefill_ranges_workspace_bytes(int total_tiles, int num_q_heads, int ranges) {
  if (total_tiles < 0 || num_q_heads < 1 || ranges < 1) return MSGL_EINVAL;
  return (int64_t)total_tiles * num_q_heads * ranges * kQTile * (kD + 4) * (int64_t)sizeof(float);  // sums; (m, l) of each lane of a row's pair
}

extern "C" int msgl_attn_prefill_ranges(void* out, const void* q, const void* k_cache, const void* v_cache, const int32_t* page_table, int64_t pt_stride,
                                              const int32_t* req_rows, const int32_t* seq_lens, const int32_t* cu_seqlens_q, const int32_t* tile_cu,
                                              int batch, int total_tiles, int num_q_heads, int num_kv_heads, int head_dim, int64_t q_stride_tok,
                                              int64_t kv_stride_tok, int64_t kv_stride_head, int64_t out_stride_tok, float sm_scale, int dtype,
                                              const int32_t* tile_order, int ranges, int range_tiles, void* workspace, int64_t workspace_bytes, void* stream) {
  MSGL_REQUIRE(ranges >= 2 && ranges <= 64 && range_tiles >= 1, "attn_prefill_ranges: %d ranges of %d tiles", ranges, range_tiles);
  MSGL_REQUIRE(num_q_heads >= 1 && total_tiles >= 0, "attn_prefill_ranges: %d tiles, %d heads", total_tiles, num_q_heads);
  MSGL_REQUIRE(workspace && aligned16(workspace) && workspace_bytes >= msgl_attn_prefill_ranges_workspace_bytes(total_tiles, num_q_heads, ranges),
               "attn_prefill_ranges: workspace of %lld bytes", (long long)workspace_bytes);
  return prefill(out, q, k_cache, v_cache, page_table, pt_stride, req_rows, seq_lens, cu_seqlens_q, tile_cu, batch, total_tiles, num_q_heads,
                 num_kv_heads, head_dim, q_stride_tok, kv_stride_tok, kv_stride_head, out_stride_tok, sm_scale, dtype, tile_order, 0, ranges, range_tiles, (float*)workspace, nullptr, stream);
}

extern "C" int msgl_attn_prefill_fresh(void* out, const void* q, const void* k, const void* v, int64_t kv_stride_new, void* k_cache, void* v_cache,
                                       const int32_t* out_loc, const int32_t* seq_lens, const int32_t* cu_seqlens_q, const int32_t* tile_cu, int batch,
                                       int total_tiles, int num_q_heads, int num_kv_heads, int head_dim, int64_t q_stride_tok, int64_t kv_stride_tok,
                                       int64_t kv_stride_head, int64_t out_stride_tok, float sm_scale, int dtype, const int32_t* tile_order, void* stream) {
  const PrefillFresh fresh{k, v, kv_stride_new, out_loc};
  return prefill(out, q, k_cache, v_cache, out_loc, 0, nullptr, seq_lens, cu_seqlens_q, tile_cu, batch, total_tiles, num_q_heads, num_kv_heads, head_dim,
                 q_stride_tok, kv_stride_tok, kv_stride_head, out_stride_tok, sm_scale, dtype, tile_order, 4, 1, 0, nullptr, &fresh, stream);
}
