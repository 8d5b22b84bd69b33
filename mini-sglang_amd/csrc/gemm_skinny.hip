// Weight-streaming projection GEMM for small decode batches (M <= 64):
//     out[M, N] = x[M, K] . w[N, K]^T        (torch F.linear layout, bf16 / fp16, fp32 accumulate)
//
// At M <= 64 a decode-step projection is a pure stream of the weight matrix (<= 64 flop per weight byte,
// ridge ~312), yet the BLAS library's kernels for these shapes reach only 1.4-4.4 TB/s on gfx950
// (profiles/r01d_gemm_sweep_small_batch.txt: down-projection 118 us for 178 MB at M = 1 .. 64).  This
// kernel is built around the stream instead of around a tile:
//   * a workgroup owns 16 consecutive weight rows; its SL waves split K between them (split-K inside the
//     workgroup: N/16 x SL waves fill the chip even for N = 5120), partial sums meet in LDS once, in a
//     fixed order (deterministic);
//   * weights go HBM -> VGPR directly (no LDS: nothing is shared between waves), 16 B per lane, in exactly
//     the v_mfma_f32_16x16x32 A-operand layout (lane = row l&15, k-group l>>4): a wave load covers
//     16 rows x 64 contiguous bytes and the two loads of a 64-k block complete the 128-B lines;
//   * activations (M x K, L2-resident, read by every workgroup) are the B operand in the same layout,
//     rows clamped to M-1 for the padding columns;
//   * a wave may take NT = 1, 2 or 4 row tiles at once: the activation fragment is then reused NT times
//     from registers (at M = 16, NT = 1 the activation re-reads through L2 -> L1 equal the weight stream);
//   * up to 4 x 64 k per step with all loads issued ahead of the MFMAs; the resident waves hide each
//     other's waits.
// The tuner (model.tune_gemms) times it against the library's best per (M, N, K) and records SL.
//
// SILU (msgl_skinny_gemm_silu_nt): `w` is a gate_up weight whose rows are interleaved in blocks of 32 (ops.interleave_gate_up:
// rows 64 j .. + 31 gate, + 32 .. + 63 up) and out[M, N/2] = silu(gate) * up: a workgroup takes NT/2 gate tiles and the NT/2
// up tiles 32 rows further (or, NT = 1, half of its waves the gate tile and half the up tile), so gate and up of one output
// column meet in one lane's accumulators (in LDS for NT = 1); both are rounded to the
// 16-bit type first, then silu_mul_f32 (common.h) -- bit for bit what msgl_skinny_gemm_nt + msgl_silu_and_mul_interleaved give,
// without the activation launch (~4.7 us of a decode step's ~200 per layer at small batch) and its round trip.
//
// NORM (msgl_skinny_norm_gemm_nt): `x` is the previous projection's output and the operand is fused_add_rmsnorm(x, residual):
// every workgroup normalises the few rows itself (skinny_stage_norm) while its first weight loads are in flight, and the
// norm's launch disappears.  See the banner of that function for the sizes where this pays.
#include <type_traits>

#include "common.h"

namespace msgl {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t W4 __attribute__((ext_vector_type(4)));

template <typename T>
__device__ __forceinline__ f32x4 mfma16(const W4& a, const W4& b, const f32x4& c) {
  if constexpr (std::is_same_v<T, BF16>)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                  0, 0);
}

constexpr int kSkinnyMaxSlices = 16;
// more column / row tiles per wave = more operand registers: the workgroup (hence the register budget per
// wave) shrinks
__host__ __device__ constexpr int skinny_max_slices(int MT, int NT) { return MT * NT <= 2 ? 16 : MT * NT <= 8 ? 8 : 4; }

// ---- fused add + RMSNorm in front of the product, by every workgroup for itself ----
// At M <= 8 rows of a small hidden size the norm is a launch of its own that computes next to nothing: 2.4 us of a captured
// step, in front of projections of 4 - 5 us (8 MB of weights), and nothing of the projection runs beside it.  Here the
// workgroup asks for x, residual and gamma, then for its first weights, and normalises while these are on their way.  Every
// workgroup does the same work again (reads from L2), so the sizes are bounded: at most kNormPieces 16-byte pieces of the
// rows per lane.  Same bits as msgl_fused_add_rmsnorm: rows of up to 128 pieces are added as rmsnorm_kernel<64, 2> adds them
// (a lane's two pieces as one chain), wider ones as rmsnorm_wide_row_kernel does (groups of 64 pieces, added in order).
// Hidden size 1024, us in a captured chain, norm and projection as two launches -> one: qkv (4096 rows) 6.6 -> 4.0 at one row,
// 7.0 -> 4.6 at eight (the projection alone: 3.8, 4.1); gate_up with SiLU.mul (6144 rows) 8.4 -> 5.0, 8.9 -> 6.0.  Where it pays is
// measured per shape (ops.norm_linear_tune): a large grid does the norm once per workgroup.
struct SkinnyNorm {
  const uint16_t* res_in;
  uint16_t* res_out;
  const uint16_t* gamma;
  float eps;
  int64_t ldr_in, ldr_out;
};
constexpr int kNormRows = 8;    // rows of x
constexpr int kNormPieces = 4;  // 16-byte pieces of (x, residual, gamma) a lane holds
constexpr int kNormPad = 32;    // elements between the staged rows beyond K: eight rows' 16-byte reads of one k cover the banks twice
constexpr int kNormLds = 159 * 1024;  // the most dynamic LDS a launch asks for
constexpr int kNormGroups = 16; // 64-piece groups of a row: K <= 8192

__host__ __device__ constexpr int norm_row_groups(int K) { return K <= 1024 ? 1 : (K / 8 + 63) / 64; }

template <typename T, bool WIDE>
struct SkinnyNormStage {
  static constexpr int P = WIDE ? 1 : 2, S = kNormPieces / P;  // pieces of a (row, group) per lane, (row, group) pairs per wave
  U4 xq[S][P], rq[S][P], gq[S][P];

  // (a wave without a pair asks for nothing: at one row of 1024 elements, eleven of twelve requests of sixteen waves)
  __device__ __forceinline__ void request(const SkinnyNorm& p, const uint16_t* x, int64_t ldx, int M, int K, int s, int SL, int lane) {
    const int pieces = K >> 3, groups = norm_row_groups(K);
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const int pair = s + i * SL;
      if (pair < M * groups) {  // the same for a whole wave
        const int m = pair / groups, g = pair - m * groups;
#pragma unroll
        for (int q = 0; q < P; ++q) {
          const int piece = min((g + q) * 64 + lane, pieces - 1);
          xq[i][q] = ldg16(x + (int64_t)m * ldx + piece * 8);
          rq[i][q] = ldg16(p.res_in + (int64_t)m * p.ldr_in + piece * 8);
          gq[i][q] = ldg16(p.gamma + piece * 8);
        }
      }
    }
  }

  // normalised rows into xs (`pitch` elements apart); workgroup 0 (`writer`) stores the new residual
  __device__ __forceinline__ void stage(const SkinnyNorm& p, uint16_t* xs, int pitch, float* sums, int M, int K, int s, int SL, int lane, bool writer) {
    const int pieces = K >> 3, groups = norm_row_groups(K), pairs = M * groups;
    float v[S][P][8];
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const int pair = s + i * SL;
      if (pair < pairs) {  // the same for a whole wave
        const int m = pair / groups, g = pair - m * groups;
        float ss = 0.f;
#pragma unroll
        for (int q = 0; q < P; ++q) {
          const int piece = (g + q) * 64 + lane;
          if (piece < pieces) {
            float rr[8];
            unpack8<T>(xq[i][q], v[i][q]);
            unpack8<T>(rq[i][q], rr);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[i][q][e] += rr[e];
            if (writer) stg16(p.res_out + (int64_t)m * p.ldr_out + piece * 8, pack8<T>(v[i][q]));
#pragma unroll
            for (int e = 0; e < 8; ++e) ss = fmaf(v[i][q][e], v[i][q][e], ss);
          }
        }
        ss = wave_sum(ss);
        if (lane == 0) sums[pair] = ss;
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < S; ++i) {
      const int pair = s + i * SL;
      if (pair < pairs) {
        const int m = pair / groups, g = pair - m * groups;
        float tot = 0.f;
        for (int j = 0; j < groups; ++j) tot += sums[m * groups + j];
        const float inv = rsqrtf(tot / (float)K + p.eps);
#pragma unroll
        for (int q = 0; q < P; ++q) {
          const int piece = (g + q) * 64 + lane;
          if (piece < pieces) {
            float w[8], y[8];
            unpack8<T>(gq[i][q], w);
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] = __fmul_rn(__fmul_rn(v[i][q][e], inv), w[e]);
            *reinterpret_cast<U4*>(xs + (size_t)m * pitch + piece * 8) = pack8<T>(y);
          }
        }
      }
    }
    __syncthreads();
  }
};

// MT = 16-token column tiles (M <= 16 MT), NT = 16-row weight tiles per wave: an activation fragment, read
// from L2 by every wave, is reused for NT weight tiles (at NT = 1 and M = 16 the activation traffic through
// L2 -> L1 equals the weight stream and halves the rate).  blockDim = 64 SL, grid = N / (16 NT),
// dynamic LDS = SL * MT * NT * 64 * 16 bytes (NORM: and behind them the M staged rows of K + kNormPad elements).
// NORM: 0 = x as it is, 1 / 2 = fused_add_rmsnorm(x, residual) of rows of up to 128 pieces / of wider ones.
template <typename T, int MT, int NT, bool SILU = false, int NORM = 0>
__global__ __launch_bounds__(64 * skinny_max_slices(MT, NT)) void skinny_gemm_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, int M, int nblk,
    int64_t ldx, int64_t ldw, int64_t ldo, const SkinnyNorm norm) {
  static_assert(NORM == 0 || MT == 1, "the norm is folded at up to eight rows");
  extern __shared__ f32x4 red[];  // [SL][NT][MT][64]
  const int lane = threadIdx.x & 63;
  const int s = threadIdx.x >> 6;
  const int SL = blockDim.x >> 6;
  const int r = lane & 15, kg = lane >> 4;
  const int blk = (int)blockIdx.x;
  // SILU with NT = 1: the first half of the workgroup's waves streams a gate tile, the second half its up tile (each half
  // splits K among its waves): one tile per wave, as the plain kernel at its fastest setting, and the pair still meets in LDS
  constexpr bool kSplitPair = SILU && NT == 1;
  const int SLk = kSplitPair ? SL >> 1 : SL;          // waves sharing one k range split
  const int up_half = kSplitPair ? (s >= SLk) : 0;
  const int sk = kSplitPair ? s - up_half * SLk : s;  // this wave's k slice
  // first weight row of the wave; SILU: NT <= 2 -> one 16-row gate tile and its up tile per workgroup, NT = 4 -> a whole 64-row group
  const int64_t n0 = !SILU ? (int64_t)blk * (16 * NT)
                     : NT <= 2 ? (int64_t)(blk >> 1) * 64 + (blk & 1) * 16 + up_half * 32 : (int64_t)blk * 64;
  // this wave's 64-k blocks
  const int b0 = (int)((int64_t)sk * nblk / SLk), b1 = (int)((int64_t)(sk + 1) * nblk / SLk);
  const uint16_t* wp = w + (n0 + r) * ldw + kg * 8;  // row tile i is 16 i rows further
  // row tile i starts 16 i rows further; SILU: the gate tiles first, the up tiles 32 rows behind their gate tile
  auto tile_off = [&](int i) { return (int64_t)(!SILU || NT == 1 ? 16 * i : (i % (NT / 2)) * 16 + (i / (NT / 2)) * 32) * ldw; };
  const uint16_t* xp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) xp[t] = x + (int64_t)min(t * 16 + r, M - 1) * ldx + kg * 8;

  // NORM: the rows' pieces are asked for first, then the first weights (loads return in order: the norm waits for its own
  // only); a wave with fewer blocks than kU asks for its last one again
  constexpr int kU = (NT + MT) <= 2 ? 4 : (NT + MT) <= 5 ? 2 : 1;  // 16-B loads in flight per lane: 2 U (NT + MT)
  W4 first[NORM ? kU : 1][NT][2];
  if constexpr (NORM != 0) {
    __shared__ float sums[kNormRows * kNormGroups];
    uint16_t* xs = reinterpret_cast<uint16_t*>(red + SL * NT * MT * 64);
    const int K = nblk * 64, pitch = K + kNormPad;
    SkinnyNormStage<T, NORM == 2> st;
    st.request(norm, x, ldx, M, K, s, SL, lane);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int64_t k = (int64_t)min(b0 + u, b1 - 1) * 64;
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        first[u][i][0] = *reinterpret_cast<const W4*>(wp + tile_off(i) + k);
        first[u][i][1] = *reinterpret_cast<const W4*>(wp + tile_off(i) + k + 32);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    st.stage(norm, xs, pitch, sums, M, K, s, SL, lane, blockIdx.x == 0);
    xp[0] = xs + (size_t)min(r, M - 1) * pitch + kg * 8;
  }

  f32x4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  // U 64-k blocks per step: all their loads are issued back to back (2 U NT weight + 2 U MT activation
  // loads of 16 B per lane), the MFMAs follow as the data arrives.  No second register set: the other
  // resident waves' loads cover this wave's wait, and straight-line steps keep the compiler's vmcnt
  // bookkeeping exact (a conditional prefetch made it drain the queue every step).
  auto step = [&](int kb, auto u_tag) {
    constexpr int U = decltype(u_tag)::value;
    W4 a[U][NT][2], b[U][MT][2];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t k = (int64_t)(kb + u) * 64;
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        a[u][i][0] = *reinterpret_cast<const W4*>(wp + tile_off(i) + k);
        a[u][i][1] = *reinterpret_cast<const W4*>(wp + tile_off(i) + k + 32);
      }
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        b[u][t][0] = *reinterpret_cast<const W4*>(xp[t] + k);
        b[u][t][1] = *reinterpret_cast<const W4*>(xp[t] + k + 32);
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // keep every load of the step ahead of its MFMAs (the scheduler
                                        // otherwise interleaves them to save registers: 5 loads in flight)
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int i = 0; i < NT; ++i) {
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          acc[i][t] = mfma16<T>(a[u][i][0], b[u][t][0], acc[i][t]);
          acc[i][t] = mfma16<T>(a[u][i][1], b[u][t][1], acc[i][t]);
        }
      }
    }
  };
  int kb = b0;
  if constexpr (NORM != 0) {
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      if (b0 + u < b1) {
        const W4 f0 = *reinterpret_cast<const W4*>(xp[0] + (b0 + u) * 64), f1 = *reinterpret_cast<const W4*>(xp[0] + (b0 + u) * 64 + 32);
#pragma unroll
        for (int i = 0; i < NT; ++i) {
          acc[i][0] = mfma16<T>(first[u][i][0], f0, acc[i][0]);
          acc[i][0] = mfma16<T>(first[u][i][1], f1, acc[i][0]);
        }
      }
    }
    kb = min(b0 + kU, b1);
  }
  for (; kb + kU <= b1; kb += kU) step(kb, std::integral_constant<int, kU>{});
  for (; kb < b1; ++kb) step(kb, std::integral_constant<int, 1>{});

  // split-K partials meet in LDS; wave 0 adds them in slice order and writes 4 consecutive columns per lane
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int t = 0; t < MT; ++t) red[((s * NT + i) * MT + t) * 64 + lane] = acc[i][t];
  __syncthreads();
  auto slice_sum = [&](int i, int t, int j0 = 0, int j1 = -1) {
    if (j1 < 0) j1 = SL;
    f32x4 v = red[((j0 * NT + i) * MT + t) * 64 + lane];
    for (int j = j0 + 1; j < j1; ++j) {
      const f32x4 o = red[((j * NT + i) * MT + t) * 64 + lane];
      v.x += o.x; v.y += o.y; v.z += o.z; v.w += o.w;
    }
    return v;
  };
  if constexpr (SILU) {
    if (s == 0) {
      const int64_t c0 = NT <= 2 ? (int64_t)(blk >> 1) * 32 + (blk & 1) * 16 : (int64_t)blk * 32;
#pragma unroll
      for (int pr = 0; pr < (NT + 1) / 2; ++pr) {
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          const f32x4 g = kSplitPair ? slice_sum(0, t, 0, SLk) : slice_sum(pr, t);
          const f32x4 u = kSplitPair ? slice_sum(0, t, SLk, SL) : slice_sum(pr + NT / 2, t);
          const int m = t * 16 + r;
          if (m < M) {
            // gate and up as the unfused path stores them (rounded to T), then the activation kernel's arithmetic
            const uint32_t g01 = Elem<T>::pack(g.x, g.y), g23 = Elem<T>::pack(g.z, g.w);
            const uint32_t u01 = Elem<T>::pack(u.x, u.y), u23 = Elem<T>::pack(u.z, u.w);
            uint2 pk;
            pk.x = Elem<T>::pack(silu_mul_f32(Elem<T>::lo(g01), Elem<T>::lo(u01)), silu_mul_f32(Elem<T>::hi(g01), Elem<T>::hi(u01)));
            pk.y = Elem<T>::pack(silu_mul_f32(Elem<T>::lo(g23), Elem<T>::lo(u23)), silu_mul_f32(Elem<T>::hi(g23), Elem<T>::hi(u23)));
            *reinterpret_cast<uint2*>(out + (int64_t)m * ldo + c0 + pr * 16 + kg * 4) = pk;
          }
        }
      }
    }
    return;
  }
  if (s == 0) {
#pragma unroll
    for (int i = 0; i < NT; ++i) {
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const f32x4 v = slice_sum(i, t);
        const int m = t * 16 + r;
        if (m < M) {
          uint2 pk;
          pk.x = Elem<T>::pack(v.x, v.y);
          pk.y = Elem<T>::pack(v.z, v.w);
          *reinterpret_cast<uint2*>(out + (int64_t)m * ldo + n0 + i * 16 + kg * 4) = pk;
        }
      }
    }
  }
}

template <typename T, int MT, int NT, bool SILU = false, int NORM = 0>
static int launch_skinny_t(uint16_t* out, const uint16_t* x, const uint16_t* w, int M, int N, int K, int64_t ldx,
                           int64_t ldw, int64_t ldo, int slices, hipStream_t s, const SkinnyNorm& norm = SkinnyNorm{}) {
  if (slices > skinny_max_slices(MT, NT)) {
    set_error("skinny_gemm_nt: at most %d k-slices for M = %d with %d row tiles per wave", skinny_max_slices(MT, NT),
              M, NT);
    return MSGL_EINVAL;
  }
  if (SILU && NT == 1 && (slices & 1)) {
    set_error("skinny_gemm_silu_nt: row_tiles 1 splits the waves between the gate and the up tile: %d k-slices is odd", slices);
    return MSGL_EINVAL;
  }
  const dim3 grid((unsigned)(N / (16 * (SILU && NT == 1 ? 2 : NT)))), block(64 * slices);
  const size_t lds = (size_t)slices * MT * NT * 64 * sizeof(f32x4) + (NORM ? (size_t)M * (K + kNormPad) * 2 : 0);
  auto* kernel = &skinny_gemm_kernel<T, MT, NT, SILU, NORM>;
  if constexpr (NORM != 0) {
    static PerDeviceOnce lds_attr;  // per instantiation and device: more than 64 KB of dynamic LDS has to be requested
    if (lds > 64 * 1024 && !lds_attr.ensure([&] {
          return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kNormLds) == hipSuccess;
        })) {
      set_error("skinny_norm_gemm_nt: cannot reserve %d bytes of LDS: %s", kNormLds, hipGetErrorString(hipGetLastError()));
      return MSGL_ELAUNCH;
    }
  }
  kernel<<<grid, block, lds, s>>>(out, x, w, M, K / 64, ldx, ldw, ldo, norm);
  return MSGL_OK;
}

template <typename T, int NT, bool SILU>
static int launch_skinny_norm(uint16_t* out, const uint16_t* x, const uint16_t* w, int M, int N, int K, int64_t ldx, int64_t ldw,
                              int64_t ldo, int slices, const SkinnyNorm& norm, hipStream_t s) {
  return K <= 1024 ? launch_skinny_t<T, 1, NT, SILU, 1>(out, x, w, M, N, K, ldx, ldw, ldo, slices, s, norm)
                   : launch_skinny_t<T, 1, NT, SILU, 2>(out, x, w, M, N, K, ldx, ldw, ldo, slices, s, norm);
}

template <typename T>
static int launch_skinny_norm(uint16_t* out, const uint16_t* x, const uint16_t* w, int M, int N, int K, int64_t ldx, int64_t ldw,
                              int64_t ldo, int slices, int row_tiles, bool silu, const SkinnyNorm& norm, hipStream_t s) {
  if (silu)
    return row_tiles == 1 ? launch_skinny_norm<T, 1, true>(out, x, w, M, N, K, ldx, ldw, ldo, slices, norm, s)
                          : launch_skinny_norm<T, 2, true>(out, x, w, M, N, K, ldx, ldw, ldo, slices, norm, s);
  return row_tiles == 1 ? launch_skinny_norm<T, 1, false>(out, x, w, M, N, K, ldx, ldw, ldo, slices, norm, s)
                        : launch_skinny_norm<T, 2, false>(out, x, w, M, N, K, ldx, ldw, ldo, slices, norm, s);
}

template <typename T, bool SILU = false>
static int launch_skinny(uint16_t* out, const uint16_t* x, const uint16_t* w, int M, int N, int K, int64_t ldx,
                         int64_t ldw, int64_t ldo, int slices, int row_tiles, hipStream_t s) {
  const int MT = M <= 16 ? 1 : M <= 32 ? 2 : 4;
#define MSGL_SKINNY(MT_, NT_) \
  if (MT == MT_ && row_tiles == NT_) return launch_skinny_t<T, MT_, NT_, SILU>(out, x, w, M, N, K, ldx, ldw, ldo, slices, s)
  MSGL_SKINNY(1, 1); MSGL_SKINNY(2, 1); MSGL_SKINNY(4, 1);
  MSGL_SKINNY(1, 2); MSGL_SKINNY(1, 4);
  MSGL_SKINNY(2, 2); MSGL_SKINNY(2, 4);
  MSGL_SKINNY(4, 2); MSGL_SKINNY(4, 4);
#undef MSGL_SKINNY
  set_error("skinny_gemm_nt: row_tiles %d unsupported (1, 2, 4)", row_tiles);
  return MSGL_EINVAL;
}

// ------------------------------------------------------------------------------------------------------------------
// The same product with FOUR weight rows per workgroup, for M <= 8 and projections of few rows.  Sixteen rows per workgroup
// leave 192 of 256 CUs without one at N = 1024 (output and down projections of a hidden size of 1024: 64 workgroups,
// 4.7 / 5.8 us for 4 / 6 MB).  v_mfma_f32_4x4x4_16b: 16 independent blocks of D[4][4] += A[4][4] . B[4][4] (gemm_rowstream.hip);
// block b takes the b-th 8-k piece of a 128-k unit, lane 4 b + i row i of it: a wave load covers 256 contiguous bytes of four
// rows.  K is split over the SL waves of the workgroup; no ring: a wave has a handful of units, all asked for at once (the
// row-streaming kernel's requests past the end of its window, one cache line for all CUs, cost it 1.5 us here).
// 1024 x 2048 / 1024 x 3072, us in a captured chain, sixteen rows -> four: 4.6 -> 3.4 / 5.8 -> 3.8 at one row of x, 5.4 -> 4.3 /
// 6.8 -> 4.9 at eight; an empty kernel takes 1.6.
// NB = 1 (M <= 4) or 2 column operands.
// ------------------------------------------------------------------------------------------------------------------
template <typename T, int NB>
__global__ __launch_bounds__(1024) void skinny_quarter_gemm_kernel(uint16_t* __restrict__ out, const uint16_t* __restrict__ x,
                                                                   const uint16_t* __restrict__ w, int M, int units, int64_t ldx,
                                                                   int64_t ldw, int64_t ldo) {
  __shared__ f32x4 part[kSkinnyMaxSlices][NB][4];  // [wave][column operand][column j] of four rows
  const int lane = threadIdx.x & 63, s = threadIdx.x >> 6, SL = blockDim.x >> 6;
  const int b = lane >> 2, ij = lane & 3;
  const int u0 = (int)((int64_t)s * units / SL), u1 = (int)((int64_t)(s + 1) * units / SL);
  const uint16_t* wp = w + ((int64_t)blockIdx.x * 4 + ij) * ldw + b * 8;
  const uint16_t* xp[NB];
#pragma unroll
  for (int n = 0; n < NB; ++n) xp[n] = x + (int64_t)min(n * 4 + ij, M - 1) * ldx + b * 8;
  f32x4 acc[NB];
#pragma unroll
  for (int n = 0; n < NB; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto step = [&](int u, auto u_tag) {
    constexpr int U = decltype(u_tag)::value;
    W4 a[U], c[U][NB];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      a[i] = *reinterpret_cast<const W4*>(wp + (int64_t)(u + i) * 128);
#pragma unroll
      for (int n = 0; n < NB; ++n) c[i][n] = *reinterpret_cast<const W4*>(xp[n] + (int64_t)(u + i) * 128);
    }
    __builtin_amdgcn_sched_barrier(0);  // every load of the step ahead of its products
#pragma unroll
    for (int i = 0; i < U; ++i) {
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        acc[n] = mfma444<T>(a[i].x, a[i].y, c[i][n].x, c[i][n].y, acc[n]);
        acc[n] = mfma444<T>(a[i].z, a[i].w, c[i][n].z, c[i][n].w, acc[n]);
      }
    }
  };
  int u = u0;
  for (; u + 4 <= u1; u += 4) step(u, std::integral_constant<int, 4>{});
  if (u + 2 <= u1) {
    step(u, std::integral_constant<int, 2>{});
    u += 2;
  }
  if (u < u1) step(u, std::integral_constant<int, 1>{});
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    f32x4 v = acc[n];
#pragma unroll
    for (int e = 0; e < 4; ++e) {  // the 16 blocks: lanes 4 b + j over b
      float t = v[e];
      t += dpp_mov<0x128>(t);  // row_ror:8
      t += dpp_mov<0x124>(t);  // row_ror:4
      t += __shfl_xor(t, 16, 64);
      t += __shfl_xor(t, 32, 64);
      v[e] = t;
    }
    if (lane < 4) part[s][n][lane] = v;
  }
  __syncthreads();
  if (threadIdx.x < 4 * NB) {  // column m: four consecutive outputs, the waves' sums in wave order
    const int m = threadIdx.x;
    f32x4 v = part[0][m >> 2][m & 3];
    for (int j = 1; j < SL; ++j) {
      const f32x4 o = part[j][m >> 2][m & 3];
      v.x += o.x; v.y += o.y; v.z += o.z; v.w += o.w;
    }
    if (m < M) {
      uint2 pk;
      pk.x = Elem<T>::pack(v.x, v.y);
      pk.y = Elem<T>::pack(v.z, v.w);
      *reinterpret_cast<uint2*>(out + (int64_t)m * ldo + (int64_t)blockIdx.x * 4) = pk;
    }
  }
}

template <typename T>
static void launch_skinny_quarter(uint16_t* out, const uint16_t* x, const uint16_t* w, int M, int N, int K, int64_t ldx, int64_t ldw,
                                  int64_t ldo, int slices, hipStream_t s) {
  const dim3 grid((unsigned)(N / 4)), block(64 * slices);
  if (M <= 4) skinny_quarter_gemm_kernel<T, 1><<<grid, block, 0, s>>>(out, x, w, M, K / 128, ldx, ldw, ldo);
  else skinny_quarter_gemm_kernel<T, 2><<<grid, block, 0, s>>>(out, x, w, M, K / 128, ldx, ldw, ldo);
}

}  // namespace msgl

using namespace msgl;

extern "C" int msgl_skinny_gemm_nt(void* out, const void* x, const void* w, int M, int N, int K, int64_t ldx,
                                   int64_t ldw, int64_t ldo, int dtype, int slices, int row_tiles, void* stream) {
  MSGL_REQUIRE(out && x && w, "skinny_gemm_nt: null pointer");
  MSGL_REQUIRE(M >= 1 && M <= 64, "skinny_gemm_nt: M = %d outside [1, 64]", M);
  MSGL_REQUIRE(row_tiles == 1 || row_tiles == 2 || row_tiles == 4, "skinny_gemm_nt: row_tiles %d (1, 2, 4)", row_tiles);
  MSGL_REQUIRE(N >= 16 * row_tiles && N % (16 * row_tiles) == 0,
               "skinny_gemm_nt: N = %d must be a multiple of %d", N, 16 * row_tiles);
  MSGL_REQUIRE(K >= 64 && K % 64 == 0, "skinny_gemm_nt: K = %d must be a multiple of 64", K);
  MSGL_REQUIRE(slices >= 1 && slices <= kSkinnyMaxSlices && slices <= K / 64,
               "skinny_gemm_nt: %d k-slices outside [1, min(%d, K/64)]", slices, kSkinnyMaxSlices);
  MSGL_REQUIRE(ldx >= K && ldw >= K && ldo >= N && ldx % 8 == 0 && ldw % 8 == 0 && ldo % 4 == 0,
               "skinny_gemm_nt: leading dimensions (%lld, %lld, %lld)", (long long)ldx, (long long)ldw,
               (long long)ldo);
  MSGL_REQUIRE(aligned16(x) && aligned16(w) && (reinterpret_cast<uintptr_t>(out) & 7u) == 0,
               "skinny_gemm_nt: x, w must be 16-byte and out 8-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  int rc;
  if (dtype == MSGL_BF16)
    rc = launch_skinny<BF16>((uint16_t*)out, (const uint16_t*)x, (const uint16_t*)w, M, N, K, ldx, ldw, ldo, slices, row_tiles, s);
  else if (dtype == MSGL_FP16)
    rc = launch_skinny<FP16>((uint16_t*)out, (const uint16_t*)x, (const uint16_t*)w, M, N, K, ldx, ldw, ldo, slices, row_tiles, s);
  else {
    set_error("skinny_gemm_nt: unsupported dtype code %d", dtype);
    return MSGL_EINVAL;
  }
  if (rc != MSGL_OK) return rc;
  MSGL_CHECK_LAUNCH("skinny_gemm_nt");
  return MSGL_OK;
}

// gate_up projection + SiLU.mul in one launch: w [N, K] with rows in ops.interleave_gate_up order (blocks of 32: gate, up),
// out [M, N / 2].  row_tiles 2 or 4: a wave holds gate and up tiles; row_tiles 1 (slices even): half of the waves stream the
// gate tile, half the up tile, slices / 2 k-slices each.  Same bits as msgl_skinny_gemm_nt (with slices / 2 k-slices for
// row_tiles 1) followed by msgl_silu_and_mul_interleaved.
extern "C" int msgl_skinny_gemm_silu_nt(void* out, const void* x, const void* w, int M, int N, int K, int64_t ldx,
                                        int64_t ldw, int64_t ldo, int dtype, int slices, int row_tiles, void* stream) {
  MSGL_REQUIRE(out && x && w, "skinny_gemm_silu_nt: null pointer");
  MSGL_REQUIRE(M >= 1 && M <= 64, "skinny_gemm_silu_nt: M = %d outside [1, 64]", M);
  MSGL_REQUIRE(row_tiles == 1 || row_tiles == 2 || row_tiles == 4, "skinny_gemm_silu_nt: row_tiles %d (1, 2, 4)", row_tiles);
  MSGL_REQUIRE(N >= 64 && N % 64 == 0, "skinny_gemm_silu_nt: N = %d must be a multiple of 64 (gate / up blocks of 32 rows)", N);
  MSGL_REQUIRE(K >= 64 && K % 64 == 0, "skinny_gemm_silu_nt: K = %d must be a multiple of 64", K);
  MSGL_REQUIRE(slices >= 1 && slices <= kSkinnyMaxSlices && (row_tiles == 1 ? slices / 2 : slices) <= K / 64,
               "skinny_gemm_silu_nt: %d k-slices outside [1, min(%d, K/64)]", slices, kSkinnyMaxSlices);
  MSGL_REQUIRE(ldx >= K && ldw >= K && ldo >= N / 2 && ldx % 8 == 0 && ldw % 8 == 0 && ldo % 4 == 0,
               "skinny_gemm_silu_nt: leading dimensions (%lld, %lld, %lld)", (long long)ldx, (long long)ldw, (long long)ldo);
  MSGL_REQUIRE(aligned16(x) && aligned16(w) && (reinterpret_cast<uintptr_t>(out) & 7u) == 0,
               "skinny_gemm_silu_nt: x, w must be 16-byte and out 8-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  int rc;
  if (dtype == MSGL_BF16)
    rc = launch_skinny<BF16, true>((uint16_t*)out, (const uint16_t*)x, (const uint16_t*)w, M, N, K, ldx, ldw, ldo, slices, row_tiles, s);
  else if (dtype == MSGL_FP16)
    rc = launch_skinny<FP16, true>((uint16_t*)out, (const uint16_t*)x, (const uint16_t*)w, M, N, K, ldx, ldw, ldo, slices, row_tiles, s);
  else {
    set_error("skinny_gemm_silu_nt: unsupported dtype code %d", dtype);
    return MSGL_EINVAL;
  }
  if (rc != MSGL_OK) return rc;
  MSGL_CHECK_LAUNCH("skinny_gemm_silu_nt");
  return MSGL_OK;
}

// Four weight rows per workgroup (M <= 8): out[M, N] = x[M, K] . w[N, K]^T, K split over `slices` waves.
extern "C" int msgl_skinny_quarter_gemm_nt(void* out, const void* x, const void* w, int M, int N, int K, int64_t ldx, int64_t ldw,
                                           int64_t ldo, int dtype, int slices, void* stream) {
  MSGL_REQUIRE(out && x && w, "skinny_quarter_gemm_nt: null pointer");
  MSGL_REQUIRE(M >= 1 && M <= 8, "skinny_quarter_gemm_nt: M = %d outside [1, 8]", M);
  MSGL_REQUIRE(N >= 4 && N % 4 == 0, "skinny_quarter_gemm_nt: N = %d must be a multiple of 4", N);
  MSGL_REQUIRE(K >= 128 && K % 128 == 0, "skinny_quarter_gemm_nt: K = %d must be a multiple of 128", K);
  MSGL_REQUIRE(slices >= 1 && slices <= kSkinnyMaxSlices && slices <= K / 128,
               "skinny_quarter_gemm_nt: %d k-slices outside [1, min(%d, K/128)]", slices, kSkinnyMaxSlices);
  MSGL_REQUIRE(ldx >= K && ldw >= K && ldo >= N && ldx % 8 == 0 && ldw % 8 == 0 && ldo % 4 == 0,
               "skinny_quarter_gemm_nt: leading dimensions (%lld, %lld, %lld)", (long long)ldx, (long long)ldw, (long long)ldo);
  MSGL_REQUIRE(aligned16(x) && aligned16(w) && (reinterpret_cast<uintptr_t>(out) & 7u) == 0,
               "skinny_quarter_gemm_nt: x, w must be 16-byte and out 8-byte aligned");
  MSGL_REQUIRE(dtype == MSGL_BF16 || dtype == MSGL_FP16, "skinny_quarter_gemm_nt: unsupported dtype code %d", dtype);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == MSGL_BF16)
    launch_skinny_quarter<BF16>((uint16_t*)out, (const uint16_t*)x, (const uint16_t*)w, M, N, K, ldx, ldw, ldo, slices, s);
  else
    launch_skinny_quarter<FP16>((uint16_t*)out, (const uint16_t*)x, (const uint16_t*)w, M, N, K, ldx, ldw, ldo, slices, s);
  MSGL_CHECK_LAUNCH("skinny_quarter_gemm_nt");
  return MSGL_OK;
}

// nullptr, or why msgl_skinny_norm_gemm_nt does not take the shape
static const char* skinny_norm_refusal(int M, int N, int K, int slices, int row_tiles, int silu) {
  if (M < 1 || M > kNormRows) return "M outside [1, 8]";
  if (row_tiles != 1 && row_tiles != 2) return "row_tiles 1 or 2";
  if (K < 192 || K % 64 || K > 1024 * kNormGroups / 2) return "K must be a multiple of 64 in [192, 8192]";
  if (N < 16 * row_tiles || N % (16 * row_tiles) || (silu && N % 64)) return "N must be a multiple of 16 row_tiles (silu: of 64)";
  const int waves_k = silu && row_tiles == 1 ? slices / 2 : slices;
  if (slices < 1 || slices > kSkinnyMaxSlices || waves_k < 1 || waves_k > K / 64 || (silu && row_tiles == 1 && (slices & 1)))
    return "k-slices outside [1, min(16, K/64)] (silu with one row tile: even)";
  if (M * norm_row_groups(K) > slices * (K <= 1024 ? kNormPieces / 2 : kNormPieces)) return "more of the rows than the workgroup's lanes hold";
  if ((int64_t)slices * row_tiles * 1024 + (int64_t)M * (K + kNormPad) * 2 > kNormLds) return "the rows do not fit the CU's LDS";
  return nullptr;
}

extern "C" int msgl_skinny_norm_gemm_supported(int M, int N, int K, int slices, int row_tiles, int silu) {
  return skinny_norm_refusal(M, N, K, slices, row_tiles, silu) == nullptr;
}

// fused_add_rmsnorm(x, res_in) (new residual to res_out) and the projection of its result -- with silu: and SiLU.mul, w in
// ops.interleave_gate_up order, out [M, N / 2] -- in one launch.  Same bits as the two (three) launches.
extern "C" int msgl_skinny_norm_gemm_nt(void* out, const void* x, const void* w, int M, int N, int K, int64_t ldx, int64_t ldw,
                                        int64_t ldo, int dtype, int slices, int row_tiles, int silu, const void* res_in, void* res_out,
                                        const void* gamma, float eps, int64_t ldr_in, int64_t ldr_out, void* stream) {
  MSGL_REQUIRE(out && x && w && res_in && res_out && gamma, "skinny_norm_gemm_nt: null pointer");
  const char* why = skinny_norm_refusal(M, N, K, slices, row_tiles, silu);
  MSGL_REQUIRE(why == nullptr, "skinny_norm_gemm_nt: M = %d, N = %d, K = %d, %d k-slices, %d row tiles: %s", M, N, K, slices, row_tiles, why);
  MSGL_REQUIRE(ldx >= K && ldw >= K && ldo >= (silu ? N / 2 : N) && ldx % 8 == 0 && ldw % 8 == 0 && ldo % 4 == 0 && ldr_in >= K &&
                   ldr_out >= K && ldr_in % 8 == 0 && ldr_out % 8 == 0,
               "skinny_norm_gemm_nt: leading dimensions (%lld, %lld, %lld, %lld, %lld)", (long long)ldx, (long long)ldw, (long long)ldo,
               (long long)ldr_in, (long long)ldr_out);
  MSGL_REQUIRE(aligned16(x) && aligned16(w) && aligned16(res_in) && aligned16(res_out) && aligned16(gamma) &&
                   (reinterpret_cast<uintptr_t>(out) & 7u) == 0,
               "skinny_norm_gemm_nt: x, w, residuals and gamma must be 16-byte and out 8-byte aligned");
  MSGL_REQUIRE(res_in != res_out && res_out != x && out != x && out != res_in,
               "skinny_norm_gemm_nt: neither result may alias x or res_in (the other workgroups are still reading them)");
  MSGL_REQUIRE(dtype == MSGL_BF16 || dtype == MSGL_FP16, "skinny_norm_gemm_nt: unsupported dtype code %d", dtype);
  const SkinnyNorm norm{(const uint16_t*)res_in, (uint16_t*)res_out, (const uint16_t*)gamma, eps, ldr_in, ldr_out};
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int rc = dtype == MSGL_BF16 ? launch_skinny_norm<BF16>((uint16_t*)out, (const uint16_t*)x, (const uint16_t*)w, M, N, K, ldx, ldw, ldo,
                                                               slices, row_tiles, silu != 0, norm, s)
                                    : launch_skinny_norm<FP16>((uint16_t*)out, (const uint16_t*)x, (const uint16_t*)w, M, N, K, ldx, ldw, ldo,
                                                               slices, row_tiles, silu != 0, norm, s);
  if (rc != MSGL_OK) return rc;
  MSGL_CHECK_LAUNCH("skinny_norm_gemm_nt");
  return MSGL_OK;
}
