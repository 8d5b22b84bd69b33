// Grouped / segmented / gathered C = act(A B^T), both operands bf16, all rows in 16-byte pieces: the expert layers and per-head products of
// msgl_mix_gemm_nt.  seqmix.hip keeps the kernels for fp32 operands, unaligned rows and odd K.
//
// Both operands come to LDS by DMA in k steps of KS = 64 (32 where K is no multiple of 64), ST stages in a ring, one barrier a step.  A DMA
// writes its 64 lanes' pieces one after the other, so a row's pieces change places by the row's number when they are fetched: 16 rows'
// fragment reads then touch every bank once.  The rows of B go to the MFMA's rows in an order that leaves a lane eight neighbouring columns
// of two tiles: 16-byte stores.
// An output element's k order is that of the other matrix-core kernel, ascending in blocks of 32, wherever its row lies: the same bits.
#include "mix_common.h"

namespace {

typedef __attribute__((address_space(1))) void glb_void_t;
typedef __attribute__((address_space(3))) void lds_void_t;

// The length of the list of row tiles, group by group.
template <int MT>
__device__ __forceinline__ int count_tiles(const int* __restrict__ seg, int groups, int M) {
  if (!seg) return groups * ((M + MT - 1) / MT);
  int n = 0;
  for (int g = threadIdx.x & 63; g < groups; g += 64) n += (seg[g + 1] - seg[g] + MT - 1) / MT;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) n += __shfl_xor(n, o, 64);
  return __builtin_amdgcn_readfirstlane(n);
}

// What bounds it: for long segments the rows' way to LDS (256 x 256 tiles: 64 KB for 2048 cycles of the matrix cores, at 8 TB/s in all, four
// fifths of what a large library product draws) and tiles that the last round of CUs and the segments' ends leave empty; for short ones the
// way of B from memory.  k steps of 64 are whole cache lines of both operands: with steps of 32 and twice the stages the same tiles are
// a quarter slower.
//   64 experts x 768 rows, N 1024, K 2048: 539 -> 265 us (777 TFLOP/s); 64 x 3 rows: 123 -> 96 us (268 MB of weights)
//   MT x NT = 256 x 256, 8 waves of 64 x 128   long segments
//             128 x 128, 4 waves of 64 x 64    middling ones: two workgroups a CU
//              64 x 128, 4 waves of 64 x 32    short ones: the ring holds 2 x 2 x 16 KB of B per CU under way
//              32 x 128, 4 waves of 32 x 32    a decode step's few rows: less of A beside B, 2 x 3 x 16 KB of B under way
// STREAM: B passes by the caches (one row tile reads it).  64 x 3 rows, N 1024, K 2048 and N 2048, K 512: 53.6 and 25.5 us, 32-row tiles
// 50.4 and 25.2, streaming 46.7 and 21.3 (5.7 and 6.3 TB/s); 32 x 256 tiles 56 and 24.5, a stage less 53 and 24.8, one more 55 and 30.
template <typename TC, int MT, int NT, int W, int WR, int KS, int ST, bool STREAM = false>
__global__ __launch_bounds__(64 * W, 2) void gemm_nt_dma_kernel(TC* __restrict__ C, const bf16_t* __restrict__ A, const bf16_t* __restrict__ Bm, int M,
                                                             int N, int K, int64_t lda, int64_t ldb, int64_t ldc, int groups, int64_t a_gs,
                                                             int64_t b_gs, int64_t c_gs, const int* __restrict__ seg,
                                                             const int* __restrict__ a_rows, int a_div, const int* __restrict__ c_rows, int act) {
  constexpr int WC = W / WR, TI = MT / WR / 16, TJ = NT / WC / 16;  // waves by rows x columns; a wave's 16 x 16 tiles
  constexpr int ROW = KS * 2, LPR = KS / 8, RPI = 64 / LPR;  // bytes of a row in LDS; lanes (pieces) of a row, rows of a DMA instruction
  constexpr int STAGE = (MT + NT) * ROW, UA = MT / RPI / W, UB = NT / RPI / W, U = UA + UB;  // bytes; DMA instructions of a wave and step
  static_assert((KS == 32 || KS == 64) && MT % (W * RPI) == 0 && NT % (W * RPI) == 0 && TJ % 2 == 0, "tiles");
  extern __shared__ __attribute__((aligned(1024))) char ring[];  // [ST][MT rows of A | NT rows of B][KS]
  const int n_cols = (N + NT - 1) / NT, total = count_tiles<MT>(seg, groups, M) * n_cols;
  // neighbours in the list share rows of A or B: a run of them to each XCD
  const int per = (total + 7) / 8, t = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || t >= total) return;
  const int rt = t / n_cols, n0 = (t - rt * n_cols) * NT;
  int g, m0, row0 = 0, rows = M;
  if (seg) {
    g = find_group_wave(seg, groups, MT, rt, &m0);
    row0 = seg[g];
    rows = seg[g + 1] - row0;
  } else {
    const int each = (M + MT - 1) / MT;
    g = rt / each;
    m0 = (rt - g * each) * MT;
  }
  const bf16_t* Ag = A + (seg ? 0 : g * a_gs);
  const bf16_t* Bg = Bm + g * b_gs;
  TC* Cg = C + (seg ? 0 : g * c_gs);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lr = lane & 15, lg = lane >> 4;
  const int wm = wave / WC * (MT / WR), wn = wave % WC * (NT / WC);
  // instruction u of this wave: LPR lanes a row; rows past the end read the last one (never stored).  A row's piece p lies at place p ^ key.
  const auto a_key = [](int r) { return KS == 32 ? (r >> 2) & 3 : (r >> 1) & 7; };
  const auto b_key = [](int r) { return KS == 32 ? (r >> 3) & 3 : ((r >> 1) & 1) | ((r >> 2) & 6); };
  const char* src[U];
#pragma unroll
  for (int u = 0; u < UA; ++u) {
    const int r = RPI * (wave + W * u) + lane / LPR, m = row0 + min(m0 + r, rows - 1);
    src[u] = reinterpret_cast<const char*>(Ag + (int64_t)(a_rows ? a_rows[m] / a_div : m) * lda) + ((lane & (LPR - 1)) ^ a_key(r)) * 16;
  }
#pragma unroll
  for (int u = 0; u < UB; ++u) {
    const int r = RPI * (wave + W * u) + lane / LPR;
    src[UA + u] = reinterpret_cast<const char*>(Bg + (int64_t)min(n0 + r, N - 1) * ldb) + ((lane & (LPR - 1)) ^ b_key(r)) * 16;
  }
  auto dma = [&](int stage) {
    char* dst = ring + stage * STAGE + wave * 1024;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      constexpr int kNonTemporal = 2;
      if (STREAM && u >= UA)
        __builtin_amdgcn_global_load_lds((glb_void_t*)src[u], (lds_void_t*)(dst + MT * ROW + (u - UA) * W * 1024), 16, 0, kNonTemporal);
      else
        __builtin_amdgcn_global_load_lds((glb_void_t*)src[u], (lds_void_t*)(dst + (u < UA ? u * W * 1024 : MT * ROW + (u - UA) * W * 1024)), 16, 0, 0);
      src[u] += ROW;
    }
  };
  f32x4_t acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const bool live = m0 + wm < rows;  // this wave has rows
  const int n_steps = K / KS;
  int a_off[KS / 32], b_off[KS / 32];  // for each block of 32 of the step
#pragma unroll
  for (int kb = 0; kb < KS / 32; ++kb) {
    const int bn = 8 * (lr >> 2) + (lr & 3);  // + 4: the pair's second tile (the same key)
    a_off[kb] = (wm + lr) * ROW + ((4 * kb + lg) ^ a_key(lr)) * 16;
    b_off[kb] = (MT + wn + bn) * ROW + ((4 * kb + lg) ^ b_key(bn)) * 16;
  }
  int at = 0;
  if constexpr (MT <= 64 && KS == 64) {
    // Short segments, few products: the fragments' reads are what is left to hide.  A step's two blocks of 32 take turns, each block's fragments
    // are read before the other one's products, and the barrier lies between them: by then the step has been read by everybody, its stage takes
    // a later one.  (64 x 3 rows, N 1024, K 2048: 100 -> 96 us, 16 x 62, N 1536, K 1024: 24.8 -> 22.8; larger tiles are 1 - 3 % slower this way.)
    bf16x8_t fa[2][TI], fb[2][TJ];
    auto read = [&](int kb) __attribute__((always_inline)) {
      const char* buf = ring + at * STAGE;
#pragma unroll
      for (int i = 0; i < TI; ++i) fa[kb][i] = *reinterpret_cast<const bf16x8_t*>(buf + a_off[kb] + i * 16 * ROW);
#pragma unroll
      for (int j = 0; j < TJ; ++j) fb[kb][j] = *reinterpret_cast<const bf16x8_t*>(buf + b_off[kb] + (j >> 1) * 32 * ROW + (j & 1) * 4 * ROW);
      __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](int kb) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < TJ; ++j)
#pragma unroll
        for (int i = 0; i < TI; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[kb][j], fa[kb][i], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int i = 0; i < ST; ++i)
      if (i < n_steps) dma(i);
    if (n_steps >= ST) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((ST - 1) * U) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    read(0);
#pragma unroll 1
    for (int step = 0; step < n_steps; ++step) {
      asm volatile("" : "+s"(step));       // or the compiler makes copies of the loop for its last steps
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): block 0's fragments, before block 1's are asked for
      read(1);
      multiply(0);
      if (step + ST <= n_steps) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((ST - 2) * U) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (step + ST < n_steps) dma(at);
      at = at == ST - 1 ? 0 : at + 1;
      read(0);  // past the last step: some stage, not used
      multiply(1);
    }
  } else {
#pragma unroll
    for (int i = 0; i < ST - 1; ++i)
      if (i < n_steps) dma(i);
    for (int step = 0; step < n_steps; ++step) {
      // this wave's pieces of the step have come when only those of the later ones are under way (memory counters retire in order)
      if (step + ST - 2 < n_steps) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((ST - 2) * U) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();  // everybody's; everybody done with the stage before
      if (step + ST - 1 < n_steps) dma(at == 0 ? ST - 1 : at - 1);
      if (live) {
        const char* buf = ring + at * STAGE;
#pragma unroll
        for (int kb = 0; kb < KS / 32; ++kb) {
          bf16x8_t fa[TI], fb[TJ];
#pragma unroll
          for (int i = 0; i < TI; ++i) fa[i] = *reinterpret_cast<const bf16x8_t*>(buf + a_off[kb] + i * 16 * ROW);
#pragma unroll
          for (int j = 0; j < TJ; ++j) fb[j] = *reinterpret_cast<const bf16x8_t*>(buf + b_off[kb] + (j >> 1) * 32 * ROW + (j & 1) * 4 * ROW);
#pragma unroll
          for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int i = 0; i < TI; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0);
        }
      }
      at = at == ST - 1 ? 0 : at + 1;
    }
  }
  // lane holds C[m = tile row lr][n = 32 pair + 8 lg .. + 7]
  int at_row[TI];
#pragma unroll
  for (int i = 0; i < TI; ++i) {
    const int m = row0 + min(m0 + wm + i * 16 + lr, rows - 1);
    at_row[i] = c_rows ? c_rows[m] : m;
  }
#pragma unroll
  for (int i = 0; i < TI; ++i) {
    if (m0 + wm + i * 16 + lr >= rows) continue;
    TC* row = Cg + (int64_t)at_row[i] * ldc;
#pragma unroll
    for (int p = 0; p < TJ / 2; ++p) {
      const int n = n0 + wn + 32 * p + 8 * lg;
      float v[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        v[c] = acc[i][2 * p + (c >> 2)][c & 3];
        if (act == MSGL_MIX_ACT_RELU2) {
          v[c] = fmaxf(v[c], 0.f);
          v[c] = v[c] * v[c];
        }
      }
      if (n >= N) continue;
      if constexpr (sizeof(TC) == 2) {
        *reinterpret_cast<Q4*>(row + n) = Q4{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7])};
      } else {
        *reinterpret_cast<float4*>(row + n) = float4{v[0], v[1], v[2], v[3]};
        *reinterpret_cast<float4*>(row + n + 4) = float4{v[4], v[5], v[6], v[7]};
      }
    }
  }
}

template <int MT, int NT, int WR, int KS, int ST, bool STREAM = false>
constexpr size_t gemm_lds() {
  return (size_t)ST * (MT + NT) * KS * 2;
}

}  // namespace

// 1: launched; 0: not this kernel's operands (the caller takes the other ones); < 0: an error code.
extern "C" __attribute__((visibility("hidden"))) int mix_gemm_nt_dma(void* C, const void* A, const void* B, int M, int N, int K, int64_t lda, int64_t ldb,
                                                                     int64_t ldc, int groups, int64_t a_gs, int64_t b_gs, int64_t c_gs, const int* seg,
                                                                     const int* a_rows, int a_div, const int* c_rows, int act, int tc, hipStream_t s) {
  const auto al = [](const void* p, int64_t ld, int64_t gs) { return ((uintptr_t)p & 15u) == 0 && ld % 8 == 0 && gs % 8 == 0; };
  if (K % 32 || N % 8 || !al(A, lda, a_gs) || !al(B, ldb, b_gs) || !al(C, ldc, c_gs)) return 0;
  const auto blocks = [&](int mt, int nt) -> int64_t {  // the most tiles there can be, in whole rounds of the XCDs
    const int64_t list = seg ? (int64_t)M / mt + groups : (int64_t)groups * ((M + mt - 1) / mt);
    return (list * ((N + nt - 1) / nt) + 7) / 8 * 8;
  };
#define GEMM_RUN(TC, MT, NT, W, ...)                                                                                                  \
  {                                                                                                                                   \
    const auto kernel = gemm_nt_dma_kernel<TC, MT, NT, W, __VA_ARGS__>;                                                               \
    constexpr size_t lds = gemm_lds<MT, NT, __VA_ARGS__>();                                                                           \
    const int64_t n = blocks(MT, NT);                                                                                                 \
    if (n > 0x7fffffff) return 0;                                                                                                     \
    MIX_REQUIRE(ensure_lds((const void*)kernel, lds) == 0, "gemm_nt: %zu bytes of LDS", lds);                                         \
    hipLaunchKernelGGL(kernel, dim3((unsigned)n), dim3(64 * W), lds, s, mp<TC>(C), cp<bf16_t>(A), cp<bf16_t>(B), M, N, K, lda, ldb, ldc, groups, \
                       a_gs, b_gs, c_gs, seg, a_rows, a_div, c_rows, act);                                                            \
  }
  // Rows per group on average, and how many of the largest tiles there are.  Groups x rows, N, K (us, weights not in cache):
  //                              64 x 128   128 x 128   256 x 256
  //   16 x 62, 1536, 1024           22.8       26.8        34.8
  //   64 x 64, 1024, 2048            114        105         106
  //   16 x 188, 1536, 1024          37.9       30.9        39.9    96 large tiles: most CUs without one
  //   32 x 188, 1024, 1024          45.2       38.5        43.7
  //   64 x 128, 1024, 2048           134        126         117
  //   16 x 1500, 1024, 768          93.1       72.6        63.0
  //   64 x 768, 1024, 2048           420        304         265
  //   64 x 256, 2048, 512            106       82.1        88.0    (the one of 19 sizes measured where the rule misses by more than 3 %)
  // Groups of uneven length, as a router fills them (random | log-normal, sigma 0.7), where a 256-row tile holds one short group:
  //   64 x 96, 1024, 2048                      72.8 | 90.5   74.7 | 112    32 x 96, 2048, 1024: 29.8 | 43.0   33.8 | 56.7
  //   64 x 112, 1024, 2048                     97.2 | 90.7   76.9 | 114    32 x 128, 2048, 1024: 46.9 | 44.6   36.1 | 57.5
  // Few rows a group, N 1024, K 2048, 64 groups (random | log-normal 0.7 | 1.3): 64-row tiles -> 32-row, B streaming -> 64-row, B streaming
  //   x 4: 61.3 | 53.5 | 47.1 -> 51.5 | 45.5 | 41.3     x 14: 62.8 | 72.8 | 55.5 -> 52.8 | 61.2 | 54.6
  //   x 20: 62.8 | 71.9 | 61.0 -> -> 56.7 | 67.4 | 57.9    x 40: 63.0 | 70.1 | 70.6 -> -> 57.2 | 66.8 | 66.8
  //   x 62: 73.2 | 70.7 | 71.6 -> -> 74.9 | 77.3 | 79.5    (second row tiles read B again)
  // A B that the last cache (256 MB) keeps from one pass to the next loses by streaming, and small ones belong to models that it holds.  Layers in
  // turn that take 200 | 800 MB, us (64-row tiles, and under 16 rows a group 32-row ones; B streaming): the line lies at 64 MB
  //   34 MB (16 x 1024 x 1024)   x 4: 9.3 | 10.5; 10.4 | 10.1     x 14: 9.6 | 11.2; 11.1 | 10.8     x 40: 10.6 | 12.7; 12.4 | 12.4
  //   50 MB (24 x 1024 x 1024)   x 4: 10.8 | 12.3; 11.3 | 11.3    x 20: 11.7 | 13.4; 12.6 | 12.6    x 40: 12.3 | 14.0; 13.1 | 13.2
  //   67 MB (32 x 1024 x 1024)   x 4 (64-row tiles): 13.4 | 15.5; 13.8 | 13.9    x 20: 13.8 | 15.8; 14.0 | 14.4    x 40: 14.6 | 16.3; 14.5 | 15.1
  const int64_t each = seg ? M / groups : M;
  const bool large = each >= 112 && blocks(256, 256) >= 256;
  const bool stream = (int64_t)groups * N * K >= 32 << 20;
#define GEMM_SIZE(TC)                                                   \
  {                                                                     \
    if (K % 64) {                                                       \
      if (each < 64) GEMM_RUN(TC, 64, 128, 4, 1, 32, 6)                 \
      else GEMM_RUN(TC, 128, 128, 4, 2, 32, 4)                          \
    } else if (each < 16) {                                             \
      if (stream) GEMM_RUN(TC, 32, 128, 4, 1, 64, 4, true)              \
      else GEMM_RUN(TC, 32, 128, 4, 1, 64, 4)                           \
    } else if (each < 48 && stream) {                                   \
      GEMM_RUN(TC, 64, 128, 4, 1, 64, 3, true)                          \
    } else if (each < 64) {                                             \
      GEMM_RUN(TC, 64, 128, 4, 1, 64, 3)                                \
    } else if (!large) {                                                \
      GEMM_RUN(TC, 128, 128, 4, 2, 64, 2)                               \
    } else {                                                            \
      GEMM_RUN(TC, 256, 256, 8, 4, 64, 2)                               \
    }                                                                   \
  }
  if (tc == MSGL_MIX_BF16) GEMM_SIZE(bf16_t)
  else GEMM_SIZE(float)
#undef GEMM_SIZE
#undef GEMM_RUN
  MIX_LAUNCHED("gemm_nt (matrix cores, DMA)");
  return 1;
}
