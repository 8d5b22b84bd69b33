// The decoder layers of a small decode batch in ONE launch: every layer's projections, norms, attention and activation by one team of resident
// workgroups that pass rows to each other through memory.
//
// At a handful of rows a layer is a chain of five products over a few MB of weights each.  As launches (add + norm inside the projections,
// qk-norm / RoPE / store inside the attention: six a layer) each of them pays its dispatch, its first memory latency and its tail, 4 - 7 us for 1 - 2.6 us
// of stream.  Here one workgroup per CU stays for all layers, and
//   * WEIGHTS do not wait for rows: a workgroup's share of each of the four products has a region of LDS (123 KB at hidden size 1024), which is refilled
//     by DMA two stages ahead, and goes to registers in front of the wait for the rows; the cache's rows of earlier tokens are there a layer ahead;
//   * ROWS go from everyone to everyone as 8-byte packets {two 16-bit values (or one fp32), number of this launch}: written and read at agent scope
//     (past the L2s, of which each XCD has its own), the number says by itself that the values have arrived: no fence, no flag, no counter.
//     Two packets travel in one aligned 16-byte access, which is no atomic operation of the memory model: what this rests on is that each 8-byte half of it
//     arrives whole, as a lane's aligned 16 bytes are one piece of one request to one line on this device (whether the halves arrive together does not
//     matter: each has its number).  As 8-byte accesses, which are atomic by the model, a step takes 8 % more (1 request of 533 tokens 676 -> 733 us, 8 of 2000
//     1229 -> 1320);
//   * every layer has packets of its own, so none is overwritten before all have read it; and as each stage needs rows of all workgroups, a workgroup that
//     has them knows its own waves done with the stages before: LDS regions need no barriers of their own against being overwritten;
//   * four waves fetch rows (and norm, rotate, stage them), four fetch weights, multiply and attend: a row's request never stands behind a weight's in
//     its own wave.
// The TEAM is who is there: a workgroup counts itself in, and the first one says how many they are, when all have come or after kGatherTicks, and for each
// layer after that until all have: latecomers join at the next layer.  All work is dealt out by the team's size, so that no workgroup ever waits for one
// that is not resident, whatever else runs on the device.
// Rounding points are those of the separate launches (msgl_fused_add_rmsnorm, the projections, msgl_qk_norm_rope_store, msgl_silu_and_mul_interleaved).
//
// Bound: latency.  A hop between 256 workgroups is 1.3 us by itself, there are five in a layer (six where a request's keys are cut into ranges), and 0.6 - 0.8 us of
// dependent instructions in each; the weights' DMAs share the way with the packets and cost 4 us a layer beside them (417 of 521 us for 28 layers
// of Qwen3-0.6B without them).  A decode step of that model, launches -> this: one request of 533 tokens 850 -> 675 us, four 882 -> 765, eight of 2000 1305 -> 1214;
// with a vocabulary of 32768, in an engine of 40960 tokens, one of 32000 1472 -> 1424, four of 16000 2263 -> 2144 (other models: HipAttnBackend.takes_layers).
// A team that misses workgroups has no weights ahead and several turns a product: the launch alone, one request of 533 tokens, takes 602 us with 256, 776 with
// 255, 1028 with 128, 1757 with 64, 18800 with 4, hence the latecomers: a step begun beside a prompt's attention (8192 tokens after 16384, 64 heads on 8, 5.0 ms)
// takes 2.0 ms (2.4 at most) where the team stayed as it began 3.2 (19.9), four requests 2.2 (2.7), 3.6 (25.9).  As launches it ends 0.8 ms behind the prompt's
// kernel, wherever it began; that kernel takes 5.7 - 6.0 ms beside this launch, which holds the compute units' LDS, and 5.0 - 5.3 beside those.
// Measured on the way (28 layers, one request of 16 tokens): a product's columns dealt out to four waves instead of its groups 545 -> 535; DMAs with 256
// cycles between them 521 -> 508; sleeping between two looks at the packets +6; all of a layer's DMAs in the attention's shadow +-0; without arguments
// read ahead, per-stage code and one barrier less 626.  Weights without nt: a step of one request of 533 tokens 676 -> 683, of four 778 -> 793, eight +-0.
#include "attn_decode_tile.h"

namespace msgl {

typedef unsigned long long u64_t;
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(1))) void dl_glb_t;
typedef __attribute__((address_space(3))) void dl_lds_t;

constexpr int kDlFetch = 4;          // waves 4 .. 7 fetch rows; waves 0 .. 3 fetch weights, multiply and attend
constexpr int kDlThreads = 512;
constexpr int kDlPad = 32;           // elements between staged rows beyond K: the rows' 16-byte reads of one column spread over the banks
constexpr int kDlRange = 2;          // 16-token tiles of a wave beyond which a request's keys are cut into (more) ranges
constexpr int kDlRow = 1024;         // columns of qkv's and gate_up's products at most,
constexpr int kDlCols = 4096;        // of the other two's: what of them a wave multiplies is kept in registers
constexpr int kDlUnits = 4;          // groups of four weight rows (gate_up: of four activated columns) of a workgroup, one of o and down
constexpr int kDlMaxLayers = 40;     // their addresses travel as kernel arguments (4 KB)
constexpr int kDlLds = 159 * 1024;   // (and the kernel's own few hundred bytes)
constexpr int kDlPart = 130;         // packets of a (task, head)'s partial sums: 128 values, reference, sum
constexpr u64_t kGatherTicks = 5000;       // 50 us (100 MHz)
// Looks of a wait at its packets, a microsecond or more each, until it gives up: seconds of the workgroup's own running time (a queue that is set aside
// meanwhile does not count).  What did not come is NaN then, as is everything made of it: whoever reads it, the rows of the results and the new keys and
// values among them; and the team's block keeps the launch's number for the host.
constexpr int kLooks = 4000000, kLooksPause = 256;
constexpr uint32_t kNaNs = 0x7fff7fffu;  // two of either type, or one of 32 bits

// words of the team's block, 64 bytes apart: counted in, left, launch number, number of the last launch in which someone gave up, and from kTeamSizes on
// {launch number, size * 2, + 1 where it stays so} of each layer
enum { kTeamCount = 0, kTeamLeft = 16, kTeamEpoch = 32, kTeamFailed = 48, kTeamSizes = 64, kTeamWords = kTeamSizes + 2 * kDlMaxLayers };

struct DlLayer {  // device addresses
  u64_t norm[2], w[4], q_norm, k_norm, k_cache, v_cache;  // w: qkv, o, gate_up, down
};
struct DlParams {
  u64_t x, y_in;  // residual stream in, and what is to be added to it first (or 0)
  u64_t y_out, res_out;
  u64_t positions, cos_sin, out_loc, page_table, req_rows, seq_lens;
  u64_t packets, team;
  int64_t pt_stride, kv_stride_tok, kv_stride_head, packets_all;
  int M, H, hq, hkv, inter, layers, ranges, interleaved;
  float eps, scale_log2;
  int layer_packets, at_part;
  int at[5];                          // packets of a layer: qkv, o, activated, down rows; attention's
  int lds_w[4], lds_rows[4];          // regions of LDS: a product's weights and rows
  int lds_images, lds_sums, lds_norms, lds_new;
  int cap[4];                         // units (groups of four rows, gate_up: of four activated columns) that a weight region holds
  int K[4];
  int looks;                          // of a wait until it ends
  DlLayer layer[kDlMaxLayers];
  int absent, most, until;            // workgroup that leaves (-1: none), and size of the team at most in the layers before `until`
};
static_assert(sizeof(DlParams) <= 4096, "kernel arguments");

// The arguments, read again where they are used: held in scalar registers over the whole kernel they do not fit (326 spilled)
typedef const __attribute__((address_space(4))) DlParams* dl_args_t;
__device__ __forceinline__ dl_args_t dl_args() {
  dl_args_t a = (dl_args_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(a));
  return a;
}
// the lane's number, whose derivatives are likewise not to be kept in registers from one stage to the next
__device__ __forceinline__ int dl_lane() {
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));
  return lane;
}
template <typename V>
__device__ __forceinline__ V* dl_ptr(u64_t a) {  // device memory, which the compiler should know
  return (V*)(__attribute__((address_space(1))) V*)a;
}

__device__ __forceinline__ u64_t dl_get(const u64_t* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void dl_put(u64_t* p, uint32_t value, uint32_t epoch) {
  __hip_atomic_store(p, (u64_t)epoch << 32 | value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// LDS is complete, memory requests stay under way
__device__ __forceinline__ void dl_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

struct DlWait {
  int* dead;  // LDS: someone of this workgroup gave up
  uint32_t epoch;

  // false once the wait has to end
  __device__ __forceinline__ bool again(int& spins) const {
    if ((++spins & (kLooksPause - 1)) == 0) {
      if (*(volatile int*)dead) return false;
      if (spins >= dl_args()->looks) {
        *(volatile int*)dead = 1;
        return false;
      }
    }
    return true;
  }
  // N pairs of packets of this lane, all asked for together; at(i): bytes from byte `from` of the packets on
  template <int N, typename AT>
  __device__ __forceinline__ void get(const __amdgpu_buffer_rsrc_t& pk, int from, uint32_t (&v)[2 * N], AT&& at) const {
    V4 q[N];
    int spins = 0;
    for (;;) {
      asm volatile("" ::: "memory");  // read again
#pragma unroll
      for (int i = 0; i < N; ++i) q[i] = __builtin_bit_cast(V4, __builtin_amdgcn_raw_buffer_load_b128(pk, at(i), from, 16));  // sc1: agent scope
      bool ok = true;
#pragma unroll
      for (int i = 0; i < N; ++i) ok &= q[i][1] == epoch && q[i][3] == epoch;
      if (ok) break;
      if (!again(spins)) {  // (in the loop: a step of eight requests of 2000 1230 us with the NaN behind it, 1214 so)
#pragma unroll
        for (int i = 0; i < N; ++i) q[i] = V4{kNaNs, 0, kNaNs, 0};
        break;
      }
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      v[2 * i] = q[i][0];
      v[2 * i + 1] = q[i][2];
    }
  }
};
__device__ __forceinline__ __amdgpu_buffer_rsrc_t dl_rsrc(u64_t at) { return __builtin_amdgcn_make_buffer_rsrc(dl_ptr<u64_t>(at), 0, -1, 0x00027000); }
// two packets
__device__ __forceinline__ void dl_put2(const __amdgpu_buffer_rsrc_t& pk, int from, int at, uint32_t lo, uint32_t hi, uint32_t epoch) {
  __builtin_amdgcn_raw_buffer_store_b128(V4{lo, epoch, hi, epoch}, pk, at, from, 16);
}

__device__ __forceinline__ void dl_dma16(const void* src, char* dst) {  // 16 bytes a lane; dst: lane 0's
  __builtin_amdgcn_global_load_lds((dl_glb_t*)src, (dl_lds_t*)dst, 16, 0, 2);  // nt: nobody reads a weight again
}
__device__ __forceinline__ void dl_fetch_vector(char* dst, const uint16_t* src, int n) {
  const int lane = threadIdx.x & 63;
  for (int i = 0; i < n; i += 512)
    if (i + lane * 8 < n) dl_dma16(src + i + lane * 8, dst + i * 2);
}
// Reads of LDS that know nothing of a DMA under way (the compiler waits for a wave's DMAs in front of every access of LDS: a wave that fetches ahead would
// wait for the next layer's weights); each waits for itself.  The barriers say what is there.  Eight pieces STEP bytes apart
__device__ __forceinline__ uint32_t dl_lds_at(const void* p) { return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p; }
template <int STEP>
__device__ __forceinline__ void dl_read8(V4 (&v)[8], uint32_t at) {
  asm volatile(
      "ds_read_b128 %0, %8\n\tds_read_b128 %1, %8 offset:%9\n\tds_read_b128 %2, %8 offset:%10\n\tds_read_b128 %3, %8 offset:%11\n\t"
      "ds_read_b128 %4, %8 offset:%12\n\tds_read_b128 %5, %8 offset:%13\n\tds_read_b128 %6, %8 offset:%14\n\tds_read_b128 %7, %8 offset:%15\n\ts_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
      : "v"(at), "i"(STEP), "i"(2 * STEP), "i"(3 * STEP), "i"(4 * STEP), "i"(5 * STEP), "i"(6 * STEP), "i"(7 * STEP) : "memory");
}
template <int STEP>
__device__ __forceinline__ void dl_read2(V4 (&v)[2], uint32_t at) {
  asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:%3\n\ts_waitcnt lgkmcnt(0)" : "=&v"(v[0]), "=&v"(v[1]) : "v"(at), "i"(STEP) : "memory");
}
template <int STEP>
__device__ __forceinline__ void dl_read4(f32x4 (&v)[4], uint32_t at) {
  asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:%5\n\tds_read_b128 %2, %4 offset:%6\n\tds_read_b128 %3, %4 offset:%7\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]) : "v"(at), "i"(STEP), "i"(2 * STEP), "i"(3 * STEP) : "memory");
}
__device__ __forceinline__ void dl_write(uint32_t at, const f32x4& v) {
  asm volatile("ds_write_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : : "v"(at), "v"(v) : "memory");
}
// sum over the sixteen blocks of a 4 x 4 x 4 product: lanes with the same low two bits
__device__ __forceinline__ f32x4 dl_over_blocks(f32x4 v) {
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] += dpp_get<0x124>(v[e]);  // row_ror:4
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] += dpp_get<kDppRor8>(v[e]);
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = sum_over_rows(v[e]);
  return v;
}
// the same of four products: sixteen lanes each
__device__ __forceinline__ f32x4 dl_over_blocks(const f32x4& v0, const f32x4& v1, const f32x4& v2, const f32x4& v3) {
  f32x4 x;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    auto halves = [](float a, float b) {  // lanes below 32: a's sum of both halves, the others: b's
      const auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
      const uint32_t w0 = w[0], w1 = w[1];
      return __uint_as_float(w0) + __uint_as_float(w1);
    };
    const auto w = __builtin_amdgcn_permlane16_swap(__float_as_uint(halves(v0[e], v2[e])), __float_as_uint(halves(v1[e], v3[e])), false, false);
    const uint32_t w0 = w[0], w1 = w[1];
    x[e] = __uint_as_float(w0) + __uint_as_float(w1);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) x[e] += dpp_get<0x124>(x[e]);
#pragma unroll
  for (int e = 0; e < 4; ++e) x[e] += dpp_get<kDppRor8>(x[e]);
  return x;
}
__device__ __forceinline__ float dl_wave_sum(float x) { return sum_over_rows(row16_sum(x)); }

// the team of layer l at most, and its size (* 2, + 1 where it stays so) if `have` have come
__device__ __forceinline__ uint32_t dl_most(int l) { return l < dl_args()->until ? min(gridDim.x, (uint32_t)dl_args()->most) : gridDim.x; }
__device__ __forceinline__ int dl_size(uint32_t have, int l) {
  const uint32_t size = min(have, dl_most(l));
  return (int)(2 * size + (size == gridDim.x || l + 1 == dl_args()->layers));
}

template <typename T, int MQ>
__global__ __launch_bounds__(kDlThreads, 2) void decode_layers_kernel(const DlParams) {
  constexpr int D = 128;
  constexpr int kRow = kDlRow / 256;         // pieces of a row of the residual stream: MQ rows a fetching wave
  constexpr int kDlAhead = 2;                // 16-token tiles of a wave in registers, asked for a layer ahead
  extern __shared__ __attribute__((aligned(16))) char lds[];
  __shared__ int s_dead, s_rank, s_size, s_from, s_last;
  __shared__ uint32_t s_epoch;
  __shared__ float2 s_stat[4][8];
  const int lane = threadIdx.x & 63;
  const int wv = sgpr((int)(threadIdx.x >> 6));
  const u64_t t0 = __builtin_amdgcn_s_memrealtime();

  // ---- the team ----
  if (threadIdx.x == 0) {
    uint32_t* team = dl_ptr<uint32_t>(dl_args()->team);
    s_dead = 0;
    const uint32_t before = __hip_atomic_load(team + kTeamEpoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t epoch = before == 0xffffffffu ? 1 : before + 1;
    u64_t* sizes = reinterpret_cast<u64_t*>(team + kTeamSizes);
    int rank = (int)__hip_atomic_fetch_add(team + kTeamCount, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), size = 0, from = 0;
    if (rank == 0) {
      const uint32_t most = dl_most(0);
      uint32_t have = 1;
      while (have < most && __builtin_amdgcn_s_memrealtime() - t0 < kGatherTicks)
        have = __hip_atomic_load(team + kTeamCount, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      size = dl_size(have, 0);
      dl_put(sizes, (uint32_t)size, epoch);
    } else {  // until there is a layer that I am in (the first one is resident)
      int left = dl_args()->looks;
      for (;;) {
        const u64_t v = dl_get(sizes + from);
        if ((uint32_t)(v >> 32) == epoch) {
          size = (int)(uint32_t)v;
          if (rank < size >> 1) break;
          if (size & 1) rank = -1;
          else ++from;
        } else if (--left <= 0) {
          s_dead = 1;
          rank = -1;
        }
        if (rank < 0) break;
      }
    }
    s_rank = rank >= 0 && rank == dl_args()->absent ? -1 : rank;
    s_size = size;
    s_from = from;
    s_epoch = epoch;
  }
  __syncthreads();
  const int rank = sgpr(s_rank), from = sgpr(s_from);
  const uint32_t epoch = (uint32_t)sgpr((int)s_epoch);

  if (rank >= 0) {
    const DlWait wait{&s_dead, epoch};
    const int M = dl_args()->M, layers = dl_args()->layers;
    const int f = wv - kDlFetch;  // fetching waves: 0 .. 3
    // my units (groups of four rows, gate_up: of four activated columns) of the products: qkv, o and down, gate_up
    const int qkv_rows = (dl_args()->hq + 2 * dl_args()->hkv) * D;
    int n, first_qkv, count_qkv, first_hid, count_hid, first_act, count_act;
    bool open, ahead;  // the team may grow; all units have a place, and what comes next is asked for ahead, else (a small team) they take turns
    auto first_of = [&](int s) { return s == 0 ? first_qkv : s == 2 ? first_act : first_hid; };
    auto count_of = [&](int s) { return s == 0 ? count_qkv : s == 2 ? count_act : count_hid; };
    auto cap_of = [&](int s) { return dl_args()->cap[s]; };
    auto passes_of = [&](int s) { return ahead ? 1 : max(1, (count_of(s) + cap_of(s) - 1) / cap_of(s)); };
    auto deal = [&](int size) {
      n = size >> 1;
      open = !(size & 1);
      auto bound = [&](int rows, int r) { return (int)((uint32_t)(rows >> 2) * (uint32_t)r / (uint32_t)n); };
      first_qkv = bound(qkv_rows, rank);
      count_qkv = bound(qkv_rows, rank + 1) - first_qkv;
      first_hid = bound(dl_args()->H, rank);
      count_hid = bound(dl_args()->H, rank + 1) - first_hid;
      first_act = bound(dl_args()->inter, rank);
      count_act = bound(dl_args()->inter, rank + 1) - first_act;
      ahead = count_qkv <= cap_of(0) && count_hid <= cap_of(1) && count_act <= cap_of(2);
    };
    deal(sgpr(s_size));
    // between two layers, in front of layer l: true if the team has another size than in the one before, during which a fetching wave has looked
    auto grown = [&](int l) {
      if (!open || l <= from) return false;
      const int size = sgpr(*(volatile int*)&s_size), before = n;
      deal(size);
      return n != before;
    };

    // ---- weights: a wave fetches, keeps and multiplies 128 columns of every 512 of all units ----
    // One 1-KB piece is 128 columns of a group of four rows: 16-byte piece (column c, row r) at (4 c + r) * 16, so that a DMA reads 256 contiguous bytes of
    // each row and lane 4 c + r of the product reads the same 16 bytes.  A group has room for a multiple of eight pieces; a unit's groups (gate_up:
    // gate rows, up rows) follow each other.
    auto fetch = [&](int s, int l, int first, int units) {
      const int lane = dl_lane();
      const dl_args_t p = dl_args();
      const int K = p->K[s], room = (K + 1023) >> 10 << 13, up = p->interleaved ? 32 : p->inter;
      char* dst = lds + p->lds_w[s];
      const uint16_t* w = dl_ptr<const uint16_t>(p->layer[l].w[s]) + (int64_t)(lane & 3) * K + (lane >> 2) * 8;
      for (int u = first; u < first + units; ++u) {
        int64_t row = 4 * u;
        if (s == 2 && p->interleaved) row = (u >> 3) * 64 + (u & 7) * 4;
        for (int h = 0; h < (s == 2 ? 2 : 1); ++h) {
#pragma unroll 1
          for (int c = wv * 128; c < K; c += 512) {
            dl_dma16(w + row * K + c, dst + c * 8);
            __builtin_amdgcn_s_sleep(4);
          }
          row += up;
          dst += room;
        }
      }
    };
    // norm weights, by wave 1: [input H][post H][q 128][k 128]
    auto fetch_norms = [&](int l, int which) {
      const dl_args_t p = dl_args();
      char* norms = lds + p->lds_norms;
      dl_fetch_vector(norms + which * p->H * 2, dl_ptr<const uint16_t>(p->layer[l].norm[which]), p->H);
      if (which == 0 && p->layer[l].q_norm) {
        dl_fetch_vector(norms + p->H * 4, dl_ptr<const uint16_t>(p->layer[l].q_norm), D);
        dl_fetch_vector(norms + p->H * 4 + D * 2, dl_ptr<const uint16_t>(p->layer[l].k_norm), D);
      }
    };
    uint32_t res[MQ][kRow][2];  // fetching wave f: rows f, f + 4 of the residual stream (lane: values 4 lane .. + 3 of each piece)
    // staged rows = norm(res += rows); from: 0 nothing to add, 1 y_in, 2 packets [row][column] from byte `at` on; which of the two norms.  (Pieces past the
    // row's end: its last one again.)
    auto add_norm = [&](int from, const __amdgpu_buffer_rsrc_t& pk, int at, int which) {
      const int lane = dl_lane();
      const dl_args_t p = dl_args();
      const int H = p->H, per_row = H >> 8;
      const char* gamma = lds + p->lds_norms + which * H * 2 + lane * 8;
      char* xs = lds + p->lds_rows[0] + lane * 8;
      const uint16_t* y_in = dl_ptr<const uint16_t>(p->y_in);
      const float eps = p->eps, width = (float)H;
      int pc[kRow];
      uint2 g[kRow];
#pragma unroll
      for (int c = 0; c < kRow; ++c) {
        pc[c] = min(c, per_row - 1);
        g[c] = *reinterpret_cast<const uint2*>(gamma + pc[c] * 512);
      }
      if (f >= M) return;
      uint32_t ys[2 * kRow * MQ];
      if (from == 2) wait.template get<kRow * MQ>(pk, at, ys, [&](int i) { return ((i >= kRow && f + 4 < M ? f + 4 : f) * per_row + pc[i % kRow]) * 1024 + lane * 16; });
#pragma unroll
      for (int q = 0; q < MQ; ++q) {
        const int m = f + 4 * q;
        if (m < M) {  // the same for a whole wave
          uint32_t y[2 * kRow];
          if (from == 2) {
#pragma unroll
            for (int c = 0; c < 2 * kRow; ++c) y[c] = ys[2 * kRow * q + c];
          } else if (from == 1) {
#pragma unroll
            for (int c = 0; c < kRow; ++c) {
              const uint2 w = *reinterpret_cast<const uint2*>(y_in + m * H + pc[c] * 256 + lane * 4);
              y[2 * c] = w.x;
              y[2 * c + 1] = w.y;
            }
          }
          float v[kRow][4], ss = 0.f;
#pragma unroll
          for (int c = 0; c < kRow; ++c) {
            float sc = 0.f;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              float a = Elem<T>::lo(res[q][c][e]), b = Elem<T>::hi(res[q][c][e]);
              if (from) {
                a = Elem<T>::lo(y[2 * c + e]) + a;
                b = Elem<T>::hi(y[2 * c + e]) + b;
                res[q][c][e] = Elem<T>::pack(a, b);
              }
              v[c][2 * e] = a;
              v[c][2 * e + 1] = b;
              sc = fmaf(a, a, sc);
              sc = fmaf(b, b, sc);
            }
            ss += c < per_row ? sc : 0.f;
          }
          const float inv = rsqrtf(dl_wave_sum(ss) / width + eps);
#pragma unroll
          for (int c = 0; c < kRow; ++c) {
            uint2 o;
            o.x = Elem<T>::pack(__fmul_rn(__fmul_rn(v[c][0], inv), Elem<T>::lo(g[c].x)), __fmul_rn(__fmul_rn(v[c][1], inv), Elem<T>::hi(g[c].x)));
            o.y = Elem<T>::pack(__fmul_rn(__fmul_rn(v[c][2], inv), Elem<T>::lo(g[c].y)), __fmul_rn(__fmul_rn(v[c][3], inv), Elem<T>::hi(g[c].y)));
            *reinterpret_cast<uint2*>(xs + m * (H + kDlPad) * 2 + pc[c] * 512) = o;
          }
        }
      }
    };
    // staged rows = K values of each row from packets as they are
    auto take_rows = [&](const __amdgpu_buffer_rsrc_t& pk, int at, int K, int rows_at) {
      const int lane = dl_lane();
      const int per = K >> 8, all = M * per;
      int m = 0, end = per;  // row of the next piece, first piece behind it
      auto some = [&](auto N_, int t) __attribute__((always_inline)) {
        constexpr int N = decltype(N_)::value;
        uint32_t y[2 * N];
        wait.template get<N>(pk, at, y, [&](int j) { return (t + 4 * j < all ? t + 4 * j : t) * 1024 + lane * 16; });
#pragma unroll
        for (int j = 0; j < N; ++j) {
          const int u = t + 4 * j;
          if (u < all) {
            while (u >= end) {
              ++m;
              end += per;
            }
            *reinterpret_cast<uint2*>(lds + rows_at + m * kDlPad * 2 + u * 512 + lane * 8) = make_uint2(y[2 * j], y[2 * j + 1]);
          }
        }
      };
      int t = f;
      if constexpr (MQ == 2)
        for (; t + 16 < all; t += 32) some(std::integral_constant<int, 8>{}, t);
      for (; t < all; t += 16) some(std::integral_constant<int, 4>{}, t);
    };

    // ---- attention: task (request, kv head, range of its keys) ----
    constexpr int W = kDlFetch;  // waves that share a task's tiles
    auto ranges_of = [&](int nt, int R) { return min(R, (nt + W * kDlRange - 1) / (W * kDlRange)); };
    struct Task {
      int b, h, r, nt, active, last, table, loc;  // table: row of the page table; loc: the new token's slot
    };
    struct Tile {
      V4 k[4], v[4];
    };
    auto task_of = [&](int id) {
      const dl_args_t p = dl_args();
      Task t;
      const int R = p->ranges, bh = id / R;
      t.r = id - bh * R;
      t.b = bh / p->hkv;
      t.h = bh - t.b * p->hkv;
      const int S = sgpr(dl_ptr<const int>(p->seq_lens)[t.b]);
      t.nt = (S + 15) >> 4;
      t.active = ranges_of(t.nt, R);
      t.last = S - 1;
      t.table = p->req_rows ? sgpr(dl_ptr<const int>(p->req_rows)[t.b]) : t.b;
      t.loc = sgpr(dl_ptr<const int>(p->out_loc)[t.b]);
      return t;
    };
    auto slot_of = [&](const Task& t, int ti) {
      const int tok = dl_lane() & 15;
      const dl_args_t p = dl_args();
      return dl_ptr<const int>(p->page_table)[(int64_t)t.table * p->pt_stride + min(ti * 16 + tok, t.last)];
    };
    auto load_tile = [&](Tile& d, const Task& t, int l, int slot) {
      const int qd = dl_lane() >> 4;
      const dl_args_t p = dl_args();
      const int64_t head = (int64_t)t.h * p->kv_stride_head, off = (int64_t)slot * p->kv_stride_tok + qd * 8;
      const uint16_t *kc = dl_ptr<const uint16_t>(p->layer[l].k_cache) + head, *vc = dl_ptr<const uint16_t>(p->layer[l].v_cache) + head;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) d.k[kk] = *reinterpret_cast<const V4*>(kc + off + kk * 32);
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) d.v[kk] = *reinterpret_cast<const V4*>(vc + off + kk * 32);
    };
    auto load_ahead = [&](Tile (&pre)[kDlAhead], const Task& t, int l, const int (&slot)[kDlAhead]) {
#pragma unroll
      for (int j = 0; j < kDlAhead; ++j)
        if (t.r * W + wv + j * t.active * W < t.nt) load_tile(pre[j], t, l, slot[j]);
    };
    auto slots_of = [&](const Task& t, int (&slot)[kDlAhead]) {
#pragma unroll
      for (int j = 0; j < kDlAhead; ++j) {
        const int ti = t.r * W + wv + j * t.active * W;
        slot[j] = ti < t.nt ? slot_of(t, ti) : 0;
      }
    };
    // fetching waves: cos and sin of a request's new position (dims 4 (lane & 15) .. + 3)
    auto angles_of = [&](const Task& t, f32x4& c, f32x4& s) {
      const int lane = dl_lane();
      const dl_args_t p = dl_args();
      const float* at = dl_ptr<const float>(p->cos_sin) + (int64_t)dl_ptr<const int>(p->positions)[t.b] * D + (lane & 15) * 4;
      c = *reinterpret_cast<const f32x4*>(at);
      s = *reinterpret_cast<const f32x4*>(at + 64);
    };
    const int tasks = M * dl_args()->hkv * dl_args()->ranges;
    const Task mine = task_of(min(rank, tasks - 1));  // my first one
    const bool works = rank < tasks && mine.r < mine.active;
    // the fetching waves' half: the new rows, norm, rotation, store; then the multiplying waves' sums
    auto attend_rows = [&](const Task& t, int l, const __amdgpu_buffer_rsrc_t& pk, const f32x4& cv, const f32x4& sv) {
      const int lane = dl_lane();
      const dl_args_t p = dl_args();
      const int hkv = p->hkv, hq = p->hq, G = hq / hkv, from = p->at[0] * 8, to = p->at[4] * 8, parts = p->at_part * 8, R = p->ranges;
      char* qbuf = lds + p->lds_new;  // G query heads, the new key, the new value
      const float* sums = reinterpret_cast<const float*>(lds + p->lds_sums);
      const bool normed = p->layer[l].q_norm != 0;
      const char* norms = lds + p->lds_norms + p->H * 4;
      const float eps = p->eps;
      const int half = lane >> 5, gl = lane & 31;  // two rows a wave, four dims a lane
      const bool stores = t.r == (t.nt - 1) % (t.active * W) / W;  // the range of the last tile stores the new rows
      const int64_t store_at = (int64_t)t.loc * p->kv_stride_tok + (int64_t)t.h * p->kv_stride_head + gl * 4;
      uint16_t *kc = dl_ptr<uint16_t>(p->layer[l].k_cache) + store_at, *vc = dl_ptr<uint16_t>(p->layer[l].v_cache) + store_at;
      auto swapped = [&](uint32_t x) {  // of the lane sixteen further or back
        const auto w = __builtin_amdgcn_permlane16_swap(x, x, false, false);
        const uint32_t w0 = w[0], w1 = w[1];
        return lane & 16 ? w0 : w1;
      };
      for (int row0 = 2 * f; row0 < G + 2; row0 += 8) {
        const int row = row0 + half, head = row < G ? t.h * G + row : row == G ? hq + t.h : hq + hkv + t.h;
        if (row < G + 2) {
          uint32_t v[2];
          const int at = (t.b * (hq + 2 * hkv) + head) * 512 + gl * 16;
          const uint2 w = *reinterpret_cast<const uint2*>(norms + (row < G ? 0 : D * 2) + gl * 8);
          wait.template get<1>(pk, from, v, [&](int) { return at; });
          if (row <= G) {
            if (normed) {
              float x[4] = {Elem<T>::lo(v[0]), Elem<T>::hi(v[0]), Elem<T>::lo(v[1]), Elem<T>::hi(v[1])};
              float ss = row16_sum(fmaf(x[3], x[3], fmaf(x[2], x[2], fmaf(x[1], x[1], x[0] * x[0]))));
              ss += __uint_as_float(swapped(__float_as_uint(ss)));
              const float inv = rsqrtf(ss / (float)D + eps);
              v[0] = Elem<T>::pack(__fmul_rn(__fmul_rn(x[0], inv), Elem<T>::lo(w.x)), __fmul_rn(__fmul_rn(x[1], inv), Elem<T>::hi(w.x)));
              v[1] = Elem<T>::pack(__fmul_rn(__fmul_rn(x[2], inv), Elem<T>::lo(w.y)), __fmul_rn(__fmul_rn(x[3], inv), Elem<T>::hi(w.y)));
            }
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              const uint32_t o = swapped(v[e]);  // dims 64 further or back
              const float s0 = gl < 16 ? -sv[2 * e] : sv[2 * e], s1 = gl < 16 ? -sv[2 * e + 1] : sv[2 * e + 1];
              v[e] = Elem<T>::pack(fmaf(Elem<T>::lo(v[e]), cv[2 * e], __fmul_rn(Elem<T>::lo(o), s0)), fmaf(Elem<T>::hi(v[e]), cv[2 * e + 1], __fmul_rn(Elem<T>::hi(o), s1)));
            }
          }
          *reinterpret_cast<uint2*>(qbuf + row * D * 2 + gl * 8) = make_uint2(v[0], v[1]);
          if (row >= G && stores) *reinterpret_cast<uint2*>(row == G ? kc : vc) = make_uint2(v[0], v[1]);
        }
      }
      dl_barrier();  // the new rows are there
      dl_barrier();  // the waves' sums are there
      const int id = (int)threadIdx.x - 64 * kDlFetch, g = id >> 5, d = (id & 31) * 4;
      if (g < G) {
        f32x4 ov[W];
        float2 ml[W];
#pragma unroll
        for (int w = 0; w < W; ++w) {
          ml[w] = s_stat[w][g];
          ov[w] = *reinterpret_cast<const f32x4*>(sums + (w * G + g) * D + d);
        }
        float top = kNegBig;
#pragma unroll
        for (int w = 0; w < W; ++w) top = fmaxf(top, ml[w].x);
        f32x4 a = {0.f, 0.f, 0.f, 0.f};
        float den = 0.f;
#pragma unroll
        for (int w = 0; w < W; ++w) {  // (a wave without a tile: weight 0 or 1, sums 0)
          const float wgt = __builtin_amdgcn_exp2f(ml[w].x - top);
#pragma unroll
          for (int e = 0; e < 4; ++e) a[e] = fmaf(wgt, ov[w][e], a[e]);
          den = fmaf(wgt, ml[w].y, den);
        }
        const int head = t.h * G + g;
        if (t.active == 1) {
          const float inv = 1.0f / den;
          dl_put2(pk, to, (t.b * hq + head) * 512 + d * 4, Elem<T>::pack(a[0] * inv, a[1] * inv), Elem<T>::pack(a[2] * inv, a[3] * inv), epoch);
        } else {
          const int at = ((t.b * R + t.r) * hq + head) * (kDlPart * 8);
          dl_put2(pk, parts, at + d * 8, __float_as_uint(a[0]), __float_as_uint(a[1]), epoch);
          dl_put2(pk, parts, at + d * 8 + 16, __float_as_uint(a[2]), __float_as_uint(a[3]), epoch);
          if (d == 0) dl_put2(pk, parts, at + 1024, __float_as_uint(top), __float_as_uint(den), epoch);
        }
      }
    };
    // the multiplying waves' half
    auto attend_tiles = [&](const Task& t, int l, Tile (&pre)[kDlAhead]) {
      const int lane = dl_lane(), tok = lane & 15, qd = lane >> 4;
      const dl_args_t p = dl_args();
      const int G = p->hq / p->hkv;
      uint16_t* qbuf = reinterpret_cast<uint16_t*>(lds + p->lds_new);  // G query heads, the new key, the new value
      const int step = t.active * W;
      const int first = t.r * W + wv;
      dl_barrier();  // the new rows are there
      float* sums = reinterpret_cast<float*>(lds + p->lds_sums);
      V4 qf[4];
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) qf[kk] = *reinterpret_cast<const V4*>(qbuf + (tok < G ? tok : 0) * D + kk * 32 + qd * 8);
      const float scale_log2 = p->scale_log2;
      float mx = kNegBig, l_sum = 0.f;
      f32x4 o[8];
#pragma unroll
      for (int db = 0; db < 8; ++db) o[db] = f32x4{0.f, 0.f, 0.f, 0.f};
      dlds_char* img = (dlds_char*)(lds + p->lds_images) + wv * 4096;
      int next[kDlAhead];
#pragma unroll
      for (int j = 0; j < kDlAhead; ++j) next[j] = first + (j + kDlAhead) * step < t.nt ? slot_of(t, first + (j + kDlAhead) * step) : 0;
#pragma unroll 1
      for (int base = first; base < t.nt; base += kDlAhead * step) {
#pragma unroll
        for (int j = 0; j < kDlAhead; ++j) {
          const int ti = base + j * step;
          if (ti < t.nt) {
            Tile& c = pre[j];
            if (ti == t.nt - 1) {  // the new token's key and value, and finite rows for the lanes past the end
              const int lt = t.last & 15;
#pragma unroll
              for (int kk = 0; kk < 4; ++kk) {
                const V4 nk = *reinterpret_cast<const V4*>(qbuf + G * D + kk * 32 + qd * 8), nv = *reinterpret_cast<const V4*>(qbuf + (G + 1) * D + kk * 32 + qd * 8);
                if (tok >= lt) {
                  c.k[kk] = nk;
                  c.v[kk] = nv;
                }
              }
            }
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
              *reinterpret_cast<__attribute__((address_space(3))) V4*>(img + vimg_off(tok, kk * 64 + qd * 16)) = c.v[kk];
            f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) s = mfma_k32<T>(c.k[kk], qf[kk], s);
            const int n1 = ti + kDlAhead * step;
            if (n1 < t.nt) {
              load_tile(c, t, l, next[j]);
              if (n1 + kDlAhead * step < t.nt) next[j] = slot_of(t, n1 + kDlAhead * step);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (ti * 16 + 4 * qd + i > t.last) s[i] = -INFINITY;
            const float sm = max_over_rows(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))) * scale_log2;
            const float mn = fmaxf(mx, sm);
            const float alpha = __builtin_amdgcn_exp2f(mx - mn);
            mx = mn;
            float pe[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) pe[i] = __builtin_amdgcn_exp2f(fmaf(s[i], scale_log2, -mx));
            l_sum = fmaf(l_sum, alpha, (pe[0] + pe[1]) + (pe[2] + pe[3]));
            uint2 pf;
            pf.x = Elem<T>::pack(pe[0], pe[1]);
            pf.y = Elem<T>::pack(pe[2], pe[3]);
#pragma unroll
            for (int db = 0; db < 8; ++db) {
#pragma unroll
              for (int i = 0; i < 4; ++i) o[db][i] *= alpha;
              const ds16x4 vt = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ds16x4*)(img + vimg_off(4 * qd + (tok >> 2), db * 32 + (tok & 3) * 8)));
              o[db] = mfma_k16<T>(__builtin_bit_cast(uint2, vt), pf, o[db]);
            }
          }
        }
      }
      l_sum = sum_over_rows(l_sum);
      if (tok < G) {
        float* so = sums + (wv * G + tok) * D + 4 * qd;
#pragma unroll
        for (int db = 0; db < 8; ++db) *reinterpret_cast<f32x4*>(so + db * 16) = o[db];
        if (qd == 0) s_stat[wv][tok] = make_float2(mx, l_sum);
      }
      dl_barrier();  // the waves' sums are there
    };
    // the ranges of one (request, query head), by one wave: lane = dims 2 lane, + 1
    auto active_of = [&](int id) { return ranges_of((dl_ptr<const int>(dl_args()->seq_lens)[id / dl_args()->hq] + 15) >> 4, dl_args()->ranges); };
    auto join = [&](int id, int active, const __amdgpu_buffer_rsrc_t& pk) {
      const int lane = dl_lane();
      const dl_args_t p = dl_args();
      const int hq = p->hq, b = id / hq, head = id - b * hq, to = p->at[4] * 8;
      const int from = p->at_part * 8 + (b * p->ranges * hq + head) * (kDlPart * 8), apart = hq * (kDlPart * 8);
      uint32_t v[10];
      wait.template get<5>(pk, from, v, [&](int j) { return j == 4 ? min(lane, active - 1) * apart + 1024 : min(j, active - 1) * apart + 16 * lane; });
      const float m_r = lane < active ? __uint_as_float(v[8]) : kNegBig;
      const float w_r = __builtin_amdgcn_exp2f(m_r - wave_max(m_r));
      const float den = dl_wave_sum(lane < active ? w_r * __uint_as_float(v[9]) : 0.f);
      float a0 = 0.f, a1 = 0.f;
      for (int r0 = 0;;) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (r0 + j < active) {
            const float w = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w_r), r0 + j));
            a0 = fmaf(w, __uint_as_float(v[2 * j]), a0);
            a1 = fmaf(w, __uint_as_float(v[2 * j + 1]), a1);
          }
        }
        r0 += 4;
        if (r0 >= active) break;
        uint32_t u[8];
        wait.template get<4>(pk, from, u, [&](int j) { return min(r0 + j, active - 1) * apart + 16 * lane; });
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = u[j];
      }
      const float inv = 1.0f / den;
      __builtin_amdgcn_raw_buffer_store_b64(u32x2_t{Elem<T>::pack(a0 * inv, a1 * inv), epoch}, pk, id * 512 + lane * 8, to, 16);
    };

    auto packets_of = [&](int l) { return dl_rsrc(dl_args()->packets + (u64_t)((int64_t)l * dl_args()->layer_packets * 8)); };
    if (f >= 0) {
      // ---- fetching waves: stage rows, meet the multiplying waves at a barrier ----
      f32x4 cosv = {0.f, 0.f, 0.f, 0.f}, sinv = cosv;
      if (works) angles_of(mine, cosv, sinv);
      const int heads = M * dl_args()->hq;
      int first_join, active0;
      auto join_of = [&] {
        first_join = f == 0 && dl_args()->ranges > 1 ? n - 1 - rank : heads;
        active0 = first_join < heads ? sgpr(active_of(first_join)) : 0;
      };
      join_of();
      {
        const dl_args_t p = dl_args();
        const int H = p->H, per_row = H >> 8;
        const uint16_t* x = dl_ptr<const uint16_t>(p->x);
#pragma unroll
        for (int q = 0; q < MQ; ++q)
#pragma unroll
          for (int c = 0; c < kRow; ++c) {
            const int m = f + 4 * q;
            res[q][c][0] = res[q][c][1] = 0;
            if (m < M) {
              const uint2 v = *reinterpret_cast<const uint2*>(x + m * H + min(c, per_row - 1) * 256 + lane * 4);
              res[q][c][0] = v.x;
              res[q][c][1] = v.y;
            }
          }
      }
      dl_barrier();  // the first norm weights are there
      auto sums_of = [&](int s) {  // (the multiplying waves')
        for (int i = passes_of(s); i > 0; --i) {
          dl_barrier();
          if (i > 1) dl_barrier();
        }
      };
      for (int l = 0; l < layers; ++l) {
        const __amdgpu_buffer_rsrc_t pk = packets_of(l);
        if (grown(l)) join_of();
        // While the team may grow, the last of these waves of the first workgroup says which size the next layer's has, and everyone's looks for it
        const bool asks = open && f == kDlFetch - 1 && l >= from && l + 1 < layers;
        uint32_t* team = dl_ptr<uint32_t>(dl_args()->team);
        u64_t* next = reinterpret_cast<u64_t*>(team + kTeamSizes) + l + 1;
        uint32_t have = 0;
        if (asks && rank == 0) have = __hip_atomic_load(team + kTeamCount, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        {
          const dl_args_t p = dl_args();
          add_norm(l ? 2 : p->y_in ? 1 : 0, packets_of(max(l - 1, 0)), p->at[3] * 8, 0);
        }
        if (asks && rank == 0) dl_put(next, (uint32_t)dl_size(have, l + 1), epoch);
        if (l >= from) {  // (a latecomer follows the residual stream to the layer that it joins at)
          dl_barrier();  // qkv's rows are there
          sums_of(0);
#pragma unroll 1
          for (int id = rank; id < tasks; id += n) {
            Task t = mine;
            f32x4 cv = cosv, sv = sinv;
            if (id != rank) {
              t = task_of(id);
              angles_of(t, cv, sv);
            }
            if (t.r < t.active) attend_rows(t, l, pk, cv, sv);
          }
#pragma unroll 1
          for (int id = first_join; id < heads; id += n) {
            const int active = id == first_join ? active0 : active_of(id);
            if (active > 1) join(id, active, pk);
          }
          take_rows(pk, dl_args()->at[4] * 8, dl_args()->K[1], dl_args()->lds_rows[1]);
          dl_barrier();  // o's rows are there
          sums_of(1);
        }
        add_norm(2, pk, dl_args()->at[1] * 8, 1);
        if (l < from) continue;
        dl_barrier();  // gate_up's rows are there
        sums_of(2);
        u64_t seen = 0;
        if (asks) seen = dl_get(next);
        take_rows(pk, dl_args()->at[2] * 8, dl_args()->K[3], dl_args()->lds_rows[3]);
        if (asks) {
          int spins = 0;
          while ((uint32_t)(seen >> 32) != epoch && wait.again(spins)) seen = dl_get(next);
          if ((uint32_t)(seen >> 32) == epoch) *(volatile int*)&s_size = (int)(uint32_t)seen;
        }
        dl_barrier();  // down's rows, and the team's next size, are there
        sums_of(3);
      }
      if (rank == 0) {
        const dl_args_t p = dl_args();
        uint16_t* out = dl_ptr<uint16_t>(p->res_out);
        const int H = p->H;
#pragma unroll
        for (int q = 0; q < MQ; ++q)
#pragma unroll
          for (int c = 0; c < kRow; ++c)
            if (const int m = f + 4 * q; m < M && c < H >> 8) *reinterpret_cast<uint2*>(out + m * H + c * 256 + lane * 4) = make_uint2(res[q][c][0], res[q][c][1]);
      }
    } else {
      // ---- multiplying waves ----
      Tile pre[kDlAhead];
      int slots[kDlAhead];  // of my first task's first tiles, the same in every layer
      if (works) {
        slots_of(mine, slots);
        load_ahead(pre, mine, from, slots);
      }
      if (wv == 1) {
        fetch_norms(from, 0);
        fetch_norms(from, 1);
      }
      auto fetch_first = [&](int l) {  // a layer's products that nothing before has asked for
        fetch(0, l, first_qkv, count_qkv);
        fetch(1, l, first_hid, count_hid);
      };
      if (ahead) fetch_first(from);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      dl_barrier();  // the first norm weights are there

      // one product of a layer.  v_mfma_f32_4x4x4_16b has block b = columns 8 b .. + 7 of 128, A = a group's four rows, B = four staged rows (MQ times); the
      // sixteen blocks' sums are added across the lanes, the four waves' in LDS, where wave u takes unit u's.
      // Weights: asked for two stages ahead, when those before them (and the rows that lay in their place) are used.
      auto stage = [&](auto S_, int l) __attribute__((always_inline)) {
        constexpr int S = decltype(S_)::value;
        constexpr bool kWide = S & 1;  // o, down: one unit, up to eight pieces of it a wave; else four units, two pieces of each group
        constexpr int kRead = S == 2 ? 2 : 1;
        const int lane = dl_lane();
        const bool more = l + 1 < layers;
        const dl_args_t p = dl_args();
        const int first = first_of(S), count = count_of(S), cap = p->cap[S], K = p->K[S], chunks = K >> 7;
        const uint32_t weights = dl_lds_at(lds) + p->lds_w[S] + wv * 1024 + lane * 16, sums = dl_lds_at(lds) + p->lds_sums;
        uint32_t rows[MQ];
#pragma unroll
        for (int q = 0; q < MQ; ++q) rows[q] = dl_lds_at(lds) + p->lds_rows[S] + min(4 * q + (lane & 3), M - 1) * (K + kDlPad) * 2 + (lane >> 2) * 16 + wv * 256;
        const int N = S == 0 ? qkv_rows : S == 2 ? p->inter : p->H, out_at = p->at[S] * 8;
        const u64_t y_out = p->y_out;
        const __amdgpu_buffer_rsrc_t pk = packets_of(l);
        V4 a[kRead][8];
        auto read_weights = [&] {
#pragma unroll
          for (int i = 0; i < kRead; ++i) dl_read8<4096>(a[i], weights + i * 32768);  // (what lies past the units is not used)
        };
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (asked for two stages ago)
        if (ahead) {
          read_weights();
          if (S == 0) fetch(2, l, first_act, count_act);
          if (S == 1) fetch(3, l, first_hid, count_hid);
          if (S == 2 && more) fetch(0, l + 1, first_qkv, count_qkv);
          if (S == 3 && more) fetch(1, l + 1, first_hid, count_hid);
        }
        if (more) {
          if (wv == 1 && (S & 1)) fetch_norms(l + 1, S >> 1);
          if (works && S == 2) load_ahead(pre, mine, l + 1, slots);
        }
        dl_barrier();  // the rows are there
        for (int pass = 0;;) {
          const int here = min(cap, count - pass);
          if (!ahead) {
            fetch(S, l, first + pass, here);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            read_weights();
          }
          constexpr int kAcc = kWide ? 2 : S == 2 ? 8 : 4;
          f32x4 acc[kAcc][MQ];
#pragma unroll
          for (int i = 0; i < kAcc; ++i)
#pragma unroll
            for (int q = 0; q < MQ; ++q) acc[i][q] = f32x4{0.f, 0.f, 0.f, 0.f};
          auto mul = [](f32x4& c, const V4& w, const V4& x) __attribute__((always_inline)) {
            c = mfma444<T>(w[0], w[1], x[0], x[1], c);
            c = mfma444<T>(w[2], w[3], x[2], x[3], c);
          };
#pragma unroll
          for (int q = 0; q < MQ; ++q) {
            if constexpr (kWide) {
              V4 b[8];
              dl_read8<1024>(b, rows[q]);
#pragma unroll
              for (int i = 0; i < 8; ++i)
                if (wv + 4 * i < chunks) mul(acc[i & 1][q], a[0][i], b[i]);
            } else {
              V4 b[2];
              dl_read2<1024>(b, rows[q]);
#pragma unroll
              for (int i = 0; i < 2; ++i) {
                if (wv + 4 * i < chunks) {
#pragma unroll
                  for (int g = 0; g < kAcc; ++g) mul(acc[g][q], a[g >> 2][2 * (g & 3) + i], b[i]);
                }
              }
            }
          }
          // sums [wave][q][unit][row of the stream] (gate_up: [wave][q][unit / 2][unit's halves][row])
#pragma unroll
          for (int q = 0; q < MQ; ++q) {
            if constexpr (kWide) {
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[0][q][e] += acc[1][q][e];
              const f32x4 v = dl_over_blocks(acc[0][q]);
              if (lane < 4) dl_write(sums + ((wv * MQ + q) * 4 + lane) * 16, v);
            } else {
#pragma unroll
              for (int h = 0; h < kRead; ++h) {
                const f32x4 v = dl_over_blocks(acc[4 * h][q], acc[4 * h + 1][q], acc[4 * h + 2][q], acc[4 * h + 3][q]);
                if ((lane & 12) == 0) dl_write(sums + (((wv * MQ + q) * kRead + h) * 16 + (lane >> 4) * 4 + (lane & 3)) * 16, v);
              }
            }
          }
          dl_barrier();  // the waves' sums are there, weights and rows are used
          if (kWide ? wv == 3 && here > 0 : wv < here) {
            const int m = lane, q = MQ == 2 ? lane >> 2 & 1 : 0, j = lane & 3;
            auto total = [&](int g) {  // of group g (gate_up: 2 units + half)
              f32x4 t[4];  // the waves'
              dl_read4<(kWide ? 4 : 16 * kRead) * MQ * 16>(t, sums + (kWide ? q * 4 + j : (q * kRead + (g >> 2)) * 16 + (g & 3) * 4 + j) * 16);
#pragma unroll
              for (int w = 1; w < 4; ++w)
#pragma unroll
                for (int e = 0; e < 4; ++e) t[0][e] += t[w][e];
              return t[0];
            };
            const int unit = first + pass + (kWide ? 0 : wv);
            const f32x4 v = total(S == 2 ? 2 * wv : wv);
            uint32_t lo = Elem<T>::pack(v[0], v[1]), hi = Elem<T>::pack(v[2], v[3]);
            if constexpr (S == 2) {  // gate and up rounded as the projection stores them
              const f32x4 w = total(2 * wv + 1);
              const uint32_t u01 = Elem<T>::pack(w[0], w[1]), u23 = Elem<T>::pack(w[2], w[3]);
              const uint32_t p01 = Elem<T>::pack(silu_mul_f32(Elem<T>::lo(lo), Elem<T>::lo(u01)), silu_mul_f32(Elem<T>::hi(lo), Elem<T>::hi(u01)));
              const uint32_t p23 = Elem<T>::pack(silu_mul_f32(Elem<T>::lo(hi), Elem<T>::lo(u23)), silu_mul_f32(Elem<T>::hi(hi), Elem<T>::hi(u23)));
              lo = p01;
              hi = p23;
            }
            if (m < M) {
              if (S < 3 || more) {
                dl_put2(pk, out_at, (m * N + 4 * unit) * 4, lo, hi, epoch);
              } else {
                *reinterpret_cast<uint2*>(dl_ptr<uint16_t>(y_out) + (int64_t)m * N + 4 * unit) = make_uint2(lo, hi);
              }
            }
          }
          pass += cap;
          if (ahead || pass >= count) break;
          dl_barrier();  // the sums are read
        }
      };
      for (int l = from; l < layers; ++l) {
        stage(std::integral_constant<int, 0>{}, l);
#pragma unroll 1
        for (int id = rank; id < tasks; id += n) {
          Task t = mine;
          if (id != rank) {  // (the first one's tiles are there)
            t = task_of(id);
            int slot[kDlAhead];
            slots_of(t, slot);
            if (t.r < t.active) load_ahead(pre, t, l, slot);
          }
          if (t.r < t.active) attend_tiles(t, l, pre);
        }
        stage(std::integral_constant<int, 1>{}, l);
        stage(std::integral_constant<int, 2>{}, l);
        stage(std::integral_constant<int, 3>{}, l);
        if (open && l + 1 < layers && grown(l + 1) && ahead) {
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (what was asked for of other shares)
          fetch_first(l + 1);
        }
      }
    }
  }

  // ---- the last one to leave opens the count for the next launch ----
  if (threadIdx.x == 0) {
    uint32_t* team = dl_ptr<uint32_t>(dl_args()->team);
    if (*(volatile int*)&s_dead) __hip_atomic_store(team + kTeamFailed, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = __hip_atomic_fetch_add(team + kTeamLeft, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
    if (s_last) {
      __hip_atomic_store(team + kTeamCount, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(team + kTeamLeft, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(team + kTeamEpoch, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if (epoch == 0xffffffffu) {  // the numbers start again: no packet of any earlier launch stays, and no size
    __syncthreads();
    if (s_last) {
      u64_t* packets = dl_ptr<u64_t>(dl_args()->packets) - kDlMaxLayers;
      const int64_t all = dl_args()->packets_all + kDlMaxLayers;
      for (int64_t i = threadIdx.x; i < all; i += kDlThreads) packets[i] = 0;
    }
  }
}

// ---- sizes ----
struct DlLayout {
  int64_t layer_packets;
  int at[5], at_part, ranges;
  int lds_w[4], lds_rows[4], lds_images, lds_sums, lds_norms, lds_new, lds_bytes, cap[4], cus, alias, mq;
};

// what a launch of `batch` rows needs; false: does not fit
static bool dl_layout(DlLayout& a, int batch, int hidden, int hq, int hkv, int inter) {
  if (batch < 1 || batch > 8 || hidden < 256 || hidden % 256 || hq < 1 || hkv < 1 || hq % hkv || hq / hkv > 8 || hq % 2 || inter < 256 || inter % 256) return false;
  if (hidden > 65536 || hq > 1024 || inter > 262144) return false;
  a.mq = batch > 4 ? 2 : 1;
  if (hidden > kDlRow || hq * 128 > kDlCols || inter > kDlCols) return false;
  a.cus = device_cu_count() > 0 ? device_cu_count() : 256;
  const int q_dim = hq * 128, qkv_dim = (hq + 2 * hkv) * 128;
  auto groups = [&](int rows) { return (rows / 4 + a.cus - 1) / a.cus; };
  const int cap_qkv = groups(qkv_dim), cap_act = groups(inter), cap_hidden = groups(hidden);
  if (cap_qkv > kDlUnits || cap_act > kDlUnits || cap_hidden > 1) return false;
  auto rows = [&](int K) { return (int64_t)batch * (K + kDlPad) * 2; };
  auto most = [](int64_t x, int64_t y) { return x > y ? x : y; };
  auto unit = [](int K) { return (int64_t)(K + 1023) / 1024 * 8192; };
  const int64_t qkv = cap_qkv * unit(hidden), gu = 2 * cap_act * unit(hidden), down = cap_hidden * unit(inter), o = cap_hidden * unit(q_dim);
  const int64_t images = kDlFetch * 4096, sums = most((int64_t)kDlFetch * (hq / hkv) * 512, kDlFetch * a.mq * 512), norms = (int64_t)hidden * 4 + 512 + (hq / hkv + 2) * 256;  // (and attention's new rows)
  int64_t xs = rows(hidden);
  // [qkv weights][rows of the hidden size][gate_up weights][down][o][V images, then rows of o and down][sums][norms], or, where that does not fit, images and rows
  // of o in the first two, rows of down in the second and third: their weights are asked for later
  int64_t at_rows = qkv + xs + gu + down + o, all = at_rows + most(images, rows(q_dim) + rows(inter)) + sums + norms;
  a.alias = all > kDlLds;
  if (a.alias) {
    xs = most(xs, most(most(rows(q_dim), images) - qkv, rows(inter) - gu));
    at_rows = qkv + xs + gu + down + o;
    all = at_rows + sums + norms;
    if (all > kDlLds) return false;
  }
  const int64_t gu_at = qkv + xs, down_at = gu_at + gu, o_at = down_at + down;
  const int64_t w[4] = {0, o_at, gu_at, down_at};
  const int64_t r[4] = {qkv, a.alias ? 0 : at_rows, qkv, !a.alias ? at_rows + rows(q_dim) : rows(inter) > gu ? down_at - rows(inter) : gu_at};
  const int cap[4] = {cap_qkv, cap_hidden, cap_act, cap_hidden};
  for (int i = 0; i < 4; ++i) {
    a.lds_w[i] = (int)w[i];
    a.lds_rows[i] = (int)r[i];
    a.cap[i] = cap[i];
  }
  a.lds_images = a.alias ? 0 : (int)at_rows;
  a.lds_sums = (int)(all - norms - sums);
  a.lds_norms = (int)(all - norms);
  a.lds_new = a.lds_norms + hidden * 4 + 512;
  a.lds_bytes = (int)all;
  // key ranges: as many as give every CU a (request, kv head, range), 64 at most (the join has one per lane)
  a.ranges = a.cus / (batch * hkv);
  a.ranges = a.ranges < 1 ? 1 : a.ranges > 64 ? 64 : a.ranges;
  const int n[5] = {qkv_dim, hidden, inter, hidden, q_dim};
  int at = 0;
  for (int i = 0; i < 5; ++i) {
    a.at[i] = at;
    at += batch * n[i] / 2;
  }
  a.at_part = at;
  a.layer_packets = at + (int64_t)batch * a.ranges * hq * kDlPart;
  return true;
}

}  // namespace msgl

using namespace msgl;

extern "C" int msgl_decode_layers_supported(int batch, int hidden, int num_q_heads, int num_kv_heads, int intermediate) {
  DlLayout a;
  return dl_layout(a, batch, hidden, num_q_heads, num_kv_heads, intermediate) ? 1 : 0;
}

extern "C" int64_t msgl_decode_layers_workspace_bytes(int batch, int layers, int hidden, int num_q_heads, int num_kv_heads, int intermediate) {
  DlLayout a;
  if (layers < 1 || !dl_layout(a, batch, hidden, num_q_heads, num_kv_heads, intermediate)) return MSGL_EINVAL;
  return kTeamWords * 4 + a.layer_packets * (layers < kDlMaxLayers ? layers : kDlMaxLayers) * 8;
}

template <typename T, int MQ>
static int dl_launch(const DlParams& p, const DlLayout& a, hipStream_t s) {
  static PerDeviceOnce once;
  const bool ok = once.ensure([] {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(&decode_layers_kernel<T, MQ>), hipFuncAttributeMaxDynamicSharedMemorySize, kDlLds) == hipSuccess;
  });
  MSGL_REQUIRE(ok, "decode_layers: no %d bytes of LDS", kDlLds);
  decode_layers_kernel<T, MQ><<<dim3((unsigned)a.cus), dim3(kDlThreads), (size_t)a.lds_bytes, s>>>(p);
  MSGL_CHECK_LAUNCH("decode_layers");
  return MSGL_OK;
}

extern "C" int64_t msgl_decode_layers_failed_at(void) { return kTeamFailed * 4; }

extern "C" int msgl_decode_layers_bounded(void* y_out, void* res_out, const void* x, const msgl_decode_layer_t* layer, int layers, const int32_t* positions,
                                          const float* cos_sin, const int32_t* out_loc, const int32_t* page_table, int64_t pt_stride, const int32_t* req_rows,
                                          const int32_t* seq_lens, void* workspace, int64_t workspace_bytes, int batch, int hidden, int num_q_heads,
                                          int num_kv_heads, int head_dim, int intermediate, int gate_up_interleaved, int64_t kv_stride_tok,
                                          int64_t kv_stride_head, float eps, float sm_scale, int dtype, int looks, int absent, int most, int until, void* stream) {
  MSGL_REQUIRE(looks >= 0 && most >= 0 && until >= 0, "decode_layers: %d looks, a team of %d before layer %d", looks, most, until);
  MSGL_REQUIRE(y_out && res_out && x && layer && positions && cos_sin && out_loc && page_table && seq_lens && workspace, "decode_layers: null pointer");
  MSGL_REQUIRE(layers >= 1, "decode_layers: %d layers", layers);
  MSGL_REQUIRE(head_dim == 128, "decode_layers: head_dim %d unsupported (128 only)", head_dim);
  MSGL_REQUIRE(dtype == MSGL_BF16 || dtype == MSGL_FP16, "decode_layers: unsupported dtype code %d", dtype);
  DlLayout a;
  MSGL_REQUIRE(dl_layout(a, batch, hidden, num_q_heads, num_kv_heads, intermediate), "decode_layers: batch %d, hidden %d, %d / %d heads, intermediate %d unsupported",
               batch, hidden, num_q_heads, num_kv_heads, intermediate);
  MSGL_REQUIRE(!gate_up_interleaved || intermediate % 32 == 0, "decode_layers: interleaved gate_up of %d columns", intermediate);
  MSGL_REQUIRE(workspace_bytes >= msgl_decode_layers_workspace_bytes(batch, layers, hidden, num_q_heads, num_kv_heads, intermediate),
               "decode_layers: workspace of %lld bytes", (long long)workspace_bytes);
  MSGL_REQUIRE(kv_stride_tok % 8 == 0 && kv_stride_head % 8 == 0, "decode_layers: strides must be multiples of 8 elements");
  bool fine = aligned16(y_out) && aligned16(res_out) && aligned16(x) && aligned16(workspace) && aligned16(cos_sin);
  for (int i = 0; i < layers; ++i) {
    const msgl_decode_layer_t& w = layer[i];
    MSGL_REQUIRE(w.input_norm && w.qkv && w.o && w.post_norm && w.gate_up && w.down && w.k_cache && w.v_cache, "decode_layers: null pointer in layer %d", i);
    MSGL_REQUIRE((w.q_norm == nullptr) == (w.k_norm == nullptr), "decode_layers: both head norm weights or neither (layer %d)", i);
    fine = fine && aligned16(w.input_norm) && aligned16(w.qkv) && aligned16(w.o) && aligned16(w.post_norm) && aligned16(w.gate_up) && aligned16(w.down) &&
           aligned16(w.k_cache) && aligned16(w.v_cache) && aligned16(w.q_norm) && aligned16(w.k_norm);
  }
  MSGL_REQUIRE(fine, "decode_layers: pointers must be 16-byte aligned");
  DlParams p{};
  auto at = [](const void* q) { return (u64_t)(uintptr_t)q; };
  p.positions = at(positions); p.cos_sin = at(cos_sin); p.out_loc = at(out_loc);
  p.page_table = at(page_table); p.req_rows = at(req_rows); p.seq_lens = at(seq_lens);
  p.team = at(workspace);
  p.packets = p.team + kTeamWords * 4;
  p.packets_all = (workspace_bytes - kTeamWords * 4) / 8;
  p.pt_stride = pt_stride; p.kv_stride_tok = kv_stride_tok; p.kv_stride_head = kv_stride_head;
  p.M = batch; p.H = hidden; p.hq = num_q_heads; p.hkv = num_kv_heads; p.inter = intermediate;
  p.ranges = a.ranges; p.interleaved = gate_up_interleaved;
  p.looks = looks > 0 ? looks : kLooks;
  p.absent = absent;
  p.most = most;
  p.until = most > 0 ? until : 0;
  p.eps = eps;
  p.scale_log2 = sm_scale * 1.4426950408889634f;
  p.layer_packets = (int)a.layer_packets; p.at_part = a.at_part;
  p.lds_images = a.lds_images; p.lds_sums = a.lds_sums; p.lds_norms = a.lds_norms; p.lds_new = a.lds_new;
  const int K[4] = {hidden, num_q_heads * 128, hidden, intermediate};
  for (int i = 0; i < 4; ++i) {
    p.lds_w[i] = a.lds_w[i];
    p.lds_rows[i] = a.lds_rows[i];
    p.cap[i] = a.cap[i];
    p.K[i] = K[i];
  }
  for (int i = 0; i < 5; ++i) p.at[i] = a.at[i];
  p.y_out = at(y_out); p.res_out = at(res_out); p.x = at(x);
  for (int first = 0; first < layers; first += kDlMaxLayers) {  // (the next launch reads the rows that this one leaves)
    p.layers = layers - first < kDlMaxLayers ? layers - first : kDlMaxLayers;
    for (int i = 0; i < p.layers; ++i) {
      const msgl_decode_layer_t& w = layer[first + i];
      p.layer[i] = DlLayer{{at(w.input_norm), at(w.post_norm)}, {at(w.qkv), at(w.o), at(w.gate_up), at(w.down)}, at(w.q_norm), at(w.k_norm), at(w.k_cache), at(w.v_cache)};
    }
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const bool two = a.mq == 2;
    const int rc = dtype == MSGL_BF16 ? (two ? dl_launch<BF16, 2>(p, a, s) : dl_launch<BF16, 1>(p, a, s))
                                      : (two ? dl_launch<FP16, 2>(p, a, s) : dl_launch<FP16, 1>(p, a, s));
    if (rc != MSGL_OK) return rc;
    p.x = p.res_out;
    p.y_in = p.y_out;
  }
  return MSGL_OK;
}

extern "C" int msgl_decode_layers(void* y_out, void* res_out, const void* x, const msgl_decode_layer_t* layer, int layers, const int32_t* positions,
                                  const float* cos_sin, const int32_t* out_loc, const int32_t* page_table, int64_t pt_stride, const int32_t* req_rows,
                                  const int32_t* seq_lens, void* workspace, int64_t workspace_bytes, int batch, int hidden, int num_q_heads,
                                  int num_kv_heads, int head_dim, int intermediate, int gate_up_interleaved, int64_t kv_stride_tok,
                                  int64_t kv_stride_head, float eps, float sm_scale, int dtype, void* stream) {
  return msgl_decode_layers_bounded(y_out, res_out, x, layer, layers, positions, cos_sin, out_loc, page_table, pt_stride, req_rows, seq_lens, workspace,
                                    workspace_bytes, batch, hidden, num_q_heads, num_kv_heads, head_dim, intermediate, gate_up_interleaved, kv_stride_tok,
                                    kv_stride_head, eps, sm_scale, dtype, 0, -1, 0, 0, stream);
}
