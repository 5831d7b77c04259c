// Wide GEMM over packed weights: Y[M,N] = X[M,K] · W[N,K]^T for M > 128 (the prefill chunks the
// reference hands to F.linear, plm/rounds.py:16, plm/fast_gemm.py:108-111), so that a caller that
// keeps only the packed copy of a weight has a compute-bound kernel for them; for single linears of a
// round on row-split tiles (packed_api.hip, wide_preferred), where its X, read once per workgroup, beats
// the packed kernel's; both with a fused gate/up projection's SiLU-and-multiply as the epilogue; and the
// gated-LoRA launch on such tiles.
//
// Every output is one MFMA chain over the K steps in ascending order (v_mfma_f32_16x16x32), the
// order of a row-split packed tile without K splits; it is also what torch's F.linear returned bit for
// bit at every prefill width measured. With K splits each range is such a chain and the ranges' sums
// are added in order, as the packed kernel does.
//
// What bounds it: a CU's vector memory path, which moves 75-100 KiB per us from L2 whatever is
// loaded (measured with the loads alone: 16 KiB per K step in 0.16-0.21 us), against 0.12 us of MFMA
// for a 128 x 128 tile's K step; then the LDS reads of X. So a tile is chosen by the bytes it loads
// per K step and by how evenly its tiles fill the CUs (wide_pick), and nothing is loaded twice inside
// a workgroup: its four wavefronts take 16*NF weight rows each over the tile's whole 16*MT rows of X.
// Weight fragments go straight to registers (a packed fragment is one contiguous KiB in operand
// order); X goes through registers into LDS as rows of 128 B (two K steps, whole cache lines) with
// 16-byte chunk c of row r at slot c ^ (r % 8), which makes the operand reads conflict-free (LDS reads
// measured at 125-131 B per clock in this pattern, 64 without the swizzle).
//
// A stage is two K steps with one barrier, in its middle: the first step's MFMAs run while the second
// step's X is read and the next stage's X written, then the barrier, then the second step's MFMAs
// while the next stage's first X is read. The 16-row tile, whose MFMAs cover none of those LDS round
// trips, takes four K steps per stage and reads the next stage whole during a stage. Where the ranges of
// K steps allow it a stage's offsets come from one multiply: a wavefront alone on its SIMD is bound by the
// instructions it issues (512x1408 at M = 42: 5.6 -> 4.7 us; 2048x8192 at M = 256: 22.7 -> 20.5, at M = 7
// unsplit 19.3 -> 16.2; four K steps per stage on 32-row tiles too: 6144x2048 at M = 56 9.45 -> 9.74, as
// their loads then go out in bursts). Memory instructions are spread between the MFMAs
// (sched_group_barrier), since a burst of them stalls a wavefront's MFMAs behind it (M = 640,
// 8192 x 2048: 26.0 us without the spreading, 24.9 with). Global loads run D stages ahead. The
// 16-bit outputs go through LDS so that a row's stores are whole 128*NF-byte segments.
//
// Measured against unpacking the weight and F.linear (us; M = 640: 6144x2048, 2048x2048, 8192x2048,
// 2048x8192): 34 / 17 / 35 / 51 -> 22 / 11 / 25 / 38; M = 256: 31 / 12 / 32 / 33 -> 16 / 7 / 15 / 23.
// Rounds, against the packed kernel's best tile (us; 6144x2048, 2048x2048, 8192x2048, 2048x8192 split 4):
// M = 56 12.8 / 9.5 / 13.6 / 15.8 -> 9.6 / 7.5 / 10.2 / 14.1, M = 110 18.4 / 12.1 / 19.2 / 21.8 -> 11.5 /
// 7.9 / 12.0 / 16.6. Rows past N or M and K past K load zeros (buffer range checks, per-lane masks) and are never stored.
#include <hip/hip_runtime.h>

#include "packed_gemm.h"
#include "plm_amd.h"
#include "tile.h"
#include "wide_gemm.h"

namespace plm {
namespace {

constexpr int kWideWaves = 4;
constexpr int kWideThreads = 64 * kWideWaves;
constexpr uint32_t kWideNoLoad = 0x80000000u;

// What the kernel's stores are: the product, a fused gate/up projection's activation, or the gated-LoRA
// launch's base linear (with the h linear's workgroups ahead of it).
constexpr int kWidePlain = 0, kWideAct = 1, kWideLora = 2;

// The gated-LoRA launch (plm_gemm_packed_lora): workgroups [0, items) form h = X A^T in the model dtype,
// the base linear's workgroups follow, wait for h once their own sums are formed, and add the rank-r
// correction as MFMAs. Against the packed kernel's launch, which adds it as scalar products (us, weights
// from memory): 3072x2048, rank 16, M = 56 13.8 -> 10.9; 11264x2048 24.1 -> 18.7; 4608x3072, rank 64,
// M = 110 55.1 -> 17.1. What is left over the base linear (7.6, 13.5, 13.0) is h's chain: X, the partial
// sums' round trip, h's own.
struct WideLora {
  const void* w;     // A, packed
  uint16_t* h;       // [M][width]
  const uint16_t* b; // [N][rank]
  uint32_t wbytes, wgroup;
  int width, split, tiles, items, rank, gated_from;
  int base_tiles;
  int shard_end[3];  // exclusive column ends of the first three shards (N past the last)
  float* partial;
  int* arrive;
  int* counters;     // the workspace's: h tiles written, base tiles past their wait, the error flag
  int spin_limit;
};

struct WideArgs {
  const void* x;
  const void* w;
  void* y;
  int64_t ldx, ldy;
  int M, N, Ks;        // N: output columns (N/2 of the weight's rows with the activation)
  int mtiles, tiles, per_xcd, out_f32;
  uint32_t wbytes, wgroup;
  int K, split;            // split > 1: an item is a tile and one of `split` ranges of K steps
  float* partial;          // split > 1: fp32 fragments [split][weight fragments][X fragments][64 lanes]
  int* arrive;             // split > 1: one arrival counter per tile
  int gate_step, up_step;  // activation: fragment g's gate rows lie in weight fragment g * gate_step,
                           // its up rows up_step fragments further
  WideLora lora;           // kWideLora only
};

template <int DT>
__device__ __forceinline__ void wide_store4_f32(const WideArgs& a, int m, int n, f32x4 v) {
  const int left = a.N - n;
  float* y = static_cast<float*>(a.y) + static_cast<int64_t>(m) * a.ldy + n;
  if (left >= 4 && (reinterpret_cast<uintptr_t>(y) & 15) == 0) {
    *reinterpret_cast<f32x4*>(y) = v;
  } else {
    for (int j = 0; j < 4 && j < left; ++j) y[j] = v[j];
  }
}

__device__ __forceinline__ void wide_sync() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Masks of sched_group_barrier.
constexpr int kMfma = 0x8, kVmemRead = 0x20, kDsRead = 0x100, kDsWrite = 0x200;

// K steps of a stage, and stages of global loads in flight: eight K steps, or four where they are long and
// the registers are taken (2048x8192 at M = 256 on 64 x 32 tiles: 29.6 us with four in flight, 23.0 with
// eight, no better with sixteen; 128 x 128 tiles: no difference).
template <int NF, int MT>
constexpr int wide_steps() {
  return NF * MT == 1 ? 4 : 2;
}
template <int NF, int MT>
constexpr int wide_depth() {
  return wide_steps<NF, MT>() == 4 ? 2 : NF * MT <= 8 ? 4 : 2;
}

// The base linear's wait (bounded) until every h tile is written.
__device__ __forceinline__ void wide_wait_h(const WideLora& z) {
  for (int i = 0;; ++i) {
    if (__builtin_amdgcn_readfirstlane(collect(z.counters + kPkLoraHDone)) >= z.tiles) return;
    if (i >= z.spin_limit) {
      if ((threadIdx.x & 63) == 0) publish(z.counters + kPkErrorSlot, 1);
      return;
    }
    if (i % kErrorCheckPolls == kErrorCheckPolls - 1 &&
        __builtin_amdgcn_readfirstlane(collect(z.counters + kPkErrorSlot)) != 0)
      return;
    __builtin_amdgcn_s_sleep(1);
  }
}

template <int DT, int NF, int MT, int EPI, bool ALIGNED>
__global__ __launch_bounds__(kWideThreads, 1) void wide_gemm_kernel(WideArgs a) {
  constexpr bool ACT = EPI == kWideAct;
  constexpr int D = wide_depth<NF, MT>(), S = wide_steps<NF, MT>();
  constexpr int CH = 4 * S;                                // 16-byte chunks of an X row of a stage
  constexpr int GR = 64 / CH;                              // rows of one load instruction
  constexpr int GROUPS = 16 * MT / GR;                     // load instructions of a stage, over the workgroup
  constexpr int XN = (GROUPS + 3) / 4;                     // and of a wavefront
  constexpr int OF = ACT ? NF / 2 : NF;                    // output fragments per wavefront
  constexpr int OC = 8 * OF;                               // 16-byte chunks of a row of the output tile
  constexpr int kStageWords = GROUPS * 64;                 // u32x4 of one stage of X
  constexpr int kOutWords = 16 * MT * OC;                  // u32x4 of the 16-bit output tile
  __shared__ __attribute__((aligned(16))) u32x4 lds[2 * kStageWords > kOutWords ? 2 * kStageWords : kOutWords];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Workgroups go round the 8 XCDs; each XCD takes a run of items, X tiles fastest, then splits, so
  // that a weight tile is read into one XCD's L2 only.
  int block = blockIdx.x;
  bool forms_h = false;
  if constexpr (EPI == kWideLora) {
    forms_h = block < a.lora.items;
    block -= a.lora.items;
    if (forms_h) {
      a.w = a.lora.w;
      a.N = a.lora.width;
      a.wbytes = a.lora.wbytes;
      a.wgroup = a.lora.wgroup;
      a.split = a.lora.split;
      a.tiles = a.lora.tiles;
      a.partial = a.lora.partial;
      a.arrive = a.lora.arrive;
    }
  }
  const int item = forms_h ? static_cast<int>(blockIdx.x) : (block & 7) * a.per_xcd + (block >> 3);
  if (item >= a.tiles * a.split) return;
  const int ns = item / a.mtiles, mt = item - ns * a.mtiles;
  const int nt = a.split == 1 ? ns : ns / a.split, sp = ns - nt * a.split;
  // K steps [lo, hi), stages of S from lo; k_tail of the last stage's 32 S K elements are real.
  const int lo = a.split == 1 ? 0 : static_cast<int>(static_cast<uint32_t>(sp * a.Ks) / static_cast<uint32_t>(a.split));
  const int hi = a.split == 1 ? a.Ks
                              : static_cast<int>(static_cast<uint32_t>((sp + 1) * a.Ks) / static_cast<uint32_t>(a.split));
  const int stages = (hi - lo + S - 1) / S;
  const int k_tail = min(a.K, 32 * hi) - 32 * lo - 32 * S * (stages - 1);
  const auto wr = make_rsrc(a.w, a.wbytes);
  const auto xr = make_rsrc(a.x, static_cast<uint32_t>(static_cast<int64_t>(a.M) * a.ldx * 2));
  const int of0 = (nt * kWideWaves + wave) * OF;           // this wavefront's first output fragment
  uint32_t wo[NF], xo[XN], xl[XN];                         // xl: the bit that puts a lane past K out of range
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int frag = ACT ? (of0 + f % OF) * a.gate_step + (f < OF ? 0 : a.up_step) : of0 + f;
    wo[f] = pack_row_offset(frag) + static_cast<uint32_t>(lane) * 16u;
  }
#pragma unroll
  for (int j = 0; j < XN; ++j) {
    const int g = wave + 4 * j;                            // rows GR g ... of the tile, CH lanes each
    const int row = mt * 16 * MT + GR * g + lane / CH;
    const int chunk = (lane % CH) ^ ((GR * wave + lane / CH) % CH);
    xo[j] = (g < GROUPS && row < a.M) ? static_cast<uint32_t>(static_cast<int64_t>(row) * a.ldx * 2) + 16u * chunk
                                      : kOutOfRange;
    xl[j] = 8 * chunk < k_tail ? 0u : kOutOfRange;
  }
  // Gated LoRA: the first 32 rank elements of this wavefront's rows of B, as MFMA operands (row lane % 16,
  // elements 8 * (lane / 16) ..), requested ahead of everything else.
  [[maybe_unused]] u32x4 b_first[NF];
  [[maybe_unused]] __amdgpu_buffer_rsrc_t br;
  [[maybe_unused]] auto load_b = [&](int f, int j) __attribute__((always_inline)) {
    const int n = 16 * (of0 + f) + (lane & 15), e = 32 * j + 8 * (lane >> 4);
    const uint32_t off = n < a.N && e < a.lora.rank ? static_cast<uint32_t>((n * a.lora.rank + e) * 2) : kOutOfRange;
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(br, static_cast<int>(off), 0, 0));
  };
  if constexpr (EPI == kWideLora) {
    if (!forms_h) {
      br = make_rsrc(a.lora.b, static_cast<uint32_t>(a.N * a.lora.rank * 2));
#pragma unroll
      for (int f = 0; f < NF; ++f) b_first[f] = load_b(f, 0);
    }
  }
  const int rd0 = (lane & 15) * CH + ((lane >> 4) ^ (lane & 15) % CH);  // K step h of a stage: rd0 ^ 4h
  u32x4 W[S * D][NF], X[D][XN];
  // A stage's scalar offsets, with the sign bit set past the last stage: it puts the whole load out of
  // range (zeros, no traffic). With ALIGNED ranges eight K steps lie in one group of the packed weight, a
  // D-stage block apart: one multiply per stage and the steps as instruction offsets. A wavefront alone
  // on its SIMD issues about one instruction per four clocks, so these counts are what short tiles run at.
  struct StageOffsets {
    int w[S], x;
    uint32_t tail;  // in the last stage, the bit that takes lanes past K out of range
  };
  auto offsets = [&](int i, int jw) __attribute__((always_inline)) {
    StageOffsets o;
    const uint32_t gone = i < stages ? 0u : kWideNoLoad;
    if constexpr (ALIGNED) {
      const uint32_t base = (static_cast<uint32_t>(lo + S * i) >> 3) * a.wgroup + static_cast<uint32_t>(jw * S) * kPackFragBytes;
      o.w[0] = static_cast<int>(base | gone);
    } else {
#pragma unroll
      for (int h = 0; h < S; ++h)
        o.w[h] = __builtin_amdgcn_readfirstlane(static_cast<int>(
            pack_step_offset(lo + S * i + h, a.wgroup) | (static_cast<uint32_t>(hi - lo - 1 - S * i - h) & kWideNoLoad)));
    }
    o.x = static_cast<int>((static_cast<uint32_t>(lo + S * i) * 64u) | gone);
    o.tail = i == stages - 1 ? kOutOfRange : 0u;
    return o;
  };
  auto load_w = [&](const StageOffsets& o, int h, int f, u32x4& w) __attribute__((always_inline)) {
    if constexpr (ALIGNED)
      w = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, wo[f] + h * kPackFragBytes, o.w[0], 0));
    else
      w = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, wo[f], o.w[h], 0));
  };
  auto load_x = [&](const StageOffsets& o, u32x4 (&x)[XN]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < XN; ++j)
      x[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, xo[j] | (xl[j] & o.tail), o.x, 0));
  };
  auto put_x = [&](int slot, const u32x4 (&x)[XN]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < XN; ++j)
      if (4 * j + 3 < GROUPS || wave + 4 * j < GROUPS) lds[slot * kStageWords + (wave + 4 * j) * 64 + lane] = x[j];
  };
  f32x4 acc[NF][MT];
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[f][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < D; ++j) {
    const StageOffsets o = offsets(j, j);
    load_x(o, X[j]);
#pragma unroll
    for (int h = 0; h < S; ++h)
#pragma unroll
      for (int f = 0; f < NF; ++f) load_w(o, h, f, W[S * j + h][f]);
    __builtin_amdgcn_sched_barrier(0);
  }
  put_x(0, X[0]);
  load_x(offsets(D, 0), X[0]);
  if constexpr (S == 4) {
    // Two buffers of operands: while a stage's MFMAs run, the next stage's X is read whole and the one
    // after it written, so a stage waits for one LDS round trip.
    u32x4 B[2][S][MT];
    wide_sync();
#pragma unroll
    for (int h = 0; h < S; ++h)
#pragma unroll
      for (int t = 0; t < MT; ++t) B[0][h][t] = lds[t * 16 * CH + (rd0 ^ (4 * h))];
    put_x(1, X[1]);
    load_x(offsets(D + 1, 1), X[1]);
    wide_sync();
    __builtin_amdgcn_sched_barrier(0);
    // Stage i in register slot j = i % D (D = 2), which is also its LDS slot.
    auto stage = [&](int j, int i) __attribute__((always_inline)) {
      const StageOffsets o = offsets(i + D, j);
#pragma unroll
      for (int h = 0; h < S; ++h)
#pragma unroll
        for (int t = 0; t < MT; ++t) B[j ^ 1][h][t] = lds[(j ^ 1) * kStageWords + t * 16 * CH + (rd0 ^ (4 * h))];
#pragma unroll
      for (int h = 0; h < S; ++h) {
#pragma unroll
        for (int f = 0; f < NF; ++f) {
#pragma unroll
          for (int t = 0; t < MT; ++t) acc[f][t] = mfma_16x16x32<DT>(W[S * j + h][f], B[j][h][t], acc[f][t]);
          load_w(o, h, f, W[S * j + h][f]);
        }
      }
      put_x(j, X[j]);  // stage i + 2: every wavefront read stage i's X before the last barrier
      load_x(offsets(i + 2 + D, j), X[j]);
      wide_sync();
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int j = 0; j < D; ++j) stage(j, j);
    for (int i = D; i < stages; i += D) {
#pragma unroll
      for (int j = 0; j < D; ++j) stage(j, i + j);
    }
  } else {
    u32x4 B0[MT], B1[MT];
    const int rd1 = rd0 ^ 4;
    wide_sync();
#pragma unroll
    for (int t = 0; t < MT; ++t) B0[t] = lds[t * 128 + rd0];
    // Stage i in register slot j = i % D. B0 holds its first K step's X operands.
    auto stage = [&](int j, int i) __attribute__((always_inline)) {
      const int slot = j & 1, jn = (j + 1) % D;
      const StageOffsets o = offsets(i + D, j), ox = offsets(i + 1 + D, jn);
#pragma unroll
      for (int t = 0; t < MT; ++t) B1[t] = lds[slot * kStageWords + t * 128 + rd1];
#pragma unroll
      for (int f = 0; f < NF; ++f) {
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[f][t] = mfma_16x16x32<DT>(W[2 * j][f], B0[t], acc[f][t]);
        load_w(o, 0, f, W[2 * j][f]);
      }
      put_x(slot ^ 1, X[jn]);
      load_x(ox, X[jn]);
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        __builtin_amdgcn_sched_group_barrier(kDsRead, 1, 0);
        __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
        if (NF == 1 && t < XN) {
          __builtin_amdgcn_sched_group_barrier(kDsWrite, 1, 0);
          __builtin_amdgcn_sched_group_barrier(kVmemRead, 1, 0);
        }
      }
#pragma unroll
      for (int t = 0; t < (NF - 1) * MT; ++t) {
        if ((t & 1) == 0 && t / 2 < XN)
          __builtin_amdgcn_sched_group_barrier(kDsWrite, 1, 0);
        else
          __builtin_amdgcn_sched_group_barrier(kVmemRead, 1, 0);
        __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
      }
      // Every wavefront has read this stage's X and written the next one's.
      wide_sync();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < MT; ++t) B0[t] = lds[(slot ^ 1) * kStageWords + t * 128 + rd0];
#pragma unroll
      for (int f = 0; f < NF; ++f) {
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[f][t] = mfma_16x16x32<DT>(W[2 * j + 1][f], B1[t], acc[f][t]);
        load_w(o, 1, f, W[2 * j + 1][f]);
      }
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        __builtin_amdgcn_sched_group_barrier(kDsRead, 1, 0);
        __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
      }
#pragma unroll
      for (int f = 1; f < NF; ++f) {
        __builtin_amdgcn_sched_group_barrier(kVmemRead, 1, 0);
#pragma unroll
        for (int t = 0; t < MT; ++t) __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    // The first D stages peeled off: the loop is entered only with its own load order in flight, so the
    // compiler's load-count waits stay exact. Stages past the last multiply zeros.
#pragma unroll
    for (int j = 0; j < D; ++j) stage(j, j);
    for (int i = D; i < stages; i += D) {
#pragma unroll
      for (int j = 0; j < D; ++j) stage(j, i + j);
    }
  }

  if (a.split > 1) {
    // This split's sums, written through; the last of the tile's splits to arrive adds all of them in
    // split order. Weight fragment wf of the packed order, X fragment xf; fragments past N or M are
    // neither stored nor loaded (out of range).
    const int wfrags = ((ACT ? 2 * a.N : a.N) + 15) >> 4, xfrags = (a.M + 15) >> 4;
    const auto pr = make_rsrc(a.partial, static_cast<uint32_t>(a.split * wfrags * xfrags) * 1024u);
    uint32_t po[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const int wf = ACT ? 2 * (of0 + f % OF) + f / OF : of0 + f;
      po[f] = wf < wfrags ? static_cast<uint32_t>(wf * xfrags + mt * MT) * 1024u + static_cast<uint32_t>(lane) * 16u
                          : kOutOfRange;
    }
    const uint32_t plane = static_cast<uint32_t>(wfrags * xfrags) * 1024u;
    const int mts = min(MT, xfrags - mt * MT);
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int t = 0; t < MT; ++t)
        if (t < mts)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[f][t]), pr, po[f] + t * 1024u,
                                                 static_cast<int>(static_cast<uint32_t>(sp) * plane), kCoherent);
    __builtin_amdgcn_s_waitcnt(0);
    wide_sync();  // every wavefront's partials are written, and no one reads X in LDS any more
    if (threadIdx.x == 0) {
      int* counter = a.arrive + nt * a.mtiles + mt;
      const int before = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const bool last = before == a.split - 1;
      if (last) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      lds[0][0] = last;
    }
    wide_sync();
    if (lds[0][0] == 0) return;
    // Four splits' loads in flight at a time (two where a wavefront holds many fragments).
    constexpr int kBatch = NF * MT <= 8 ? 4 : 2;
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[f][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < a.split; s0 += kBatch) {
      u32x4 v[kBatch][NF][MT];
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        const int so = static_cast<int>(s0 + b < a.split ? static_cast<uint32_t>(s0 + b) * plane : kWideNoLoad);
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
          for (int t = 0; t < MT; ++t)
            v[b][f][t] = __builtin_bit_cast(
                u32x4, __builtin_amdgcn_raw_buffer_load_b128(pr, t < mts ? po[f] + t * 1024u : kOutOfRange, so, kCoherent));
      }
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        if (s0 + b >= a.split) break;
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
          for (int t = 0; t < MT; ++t) acc[f][t] += __builtin_bit_cast(f32x4, v[b][f][t]);
      }
    }
  }

  if constexpr (EPI == kWideLora) {
    const WideLora& z = a.lora;
    if (forms_h) {
      // Written through for the base workgroups of every XCD, then counted in.
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          const int m = mt * 16 * MT + 16 * t + (lane & 15), n = 16 * (of0 + f) + 4 * (lane >> 4);
          if (m >= a.M || n >= a.N) continue;  // the width is a multiple of 8: all four columns are in range
          const f32x4 v = acc[f][t];
          const uint64_t lo2 = static_cast<uint64_t>(to_bits16<DT>(v[0])) | (static_cast<uint64_t>(to_bits16<DT>(v[1])) << 16);
          const uint64_t hi2 = static_cast<uint64_t>(to_bits16<DT>(v[2])) | (static_cast<uint64_t>(to_bits16<DT>(v[3])) << 16);
          publish(reinterpret_cast<uint64_t*>(z.h + static_cast<int64_t>(m) * z.width + n), lo2 | (hi2 << 32));
        }
      __builtin_amdgcn_s_waitcnt(0);
      wide_sync();
      if (threadIdx.x == 0)
        __hip_atomic_fetch_add(z.counters + kPkLoraHDone, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
    wide_wait_h(z);
    // Rows m >= gated_from: the base value rounded to the model dtype plus sum_j h[m, s rank + j] B[n, j],
    // s the shard of column n, as MFMAs over 32 rank elements. A fragment that straddles shards forms the
    // product with each shard's h by itself and takes a column's value from its own shard's (the other
    // shards' columns are zero rows of B, but an overflowed h times zero is NaN).
    const auto hr = make_rsrc(z.h, static_cast<uint32_t>(a.M * z.width * 2));
    auto shard_of = [&](int n) { return (n >= z.shard_end[0]) + (n >= z.shard_end[1]) + (n >= z.shard_end[2]); };
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const int nf = __builtin_amdgcn_readfirstlane(16 * (of0 + f));
      const int s_lo = shard_of(min(nf, a.N - 1)), s_hi = shard_of(min(nf + 15, a.N - 1));
      const int s_own = shard_of(nf + (lane & 15));
      // Over the fragment's shards, and for each over 32 rank elements at a time, in one copy of the code (a
      // second, for straddling fragments only, took 11.3 us at 3072x2048, rank 16, M = 56, this 10.9); `done`
      // holds the columns of the shards before.
      f32x4 corr[MT], done[MT];
#pragma unroll
      for (int t = 0; t < MT; ++t) corr[t] = done[t] = f32x4{0.f, 0.f, 0.f, 0.f};
      int s = s_lo;
      for (int j = 0;;) {
        const u32x4 row = j == 0 ? b_first[f] : load_b(f, j);
        const u32x4 bs = s_own == s ? row : u32x4{0u, 0u, 0u, 0u};
        const int e = 32 * j + 8 * (lane >> 4);
        u32x4 hv[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          const int m = mt * 16 * MT + 16 * t + (lane & 15);
          const uint32_t off = m < a.M && e < z.rank ? static_cast<uint32_t>((m * z.width + s * z.rank + e) * 2) : kOutOfRange;
          hv[t] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(hr, static_cast<int>(off), 0, kCoherent));
        }
#pragma unroll
        for (int t = 0; t < MT; ++t) corr[t] = mfma_16x16x32<DT>(bs, hv[t], corr[t]);
        if (32 * ++j < z.rank) continue;
        if (s_lo != s_hi) {
#pragma unroll
          for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int own = shard_of(nf + 4 * (lane >> 4) + r);
              done[t][r] = own == s ? corr[t][r] : done[t][r];
              corr[t][r] = s == s_hi ? done[t][r] : 0.f;
            }
        }
        if (++s > s_hi) break;
        j = 0;
      }
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const bool gated = mt * 16 * MT + 16 * t + (lane & 15) >= z.gated_from;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          acc[f][t][r] = gated ? from_bits16<DT>(to_bits16<DT>(acc[f][t][r])) + corr[t][r] : acc[f][t][r];
      }
    }
    // The last base tile to pass its wait leaves both counters ready for the next launch.
    wide_sync();
    if (threadIdx.x == 0 && __hip_atomic_fetch_add(z.counters + kPkLoraPast, 1, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT) == z.base_tiles - 1) {
      publish(z.counters + kPkLoraHDone, 0);
      publish(z.counters + kPkLoraPast, 0);
    }
  }

  // Fragment (f, t): output columns n0 + 16f + 4*(lane/16) + r, row m0 + 16t + lane%16.
  const int m0 = mt * 16 * MT;
  if constexpr (!ACT) {
    if (a.out_f32) {
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          const int m = m0 + 16 * t + (lane & 15), n = 16 * (of0 + f) + 4 * (lane >> 4);
          if (m < a.M && n < a.N) wide_store4_f32<DT>(a, m, n, acc[f][t]);
        }
      return;
    }
  }
  // 16-bit output: the tile in LDS as rows of OC 16-byte chunks, chunk c of row m at slot c ^ (m % 8).
  wide_sync();
  u32x2* half = reinterpret_cast<u32x2*>(lds);
#pragma unroll
  for (int f = 0; f < OF; ++f)
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      uint16_t h[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if constexpr (ACT)
          h[r] = silu_mul_bits<DT>(acc[f][t][r], acc[f + OF][t][r]);
        else
          h[r] = to_bits16<DT>(acc[f][t][r]);
      }
      const int m = 16 * t + (lane & 15), q = 4 * (OF * wave + f) + (lane >> 4);  // q: 8-byte piece of the row
      half[(m * OC + ((q >> 1) ^ (m & 7))) * 2 + (q & 1)] =
          u32x2{static_cast<uint32_t>(h[0]) | (static_cast<uint32_t>(h[1]) << 16),
                static_cast<uint32_t>(h[2]) | (static_cast<uint32_t>(h[3]) << 16)};
    }
  wide_sync();
  uint16_t* y = static_cast<uint16_t*>(a.y);
  const bool wide16 = (reinterpret_cast<uintptr_t>(y) & 15) == 0 && (a.ldy & 7) == 0;
  for (int i = threadIdx.x; i < kOutWords; i += kWideThreads) {
    const int row = i / OC, c = i - row * OC;
    const int m = m0 + row, n = 16 * (nt * kWideWaves * OF) + 8 * c;
    if (m >= a.M || n >= a.N) continue;
    const u32x4 v = lds[row * OC + (c ^ (row & 7))];
    uint16_t* dst = y + static_cast<int64_t>(m) * a.ldy + n;
    if (wide16 && n + 8 <= a.N) {
      *reinterpret_cast<u32x4*>(dst) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t word = v[e >> 1];
        if (n + e < a.N) dst[e] = static_cast<uint16_t>(e & 1 ? word >> 16 : word & 0xffffu);
      }
    }
  }
}

// The compiled tiles: 64*nf weight rows by 16*mt rows of X.
struct WideTile {
  int nf, mt;
};
constexpr WideTile kWideTiles[] = {{1, 1}, {1, 2}, {1, 3}, {1, 4}, {1, 5}, {1, 8}, {2, 1}, {2, 2},
                                   {2, 3}, {2, 4}, {2, 5}, {2, 6}, {2, 8}, {2, 10}, {4, 8}};
constexpr int kWideCus = 256;

// The tile with the least modelled time per K step: the rounds of tiles a CU runs times the KiB each
// loads per K step (4*nf of W, mt of X), the rate of the CU's memory path being the bound. Against the
// best of all tiles timed one by one at M = 640 and 256 of the 1.3B block's linears and M = 200 and 110
// of the 3B gate/up, its choice was the fastest or within 4 %; M = 7 to 110 of the round linears within
// 10 % (a few of the shortest, by 0.1-0.3 us). The activation needs gate and up
// fragments in one wavefront, hence an even nf.
WideTile wide_pick(int64_t M, int64_t N, int64_t split, bool act) {
  WideTile best{0, 0};
  int64_t best_cost = INT64_MAX;
  for (const WideTile& t : kWideTiles) {
    if (act && t.nf % 2 != 0) continue;
    const int64_t tn = 64 * t.nf / (act ? 2 : 1);
    const int64_t tiles = ((N + tn - 1) / tn) * ((M + 16 * t.mt - 1) / (16 * t.mt)) * split;
    const int64_t cost = (tiles + kWideCus - 1) / kWideCus * (4 * t.nf + t.mt);
    if (cost < best_cost) {
      best_cost = cost;
      best = t;
    }
  }
  return best;
}

template <int DT, int NF, int MT, int EPI>
hipError_t wide_go(WideArgs a, hipStream_t stream) {
  constexpr int tn = 64 * NF / (EPI == kWideAct ? 2 : 1), tm = 16 * MT;
  const int64_t mtiles = (a.M + tm - 1) / tm, ntiles = (static_cast<int64_t>(a.N) + tn - 1) / tn;
  int64_t counters = a.split > 1 ? mtiles * ntiles : 0;
  if (mtiles * ntiles * a.split > (int64_t(1) << 28)) return hipErrorInvalidConfiguration;
  a.mtiles = static_cast<int>(mtiles);
  a.tiles = static_cast<int>(mtiles * ntiles);
  a.per_xcd = (a.tiles * a.split + 7) / 8;
  unsigned grid = static_cast<unsigned>(8 * a.per_xcd);
  if constexpr (EPI == kWideLora) {
    a.lora.base_tiles = a.tiles;
    a.lora.tiles = static_cast<int>(mtiles * ((a.lora.width + tn - 1) / tn));
    a.lora.items = a.lora.tiles * a.lora.split;
    a.lora.arrive = a.lora.counters + kPackedArriveBase + counters;
    counters += a.lora.split > 1 ? a.lora.tiles : 0;
    grid += static_cast<unsigned>(a.lora.items);
  }
  if (counters > kPackedBarrierBase - kPackedArriveBase) return hipErrorInvalidConfiguration;
  // Every range of K steps starts at a group of the packed weight and, but for K's end (zero fragments
  // follow), ends at one.
  auto aligned = [&](int split) { return split == 1 || a.Ks % (kPackGroup * split) == 0; };
  constexpr bool block = wide_steps<NF, MT>() * wide_depth<NF, MT>() == kPackGroup;
  auto kern = wide_gemm_kernel<DT, NF, MT, EPI, false>;
  if constexpr (block)
    if (aligned(a.split) && (EPI != kWideLora || aligned(a.lora.split))) kern = wide_gemm_kernel<DT, NF, MT, EPI, true>;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(kWideThreads), 0, stream, a);
  return hipGetLastError();
}

template <int DT, int EPI>
hipError_t wide_dispatch(const WideArgs& a, WideTile t, hipStream_t s) {
  switch (16 * t.nf + t.mt) {
    case 16 * 2 + 1: return wide_go<DT, 2, 1, EPI>(a, s);
    case 16 * 2 + 2: return wide_go<DT, 2, 2, EPI>(a, s);
    case 16 * 2 + 3: return wide_go<DT, 2, 3, EPI>(a, s);
    case 16 * 2 + 4: return wide_go<DT, 2, 4, EPI>(a, s);
    case 16 * 2 + 5: return wide_go<DT, 2, 5, EPI>(a, s);
    case 16 * 2 + 6: return wide_go<DT, 2, 6, EPI>(a, s);
    case 16 * 2 + 8: return wide_go<DT, 2, 8, EPI>(a, s);
    default: break;
  }
  if constexpr (EPI != kWideLora) {  // past 128 rows, or more than 256 tiles of 128 x 128
    switch (16 * t.nf + t.mt) {
      case 16 * 2 + 10: return wide_go<DT, 2, 10, EPI>(a, s);
      case 16 * 4 + 8: return wide_go<DT, 4, 8, EPI>(a, s);
      default: break;
    }
  }
  if constexpr (EPI != kWideAct) {
    switch (16 * t.nf + t.mt) {
      case 16 + 1: return wide_go<DT, 1, 1, EPI>(a, s);
      case 16 + 2: return wide_go<DT, 1, 2, EPI>(a, s);
      case 16 + 3: return wide_go<DT, 1, 3, EPI>(a, s);
      case 16 + 4: return wide_go<DT, 1, 4, EPI>(a, s);
      case 16 + 5: return wide_go<DT, 1, 5, EPI>(a, s);
      case 16 + 8: return wide_go<DT, 1, 8, EPI>(a, s);
      default: break;
    }
  }
  return hipErrorInvalidConfiguration;
}

// Fills what every launch needs; N: the weight's rows.
WideArgs wide_args(const void* x, int64_t ldx, const void* wp, void* y, int64_t ldy, int64_t M, int64_t N, int64_t K,
                   WideOut out, int split, void* workspace) {
  const bool act = out == WideOut::kActPlain || out == WideOut::kActInterleaved;
  WideArgs a{};
  a.x = x;
  a.w = wp;
  a.y = y;
  a.ldx = ldx;
  a.ldy = ldy;
  a.M = static_cast<int>(M);
  a.N = static_cast<int>(act ? N / 2 : N);
  a.K = static_cast<int>(K);
  a.Ks = static_cast<int>((K + 31) / 32);
  a.out_f32 = out == WideOut::kF32;
  a.wbytes = static_cast<uint32_t>(pack_bytes(N, a.Ks));
  a.wgroup = pack_group_bytes(N);
  a.gate_step = out == WideOut::kActInterleaved ? 2 : 1;
  a.up_step = out == WideOut::kActInterleaved ? 1 : a.N / 16;
  a.split = split;
  if (split > 1) {
    a.arrive = static_cast<int*>(workspace) + kPackedArriveBase;
    a.partial = reinterpret_cast<float*>(static_cast<char*>(workspace) + kCounterBytes);
  }
  return a;
}

int wide_status(hipError_t err) {
  return err == hipSuccess ? PLM_OK : err == hipErrorInvalidConfiguration ? PLM_ERR_ARGUMENT : PLM_ERR_LAUNCH;
}

}  // namespace

// The scratch a caller of plm_gemm_packed provides above 128 rows. The kernel itself needs none (a K
// split would change the sums' order); the sizes callers reserve and the refusal of a smaller
// workspace are the interface's and stay.
int64_t wide_workspace(int64_t M, int64_t N, int64_t K, int64_t cap) {
  const int64_t tiles = ((N + 127) / 128) * ((M + 127) / 128), ks = (K + 31) / 32;
  const auto bytes = [&](int64_t s) { return static_cast<int64_t>(kCounterBytes) + tiles * s * 64 * 1024; };
  int64_t split = 1;
  while (tiles * split * 2 <= 320 && ks / (split * 2) >= 16 && split < 8 && bytes(split * 2) <= cap) split *= 2;
  return split == 1 ? 0 : bytes(split);
}

int wide_gemm(int32_t dtype, const void* x, int64_t ldx, const void* wp, void* y, int64_t ldy, int64_t M, int64_t N,
              int64_t K, hipStream_t stream, WideOut out, int split, void* workspace) {
  const WideArgs a = wide_args(x, ldx, wp, y, ldy, M, N, K, out, split, workspace);
  const bool act = out == WideOut::kActPlain || out == WideOut::kActInterleaved;
  const WideTile t = wide_pick(M, a.N, split, act);
  if (dtype == PLM_BF16)
    return wide_status(act ? wide_dispatch<DT_BF16, kWideAct>(a, t, stream) : wide_dispatch<DT_BF16, kWidePlain>(a, t, stream));
  return wide_status(act ? wide_dispatch<DT_F16, kWideAct>(a, t, stream) : wide_dispatch<DT_F16, kWidePlain>(a, t, stream));
}

int wide_lora(int32_t dtype, const void* x, int64_t ldx, const void* wp, void* y, int64_t ldy, int64_t M, int64_t N,
              int64_t K, int split, const WideLoraCall& c, hipStream_t stream) {
  WideArgs a = wide_args(x, ldx, wp, y, ldy, M, N, K, WideOut::kModel, split, c.workspace);
  char* ws = static_cast<char*>(c.workspace);
  WideLora& z = a.lora;
  z.w = c.packed_a;
  z.h = reinterpret_cast<uint16_t*>(ws + c.h_offset);
  z.b = c.b;
  z.width = c.width;
  z.wbytes = static_cast<uint32_t>(pack_bytes(c.width, a.Ks));
  z.wgroup = pack_group_bytes(c.width);
  z.split = c.h_split;
  z.rank = c.rank;
  z.gated_from = c.gated_from;
  for (int i = 0; i < 3; ++i) z.shard_end[i] = c.shard_end[i];
  z.partial = reinterpret_cast<float*>(ws + kCounterBytes) + c.h_partial;
  z.counters = reinterpret_cast<int*>(ws);
  z.spin_limit = c.spin_limit;
  const WideTile t = wide_pick(M, N, split, false);
  return wide_status(dtype == PLM_BF16 ? wide_dispatch<DT_BF16, kWideLora>(a, t, stream)
                                       : wide_dispatch<DT_F16, kWideLora>(a, t, stream));
}

}  // namespace plm
