// The wide GEMM over packed weights: behind plm_gemm_wide, behind plm_gemm_packed and its variants above 128
// rows and for row-split tiles, and behind plm_gemm_packed_silu_mul, plm_gemm_packed_lora and the links of
// plm_gemm_chain_packed on such tiles. Arguments are checked by the caller (csrc/packed_api.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace plm {

// The workspace bytes plm_gemm_packed asks its callers for above 128 rows; a caller whose scratch is
// fixed gives its size as `cap`.
constexpr int64_t kNoCap = INT64_MAX;
int64_t wide_workspace(int64_t M, int64_t N, int64_t K, int64_t cap = kNoCap);

// What is written: Y in the input dtype, the fp32 accumulator, or the SiLU-and-multiply Y[M, N/2] of a
// fused gate/up weight packed as it is (gate rows first) or with its halves interleaved by fragment.
enum class WideOut { kModel, kF32, kActPlain, kActInterleaved };

// Y = X W^T; returns a PLM_* status. With split > 1 each of `split` ranges of K steps is one chain and
// the ranges' sums are added in order (the sums of a row-split packed tile with that split_k, bit for
// bit); `workspace` then holds the counter area and split * ceil(N/16) * ceil(M/16) fp32 fragments.
int wide_gemm(int32_t dtype, const void* x, int64_t ldx, const void* wp, void* y, int64_t ldy, int64_t M, int64_t N,
              int64_t K, hipStream_t stream, WideOut out, int split = 1, void* workspace = nullptr);

// The gated-LoRA launch's second half: h = X A^T and the correction (plm_gemm_packed_lora).
struct WideLoraCall {
  const void* packed_a;
  const uint16_t* b;          // [N][rank]
  int width, rank, gated_from;
  int shard_end[3];
  int h_split;                // K splits of the h linear
  int64_t h_partial;          // its partials' float offset behind the counter area
  int64_t h_offset;           // h's byte offset in the workspace
  int spin_limit;
  void* workspace;
};
int wide_lora(int32_t dtype, const void* x, int64_t ldx, const void* wp, void* y, int64_t ldy, int64_t M, int64_t N,
              int64_t K, int split, const WideLoraCall& c, hipStream_t stream);

}  // namespace plm
