// The int4 GEMM at prefill sizes (gptq_tall.hip): host interface.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gptq {

// Can the tall kernel run this GEMM?  (K in whole k64-steps, groups of 64 * 2^n rows, no act-order permutation, act 0 or 2)
bool tall_serves(int64_t K, int64_t groups, bool act_order, int act);
// ... and does it, at M rows?  (from tall_min_m(); up to 256 rows where the streaming passes would take longer)
bool tall_ok(int64_t M, int64_t K, int64_t N, int64_t groups, bool act_order, int act);
// ... and is it, where it serves, the faster way than dequantising and a library GEMM?
bool tall_before_library(int64_t M, int64_t K, int64_t N, int act);
int64_t tall_min_m(int act);
int64_t tall_max_m();
// fp32 scratch of launch_tall
int64_t tall_workspace_bytes(int64_t M, int64_t K, int64_t N);
int launch_tall(const void* x, int64_t ldx, const void* prepared, const void* bias, void* out, int64_t ldo, int64_t M, int64_t K,
                int64_t N, int64_t groups, int act, float* scratch, hipStream_t st);

}  // namespace gptq
