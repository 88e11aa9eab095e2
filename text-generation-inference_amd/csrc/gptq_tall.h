// The int4 GEMM at prefill sizes (gptq_tall.hip): host interface.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gptq {

// Can the tall kernel run this GEMM?  (K in whole k64-steps, groups of 64 * 2^n rows, no act-order permutation, act 0 or 2)
bool tall_serves(int64_t K, int64_t groups, bool act_order, int act);
// ... and does it, at M rows?  (from tall_min_m(); up to 256 rows where the streaming passes would take longer)
bool tall_ok(int64_t M, int64_t K, int64_t N, int64_t groups, bool act_order, int act);
// ... and its deferred form?  (up to 256 rows the streaming passes leave fewer and smaller slabs)
bool tall_partial_ok(int64_t M, int64_t K, int64_t groups, const int32_t* perm, int act);
int64_t tall_min_m(int act);
int64_t tall_max_m();
// fp32 scratch of launch_tall
int64_t tall_workspace_bytes(int64_t M, int64_t K, int64_t N);
int launch_tall(const void* x, int64_t ldx, const void* prepared, const void* bias, void* out, int64_t ldo, int64_t M, int64_t K,
                int64_t N, int64_t groups, int act, float* scratch, hipStream_t st);
// deferred form: tall_partial_splits() fp32 slabs in 32-row units [unit][S][32][N rounded up to 32]
int tall_partial_splits(int64_t M, int64_t K, int64_t N);
int64_t tall_slab_bytes(int64_t M, int64_t N, int S);
int launch_tall_partial(const void* x, int64_t ldx, const void* prepared, int64_t M, int64_t K, int64_t N, int64_t groups, float* slabs,
                        hipStream_t st);

}  // namespace gptq
