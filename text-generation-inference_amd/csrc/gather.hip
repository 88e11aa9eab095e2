// Column gather of a two-byte activation: out[m][k] = x[m][perm[k]] (0 where perm[k] is outside x), row-major or in fragment order.
//
// An act-order (g_idx) int4 matrix has its rows sorted by group when its image is prepared, so its operand has to be gathered with
// the same permutation.  A GEMM that gathers while it stages its operand does so once per workgroup that reads a row and cannot take
// the operand in fragment order: 32 - 59 us per launch at 11 rows of the 7B shapes against 8 - 16 us for the fragment-order kernel.
// Gathering once, in front of it, costs one launch of a few us.
//
// A row is staged in LDS, because the gather itself is one two-byte read per element at a random place: from the vector cache that is
// a line per lane, from LDS a handful of cycles per wave.  A thread writes eight neighbouring columns, 16 bytes in either layout.
#include "common.h"

namespace {

constexpr int GT = 512;                 // threads
constexpr int64_t GATHER_LDS = 65536;   // bytes of LDS a row may take; longer rows are gathered from memory

template <bool STAGED>
__global__ __launch_bounds__(GT) void gather_columns_kernel(const uint16_t* __restrict__ x, int64_t ldx,
                                                            const int32_t* __restrict__ perm, uint16_t* __restrict__ out,
                                                            int64_t ldo, int M, int in_cols, int K, int vec, int frag) {
    using U8 = uint16_t __attribute__((ext_vector_type(8)));
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    uint16_t* row = reinterpret_cast<uint16_t*>(smem);
    // the first (up to 4096 columns the only) indices of a thread: asked for in front of the row, kept for all rows
    int first[8];
    if ((int)threadIdx.x * 8 < K) {
#pragma unroll
        for (int e = 0; e < 8; ++e) first[e] = perm[threadIdx.x * 8 + e];
    }
    for (int m = blockIdx.x; m < M; m += gridDim.x) {
        const uint16_t* xr = x + (int64_t)m * ldx;
        if (STAGED) {
            if (vec) {
                for (int c = threadIdx.x; c * 8 < in_cols; c += GT)
                    *reinterpret_cast<U8*>(row + c * 8) = *reinterpret_cast<const U8*>(xr + c * 8);
            } else {
                for (int c = threadIdx.x; c < in_cols; c += GT) row[c] = xr[c];
            }
            __syncthreads();
        }
        for (int c = threadIdx.x; c * 8 < K; c += GT) {
            U8 o;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int s = c < GT ? first[e] : perm[c * 8 + e];
                const bool in = (unsigned)s < (unsigned)in_cols;
                const uint16_t v = STAGED ? row[in ? s : 0] : xr[in ? s : 0];
                o[e] = in ? v : (uint16_t)0;
            }
            *reinterpret_cast<U8*>(out + (frag ? xf_off(m, c * 8, K) : (int64_t)m * ldo + c * 8)) = o;
        }
        if (STAGED) __syncthreads();
    }
}

}  // namespace

extern "C" int tgis_gather_columns(const void* x, int64_t ldx, const int32_t* perm, void* out, int64_t ldo, int64_t M,
                                   int64_t in_cols, int64_t K, void* stream) {
    const bool frag = ldo == TGIS_LD_FRAGMENTS;
    TGIS_CHECK_ARG(x && perm && out, "tgis_gather_columns: null tensor");
    TGIS_CHECK_ARG(M >= 0 && M <= 2147483647LL && in_cols >= 1 && in_cols <= 2147483647LL && ldx >= in_cols && K >= 8 &&
                       K <= 2147483647LL && K % 8 == 0,
                   "tgis_gather_columns: bad shape (M=%ld in_cols=%ld ldx=%ld K=%ld)", (long)M, (long)in_cols, (long)ldx, (long)K);
    TGIS_CHECK_ARG(((uintptr_t)out % 16) == 0 && (frag ? (M <= 64 && K % 64 == 0) : (ldo >= K && ldo % 8 == 0)),
                   "tgis_gather_columns: out has 16-byte aligned rows, or — M <= 64, K %% 64 == 0 — is in fragment order");
    if (M == 0) return TGIS_OK;
    const int vec = in_cols % 8 == 0 && ldx % 8 == 0 && ((uintptr_t)x % 16) == 0;
    const bool staged = in_cols * 2 <= GATHER_LDS;
    // 8 workgroups of 8 KiB rows share a CU's threads: 2048 keep the chip full, each takes every 2048th row
    const dim3 grid((unsigned)std::min<int64_t>(M, 2048));
    TgisTimedScope timed(TGIS_OP_ACT, (hipStream_t)stream);
    if (staged)
        hipLaunchKernelGGL((gather_columns_kernel<true>), grid, dim3(GT), (size_t)((in_cols * 2 + 15) & ~15LL), (hipStream_t)stream,
                           (const uint16_t*)x, ldx, perm, (uint16_t*)out, ldo, (int)M, (int)in_cols, (int)K, vec, (int)frag);
    else
        hipLaunchKernelGGL((gather_columns_kernel<false>), grid, dim3(GT), 0, (hipStream_t)stream, (const uint16_t*)x, ldx, perm,
                           (uint16_t*)out, ldo, (int)M, (int)in_cols, (int)K, vec, (int)frag);
    TGIS_CHECK_LAUNCH();
    return TGIS_OK;
}
