// Dense products of a decode step of a few rows (up to 4) with the norm in front of them and the residual add behind them.
//
// A layer of a small model at one row is seven dependent launches of 3.5 - 11 us for 88 MB of weights, 14 us at the rate of a large copy: split sums
// that a norm launch adds up, norms of one row on one CU, and projections of 64 column tiles that leave three quarters of the chip idle.  For
// a few rows the operand is small enough (8 KiB of fp32 per row at width 2048) for every workgroup to have all of it, so that
//   * a workgroup owns 8 or 16 columns and the whole k range: 256 workgroups for 2048 columns, no split sums, and the norm of the rows is
//     done by each workgroup for itself while its weights are on their way;
//   * a lane asks for 16 bytes of one column (8 lanes: 128 bytes of neighbouring columns of the image, 8 such runs an instruction), DEPTH of
//     them from the start (all it will ever need up to k = 64 waves DEPTH), and multiplies by vector FMA: at this size the matrix instruction would
//     be fed rows of zeros, and x is a broadcast from LDS;
//   * the residual stream stays in fp32 between the launches: o_proj and down add to it in place, each workgroup its own columns.
// The values and their roundings are those of the launches replaced (norm.hip, dense_finish in dense_gemm_body.h); sums are fp32 in another order.
#include <algorithm>
#include "common.h"
#include "kv_layout.h"

namespace {

enum { ROWS_RESIDUAL = 0, ROWS_HEAD = 1, ROWS_SILU = 2, ROWS_ROPE = 3 };

// waves of a workgroup (us at one row of 2048 x 2048 / 5632 x 2048 / norm + SiLU 2048 x 11264: 8 waves 3.9 / 7.1 / 9.8, 16 waves 3.7 / 6.7 / 10.2)
constexpr int rows_waves(int kind) { return kind == ROWS_RESIDUAL ? 16 : 8; }

struct RowsArgs {
    const void* x;      // RESIDUAL: [M][ldx] of the model dtype
    int64_t ldx;
    float* h;           // [M][width] fp32: what the norm reads (width = K), or what RESIDUAL adds to (width = N)
    const void* norm_w;
    float eps;
    const uint8_t* prep;
    int M, K, N, NT;
    void* out;
    int64_t ldo;
    // ROPE (as tgis_dense_gemm_rope)
    const void* bias;
    const int32_t *positions, *slots;
    const void *cosb, *sinb;
    void *kpool, *vpool;
    int H, Hkv, D;
};

// v summed over the lanes with the same lane % 8, in every one of them
__device__ __forceinline__ float sum_of_eighths(float v) {
    const uint32_t x = __builtin_bit_cast(uint32_t, v);
    const auto a = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    const uint32_t a0 = a[0], a1 = a[1];
    v = __builtin_bit_cast(float, a0) + __builtin_bit_cast(float, a1);
    const uint32_t y = __builtin_bit_cast(uint32_t, v);
    const auto b = __builtin_amdgcn_permlane16_swap(y, y, false, false);
    const uint32_t b0 = b[0], b1 = b[1];
    v = __builtin_bit_cast(float, b0) + __builtin_bit_cast(float, b1);
    return v + row_moved<0x128>(v);
}

// MR rows (M <= MR); KIND decides the operand and the epilogue; PASS: 16-byte loads per thread that bring one row of the operand
template <typename T, int MR, int KIND, int DEPTH, int PASS>
__global__ __launch_bounds__(64 * rows_waves(KIND)) void dense_rows_kernel(RowsArgs a) {
    using V8 = typename VecT<T>::x8;
    using V4 = typename VecT<T>::x4;
    constexpr bool NORM = KIND != ROWS_RESIDUAL;
    constexpr int CPL = NORM ? 2 : 1;  // columns per lane: c and c + 16 of a tile (gate and up, the halves of a rotation), or one
    constexpr int COLS = 8 * CPL, WAVES = rows_waves(KIND), THREADS = 64 * WAVES;
    extern __shared__ __attribute__((aligned(16))) float rows_lds[];
    float* xs = rows_lds;  // [MR][K]
    __shared__ float red[WAVES * MR * COLS], part[WAVES * MR];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = a.K, steps = K >> 6, mine = (steps - w + WAVES - 1) / WAVES;
    const int tile = blockIdx.x / (4 / CPL), c0 = blockIdx.x % (4 / CPL) * 8;  // columns c0 .. c0 + 7 of the tile (and c0 + 16 ..)
    const int c = lane & 7, seg = lane >> 3;

    // the operand, asked for in front of the weights: loads come back in order, and it is needed first
    f32x4 hv[NORM ? MR : 1][NORM ? PASS : 1];
    V4 nw[NORM ? PASS : 1];
    V8 xv[NORM ? 1 : MR][NORM ? 1 : PASS];
#pragma unroll
    for (int p = 0; p < PASS; ++p) {
        if (NORM) {
            const int k = min((p * THREADS + tid) * 4, K - 4);
            nw[p] = *reinterpret_cast<const V4*>(reinterpret_cast<const T*>(a.norm_w) + k);
#pragma unroll
            for (int m = 0; m < MR; ++m) hv[m][p] = *reinterpret_cast<const f32x4*>(a.h + (int64_t)min(m, a.M - 1) * K + k);
        } else {
            const int k = min((p * THREADS + tid) * 8, K - 8);
#pragma unroll
            for (int m = 0; m < MR; ++m) xv[m][p] = ld16<V8>(reinterpret_cast<const T*>(a.x) + (int64_t)min(m, a.M - 1) * a.ldx + k);
        }
    }
    // who finishes which output: (row, column of the workgroup's COLS)
    const int fm = min(lane / COLS, a.M - 1), fc = lane % COLS, fcol = c0 + (fc & 7) + (fc >> 3) * 16;
    int32_t pos = 0, slot = 0;
    if (KIND == ROWS_ROPE) {
        pos = a.positions[fm];
        slot = a.slots[fm];
    }

    const char* wbase = reinterpret_cast<const char*>(a.prep) + (int64_t)tile * steps * 4096 + (seg & 3) * 1024 + (seg >> 2) * 512 + (c0 + c) * 16;
    const int last = mine > 0 ? w + WAVES * (mine - 1) : 0;
    V8 wq[DEPTH][CPL];
    auto ask = [&](int j, V8 (&dst)[CPL]) {
        const char* p = wbase + (int64_t)min(w + WAVES * j, last) * 4096;  // (past the wave's range: its last step again)
#pragma unroll
        for (int t = 0; t < CPL; ++t) dst[t] = __builtin_nontemporal_load(reinterpret_cast<const V8*>(p + t * 256));
    };
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) ask(d, wq[d]);

    if (NORM) {
        float ss[MR];
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            ss[m] = 0.f;
#pragma unroll
            for (int p = 0; p < PASS; ++p)
                if ((p * THREADS + tid) * 4 < K) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) ss[m] += hv[m][p][e] * hv[m][p][e];
                }
            ss[m] = wave_sum(ss[m]);
            if (lane == 0) part[w * MR + m] = ss[m];
        }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            float tot = 0.f;
#pragma unroll
            for (int k = 0; k < WAVES; ++k) tot += part[k * MR + m];
            const float rstd = rsqrtf(tot / K + a.eps);
#pragma unroll
            for (int p = 0; p < PASS; ++p) {
                const int k = (p * THREADS + tid) * 4;
                f32x4 y;
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] = to_f32(from_f32<T>(hv[m][p][e] * rstd * to_f32(nw[p][e])));
                if (k < K) *reinterpret_cast<f32x4*>(xs + m * K + k) = y;
            }
        }
    } else {
#pragma unroll
        for (int m = 0; m < MR; ++m)
#pragma unroll
            for (int p = 0; p < PASS; ++p) {
                const int k = (p * THREADS + tid) * 8;
                if (k < K) {
                    f32x4 lo, hi;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        lo[e] = to_f32(xv[m][p][e]);
                        hi[e] = to_f32(xv[m][p][e + 4]);
                    }
                    *reinterpret_cast<f32x4*>(xs + m * K + k) = lo;
                    *reinterpret_cast<f32x4*>(xs + m * K + k + 4) = hi;
                }
            }
    }
    // what the epilogue reads
    float res = 0.f, cf = 1.f, sf = 0.f;
    bool roth = false;
    int head = 0, dim = 0;
    if (KIND == ROWS_RESIDUAL) res = a.h[(int64_t)fm * a.N + min(tile * 32 + fcol, a.N - 1)];
    if (KIND == ROWS_ROPE) {
        const int per = a.D >> 5, tt = tile % per;
        head = tile / per;
        roth = head < a.H + a.Hkv;
        dim = roth ? ((fcol < 16) ? 16 * tt + fcol : (a.D >> 1) + 16 * tt + (fcol - 16)) : 32 * tt + fcol;
        if (roth) {
            const int64_t at = (int64_t)pos * (a.D >> 1) + 16 * tt + (fcol & 15);
            cf = to_f32(reinterpret_cast<const T*>(a.cosb)[at]);
            sf = to_f32(reinterpret_cast<const T*>(a.sinb)[at]);
        }
    }
    __syncthreads();

    float acc[CPL][MR];
#pragma unroll
    for (int t = 0; t < CPL; ++t)
#pragma unroll
        for (int m = 0; m < MR; ++m) acc[t][m] = 0.f;
    const float* xk = xs + ((seg >> 2) * 4 + (seg & 3)) * 8;
    for (int j0 = 0; j0 < mine; j0 += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            const int j = j0 + d;
            if (j < mine) {
                float wf[CPL][8];
#pragma unroll
                for (int t = 0; t < CPL; ++t)
#pragma unroll
                    for (int e = 0; e < 8; ++e) wf[t][e] = to_f32(wq[d][t][e]);
                const float* xp = xk + (w + WAVES * j) * 64;
#pragma unroll
                for (int m = 0; m < MR; ++m) {
                    const f32x4 lo = *reinterpret_cast<const f32x4*>(xp + m * K), hi = *reinterpret_cast<const f32x4*>(xp + m * K + 4);
#pragma unroll
                    for (int t = 0; t < CPL; ++t)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            acc[t][m] += wf[t][e] * lo[e];
                            acc[t][m] += wf[t][e + 4] * hi[e];
                        }
                }
                if (j + DEPTH < mine) ask(j + DEPTH, wq[d]);
            }
        }
    }
#pragma unroll
    for (int t = 0; t < CPL; ++t)
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            const float v = sum_of_eighths(acc[t][m]);
            if (seg == 0) red[(w * MR + m) * COLS + t * 8 + c] = v;
        }
    __syncthreads();
    if (w != 0) return;
    const bool live = lane / COLS < a.M;  // (lanes without an output repeat the last row's)
    float v = 0.f;
#pragma unroll
    for (int k = 0; k < WAVES; ++k) v += red[(k * MR + fm) * COLS + fc];
    const int n = tile * 32 + fcol;
    if (KIND == ROWS_RESIDUAL) {
        if (live && n < a.N) a.h[(int64_t)fm * a.N + n] = to_f32(from_f32<T>(v)) + to_f32(from_f32<T>(res));
    } else if (KIND == ROWS_HEAD) {
        if (live && n < a.N) reinterpret_cast<float*>(a.out)[(int64_t)fm * a.ldo + n] = v;
    } else if (KIND == ROWS_SILU) {
        const float mine_ = to_f32(from_f32<T>(v)), up = __shfl_xor(mine_, 8, 64);
        const int j = tile * 16 + fcol;
        if (live && fc < 8 && j < (a.N >> 1)) {
            const float sl = mine_ / (1.f + __expf(-mine_));
            reinterpret_cast<T*>(a.out)[(int64_t)fm * a.ldo + j] = from_f32<T>(to_f32(from_f32<T>(sl)) * up);
        }
    } else {
        const int col = head * a.D + dim;
        const float bv = a.bias ? to_f32(reinterpret_cast<const T*>(a.bias)[col]) : 0.f;
        const float own = to_f32(from_f32<T>(v + bv)), other = __shfl_xor(own, 8, 64);
        float o = own;
        if (roth) o = (fcol < 16) ? own * cf - other * sf : other * sf + own * cf;
        const T oh = from_f32<T>(o);
        if (!live) return;
        if (head < a.H) {
            reinterpret_cast<T*>(a.out)[(int64_t)fm * a.ldo + col] = oh;
        } else {
            const int64_t page = slot >> 5;
            const int tok = slot & 31;
            if (roth)
                reinterpret_cast<T*>(a.kpool)[(page * a.Hkv + (head - a.H)) * 32 * a.D + k_off(tok, dim, a.D)] = oh;
            else
                reinterpret_cast<T*>(a.vpool)[(page * a.Hkv + (head - a.H - a.Hkv)) * 32 * a.D + v_off(tok, dim, a.D)] = oh;
        }
    }
}

constexpr int64_t ROWS_LDS = 144 * 1024;

template <typename T, int MR, int KIND, int DEPTH, int PASS>
int launch_rows_one(const RowsArgs& a, hipStream_t st) {
    static const hipError_t attr = hipFuncSetAttribute((const void*)dense_rows_kernel<T, MR, KIND, DEPTH, PASS>,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)ROWS_LDS);
    TGIS_CHECK_HIP(attr);
    hipLaunchKernelGGL((dense_rows_kernel<T, MR, KIND, DEPTH, PASS>), dim3((unsigned)(a.NT * (KIND == ROWS_RESIDUAL ? 4 : 2))), dim3(64 * rows_waves(KIND)),
                       (size_t)MR * a.K * sizeof(float), st, a);
    TGIS_CHECK_LAUNCH();
    return TGIS_OK;
}
template <typename T, int MR, int KIND>
int launch_rows_k(const RowsArgs& a, hipStream_t st) {
    if constexpr (KIND == ROWS_RESIDUAL) {
        if (a.K <= 2048) return launch_rows_one<T, MR, KIND, 2, 1>(a, st);
        if (a.K <= 4096) return launch_rows_one<T, MR, KIND, 4, 1>(a, st);
        if (a.K <= 6144) return launch_rows_one<T, MR, KIND, 6, 1>(a, st);
        return launch_rows_one<T, MR, KIND, 6, 2>(a, st);
    } else {
        if (a.K <= 2048) return launch_rows_one<T, MR, KIND, 4, 1>(a, st);
        if constexpr (MR <= 2) {
            if (a.K <= 3072) return launch_rows_one<T, MR, KIND, 6, 2>(a, st);
            return launch_rows_one<T, MR, KIND, 8, 2>(a, st);
        }
        return TGIS_EINVAL;  // (rows_fits)
    }
}
template <int KIND>
int launch_rows(const RowsArgs& a, int dtype, hipStream_t st) {
#define TGIS_ROWS(TT) (a.M == 1 ? launch_rows_k<TT, 1, KIND>(a, st) : a.M == 2 ? launch_rows_k<TT, 2, KIND>(a, st) : launch_rows_k<TT, 4, KIND>(a, st))
    return dtype == TGIS_F16 ? TGIS_ROWS(f16) : TGIS_ROWS(bf16);
#undef TGIS_ROWS
}

int64_t rows_height(int64_t M) { return M <= 2 ? M : 4; }

// Whole steps, us, seven launches a layer / these: 2048 wide, inner 5632, 22 layers: 1, 2, 3, 4 rows 920 / 729, 945 / 769, 980 / 948, 1008 / 981;
// 4096, 11008, 6 layers: 1, 2 rows 656 / 598, 663 / 626; 2560, 6912, 8 layers: 1, 2, 4 rows 489 / 462, 494 / 484, 500 / 622; 3072, 8192: 531 / 507, 543 /
// 522, 545 / 735.  Beyond two rows of 2048 columns the vector unit and the reads of x from LDS outlast the weights.  Narrower ones, 1, 2, 4 rows: 768, 2048,
// 12 layers 431 / 285, 445 / 302, 452 / 348; 1024, 2816, 16 layers 531 / 406, 540 / 427, 559 / 495; 1536, 4096, 16 layers 606 / 449, 621 / 470, 640 / 544.
bool rows_fits(int64_t M, int64_t K, bool norm) {
    return M >= 1 && M <= 4 && K >= 64 && K % 64 == 0 && K <= (norm ? (M <= 2 ? 4096 : 2048) : 12288) && rows_height(M) * K * 4 <= ROWS_LDS;
}

int rows_check(const char* what, int64_t M, int64_t K, int64_t N, int dtype, bool norm, const void* operand, const void* prepared, const float* h) {
    TGIS_CHECK_ARG(operand && prepared && h && N > 0 && N < (1ll << 31), "%s: null tensor or bad shape", what);
    TGIS_CHECK_ARG(dtype == TGIS_F16 || dtype == TGIS_BF16, "%s: bad dtype", what);
    TGIS_CHECK_ARG(rows_fits(M, K, norm), "%s: up to 4 rows, K a multiple of 64 up to %d that fits LDS (M=%ld K=%ld)", what, norm ? 4096 : 12288,
                   (long)M, (long)K);
    TGIS_CHECK_ARG((uintptr_t)operand % 16 == 0 && (uintptr_t)h % 16 == 0, "%s: operands must be 16-byte aligned", what);
    return TGIS_OK;
}

RowsArgs rows_args(float* h, const void* norm_w, float eps, const void* prepared, int64_t M, int64_t K, int64_t N, void* out, int64_t ldo) {
    RowsArgs a{};
    a.h = h;
    a.norm_w = norm_w;
    a.eps = eps;
    a.prep = (const uint8_t*)prepared;
    a.M = (int)M;
    a.K = (int)K;
    a.N = (int)N;
    a.NT = (int)cdiv64(N, 32);
    a.out = out;
    a.ldo = ldo;
    return a;
}

}  // namespace

extern "C" int tgis_dense_rows_ok(int64_t M, int64_t K, int norm) { return rows_fits(M, K, norm != 0) ? 1 : 0; }

extern "C" int tgis_dense_rows_residual(const void* x, int64_t ldx, const void* prepared, float* h, int64_t M, int64_t K, int64_t N, int dtype,
                                        void* stream) {
    const int rc = rows_check("tgis_dense_rows_residual", M, K, N, dtype, false, x, prepared, h);
    if (rc != TGIS_OK) return rc;
    TGIS_CHECK_ARG(ldx >= K && ldx % 8 == 0, "tgis_dense_rows_residual: x rows must be 16-byte aligned");
    TgisTimedScope timed(TGIS_OP_DENSE_GEMM, (hipStream_t)stream);
    RowsArgs a = rows_args(h, nullptr, 0.f, prepared, M, K, N, nullptr, 0);
    a.x = x;
    a.ldx = ldx;
    return launch_rows<ROWS_RESIDUAL>(a, dtype, (hipStream_t)stream);
}

extern "C" int tgis_dense_rows_norm_head(const float* h, const void* norm_w, float eps, const void* prepared, float* out, int64_t ldo, int64_t M,
                                         int64_t K, int64_t N, int dtype, void* stream) {
    const int rc = rows_check("tgis_dense_rows_norm_head", M, K, N, dtype, true, norm_w, prepared, h);
    if (rc != TGIS_OK) return rc;
    TGIS_CHECK_ARG(out && ldo >= N, "tgis_dense_rows_norm_head: bad output");
    TgisTimedScope timed(TGIS_OP_DENSE_GEMM, (hipStream_t)stream);
    return launch_rows<ROWS_HEAD>(rows_args(const_cast<float*>(h), norm_w, eps, prepared, M, K, N, out, ldo), dtype, (hipStream_t)stream);
}

extern "C" int tgis_dense_rows_norm_silu(const float* h, const void* norm_w, float eps, const void* prepared, void* out, int64_t ldo, int64_t M,
                                         int64_t K, int64_t N, int dtype, void* stream) {
    const int rc = rows_check("tgis_dense_rows_norm_silu", M, K, N, dtype, true, norm_w, prepared, h);
    if (rc != TGIS_OK) return rc;
    TGIS_CHECK_ARG(out && N % 32 == 0 && ldo >= N / 2, "tgis_dense_rows_norm_silu: needs a gate|up image (N / 2 a multiple of 16) and its output");
    TgisTimedScope timed(TGIS_OP_DENSE_GEMM, (hipStream_t)stream);
    return launch_rows<ROWS_SILU>(rows_args(const_cast<float*>(h), norm_w, eps, prepared, M, K, N, out, ldo), dtype, (hipStream_t)stream);
}

extern "C" int tgis_dense_rows_norm_rope(const float* h, const void* norm_w, float eps, const void* prepared, const void* bias,
                                         const int32_t* positions, const int32_t* slots, const void* cos, const void* sin, void* q_out, int64_t ldq,
                                         void* k_pool, void* v_pool, int64_t M, int64_t K, int64_t H, int64_t Hkv, int64_t D, int dtype,
                                         void* stream) {
    const int64_t N = (H + 2 * Hkv) * D;
    const int rc = rows_check("tgis_dense_rows_norm_rope", M, K, N, dtype, true, norm_w, prepared, h);
    if (rc != TGIS_OK) return rc;
    TGIS_CHECK_ARG(positions && slots && cos && sin && q_out && k_pool && v_pool, "tgis_dense_rows_norm_rope: null tensor");
    TGIS_CHECK_ARG(H >= 1 && Hkv >= 1 && D >= 32 && D % 32 == 0 && ldq >= H * D, "tgis_dense_rows_norm_rope: bad head geometry");
    TgisTimedScope timed(TGIS_OP_DENSE_GEMM, (hipStream_t)stream);
    RowsArgs a = rows_args(const_cast<float*>(h), norm_w, eps, prepared, M, K, N, q_out, ldq);
    a.bias = bias;
    a.positions = positions;
    a.slots = slots;
    a.cosb = cos;
    a.sinb = sin;
    a.kpool = k_pool;
    a.vpool = v_pool;
    a.H = (int)H;
    a.Hkv = (int)Hkv;
    a.D = (int)D;
    return launch_rows<ROWS_ROPE>(a, dtype, (hipStream_t)stream);
}
