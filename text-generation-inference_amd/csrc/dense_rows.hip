// Dense products of a decode step of a few rows (up to 4; in bf16 up to 64, below) with the norm in front of them and the residual add behind them.
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
#include "gptq_gemm_body.h"
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

// v summed over the lanes with the same lane % 16, in every one of them
__device__ __forceinline__ float sum_of_quarters(float v) {
    const uint32_t x = __builtin_bit_cast(uint32_t, v);
    const auto a = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    const uint32_t a0 = a[0], a1 = a[1];
    v = __builtin_bit_cast(float, a0) + __builtin_bit_cast(float, a1);
    const uint32_t y = __builtin_bit_cast(uint32_t, v);
    const auto b = __builtin_amdgcn_permlane16_swap(y, y, false, false);
    const uint32_t b0 = b[0], b1 = b[1];
    return __builtin_bit_cast(float, b0) + __builtin_bit_cast(float, b1);
}
// v summed over the lanes with the same lane % 8, in every one of them
__device__ __forceinline__ float sum_of_eighths(float v) {
    v = sum_of_quarters(v);
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

// ---- up to 16 RB rows in bf16, on the matrix instruction ----
// The same five launches with v_mfma_f32_16x16x32: sixteen weight columns are its rows, the batch its columns.  A unit is sixteen columns c0 .. +7 and c0 + 16 .. +23 of
// a tile (ROPE, SILU, HEAD), or eight columns whose two halves of a k64-step lie beside each other (RESIDUAL: each half is multiplied by its own x, and the halves that met
// the other's x are never read).  Nobody shares x: the waves of a workgroup split the k range, and a wave reads x of its own k64-steps straight into the operand's registers;
// a workgroup keeps it and takes units in turn.
// What bounds these launches is each workgroup's own copy of x beside its share of the weights, so
//   * x is 16 bits: behind a sum of the stream h (fp32 in registers) RESIDUAL leaves T(h), which the next sum adds to, T(h w) of the norm weight
//     behind it, and the sums of h^2 of its eight columns.  The norm's 1 / rms is a factor of the finished sums; an operand is rounded once either way.  (h itself in
//     fp32, normed by each workgroup: 16 rows of a 1.1B model 890 us a step for 850 at two units on their way.)
//   * x is in fragment order (xf_off): a load is four runs of 256 bytes.  From rows of x, whose cache lines the same loads take by halves, that step took
//     1056 us in the place of 890;
//   * a wave has one unit, or one k64-step of RESIDUAL, on its way, not more: gate | up of 2048 x 11264 at 16 rows with one, two, three units 9.9 / 11.2 / 11.1 us (the other
//     waves of the CU ask meanwhile), the residual products with one, two, four steps 6.2 / 6.4 / 7.2.  Fewer units a workgroup than fill one round of 256 take x in more often: one
//     11.1, two 11.5, three 9.9.
// bf16 only: T(h w) has its range.
constexpr int STREAM_ROWS = 64;
struct Rows16Args {
    const bf16* x;       // T(h w) or an activation, fragment order
    const float* sums;   // [K / 32][64 rows][4]: sums of h^2 of eight columns each
    float eps;
    const uint8_t* prep;
    int M, K, N, NT;
    void* out;
    int64_t ldo;
    // RESIDUAL: the stream behind it
    const bf16* norm_w;
    bf16 *h, *hw;        // T(h), T(h w), fragment order
    float* sums_out;
    // ROPE (as tgis_dense_gemm_rope)
    const bf16* bias;
    const int32_t *positions, *slots;
    const bf16 *cosb, *sinb;
    bf16 *kpool, *vpool;
    int H, Hkv, D;
};
// byte offset of a lane's piece of row `row` (chunk kq of the first 32 k) within a k64-step in fragment order of an operand of K columns
__device__ __forceinline__ uint32_t frag_lane(int row, int kq, int K) { return (uint32_t)(row >> 5) * 64 * K + kq * 1024 + (row & 31) * 16; }
__device__ __forceinline__ int64_t sums_off(int m, int k) { return ((int64_t)(k >> 5) * STREAM_ROWS + m) * 4 + ((k >> 3) & 3); }

// What is left of eight columns k .. k + 7 of row m of h = f: T(h), T(h w) and the sum of h^2
__device__ __forceinline__ void leave_stream(const float (&f)[8], int m, int k, int K, const bf16* norm_w, bf16* h, bf16* hw, float* sums) {
    const bf16x8 nw = ld16<bf16x8>(norm_w + k);
    bf16x8 v, y;
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        ss += f[e] * f[e];
        v[e] = (bf16)f[e];
        y[e] = (bf16)(f[e] * to_f32(nw[e]));
    }
    st16(h + xf_off(m, k, K), v);
    st16(hw + xf_off(m, k, K), y);
    sums[sums_off(m, k)] = ss;
}
// the stream of tokens (ids), or of rows x [M][K] (ids null); R: M rounded up to sixteen
__global__ __launch_bounds__(256) void rows16_embed_kernel(const int64_t* __restrict__ ids, const bf16* __restrict__ x, const bf16* __restrict__ norm_w,
                                                           bf16* __restrict__ h, bf16* __restrict__ hw, float* __restrict__ sums, int M, int K, int64_t vocab, int R) {
    const int at = blockIdx.x * 256 + threadIdx.x, m = at % R, k = at / R * 8;
    if (m >= M || k >= K) return;
    const int64_t id = ids ? ids[m] : m;
    bf16x8 v{};
    if (id >= 0 && id < vocab) v = ld16<bf16x8>(x + id * K + k);
    float f[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = to_f32(v[e]);
    leave_stream(f, m, k, K, norm_w, h, hw, sums);
}

// SPW: k64-steps of a wave at most
template <int KIND, int SPW, int RB>
__global__ __launch_bounds__(512) void dense_rows16_kernel(Rows16Args a, int units, int per) {
    constexpr int W = 8;
    static_assert(KIND != ROWS_RESIDUAL && RB <= 4, "the kernels below");
    constexpr int BUFS = RB <= 2 ? 2 : 1;                 // of the waves' sums
    constexpr int FW = RB == 1 ? 1 : RB == 2 ? 2 : 4;     // a unit's outputs are finished by FW waves, unit i's by the (i mod 8 / FW)-th FW
    __shared__ __attribute__((aligned(16))) float red[BUFS][W][RB][64 * 4];
    __shared__ float part[W][16 * RB];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int K = a.K, steps = K >> 6, mine = (steps - w + W - 1) / W;  // k64-steps w, w + 8, ..
    const int m = lane & 15, kq = lane >> 4;
    const int u0 = blockIdx.x * per, n = min(per, units - u0);

    const int fb = w & (FW - 1), frow = fb * 16 + m;  // the block of rows whose outputs this wave finishes (RB 3: the fourth wave none)
    int32_t pos = 0, slot = 0;
    if (KIND == ROWS_ROPE) {
        pos = a.positions[min(frow, a.M - 1)];
        slot = a.slots[min(frow, a.M - 1)];
    }
    bf16x8 x[RB][SPW][2];
    uint32_t xoff[RB];
#pragma unroll
    for (int b = 0; b < RB; ++b) xoff[b] = frag_lane(min(b * 16 + m, a.M - 1), kq, a.K);
#pragma unroll
    for (int j = 0; j < SPW; ++j) {
        const char* xp = reinterpret_cast<const char*>(a.x) + (int64_t)min(w + W * j, steps - 1) * 4096;
        PIN_SGPR(xp);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int b = 0; b < RB; ++b) x[b][j][h] = *(const GLOBAL_AS bf16x8*)(xp + xoff[b] + h * 512);
    }
    // the sums of h^2: SPW / 2 groups of 4 x 32 columns a wave
    constexpr int SG = (SPW + 1) / 2;
    f32x4 sq[RB][SG];
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int t = 0; t < SG; ++t)
            sq[b][t] = *reinterpret_cast<const f32x4*>(a.sums + sums_off(min(b * 16 + m, a.M - 1), min((t * W + w) * 4 + kq, (K >> 5) - 1) * 32));
    const uint32_t woff = kq * 1024 + ((lane & 7) + ((lane >> 3) & 1) * 16) * 16;
    bf16x8 wq[SPW][2];
    auto ask = [&](int u) {
        const char* base = reinterpret_cast<const char*>(a.prep) + (int64_t)(u >> 1) * steps * 4096 + (u & 1) * 128;
#pragma unroll
        for (int j = 0; j < SPW; ++j) {
            const char* p = base + (int64_t)min(w + W * j, steps - 1) * 4096;
            PIN_SGPR(p);
#pragma unroll
            for (int h = 0; h < 2; ++h) wq[j][h] = __builtin_nontemporal_load((const GLOBAL_AS bf16x8*)(p + h * 512 + woff));
        }
    };
    ask(u0);
    // ROPE: what unit u's outputs are rotated by, and the bias; asked for early for the first unit that this wave finishes
    const bool second = kq >= 2;  // this lane's columns are of the tile's second half
    bf16x4 cf{}, sf{}, bv{};
    int head = 0, dim = 0;
    auto rope_inputs = [&](int u) {
        const int tile = u >> 1, c = (u & 1) * 8 + (kq & 1) * 4, per_head = a.D >> 5, tt = tile % per_head;
        head = tile / per_head;
        const bool roth = head < a.H + a.Hkv;
        dim = roth ? (second ? (a.D >> 1) : 0) + 16 * tt + c : 32 * tt + c + (second ? 16 : 0);
        const int64_t at = (int64_t)pos * (a.D >> 1) + 16 * tt + c;
        if (roth) {
            cf = *reinterpret_cast<const bf16x4*>(a.cosb + at);
            sf = *reinterpret_cast<const bf16x4*>(a.sinb + at);
        }
        if (a.bias) bv = *reinterpret_cast<const bf16x4*>(a.bias + head * a.D + dim);
    };
    if (KIND == ROWS_ROPE) rope_inputs(u0 + min(w / FW, n - 1));

#pragma unroll
    for (int b = 0; b < RB; ++b) {
        float ss = 0.f;
#pragma unroll
        for (int t = 0; t < SG; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) ss += (t * W + w) * 4 + kq < (K >> 5) ? sq[b][t][e] : 0.f;
        ss = sum_of_quarters(ss);
        if (kq == 0) part[w][b * 16 + m] = ss;  // (read behind the first unit's barrier)
    }

    auto unit = [&](int i, bool more) {
        f32x4 acc[RB];
#pragma unroll
        for (int b = 0; b < RB; ++b) acc[b] = f32x4{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < SPW; ++j)
            if (j < mine) {
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int b = 0; b < RB; ++b) acc[b] = mfma16(wq[j][h], x[b][j][h], acc[b]);
            }
        if (more) ask(u0 + i + 1);
        const int r = i & (BUFS - 1);
        if (BUFS == 1 && i > 0) __syncthreads();  // the unit before has been read
#pragma unroll
        for (int b = 0; b < RB; ++b) *reinterpret_cast<f32x4*>(&red[r][w][b][lane * 4]) = acc[b];
        __syncthreads();  // (two buffers: the one before last was read in front of a barrier since)
        if (w / FW != i % (W / FW) || fb >= RB) return;
        float tot = 0.f;
#pragma unroll
        for (int k = 0; k < W; ++k) tot += part[k][frow];
        const float rstd = rsqrtf(tot / K + a.eps);
        f32x4 v = *reinterpret_cast<const f32x4*>(&red[r][0][fb][lane * 4]);
#pragma unroll
        for (int k = 1; k < W; ++k) v += *reinterpret_cast<const f32x4*>(&red[r][k][fb][lane * 4]);
        v *= rstd;
        // v[e]: row frow, column c + e of its half of the tile
        const int u = u0 + i, tile = u >> 1, c = (u & 1) * 8 + (kq & 1) * 4;
        const bool live = frow < a.M;
        if (KIND == ROWS_HEAD) {
            const int col = tile * 32 + c + (second ? 16 : 0);
            float* o = reinterpret_cast<float*>(a.out) + (int64_t)frow * a.ldo + col;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (live && col + e < a.N) o[e] = v[e];
        } else if (KIND == ROWS_SILU) {
            bf16x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float own = to_f32((bf16)v[e]), up = __shfl_xor(own, 32, 64);
                const float sl = own / (1.f + __expf(-own));
                o[e] = (bf16)(to_f32((bf16)sl) * up);
            }
            if (live && !second) *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16*>(a.out) + xf_off(frow, tile * 16 + c, a.N >> 1)) = o;
        } else {
            if (i >= W / FW) rope_inputs(u);
            const bool roth = head < a.H + a.Hkv;
            bf16x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float own = to_f32((bf16)(v[e] + to_f32(bv[e]))), other = __shfl_xor(own, 32, 64);
                const float co = to_f32(cf[e]), si = to_f32(sf[e]);
                o[e] = (bf16)(!roth ? own : second ? other * si + own * co : own * co - other * si);
            }
            if (!live) return;
            const int64_t page = slot >> 5;
            const int tok = slot & 31;
            if (head < a.H) {
                *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16*>(a.out) + (int64_t)frow * a.ldo + head * a.D + dim) = o;
            } else if (roth) {
                *reinterpret_cast<bf16x4*>(a.kpool + (page * a.Hkv + (head - a.H)) * 32 * a.D + k_off(tok, dim, a.D)) = o;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) a.vpool[(page * a.Hkv + (head - a.H - a.Hkv)) * 32 * a.D + v_off(tok, dim + e, a.D)] = o[e];
            }
        }
    };
    for (int i = 0; i + 1 < n; ++i) unit(i, true);
    unit(n - 1, false);
}

template <int RB>
__global__ __launch_bounds__(1024) void dense_rows16_residual_kernel(Rows16Args a) {
    constexpr int W = 16;
    __shared__ __attribute__((aligned(16))) float red[W][RB][64 * 4];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int steps = a.K >> 6;  // this wave's: w, w + 16, ..
    const int m = lane & 15, kq = lane >> 4, tile = blockIdx.x >> 2, c0 = (blockIdx.x & 3) * 8;
    const char* wbase = reinterpret_cast<const char*>(a.prep) + (int64_t)tile * steps * 4096;
    const uint32_t woff = kq * 1024 + ((lane >> 3) & 1) * 512 + (c0 + (lane & 7)) * 16;
    uint32_t xoff[RB];
#pragma unroll
    for (int b = 0; b < RB; ++b) xoff[b] = frag_lane(min(b * 16 + m, a.M - 1), kq, a.K);
    bf16x8 wq, x[RB][2];
    auto ask = [&](int s) {
        const char *p = wbase + (int64_t)s * 4096, *xp = reinterpret_cast<const char*>(a.x) + (int64_t)s * 4096;
        PIN_SGPR(p);
        PIN_SGPR(xp);
        wq = __builtin_nontemporal_load((const GLOBAL_AS bf16x8*)(p + woff));
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
            for (int h = 0; h < 2; ++h) x[b][h] = *(const GLOBAL_AS bf16x8*)(xp + xoff[b] + h * 512);
    };
    ask(min(w, steps - 1));
    const int frow = w * 16 + m, col = tile * 32 + c0 + (kq & 1) * 4;
    const int64_t at = xf_off(min(frow, a.M - 1), col, a.N);
    bf16x4 res{}, nw{};
    if (w < RB) {
        res = *reinterpret_cast<const bf16x4*>(a.h + at);
        nw = *reinterpret_cast<const bf16x4*>(a.norm_w + col);
    }
    f32x4 acc[RB][2];
#pragma unroll
    for (int b = 0; b < RB; ++b) acc[b][0] = acc[b][1] = f32x4{0, 0, 0, 0};
    for (int s = w; s < steps; s += W) {
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
            for (int h = 0; h < 2; ++h) acc[b][h] = mfma16(wq, x[b][h], acc[b][h]);
        if (s + W < steps) ask(s + W);
    }
#pragma unroll
    for (int b = 0; b < RB; ++b) {
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = kq < 2 ? acc[b][0][e] : acc[b][1][e];
        *reinterpret_cast<f32x4*>(&red[w][b][lane * 4]) = v;
    }
    __syncthreads();
    if (w >= RB) return;
    f32x4 v = *reinterpret_cast<const f32x4*>(&red[0][w][lane * 4]);
#pragma unroll
    for (int k = 1; k < W; ++k) v += *reinterpret_cast<const f32x4*>(&red[k][w][lane * 4]);
    bf16x4 h, hw;
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float f = to_f32((bf16)(v[e] + __shfl_xor(v[e], 32, 64))) + to_f32(res[e]);
        ss += f * f;
        h[e] = (bf16)f;
        hw[e] = (bf16)(f * to_f32(nw[e]));
    }
    ss += __shfl_xor(ss, 16, 64);
    if (kq >= 2 || frow >= a.M) return;
    *reinterpret_cast<bf16x4*>(a.h + at) = h;
    *reinterpret_cast<bf16x4*>(a.hw + at) = hw;
    if (kq == 0) a.sums_out[sums_off(frow, col)] = ss;
}

// RESIDUAL with the k range split over S workgroups a tile, for as many rows as make x of a whole range the larger part of what a workgroup takes in: a tile of 32 columns
// a workgroup, sums left as slabs [S][N / 4][64 rows][4], which the launch behind adds up: T(x W^T) + T(h) as above, or (`leave`, behind the last layer) the
// sum as one slab of rows and T(h) as rows for a norm of its own.
template <int RB>
__global__ __launch_bounds__(512) void dense_rows16_parts_kernel(Rows16Args a, int S, float* slabs) {
    constexpr int W = 8;
    __shared__ __attribute__((aligned(16))) float red[W][2 * RB][64 * 4];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int steps = a.K >> 6, tile = blockIdx.x, split = blockIdx.y, sb = steps * split / S, se = steps * (split + 1) / S;
    const int m = lane & 15, kq = lane >> 4;
    const char* wbase = reinterpret_cast<const char*>(a.prep) + (int64_t)tile * steps * 4096;
    const uint32_t woff = kq * 1024 + m * 16;
    uint32_t xoff[RB];
#pragma unroll
    for (int b = 0; b < RB; ++b) xoff[b] = frag_lane(min(b * 16 + m, a.M - 1), kq, a.K);
    bf16x8 wq[2][2], x[RB][2];
    auto ask = [&](int s) {
        const char *p = wbase + (int64_t)s * 4096, *xp = reinterpret_cast<const char*>(a.x) + (int64_t)s * 4096;
        PIN_SGPR(p);
        PIN_SGPR(xp);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int u = 0; u < 2; ++u) wq[u][h] = __builtin_nontemporal_load((const GLOBAL_AS bf16x8*)(p + woff + h * 512 + u * 256));
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
            for (int h = 0; h < 2; ++h) x[b][h] = *(const GLOBAL_AS bf16x8*)(xp + xoff[b] + h * 512);
    };
    ask(min(sb + w, steps - 1));
    f32x4 acc[2][RB];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int b = 0; b < RB; ++b) acc[u][b] = f32x4{0, 0, 0, 0};
    for (int s = sb + w; s < se; s += W) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int b = 0; b < RB; ++b) acc[u][b] = mfma16(wq[u][h], x[b][h], acc[u][b]);
        if (s + W < se) ask(s + W);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int b = 0; b < RB; ++b) *reinterpret_cast<f32x4*>(&red[w][u * RB + b][lane * 4]) = acc[u][b];
    __syncthreads();
    const int u = w / RB, b = w % RB, row = b * 16 + m;
    if (u >= 2 || row >= a.M) return;
    f32x4 v = *reinterpret_cast<const f32x4*>(&red[0][w][lane * 4]);
#pragma unroll
    for (int k = 1; k < W; ++k) v += *reinterpret_cast<const f32x4*>(&red[k][w][lane * 4]);
    *reinterpret_cast<f32x4*>(slabs + (((int64_t)split * (a.N >> 2) + tile * 8 + u * 4 + kq) * STREAM_ROWS + row) * 4) = v;
}
template <int SB, bool LEAVE>
__global__ __launch_bounds__(256) void rows16_sum_kernel(const float* __restrict__ slabs, int S, const bf16* __restrict__ norm_w, bf16* __restrict__ h, bf16* __restrict__ hw,
                                                         float* __restrict__ sums, int M, int N, int R) {
    const int at = blockIdx.x * 256 + threadIdx.x, m = at % R, k = at / R * 8;
    if (m >= M || k >= N) return;
    const bf16x8 res = ld16<bf16x8>(h + xf_off(m, k, N));
    f32x4 lo[SB], hi[SB];
#pragma unroll
    for (int s = 0; s < SB; ++s) {
        const float* p = slabs + (((int64_t)min(s, S - 1) * (N >> 2) + (k >> 2)) * STREAM_ROWS + m) * 4;
        lo[s] = *reinterpret_cast<const f32x4*>(p);
        hi[s] = *reinterpret_cast<const f32x4*>(p + STREAM_ROWS * 4);
    }
#pragma unroll
    for (int s = 1; s < SB; ++s)
        if (s < S) {
            lo[0] += lo[s];
            hi[0] += hi[s];
        }
    if (LEAVE) {  // hw: rows of T(h); sums: [32-row block][32][N]
        st16(hw + (int64_t)m * N + k, res);
        float* o = sums + (int64_t)m * N + k;
        *reinterpret_cast<f32x4*>(o) = lo[0];
        *reinterpret_cast<f32x4*>(o + 4) = hi[0];
    } else {
        float f[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = to_f32((bf16)(e < 4 ? lo[0][e & 3] : hi[0][e & 3])) + to_f32(res[e]);
        leave_stream(f, m, k, N, norm_w, h, hw, sums);
    }
}

// Whole steps, us, the other launches of a layer / these (2048 wide, inner 5632, 22 layers; ctx 137): 3, 4 rows 881 / 746 (the launches of up to four rows), 8 rows 964 / 761, 16
// 990 / 814, 24 1053 / 906, 32 1077 / 965, 48 1284 / 1059, 64 1355 / 1135; 768, 2048, 12 layers, 8, 16, 32, 48, 64 rows: 461 / 302, 479 / 318, 541 / 397, 653 /
// 453, 679 / 503; 1024, 2816, 16 layers: 568 / 453, 589 / 484, 658 / 595;
// 1536, 4096, 16 layers: 673 / 520, 701 / 564, 816 / 706, 977 / 826, 1052 / 897.  Wider ones, 4, 8, 16 rows: 2560, 6912, 8 layers 504 / 471, 531 / 480, 569 / 540; 3072,
// 8192: 543 / 542, 574 / 548, 597 / 585; 4096, 11008, 6 layers 664 / 617, 705 / 615, 748 / 676; there 32 rows 635 / 767, 654 / 776, 828 / 915 by more x than weights.  One and two rows: 716 / 744, 754 / 745, narrower ones 4 -
// 10 % behind the launches of up to four rows, which keep them.
bool rows16_fits(int64_t M, int64_t K, bool norm) {
    return M >= 1 && M <= STREAM_ROWS && K >= 64 && K % 64 == 0 && K <= (!norm ? 12288 : M <= 16 ? 4096 : 2048);
}
// Splits of a residual product's k range: as many as fill the chip with a tile a workgroup, a step for each wave of it; none where x of the whole range is less than 320 KiB.  Whole
// steps, us, unsplit / these products split: down of 5632 x 2048 at 32, 48, 64 rows 978 / 965, 1094 / 1059, 1211 / 1135, at 24 906 / 909; o of 2048 x 2048 besides at 48, 64 rows 1059 / 1084,
// 1135 / 1139; down of 4096 x 1536 at 24, 32 rows 659 / 673, 706 / 718, at 48 845 / 826; of 11008 x 4096 at 8, 16 rows 614 / 615, 700 / 676.  `must`: whatever the rows.
int rows16_splits(int64_t M, int64_t K, int64_t N, bool must) {
    if (!must && M * K < 160 * 1024) return 0;
    const int64_t tiles = N / 32;
    return (int)std::max<int64_t>(1, std::min<int64_t>({(256 + tiles / 2) / tiles, K / 512, 8}));
}
int64_t rows16_slab_bytes(int64_t N, int S) { return (int64_t)S * N * STREAM_ROWS * 4; }

template <int KIND, int RB, int SPW>
void launch_rows16_k(const Rows16Args& a, hipStream_t st) {
    const int units = a.NT * 2, per = (units + 255) / 256;
    hipLaunchKernelGGL((dense_rows16_kernel<KIND, SPW, RB>), dim3((unsigned)((units + per - 1) / per)), dim3(512), 0, st, a, units, per);
}
template <int KIND, int RB>
void launch_rows16_rb(const Rows16Args& a, hipStream_t st) {
    if constexpr (KIND == ROWS_RESIDUAL) {
        hipLaunchKernelGGL((dense_rows16_residual_kernel<RB>), dim3((unsigned)(a.NT * 4)), dim3(1024), 0, st, a);
    } else {
        const int spw = (a.K + 511) / 512;
        if (spw <= 2) return launch_rows16_k<KIND, RB, 2>(a, st);
        if (spw == 3) return launch_rows16_k<KIND, RB, 3>(a, st);
        if constexpr (RB == 1) {
            if (spw == 5) return launch_rows16_k<KIND, RB, 5>(a, st);
            if (spw == 6) return launch_rows16_k<KIND, RB, 6>(a, st);
            if (spw > 6) return launch_rows16_k<KIND, RB, 8>(a, st);
        }
        launch_rows16_k<KIND, RB, 4>(a, st);
    }
}
template <int KIND>
int launch_rows16(const Rows16Args& a, hipStream_t st) {
    TgisTimedScope timed(TGIS_OP_DENSE_GEMM, st);
    if (a.M <= 16)
        launch_rows16_rb<KIND, 1>(a, st);
    else if (a.M <= 32)
        launch_rows16_rb<KIND, 2>(a, st);
    else if (a.M <= 48)
        launch_rows16_rb<KIND, 3>(a, st);
    else
        launch_rows16_rb<KIND, 4>(a, st);
    TGIS_CHECK_LAUNCH();
    return TGIS_OK;
}
template <bool LEAVE>
int launch_rows16_split(const Rows16Args& a, int S, float* slabs, hipStream_t st) {
    TgisTimedScope timed(TGIS_OP_DENSE_GEMM, st);
    const dim3 grid((unsigned)a.NT, (unsigned)S);
    const int R = (a.M + 15) / 16 * 16;
    const auto parts = R == 16 ? dense_rows16_parts_kernel<1> : R == 32 ? dense_rows16_parts_kernel<2> : R == 48 ? dense_rows16_parts_kernel<3> : dense_rows16_parts_kernel<4>;
    hipLaunchKernelGGL(parts, grid, dim3(512), 0, st, a, S, slabs);
    TGIS_CHECK_LAUNCH();
    const dim3 sgrid((unsigned)cdiv64((int64_t)R * (a.N >> 3), 256));
    if (S <= 4)
        hipLaunchKernelGGL((rows16_sum_kernel<4, LEAVE>), sgrid, dim3(256), 0, st, slabs, S, a.norm_w, a.h, a.hw, a.sums_out, a.M, a.N, R);
    else
        hipLaunchKernelGGL((rows16_sum_kernel<8, LEAVE>), sgrid, dim3(256), 0, st, slabs, S, a.norm_w, a.h, a.hw, a.sums_out, a.M, a.N, R);
    TGIS_CHECK_LAUNCH();
    return TGIS_OK;
}

int64_t rows_height(int64_t M) { return M <= 2 ? M : 4; }

// Whole steps, us, seven launches a layer / these: 2048 wide, inner 5632, 22 layers: 1, 2, 3, 4 rows 920 / 729, 945 / 769, 980 / 948, 1008 / 981;
// 4096, 11008, 6 layers: 1, 2 rows 656 / 598, 663 / 626; 2560, 6912, 8 layers: 1, 2, 4 rows 489 / 462, 494 / 484, 500 / 622; 3072, 8192: 531 / 507, 543 /
// 522, 545 / 735.  Beyond two rows of 2048 columns the vector unit and the reads of x from LDS outlast the weights.  Narrower ones, 1, 2, 4 rows: 768, 2048,
// 12 layers 431 / 285, 445 / 302, 452 / 348; 1024, 2816, 16 layers 531 / 406, 540 / 427, 559 / 495; 1536, 4096, 16 layers 606 / 449, 621 / 470, 640 / 544.
// Of bf16, steps of three and four rows are those of the launches of more rows, above; they come here where no product may split its sums (TGIS_DEFER_REDUCE=0).
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

// ---- the launches of up to 64 rows ----

extern "C" int tgis_dense_rows16_ok(int64_t M, int64_t K, int norm) { return rows16_fits(M, K, norm != 0) ? 1 : 0; }

namespace {

int rows16_check(const char* what, int64_t M, int64_t K, int64_t N, bool norm, const void* x, const void* prepared, const void* other) {
    TGIS_CHECK_ARG(x && prepared && other && N > 0 && N < (1ll << 31), "%s: null tensor or bad shape", what);
    TGIS_CHECK_ARG(rows16_fits(M, K, norm), "%s: up to %d rows, K a multiple of 64 up to %d (M=%ld K=%ld)", what, STREAM_ROWS,
                   !norm ? 12288 : M <= 16 ? 4096 : 2048, (long)M, (long)K);
    TGIS_CHECK_ARG(((uintptr_t)x | (uintptr_t)prepared | (uintptr_t)other) % 16 == 0, "%s: operands must be 16-byte aligned", what);
    return TGIS_OK;
}
Rows16Args rows16_args(const void* x, const float* sums, float eps, const void* prepared, int64_t M, int64_t K, int64_t N, void* out, int64_t ldo) {
    Rows16Args a{};
    a.x = (const bf16*)x;
    a.sums = sums;
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

extern "C" int tgis_dense_rows16_embed(const int64_t* ids, const void* x, const void* norm_w, void* h, void* hw, float* sums, int64_t M, int64_t K,
                                       int64_t vocab, void* stream) {
    const int rc = rows16_check("tgis_dense_rows16_embed", M, K, ids ? vocab : M, true, x, norm_w, h);
    if (rc != TGIS_OK) return rc;
    TGIS_CHECK_ARG(hw && sums && ((uintptr_t)hw | (uintptr_t)sums) % 16 == 0, "tgis_dense_rows16_embed: null or unaligned tensor");
    const int R = ((int)M + 15) / 16 * 16;
    hipLaunchKernelGGL(rows16_embed_kernel, dim3((unsigned)cdiv64(K / 8 * R, 256)), dim3(256), 0, (hipStream_t)stream, ids, (const bf16*)x,
                       (const bf16*)norm_w, (bf16*)h, (bf16*)hw, sums, (int)M, (int)K, ids ? vocab : M, R);
    TGIS_CHECK_LAUNCH();
    return TGIS_OK;
}

extern "C" int64_t tgis_dense_rows16_slab_bytes(int64_t M, int64_t K, int64_t N, int leave) {
    return rows16_slab_bytes(N, rows16_splits(M, K, N, leave != 0));
}

extern "C" int tgis_dense_rows16_residual(const void* x, const void* prepared, const void* norm_w, void* h, void* hw, float* sums, float* slabs,
                                          int64_t slabs_bytes, int64_t M, int64_t K, int64_t N, void* stream) {
    const char* what = "tgis_dense_rows16_residual";
    const int rc = rows16_check(what, M, K, N, false, x, prepared, h);
    if (rc != TGIS_OK) return rc;
    TGIS_CHECK_ARG(norm_w && hw && sums && ((uintptr_t)norm_w | (uintptr_t)hw | (uintptr_t)sums) % 16 == 0 && N % 64 == 0,
                   "%s: null or unaligned tensor, or a width that is no multiple of 64", what);
    Rows16Args a = rows16_args(x, nullptr, 0.f, prepared, M, K, N, nullptr, 0);
    a.norm_w = (const bf16*)norm_w;
    a.h = (bf16*)h;
    a.hw = (bf16*)hw;
    a.sums_out = sums;
    const int S = rows16_splits(M, K, N, false);
    if (S == 0) return launch_rows16<ROWS_RESIDUAL>(a, (hipStream_t)stream);
    TGIS_CHECK_ARG(slabs && (uintptr_t)slabs % 16 == 0 && slabs_bytes >= rows16_slab_bytes(N, S), "%s: no room for %d partial sums", what, S);
    return launch_rows16_split<false>(a, S, slabs, (hipStream_t)stream);
}

extern "C" int tgis_dense_rows16_leave(const void* x, const void* prepared, const void* h, void* h_rows, float* sum_rows, float* slabs, int64_t slabs_bytes,
                                       int64_t M, int64_t K, int64_t N, void* stream) {
    const char* what = "tgis_dense_rows16_leave";
    const int rc = rows16_check(what, M, K, N, false, x, prepared, h);
    if (rc != TGIS_OK) return rc;
    const int S = rows16_splits(M, K, N, true);
    TGIS_CHECK_ARG(h_rows && sum_rows && ((uintptr_t)h_rows | (uintptr_t)sum_rows) % 16 == 0 && N % 64 == 0 && slabs && (uintptr_t)slabs % 16 == 0 &&
                       slabs_bytes >= rows16_slab_bytes(N, S),
                   "%s: null or unaligned tensor, a width that is no multiple of 64, or no room for %d partial sums", what, S);
    Rows16Args a = rows16_args(x, nullptr, 0.f, prepared, M, K, N, nullptr, 0);
    a.h = const_cast<bf16*>((const bf16*)h);
    a.hw = (bf16*)h_rows;
    a.sums_out = sum_rows;
    return launch_rows16_split<true>(a, S, slabs, (hipStream_t)stream);
}

extern "C" int tgis_dense_rows16_norm_head(const void* hw, const float* sums, float eps, const void* prepared, float* out, int64_t ldo, int64_t M, int64_t K,
                                           int64_t N, void* stream) {
    const int rc = rows16_check("tgis_dense_rows16_norm_head", M, K, N, true, hw, prepared, sums);
    if (rc != TGIS_OK) return rc;
    TGIS_CHECK_ARG(out && ldo >= N, "tgis_dense_rows16_norm_head: bad output");
    return launch_rows16<ROWS_HEAD>(rows16_args(hw, sums, eps, prepared, M, K, N, out, ldo), (hipStream_t)stream);
}

extern "C" int tgis_dense_rows16_norm_silu(const void* hw, const float* sums, float eps, const void* prepared, void* out, int64_t M, int64_t K, int64_t N,
                                           void* stream) {
    const int rc = rows16_check("tgis_dense_rows16_norm_silu", M, K, N, true, hw, prepared, sums);
    if (rc != TGIS_OK) return rc;
    TGIS_CHECK_ARG(out && (uintptr_t)out % 16 == 0 && N % 128 == 0, "tgis_dense_rows16_norm_silu: needs a gate|up image (N / 2 a multiple of 64) and its output");
    return launch_rows16<ROWS_SILU>(rows16_args(hw, sums, eps, prepared, M, K, N, out, 0), (hipStream_t)stream);
}

extern "C" int tgis_dense_rows16_norm_rope(const void* hw, const float* sums, float eps, const void* prepared, const void* bias, const int32_t* positions,
                                           const int32_t* slots, const void* cos, const void* sin, void* q_out, int64_t ldq, void* k_pool, void* v_pool,
                                           int64_t M, int64_t K, int64_t H, int64_t Hkv, int64_t D, void* stream) {
    const int64_t N = (H + 2 * Hkv) * D;
    const int rc = rows16_check("tgis_dense_rows16_norm_rope", M, K, N, true, hw, prepared, sums);
    if (rc != TGIS_OK) return rc;
    TGIS_CHECK_ARG(positions && slots && cos && sin && q_out && k_pool && v_pool, "tgis_dense_rows16_norm_rope: null tensor");
    TGIS_CHECK_ARG(H >= 1 && Hkv >= 1 && D >= 32 && D % 32 == 0 && ldq >= H * D, "tgis_dense_rows16_norm_rope: bad head geometry");
    TGIS_CHECK_ARG(ldq % 4 == 0 && ((uintptr_t)q_out | (uintptr_t)cos | (uintptr_t)sin | (uintptr_t)bias | (uintptr_t)k_pool) % 8 == 0,
                   "tgis_dense_rows16_norm_rope: q, its rows, bias, tables and pages must be 8-byte aligned");
    Rows16Args a = rows16_args(hw, sums, eps, prepared, M, K, N, q_out, ldq);
    a.bias = (const bf16*)bias;
    a.positions = positions;
    a.slots = slots;
    a.cosb = (const bf16*)cos;
    a.sinb = (const bf16*)sin;
    a.kpool = (bf16*)k_pool;
    a.vpool = (bf16*)v_pool;
    a.H = (int)H;
    a.Hkv = (int)Hkv;
    a.D = (int)D;
    return launch_rows16<ROWS_ROPE>(a, (hipStream_t)stream);
}
