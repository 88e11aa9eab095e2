// Int4 products of a decode step of up to 32 rows with the norm in front of them and the residual add behind them.
// Replaces exllamav2_kernels.gemm_half_q_half (utils/gptq/exllamav2.py:139-144) and the add + RMSNorm launches (custom_modeling/flash_llama_modeling.py:132-152)
// of such a step: five launches a layer, as csrc/dense_rows.hip does for dense weights, on the image of gptq_gemm_body.h.
//
// A layer of 4096, 11008 at 11 rows was seven launches: 38 us of products for 105 MB and two norm launches of 4.7 us, each a row on a CU and a boundary.  Here
//   * a unit is sixteen columns and the whole k range, so that nothing is left to add up: 256 units for 4096 columns, one a workgroup; the stream's T(h), the norm's
//     operand T(h w) and sums of h^2 leave from there, and 1 / rms is a factor of the next product's finished sums.  T(h w) is f16, which 1 / rms would bring into range:
//     two powers of two do, `unit`, which makes the largest |w| at most one, and one of each row, from a bound on the row's |h| that every workgroup of a launch
//     knows: sqrt(sum h^2) in front of the add, which the norm's product has left, and |x| times the largest column of W behind it (Cauchy and Schwarz; |x|^2 is the
//     diagonal of an instruction x x^T, which the matrix unit has time for).  The bound is set to 2^14 .. 2^15, and may be 2^10 above what a row holds: f16 is
//     normal down to 2^-14.  An operand is rounded once either way.  (With `unit` alone rows of small h left f16's normal range: error of a product of 4096 columns, one weight
//     of the norm 20 times the others, h of 1e-3 5.4e-4 and of 1e-4 6.4e-3, where the norm's own launch has 2e-4);
//   * the product is v_mfma_f32_16x16x32 with the weights as rows.  A lane's sixteen bytes are 32 k of one column; lanes l / 16 hold the four halves of two k64-steps, so that word i of
//     all of them is one operand against chunk i of x of the same halves: no rows of lanes to swap (gptq_wide_body.h), and 1 KiB of image to four instructions;
//   * in front of a norm a wave keeps x of its k-steps in registers (16 VGPR each) and takes units in turn; behind, x is asked for a step ahead.
// us a launch of 4096, 11008 at 16 rows, the other launches and the norm behind them / these: qkv 10.1 / 9.6, o 8.8 / 5.6, gate | up 13.8 / 13.3, down 11.7 / 10.7 (of these two x x^T
// and the bound 0.2 and 0.6): 2.7 TB/s of
// weights, bound by the launch's own ends and, of what is left, by the round trip of a turn's loads (weights of a turn ahead in registers of their own cost 0.7 us: x holds 64).
// Whole steps at ctx 137, 1, 4, 16 rows: eight layers of 4096, 11008 440 / 419, 471 / 424, 526 / 483; of 2048, 5632 294 / 238, 295 / 239, 308 / 253; of 3072, 8192 349 / 330, 365 /
// 335, 379 / 349; of 1536, 4096 272 / 227, 279 / 231, 300 / 251; of 1024, 2816 230 / 204, 237 / 207, 246 / 214; of 768, 2048 224 / 190, 230 / 193, 244 / 203; of 512, 1536 209 / 184,
// 214 / 186, 223 / 192; four of 8192, 28672 572 / 526, 569 / 518, 572 / 535; between 4096 and 6144 columns FlashLlamaModel.serves_int4_rows.  At 17 - 32 rows a weight feeds two instructions
// and x of a whole k range takes as long as the weights: products as above at 32 rows 12.0 / 11.8, 9.6 / 6.8, 16.4 / 16.1, 13.3 / 14.1.
// Steps at 24, 32 rows: 4096, 11008 608 / 575, 634 / 617; 3072, 8192 418 / 402, 429 / 421; 2048, 5632 334 / 284, 340 / 299; 1536, 4096 345 / 301, 358 / 320; 1024, 2816 268 / 245, 276 /
// 258; 768, 2048 280 / 236, 286 / 250; 512, 1536 241 / 214, 247 / 223.  Past 4096 columns x of two blocks leaves the registers of one unit: not served.
#include <algorithm>
#include "gptq_gemm_body.h"

namespace {

constexpr int GROWS_M = 32;
enum { GROWS_ROPE, GROWS_SILU };
struct GRowsArgs {
    const f16* x;       // T(h w unit) or an activation, fragment order (xf_off)
    float* sums;        // [K / 64][32 rows][4]: sums of h^2 of sixteen columns; behind them of whole rows [32], and what a row's operand is to be multiplied by [32]
    float eps, unit;
    const uint8_t* prep;
    int64_t offB;
    int M, K, N, KS, G, spg_shift;
    f16* out;
    int64_t ldo;
    // the stream behind a residual product
    const f16* norm_w;
    const int32_t* places;  // where the next product wants column k of its operand (null: at k)
    f16 *h, *hw;            // T(h) [M][N]; T(h w unit), fragment order
    float w_norm;           // at least the largest 2-norm of a column of W
    // ROPE (as tgis_gptq_gemm_rope_f16)
    const f16* bias;
    const int32_t *positions, *slots;
    const f16 *cosb, *sinb;
    f16 *kpool, *vpool;
    int H, Hkv, D;
};
__device__ __forceinline__ int64_t sums16_off(int m, int k) { return ((int64_t)(k >> 6) * GROWS_M + m) * 4 + ((k >> 4) & 3); }
__device__ __forceinline__ float* row_sums(float* sums, int width) { return sums + (int64_t)(width >> 4) * GROWS_M; }
__device__ __forceinline__ float* row_factors(float* sums, int width) { return row_sums(sums, width) + GROWS_M; }

// c of the 2^c that brings a bound on a row's |h|, given by its square, to 2^14 .. 2^15 (squares that are zero, infinite or NaN: an end of a range whose powers fp32 holds)
__device__ __forceinline__ int row_power(float square) {
    const int e = (int)(__builtin_bit_cast(uint32_t, square) >> 23 & 255) - 127;
    return min(max(14 - (e >> 1), -64), 64);
}
__device__ __forceinline__ f16 operand(float h, f16 w, float unit, int c) { return (f16)ldexpf(h * ((float)w * unit), c); }

// byte offset of a lane's part (32 k of one column `col` of the tile) within the two k64-steps of a tile, and of x's (row m) within its two
__device__ __forceinline__ uint32_t grows_w_off(int kq, int col) { return (kq >> 1) * 1024 + ((kq & 1) * 32 + col) * 16; }
__device__ __forceinline__ uint32_t grows_x_off(int kq, int m) { return (kq >> 1) * 4096 + ((kq & 1) * 32 + m) * 16; }

struct GRowsDequant {
    uint32_t EX = 0x64006400u, M0 = 0x000F000Fu, M1 = 0x00F000F0u;
    __device__ __forceinline__ GRowsDequant() {
        asm volatile("" : "+v"(EX));
        asm volatile("" : "+s"(M0), "+s"(M1));
    }
    // acc += (a lane's 32 k of a column) x (x of the same, each block of sixteen rows)
    template <int RB>
    __device__ __forceinline__ void mma(const u32x4& q, uint32_t sz, const f16x8 (&x)[RB][4], f32x4 (&acc)[RB]) const {
        const f16x2 s = __builtin_bit_cast(f16x2, sz);
        const f16 zc1 = s[1], zd1 = (f16)960.f - zc1;
        const f16x2 zc = {zc1, zc1}, zd = {zd1, zd1}, sc = {s[0], s[0]};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const f16x8 w = gptq::dequant8(q[i], zc, zd, sc, EX, M0, M1);
#pragma unroll
            for (int b = 0; b < RB; ++b) acc[b] = mfma16(w, x[b][i], acc[b]);
        }
    }
};

// the largest of v over a workgroup of T threads
template <int T>
__device__ __forceinline__ float block_max(float v, float (&red)[T / 64]) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) v = fmaxf(v, __shfl_xor(v, d, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < T / 64; ++k) v = fmaxf(v, red[k]);
    return v;
}

// the stream of tokens, a row a workgroup
__global__ __launch_bounds__(256) void gptq_rows_embed_kernel(const int64_t* __restrict__ ids, const f16* __restrict__ table, int64_t vocab, GRowsArgs a) {
    __shared__ float red[4];
    const int m = blockIdx.x;
    const int64_t id = ids[m];
    const bool known = id >= 0 && id < vocab;
    auto columns = [&](int k) { return known ? ld16<f16x8>(table + id * a.K + k) : f16x8{}; };
    float top = 0.f;
    for (int k = threadIdx.x * 8; k < a.K; k += 2048) {
        const f16x8 v = columns(k);
#pragma unroll
        for (int e = 0; e < 8; ++e) top = fmaxf(top, fabsf((float)v[e]));
    }
    const int c = row_power(block_max<256>(top * top, red));
    for (int k = threadIdx.x * 8; k < a.K; k += 2048) {
        const f16x8 v = columns(k), w = ld16<f16x8>(a.norm_w + k);
        f16x8 y;
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            ss += (float)v[e] * (float)v[e];
            y[e] = operand((float)v[e], w[e], a.unit, c);
        }
        st16(a.h + (int64_t)m * a.K + k, v);
        if (a.places) {
#pragma unroll
            for (int e = 0; e < 8; ++e) a.hw[xf_off(m, a.places[k + e], a.K)] = y[e];
        } else {
            st16(a.hw + xf_off(m, k, a.K), y);
        }
        ss += __shfl_xor(ss, 1, 64);
        if ((threadIdx.x & 1) == 0) a.sums[sums16_off(m, k)] = ss;
    }
    if (threadIdx.x == 0) row_factors(a.sums, a.K)[m] = ldexpf(1.f, -c);
}

// Products of a normed operand.  A unit is columns c0 .. +7 and c0 + 16 .. +23 of a tile: the halves of a rotation, or gate and up.  DS: double k64-steps of a wave at most;
// P: units a workgroup
// takes at a time, with one exchange of its waves' sums.
template <int KIND, int W, int RB, int DS, int P>
__global__ __launch_bounds__(64 * W) void gptq_rows_kernel(GRowsArgs a, int units, int per) {
    __shared__ __attribute__((aligned(16))) float red[2][P][RB][W][64 * 4];
    __shared__ float part[W][16 * RB];
    constexpr int FW = P * RB <= 4 ? 4 : 8;  // a turn's outputs are finished by FW waves, a unit's block of rows each
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int steps = a.K >> 7, mine = (steps - w + W - 1) / W;  // of 128 k: w, w + W, ..
    const int m = lane & 15, kq = lane >> 4;
    const int fp = w % FW / RB, fb = w % RB, frow = fb * 16 + m;  // the unit of a turn and the row that this lane finishes
    const int u0 = blockIdx.x * per, n = min(per, units - u0);

    const float factor = row_factors(a.sums, a.K)[min(frow, a.M - 1)] / a.unit;
    int32_t pos = 0, slot = 0;
    if (KIND == GROWS_ROPE) {
        pos = a.positions[min(frow, a.M - 1)];
        slot = a.slots[min(frow, a.M - 1)];
    }
    f16x8 x[DS][RB][4];
    uint32_t xoff[RB];
#pragma unroll
    for (int b = 0; b < RB; ++b) xoff[b] = grows_x_off(kq, min(b * 16 + m, a.M - 1));
#pragma unroll
    for (int j = 0; j < DS; ++j) {
        const char* p = reinterpret_cast<const char*>(a.x) + (int64_t)min(w + W * j, steps - 1) * 8192;
        PIN_SGPR(p);
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) x[j][b][i] = *(const GLOBAL_AS f16x8*)(p + xoff[b] + i * 1024);
    }
    constexpr int SG = (DS + 1) / 2;  // groups of 4 x 16 columns of a lane
    f32x4 sq[RB][SG];
    const int groups64 = a.K >> 6;
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int t = 0; t < SG; ++t)
            sq[b][t] = *reinterpret_cast<const f32x4*>(a.sums + ((int64_t)min((t * W + w) * 4 + kq, groups64 - 1) * GROWS_M + min(b * 16 + m, a.M - 1)) * 4);

    const int cl = (lane & 7) + ((lane >> 3) & 1) * 16;
    u32x4 wq[P][DS];
    uint32_t sz[P][DS];
    auto ask = [&](int slot_, int u) {
        const int tile = u >> 1, col = cl + (u & 1) * 8;
        const char* base = reinterpret_cast<const char*>(a.prep) + (int64_t)tile * a.KS * 1024;
        const char* sbase = reinterpret_cast<const char*>(a.prep + a.offB) + (int64_t)tile * a.G * 128;
        PIN_SGPR(sbase);
        const uint32_t woff = grows_w_off(kq, col);
#pragma unroll
        for (int j = 0; j < DS; ++j) {
            const int s = min(w + W * j, steps - 1);
            const int g = min((2 * s + (kq >> 1)) >> a.spg_shift, a.G - 1);
            const uint32_t v = *(const GLOBAL_AS uint32_t*)(sbase + (uint32_t)(g * 128 + col * 4));
            sz[slot_][j] = j < mine ? v : 0u;
        }
#pragma unroll
        for (int j = 0; j < DS; ++j) {
            const char* p = base + (int64_t)min(w + W * j, steps - 1) * 2048;
            PIN_SGPR(p);
            wq[slot_][j] = __builtin_nontemporal_load((const GLOBAL_AS u32x4*)(p + woff));
        }
    };
#pragma unroll
    for (int d = 0; d < P; ++d) ask(d, min(u0 + d, units - 1));

    const bool second = kq >= 2;  // this lane's finished columns are of the tile's second half
    f16x4 cf{}, sf{}, bv{};
    int head = 0, dim = 0;
    auto rope_inputs = [&](int u) {
        const int tile = u >> 1, c = (u & 1) * 8 + (kq & 1) * 4, per_head = a.D >> 5, tt = tile % per_head;
        head = tile / per_head;
        const bool roth = head < a.H + a.Hkv;
        dim = roth ? (second ? (a.D >> 1) : 0) + 16 * tt + c : 32 * tt + c + (second ? 16 : 0);
        if (roth) {
            const int64_t at = (int64_t)pos * (a.D >> 1) + 16 * tt + c;
            cf = *reinterpret_cast<const f16x4*>(a.cosb + at);
            sf = *reinterpret_cast<const f16x4*>(a.sinb + at);
        }
        if (a.bias) bv = *reinterpret_cast<const f16x4*>(a.bias + head * a.D + dim);
    };
    if (KIND == GROWS_ROPE) rope_inputs(u0 + min(w / FW * P + fp, n - 1));  // of the first unit that this wave finishes

#pragma unroll
    for (int b = 0; b < RB; ++b) {
        float ss = 0.f;
#pragma unroll
        for (int t = 0; t < SG; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) ss += (t * W + w) * 4 + kq < groups64 ? sq[b][t][e] : 0.f;
        ss += __shfl_xor(ss, 16, 64);
        ss += __shfl_xor(ss, 32, 64);
        if (kq == 0) part[w][b * 16 + m] = ss;  // (read behind the first turn's barrier)
    }

    const GRowsDequant dq;
    // P units from i on; what the next P take is asked for as each is done with
    auto turn = [&](const int i, auto more_tag) {
        constexpr bool MORE = decltype(more_tag)::value;
        const int r = (i / P) & 1;
#pragma unroll
        for (int p = 0; p < P; ++p) {
            f32x4 acc[RB] = {};
#pragma unroll
            for (int j = 0; j < DS; ++j) dq.mma(wq[p][j], sz[p][j], x[j], acc);
            if (MORE) ask(p, min(u0 + i + P + p, units - 1));
#pragma unroll
            for (int b = 0; b < RB; ++b) *reinterpret_cast<f32x4*>(&red[r][p][b][w][lane * 4]) = acc[b];
        }
        __syncthreads();  // (the buffer before last was read in front of a barrier since)
        const int at = i + fp;
        if (w / FW != (i / P) % (W / FW) || fp >= P || at >= n) return;
        float tot = 0.f;
#pragma unroll
        for (int k = 0; k < W; ++k) tot += part[k][frow];
        if (blockIdx.x == 0 && at == 0 && kq == 0 && frow < a.M) row_sums(a.sums, a.K)[frow] = tot;  // (for the residual product behind)
        const float rstd = rsqrtf(tot / a.K + a.eps) * factor;
        f32x4 v = *reinterpret_cast<const f32x4*>(&red[r][fp][fb][0][lane * 4]);
#pragma unroll
        for (int k = 1; k < W; ++k) v += *reinterpret_cast<const f32x4*>(&red[r][fp][fb][k][lane * 4]);
        v *= rstd;
        // v[e]: row frow, column c + e of its half of the tile
        const int u = u0 + at, tile = u >> 1, c = (u & 1) * 8 + (kq & 1) * 4;
        const bool live = frow < a.M;
        f16x4 o;
        if (KIND == GROWS_SILU) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float own = (float)(f16)v[e], up = __shfl_xor(own, 32, 64);
                const float sl = own / (1.f + __expf(-own));
                o[e] = (f16)((float)(f16)sl * up);
            }
            if (live && !second) *reinterpret_cast<f16x4*>(a.out + xf_off(frow, tile * 16 + c, a.N >> 1)) = o;
        } else {
            if (i >= P * (W / FW)) rope_inputs(u);
            const bool roth = head < a.H + a.Hkv;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float own = (float)(f16)(v[e] + (float)bv[e]), other = __shfl_xor(own, 32, 64);
                const float co = (float)cf[e], si = (float)sf[e];
                o[e] = (f16)(!roth ? own : second ? other * si + own * co : own * co - other * si);
            }
            if (!live) return;
            const int64_t page = slot >> 5;
            const int tok = slot & 31;
            if (head < a.H) {
                *reinterpret_cast<f16x4*>(a.out + (int64_t)frow * a.ldo + head * a.D + dim) = o;
            } else if (roth) {
                *reinterpret_cast<f16x4*>(a.kpool + (page * a.Hkv + (head - a.H)) * 32 * a.D + k_off(tok, dim, a.D)) = o;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) a.vpool[(page * a.Hkv + (head - a.H - a.Hkv)) * 32 * a.D + v_off(tok, dim + e, a.D)] = o[e];
            }
        }
    };
    int i = 0;
    for (; i + P < n; i += P) turn(i, std::true_type{});
    turn(i, std::false_type{});
}

// h += T(x W) and what the next norm's product needs of it; a unit of sixteen columns a workgroup.  DS: double k64-steps of a wave at most.  us at 16 rows, eight waves / sixteen (without x x^T): 4096
// x 4096 5.5 / 5.8, 11008 x 4096 10.0 / 10.3, 2048 x 2048 3.7 / 4.6, 8192 x 8192 15.0 / 16.3; x asked for one, three, five steps ahead 10.0 / 10.3 / 10.5 (11008 x 4096).
template <int RB, int DS>
__global__ __launch_bounds__(512) void gptq_rows_residual_kernel(GRowsArgs a) {
    constexpr int W = 8;
    __shared__ __attribute__((aligned(16))) float red[RB][W][64 * 4];
    __shared__ __attribute__((aligned(16))) float squares[16 * RB][W];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int steps = a.K >> 7, mine = (steps - w + W - 1) / W;
    const int m = lane & 15, kq = lane >> 4;
    const int tile = blockIdx.x >> 1, c0 = (blockIdx.x & 1) * 16;
    const char* base = reinterpret_cast<const char*>(a.prep) + (int64_t)tile * a.KS * 1024;
    const char* sbase = reinterpret_cast<const char*>(a.prep + a.offB) + (int64_t)tile * a.G * 128;
    PIN_SGPR(sbase);
    const uint32_t woff = grows_w_off(kq, c0 + m);
    uint32_t xoff[RB];
#pragma unroll
    for (int b = 0; b < RB; ++b) xoff[b] = grows_x_off(kq, min(b * 16 + m, a.M - 1));
    auto step_at = [&](int j) { return min(w + W * j, steps - 1); };
    f16x8 x[2][RB][4];
    auto ask_x = [&](int d, int j) {
        const char* p = reinterpret_cast<const char*>(a.x) + (int64_t)step_at(j) * 8192;
        PIN_SGPR(p);
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) x[d][b][i] = *(const GLOBAL_AS f16x8*)(p + xoff[b] + i * 1024);
    };
    ask_x(0, 0);
    u32x4 wq[DS];
    uint32_t sz[DS];
#pragma unroll
    for (int j = 0; j < DS; ++j) {
        const int s = step_at(j), g = min((2 * s + (kq >> 1)) >> a.spg_shift, a.G - 1);
        const uint32_t v = *(const GLOBAL_AS uint32_t*)(sbase + (uint32_t)(g * 128 + (c0 + m) * 4));
        sz[j] = j < mine ? v : 0u;
        const char* p = base + (int64_t)s * 2048;
        PIN_SGPR(p);
        wq[j] = __builtin_nontemporal_load((const GLOBAL_AS u32x4*)(p + woff));
    }
    if (DS > 1) ask_x(1, 1);
    const int col = tile * 32 + c0 + kq * 4;  // .. + 3: what this lane of the first RB waves finishes, of its row
    const int frow = w * 16 + m;
    f16x4 res{}, nw{};
    int32_t at[4] = {};
    float before = 0.f;
    if (w < RB) {
        before = row_sums(a.sums, a.N)[min(frow, a.M - 1)];
        res = *reinterpret_cast<const f16x4*>(a.h + (int64_t)min(frow, a.M - 1) * a.N + col);
        nw = *reinterpret_cast<const f16x4*>(a.norm_w + col);
        if (a.places) {
#pragma unroll
            for (int e = 0; e < 4; ++e) at[e] = a.places[col + e];
        }
    }
    const GRowsDequant dq;
    f32x4 acc[RB] = {}, gram[RB] = {};  // gram: rows by rows of x
#pragma unroll
    for (int j = 0; j < DS; ++j) {
        dq.mma(wq[j], sz[j], x[j & 1], acc);
#pragma unroll
        for (int b = 0; b < RB; ++b)  // (of steps past this wave's last, too, which are another's: the bound is only higher)
#pragma unroll
            for (int i = 0; i < 4; ++i) gram[b] = mfma16(x[j & 1][b][i], x[j & 1][b][i], gram[b]);
        if (j + 2 < DS) ask_x(j & 1, j + 2);
    }
#pragma unroll
    for (int b = 0; b < RB; ++b) {
        *reinterpret_cast<f32x4*>(&red[b][w][lane * 4]) = acc[b];
        const float lo = m & 1 ? gram[b][1] : gram[b][0], hi = m & 1 ? gram[b][3] : gram[b][2];
        if (kq == m >> 2) squares[b * 16 + m][w] = m & 2 ? hi : lo;
    }
    __syncthreads();
    if (w >= RB) return;
    float xx = 0.f;
#pragma unroll
    for (int k = 0; k < W; ++k) xx += squares[frow][k];
    const int c = row_power(2.f * (before + xx * a.w_norm * a.w_norm));  // (a + b)^2 <= 2 (a^2 + b^2)
    f32x4 v = *reinterpret_cast<const f32x4*>(&red[w][0][lane * 4]);
#pragma unroll
    for (int k = 1; k < W; ++k) v += *reinterpret_cast<const f32x4*>(&red[w][k][lane * 4]);
    f16x4 h, hw;
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float f = (float)(f16)v[e] + (float)res[e];
        ss += f * f;
        h[e] = (f16)f;
        hw[e] = operand(f, nw[e], a.unit, c);
    }
    ss += __shfl_xor(ss, 16, 64);
    ss += __shfl_xor(ss, 32, 64);
    if (frow >= a.M) return;
    *reinterpret_cast<f16x4*>(a.h + (int64_t)frow * a.N + col) = h;
    if (a.places) {
#pragma unroll
        for (int e = 0; e < 4; ++e) a.hw[xf_off(frow, at[e], a.N)] = hw[e];
    } else {
        *reinterpret_cast<f16x4*>(a.hw + xf_off(frow, col, a.N)) = hw;
    }
    if (kq == 0) a.sums[sums16_off(frow, col)] = ss;
    if (kq == 0 && blockIdx.x == 0) row_factors(a.sums, a.N)[frow] = ldexpf(1.f, -c);
}

// The same behind a product whose k range was split: S slabs [32][ld] of a tgis_gptq_gemm_partial.  A row a workgroup, which has its largest |h| then: 11 - 32 rows of 4096 3.6 - 3.9 us (a
// thread per sixteen columns wherever it runs, which has not, 3.1).
__global__ __launch_bounds__(1024) void gptq_rows_sum_kernel(const float* __restrict__ slabs, int S, int64_t ld, GRowsArgs a) {
    __shared__ float red[16];
    const int m = blockIdx.x;
    float f[8];
    f16x8 w;
    int32_t at[8];
    auto columns = [&](int k) {
        const f16x8 res = ld16<f16x8>(a.h + (int64_t)m * a.N + k);
        w = ld16<f16x8>(a.norm_w + k);
        if (a.places) {
#pragma unroll
            for (int e = 0; e < 8; ++e) at[e] = a.places[k + e];
        }
        f32x4 lo, hi;
        sum_slabs8(slabs + (int64_t)m * ld + k, 32 * ld, S, lo, hi);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = (float)(f16)(e < 4 ? lo[e & 3] : hi[e & 3]) + (float)res[e];
    };
    float top = 0.f;
    for (int k = threadIdx.x * 8; k < a.N; k += 8192) {
        columns(k);
#pragma unroll
        for (int e = 0; e < 8; ++e) top = fmaxf(top, fabsf(f[e]));
    }
    const int c = row_power(block_max<1024>(top * top, red));
    for (int k = threadIdx.x * 8; k < a.N; k += 8192) {
        if (a.N > 8192) columns(k);
        f16x8 h, hw;
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            ss += f[e] * f[e];
            h[e] = (f16)f[e];
            hw[e] = operand(f[e], w[e], a.unit, c);
        }
        st16(a.h + (int64_t)m * a.N + k, h);
        if (a.places) {
#pragma unroll
            for (int e = 0; e < 8; ++e) a.hw[xf_off(m, at[e], a.N)] = hw[e];
        } else {
            st16(a.hw + xf_off(m, k, a.N), hw);
        }
        ss += __shfl_xor(ss, 1, 64);
        if ((threadIdx.x & 1) == 0) a.sums[sums16_off(m, k)] = ss;
    }
    if (threadIdx.x == 0) row_factors(a.sums, a.N)[m] = ldexpf(1.f, -c);
}

// groups of 64 2^n rows, as gptq_wide_body.h; K of whole double steps, as many as a wave's registers hold of x (or, where steps of 5120 columns and more
// than 16 rows are no sooner done, 4096), or of one unit's weights
bool grows_fits(int64_t M, int64_t K, int64_t N, int64_t groups, bool norm) {
    if (M < 1 || M > GROWS_M || K < 128 || K % 128 || N < 32 || N % 32 || N >= (1ll << 31) || groups < 1 || K % groups) return false;
    if (K > (!norm ? 12288 : M <= 16 ? 8192 : 4096)) return false;
    const int64_t spg = K / groups / 64;
    return groups == 1 || (K / groups % 64 == 0 && (spg & (spg - 1)) == 0);
}

int grows_args(const char* what, GRowsArgs& a, const void* x, float* sums, float eps, float unit, const void* prepared, int64_t M, int64_t K, int64_t N,
               int64_t groups, bool norm) {
    TGIS_CHECK_ARG(x && prepared && sums && unit > 0.f, "%s: null tensor or bad factor", what);
    TGIS_CHECK_ARG(grows_fits(M, K, N, groups, norm), "%s: up to %d rows, K a multiple of 128 up to %d, groups of 64 2^n (M=%ld K=%ld N=%ld groups=%ld)", what, GROWS_M,
                   !norm ? 12288 : M <= 16 ? 8192 : 4096, (long)M, (long)K, (long)N, (long)groups);
    TGIS_CHECK_ARG(((uintptr_t)x | (uintptr_t)prepared | (uintptr_t)sums) % 16 == 0, "%s: operands must be 16-byte aligned", what);
    const gptq::PrepLayout p = gptq::prep_layout(K, N, groups);
    a = GRowsArgs{};
    a.x = (const f16*)x;
    a.sums = sums;
    a.eps = eps;
    a.unit = unit;
    a.prep = (const uint8_t*)prepared;
    a.offB = p.offB;
    a.M = (int)M;
    a.K = (int)K;
    a.N = (int)N;
    a.KS = (int)p.KS;
    a.G = (int)groups;
    a.spg_shift = 30;
    if (groups > 1)
        for (a.spg_shift = 0; (64 << a.spg_shift) < K / groups; ++a.spg_shift) {}
    return TGIS_OK;
}

template <int KIND, int W, int RB, int DS, int P>
void launch_grows_k(const GRowsArgs& a, int per, hipStream_t st) {
    const int units = a.N / 16;
    hipLaunchKernelGGL((gptq_rows_kernel<KIND, W, RB, DS, P>), dim3((unsigned)((units + per - 1) / per)), dim3(64 * W), 0, st, a, units, per);
}
template <int KIND, int RB, int DS>
void launch_grows_p(const GRowsArgs& a, int per, hipStream_t st) {
    if (per % 2 == 0) return launch_grows_k<KIND, 8, RB, DS, 2>(a, per, st);
    if constexpr (RB == 1 || DS <= 2)
        if (per % 3 == 0) return launch_grows_k<KIND, 8, RB, DS, 3>(a, per, st);
    launch_grows_k<KIND, 8, RB, DS, 1>(a, per, st);
}
// One workgroup a CU.  us at 16 rows, turns of one, two, three units: gate | up of 4096 x 22016 (6 units a workgroup) 14.3 / 12.9 / 13.3, of 2048 x 11264 (3) 6.6 / 6.5 / 5.8; qkv of
// 4096 x 12288 (3) 10.0 / 11.7 / 9.6, at 32 rows 11.5 / 13.4 / 12.0; from K 5120 on x leaves the registers of one: 5120 x 27648 (7) 19.7 / 21.2 / 22.5.  Sixteen waves take less of x each: 8192 x 57344
// 54.2 -> 49.1, but 4096 x 22016 14.8 and, with what a rotation needs besides, 8192 x 10240 17.9 -> 36.5.
template <int KIND>
int launch_grows(const GRowsArgs& a, hipStream_t st) {
    TgisTimedScope timed(TGIS_OP_GPTQ_GEMM, st);
    const int units = a.N / 16, per = (units + 255) / 256, ds = (a.K + 1023) / 1024;
    if (a.M > 16) {
        if (ds <= 2)
            launch_grows_p<KIND, 2, 2>(a, per, st);
        else
            launch_grows_p<KIND, 2, 4>(a, per, st);
    } else if (ds <= 2)
        launch_grows_p<KIND, 1, 2>(a, per, st);
    else if (ds <= 4)
        launch_grows_p<KIND, 1, 4>(a, per, st);
    else
        launch_grows_k<KIND, KIND == GROWS_SILU ? 16 : 8, 1, KIND == GROWS_SILU ? 4 : 8, 1>(a, per, st);
    TGIS_CHECK_LAUNCH();
    return TGIS_OK;
}
template <int RB>
void launch_grows_residual(const GRowsArgs& a, hipStream_t st) {
    const int ds = (a.K + 1023) / 1024;
    const auto kernel = ds <= 2   ? gptq_rows_residual_kernel<RB, 2>
                        : ds <= 4 ? gptq_rows_residual_kernel<RB, 4>
                        : ds <= 6 ? gptq_rows_residual_kernel<RB, 6>
                        : ds <= 8 ? gptq_rows_residual_kernel<RB, 8>
                                  : gptq_rows_residual_kernel<RB, 12>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(a.N / 16)), dim3(512), 0, st, a);
}

}  // namespace

extern "C" int tgis_gptq_rows_ok(int64_t M, int64_t K, int64_t N, int64_t groups, int norm) { return grows_fits(M, K, N, groups, norm != 0) ? 1 : 0; }

extern "C" int tgis_gptq_rows_embed(const int64_t* ids, const void* table, const void* norm_w, const int32_t* places, float unit, void* h, void* hw, float* sums,
                                    int64_t M, int64_t K, int64_t vocab, void* stream) {
    TGIS_CHECK_ARG(ids && table && norm_w && h && hw && sums && unit > 0.f, "tgis_gptq_rows_embed: null tensor or bad factor");
    TGIS_CHECK_ARG(M >= 1 && M <= GROWS_M && K >= 64 && K % 64 == 0 && K <= (1 << 20) && vocab > 0, "tgis_gptq_rows_embed: up to %d rows of a multiple of 64 columns", GROWS_M);
    TGIS_CHECK_ARG(((uintptr_t)table | (uintptr_t)norm_w | (uintptr_t)h | (uintptr_t)hw | (uintptr_t)sums) % 16 == 0, "tgis_gptq_rows_embed: tensors must be 16-byte aligned");
    GRowsArgs a{};
    a.M = (int)M;
    a.K = (int)K;
    a.norm_w = (const f16*)norm_w;
    a.places = places;
    a.unit = unit;
    a.h = (f16*)h;
    a.hw = (f16*)hw;
    a.sums = sums;
    hipLaunchKernelGGL(gptq_rows_embed_kernel, dim3((unsigned)M), dim3(256), 0, (hipStream_t)stream, ids, (const f16*)table, vocab, a);
    TGIS_CHECK_LAUNCH();
    return TGIS_OK;
}

extern "C" int tgis_gptq_rows_residual(const void* x, const void* prepared, float w_norm, const void* norm_w, const int32_t* places, float unit, void* h, void* hw,
                                       float* sums, int64_t M, int64_t K, int64_t N, int64_t groups, void* stream) {
    const char* what = "tgis_gptq_rows_residual";
    GRowsArgs a;
    const int rc = grows_args(what, a, x, sums, 0.f, unit, prepared, M, K, N, groups, false);
    if (rc != TGIS_OK) return rc;
    TGIS_CHECK_ARG(norm_w && h && hw && ((uintptr_t)norm_w | (uintptr_t)h | (uintptr_t)hw) % 16 == 0 && N % 64 == 0 && w_norm >= 0.f,
                   "%s: null or unaligned tensor, a width that is no multiple of 64, or no bound on the columns", what);
    a.norm_w = (const f16*)norm_w;
    a.places = places;
    a.h = (f16*)h;
    a.hw = (f16*)hw;
    a.w_norm = w_norm;
    TgisTimedScope timed(TGIS_OP_GPTQ_GEMM, (hipStream_t)stream);
    if (M <= 16)
        launch_grows_residual<1>(a, (hipStream_t)stream);
    else
        launch_grows_residual<2>(a, (hipStream_t)stream);
    TGIS_CHECK_LAUNCH();
    return TGIS_OK;
}

extern "C" int tgis_gptq_rows_sum(const float* slabs, int num_slabs, int64_t ld, const void* norm_w, const int32_t* places, float unit, void* h, void* hw, float* sums,
                                  int64_t M, int64_t N, void* stream) {
    const char* what = "tgis_gptq_rows_sum";
    TGIS_CHECK_ARG(slabs && norm_w && h && hw && sums && unit > 0.f && num_slabs >= 1 && ld >= N && ld % 4 == 0, "%s: null tensor, bad factor or bad slabs", what);
    TGIS_CHECK_ARG(M >= 1 && M <= GROWS_M && N >= 64 && N % 64 == 0 && N <= (1 << 20), "%s: up to %d rows of a multiple of 64 columns", what, GROWS_M);
    TGIS_CHECK_ARG(((uintptr_t)slabs | (uintptr_t)norm_w | (uintptr_t)h | (uintptr_t)hw | (uintptr_t)sums) % 16 == 0, "%s: tensors must be 16-byte aligned", what);
    GRowsArgs a{};
    a.M = (int)M;
    a.N = (int)N;
    a.norm_w = (const f16*)norm_w;
    a.places = places;
    a.unit = unit;
    a.h = (f16*)h;
    a.hw = (f16*)hw;
    a.sums = sums;
    hipLaunchKernelGGL(gptq_rows_sum_kernel, dim3((unsigned)M), dim3(1024), 0, (hipStream_t)stream, slabs, num_slabs, ld, a);
    TGIS_CHECK_LAUNCH();
    return TGIS_OK;
}

extern "C" int tgis_gptq_rows_norm_silu(const void* hw, float* sums, float eps, float unit, const void* prepared, void* out, int64_t M, int64_t K, int64_t N,
                                        int64_t groups, void* stream) {
    const char* what = "tgis_gptq_rows_norm_silu";
    GRowsArgs a;
    const int rc = grows_args(what, a, hw, sums, eps, unit, prepared, M, K, N, groups, true);
    if (rc != TGIS_OK) return rc;
    TGIS_CHECK_ARG(out && (uintptr_t)out % 16 == 0 && N % 128 == 0, "%s: needs a gate|up image (N / 2 a multiple of 64) and its output", what);
    a.out = (f16*)out;
    return launch_grows<GROWS_SILU>(a, (hipStream_t)stream);
}

extern "C" int tgis_gptq_rows_norm_rope(const void* hw, float* sums, float eps, float unit, const void* prepared, const void* bias, const int32_t* positions,
                                        const int32_t* slots, const void* cos, const void* sin, void* q_out, int64_t ldq, void* k_pool, void* v_pool, int64_t M,
                                        int64_t K, int64_t groups, int64_t H, int64_t Hkv, int64_t D, void* stream) {
    const char* what = "tgis_gptq_rows_norm_rope";
    TGIS_CHECK_ARG(H >= 1 && Hkv >= 1 && D >= 32 && D % 32 == 0 && ldq >= H * D, "%s: bad head geometry", what);
    GRowsArgs a;
    const int rc = grows_args(what, a, hw, sums, eps, unit, prepared, M, K, (H + 2 * Hkv) * D, groups, true);
    if (rc != TGIS_OK) return rc;
    TGIS_CHECK_ARG(positions && slots && cos && sin && q_out && k_pool && v_pool, "%s: null tensor", what);
    TGIS_CHECK_ARG(ldq % 4 == 0 && ((uintptr_t)q_out | (uintptr_t)cos | (uintptr_t)sin | (uintptr_t)bias | (uintptr_t)k_pool) % 8 == 0,
                   "%s: q, its rows, bias, tables and pages must be 8-byte aligned", what);
    a.out = (f16*)q_out;
    a.ldo = ldq;
    a.bias = (const f16*)bias;
    a.positions = positions;
    a.slots = slots;
    a.cosb = (const f16*)cos;
    a.sinb = (const f16*)sin;
    a.kpool = (f16*)k_pool;
    a.vpool = (f16*)v_pool;
    a.H = (int)H;
    a.Hkv = (int)Hkv;
    a.D = (int)D;
    return launch_grows<GROWS_ROPE>(a, (hipStream_t)stream);
}
