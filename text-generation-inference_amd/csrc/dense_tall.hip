// The dense (f16 / bf16) GEMM of prefills, on the image that the weight-streaming kernel of decode steps reads (tgis_dense_prepare): more rows
// than that one takes in a pass, and the products for which a library's 256 x 256 tiles leave most of the chip idle or need a launch of
// their own for the activation.
//
// A block of 4 waves owns a tile of 64, 96 or 128 rows x 128 or 256 columns; wave w its columns, TW tiles of 32, whose fragments it loads
// straight from the image into registers, WR k64-steps ahead: no other wave reads them, so they need no LDS.  x, which all four read, goes to
// LDS with direct loads, a ring of four k64-steps of 128-byte rows whose 16-byte pieces are permuted (piece ^ row / 2 mod 8) so that the fragment
// reads of 16 rows fill all banks.  One barrier a step, which is two slices of 32 k in two halves of the rows; while one half is multiplied the A fragments of
// the next are read.
//
// Products by the 16x16x32 instruction: under the card's power limit it does more than 32x32x16 (bare loops on random values, PFLOP/s: bf16 2.10 against 1.77, f16
// 1.95, 1.71).  us, 32x32x16 / now: 2048 x 11264 with SiLU at 1024, 1393, 4096 rows 55.9 / 53.2, 65.2 / 60.8, 173 / 160; 4096 x 22016 with SiLU at 2048 327 / 305;
// 6144 x 24576 at 400 165 / 156; where a SIMD has one wave, twice the products to issue cost 2 - 6 % of tiles of 256 columns (24576 x 6144 at 128 rows 307 / 321):
// of the plans those of 193 - 256 rows of some 20000 columns and more (4096 x 22016 with SiLU at 256, 172 tiles, 63.0 / 64.0; 4096 x 28672 at 224 72.2 / 74.2).
//
// Bound: the matrix cores and their power from about 1000 rows on (1.15 - 1.35 PFLOP/s; with nothing to load 1.55 - 1.9, with the weights in L1 1.3 - 1.6, with no x
// 1.25 - 1.5), before that the weights' way from HBM and the latency of the blocks' serial chains: hence the choice of tiles, and the split of a last round's tiles
// over k (plan_tall).  (Tiles of 256 x 256 by eight waves, the weights shared in L1: 2 - 8 % slower.)  Tiles are walked in groups of 8 row
// blocks, each XCD its own run of them, so that its L2 serves a tile of weights to 8 blocks: with columns fastest over the whole chip 4096 x
// 22016 at 4096 rows took 844 us, 627 so (and 551 by the other instruction).
#include <stdio.h>
#include <stdlib.h>
#include <algorithm>
#include <cmath>
#include "common.h"
#include "dense_gemm_body.h"
#include "tall_ring.h"

namespace {

struct DTallArgs {
    const void* x;
    int64_t ldx;
    const uint8_t* prep;
    const void* bias;
    void* out;
    int64_t ldo;
    int M, K, N, NT;
    int gelu;                    // act 0: as DenseArgs::gelu (0, 1, 2)
    float glu_alpha, glu_limit;  // act 2: as DenseArgs
    int tile0, col_blocks;  // this launch: tiles tile0 + 0 .. gridDim.x - 1 in the order of tile_at
    int per, S;             // k64-steps per split, splits (blockIdx.y)
    int part;               // instead of the finished output, fp32 sums in `scratch`: 1 tiles [blockIdx.x][split][BM][BN], 2 slabs [row block of
                            // 32][split][32][32 NT]
    int vec;                // rows of `out` take 16-byte stores
    int out_f32;            // act 0: `out` takes the fp32 sums (+ bias)
    float* scratch;
};

constexpr int X_RING = tall::RING;  // buffers of x

template <typename T> __device__ __forceinline__ float act2_of(const DTallArgs& a, float gate, float up) {
    if (a.glu_limit > 0.f) {
        const float g = fminf(gate, a.glu_limit), u = fminf(fmaxf(up, -a.glu_limit), a.glu_limit);
        return g / (1.f + __expf(-a.glu_alpha * g)) * (u + 1.f);
    }
    const float sl = gate / (1.f + __expf(-gate));
    return to_f32(from_f32<T>(sl)) * up;
}

// (groups of 4 against 8 row blocks: 4096 x 22016 at 4096 rows 634 / 627 us, 6144 x 6400 at 300 45 / 43)
using tall::tile_at;
using tall::xcd_run;

template <typename T, int BMR, int ACT, int TW> __device__ __forceinline__ void dense_tall_tile(const DTallArgs& a, int tile, int split) {
    using V8 = typename VecT<T>::x8;
    constexpr int BM = 32 * BMR;
    constexpr int WR = TW == 2 ? 2 : 4;  // k64-steps of weights in flight per wave
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];  // [X_RING][BM][128 bytes]
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    int row_block, col_block;
    tile_at(tile, (a.M + BM - 1) / BM, a.col_blocks, row_block, col_block);
    const int m0 = row_block * BM;
    const int mrows = min(BM, a.M - m0);
    const int nt_raw0 = (col_block * 4 + w) * TW;
    const int ksteps = a.K >> 6;                                         // K % 64 == 0 (host)
    const int ks0 = split * a.per, n = min(ksteps, ks0 + a.per) - ks0;   // n >= 1 (host)

    const uint8_t* wtile[TW];
#pragma unroll
    for (int t = 0; t < TW; ++t) wtile[t] = a.prep + (int64_t)min(nt_raw0 + t, a.NT - 1) * ksteps * 4096;
    // lane (c, q) of B fragment 2 m + h of a tile holds column 16 h + c and eight k of slice m: piece `chunk(m)` of the step's eight, which lies in the image's
    // fragment chunk % 4, half chunk / 4 (four runs of 256 bytes a load, the lines of a whole KiB)
    const int c = lane & 15, q = lane >> 4;
    auto chunk = [&](int m) { return (q >> 1) * 4 + m * 2 + (q & 1); };
    const uint32_t woff = (q & 1) * 1024 + (q >> 1) * 512 + c * 16;
    auto w_at = [&](int t, int ks, int f) -> V8 {
        const int at = min(ks, ksteps - 1) * 4096, in = (f >> 1) * 2048 + (f & 1) * 256;
        if constexpr (BMR == 4 && TW == 2) {  // (no registers to spare for addresses; the smaller tiles are a little faster without: gptq_tall.hip)
            return __builtin_bit_cast(V8, tall::buffer_piece<0>(wtile[t], ksteps * 4096, woff + in, at));
        } else {
            const uint8_t* p = wtile[t] + at + in;
            PIN_SGPR(p);
            return *(const GLOBAL_AS V8*)(p + woff);
        }
    };
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
    uint32_t rowoff[BMR];
#pragma unroll
    for (int j = 0; j < BMR; ++j)
        rowoff[j] = (uint32_t)(min(8 * (4 * j + w) + (lane >> 3), mrows - 1) * (int)a.ldx * 2 + ((lane & 7) ^ (4 * (w & 1) + (lane >> 4))) * 16);
    const char* xbase = reinterpret_cast<const char*>(a.x) + (int64_t)m0 * a.ldx * 2;
    auto x_load = [&](int step, int buf) {
        const char* xb = xbase + (int64_t)min(ks0 + step, ksteps - 1) * 128;
        PIN_SGPR(xb);
#pragma unroll
        for (int j = 0; j < BMR; ++j)
            kib_to_lds(xb, rowoff[j], __builtin_amdgcn_readfirstlane(lds0 + buf * (BM * 128) + (4 * j + w) * 1024));
    };
    f32x4 acc[TW][2][2 * BMR];  // [tile][its left, right columns][rows 16 i .. + 15]
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int rf = 0; rf < 2 * BMR; ++rf) acc[t][h][rf] = f32x4{0, 0, 0, 0};
    uint32_t apos[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) apos[m] = (uint32_t)(c * 128 + (chunk(m) ^ (c >> 1)) * 16);

    x_load(0, 0);
    x_load(1, 1);
    x_load(2, 2);
    V8 wq[WR][TW][4];
#pragma unroll
    for (int s = 0; s < WR; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int t = 0; t < TW; ++t) wq[s][t][i] = w_at(t, ks0 + s, i);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(WR * TW * 4) : "memory");
    __syncthreads();
    V8 av[2][BMR];
    auto read_a = [&](V8 (&dst)[BMR], int buf, int i) {
#pragma unroll
        for (int rb = 0; rb < BMR; ++rb) dst[rb] = ld16<V8>(smem + buf * (BM * 128) + ((i & 1) * BMR + rb) * 2048 + apos[i >> 1]);
    };
    read_a(av[0], 0, 0);
    auto step = [&](int s, auto slot_, auto tail_) {
        constexpr int SL = decltype(slot_)::value;
        constexpr bool TAIL = decltype(tail_)::value;  // (at most RING - 1 steps, the first at slot 0)
        constexpr int NX = (SL + 1) % X_RING, WS = SL % WR;
        constexpr bool REFILL = !TAIL || SL + WR < X_RING - 1;
        if constexpr (!TAIL) x_load(s + 3, (SL + 3) % X_RING);  // everyone is done with that buffer since the barrier of the step before
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            read_a(av[(i + 1) & 1], i < 3 ? SL : NX, (i + 1) & 3);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int rb = 0; rb < BMR; ++rb)
#pragma unroll
                for (int f = 0; f < 2 * TW; ++f) {
                    f32x4& sum = acc[f >> 1][f & 1][(i & 1) * BMR + rb];
                    sum = mfma16(av[i & 1][rb], wq[WS][f >> 1][(i & 2) + (f & 1)], sum);
                }
            if constexpr (REFILL) {
                if (i & 1) {
#pragma unroll
                    for (int f = 0; f < 2 * TW; ++f) wq[WS][f >> 1][(i & 2) + (f & 1)] = w_at(f >> 1, ks0 + s + WR, (i & 2) + (f & 1));
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // the x loads of step s + 2 were issued a step ago: behind them are that step's weights and, in whole turns, everything of this step
        tall::meet<TAIL ? 0 : BMR + 8 * TW>();
    };
    tall::ring_steps(n, step);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no direct load may still be on its way to LDS when the block ends

    auto row_of = [&](int rf, int r) { return rf * 16 + 4 * q + r; };
    constexpr int BN = 128 * TW;
    if (a.part == 1) {
        float* dst = a.scratch + ((int64_t)(tile - a.tile0) * a.S + split) * (BM * BN) + w * (32 * TW) + c;
#pragma unroll
        for (int f = 0; f < 2 * TW; ++f)
#pragma unroll
            for (int rf = 0; rf < 2 * BMR; ++rf)
#pragma unroll
                for (int r = 0; r < 4; ++r) dst[(int64_t)row_of(rf, r) * BN + f * 16] = acc[f >> 1][f & 1][rf][r];
        return;
    }
    if (ACT == 0 && a.part == 2) {
        const int ld = a.NT * 32, blocks = (a.M + 31) >> 5;
#pragma unroll
        for (int f = 0; f < 2 * TW; ++f) {
            if (nt_raw0 + (f >> 1) >= a.NT) continue;
#pragma unroll
            for (int rf = 0; rf < 2 * BMR; ++rf) {
                const int block = row_block * BMR + (rf >> 1);
                if (block >= blocks) continue;
                float* dst = a.scratch + ((int64_t)block * a.S + split) * 32 * ld + nt_raw0 * 32 + f * 16 + c;
#pragma unroll
                for (int r = 0; r < 4; ++r) dst[(int64_t)row_of(rf & 1, r) * ld] = acc[f >> 1][f & 1][rf][r];
            }
        }
        return;
    }
    if (ACT == 0 && a.out_f32) {
#pragma unroll
        for (int f = 0; f < 2 * TW; ++f) {
            const int n = nt_raw0 * 32 + f * 16 + c;
            if (n >= a.N) continue;
            const float bv = a.bias ? to_f32(reinterpret_cast<const T*>(a.bias)[n]) : 0.f;
            float* dst = reinterpret_cast<float*>(a.out) + n;
#pragma unroll
            for (int rf = 0; rf < 2 * BMR; ++rf)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = m0 + row_of(rf, r);
                    if (m < a.M) dst[(int64_t)m * a.ldo] = acc[f >> 1][f & 1][rf][r] + bv;
                }
        }
        return;
    }
    constexpr int BO = ACT == 2 ? BN / 2 : BN, OS = BO + 8;
    const int n_out = ACT == 2 ? a.N >> 1 : a.N, n0 = col_block * BO;
    __syncthreads();
    T* tile_out = reinterpret_cast<T*>(smem);  // [BM][OS]
    const T* bias = reinterpret_cast<const T*>(a.bias);
    if (ACT == 2) {  // a tile's left columns are those of the gate, the right ones the same of up
#pragma unroll
        for (int t = 0; t < TW; ++t) {
            const int j = min(nt_raw0 + t, a.NT - 1) * 16 + c;
            const float bg = bias ? to_f32(bias[j]) : 0.f, bu = bias ? to_f32(bias[(a.N >> 1) + j]) : 0.f;
#pragma unroll
            for (int rf = 0; rf < 2 * BMR; ++rf)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float gate = to_f32(from_f32<T>(acc[t][0][rf][r] + bg)), up = to_f32(from_f32<T>(acc[t][1][rf][r] + bu));
                    tile_out[row_of(rf, r) * OS + (w * TW + t) * 16 + c] = from_f32<T>(act2_of<T>(a, gate, up));
                }
        }
    } else {
#pragma unroll
        for (int f = 0; f < 2 * TW; ++f) {
            const int n = nt_raw0 * 32 + f * 16 + c;
            const float bv = bias && n < a.N ? to_f32(bias[n]) : 0.f;
#pragma unroll
            for (int rf = 0; rf < 2 * BMR; ++rf)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    tile_out[row_of(rf, r) * OS + w * (32 * TW) + f * 16 + c] = dense::finish_out<T>(acc[f >> 1][f & 1][rf][r] + bv, a.gelu);
        }
    }
    __syncthreads();
    constexpr int PIECES = BO / 8;
    for (int p = tid; p < mrows * PIECES; p += 256) {
        const int m = p / PIECES, col = (p % PIECES) * 8;
        if (n0 + col >= n_out) continue;
        const V8 v = *reinterpret_cast<const V8*>(tile_out + m * OS + col);
        T* o = reinterpret_cast<T*>(a.out) + (int64_t)(m0 + m) * a.ldo + n0 + col;
        if (a.vec && n0 + col + 8 <= n_out) {
            st16(o, v);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (n0 + col + e < n_out) o[e] = v[e];
        }
    }
}

template <typename T, int BMR, int ACT, int TW>
__global__ __launch_bounds__(256, 2) void dense_tall_kernel(DTallArgs a) {
    dense_tall_tile<T, BMR, ACT, TW>(a, a.tile0 + xcd_run(blockIdx.x, gridDim.x), blockIdx.y);
}

// Several products in one launch, each of its own operand, on neighbouring tiles of one image: the tiles of the first, then those of the second, ...
// NARROW: a last product of up to 128 columns goes first, in tiles of 64 x 128: where rows times width make several rounds, a column of whole tiles for it tends to be a
// round of its own; where they are few it takes the slots of larger tiles.  Four of a width and one of 64, bf16, us, whole tiles behind the others / this: 2048 at 2100, 2500,
// 3000, 4096 rows 72 / 79, 89 / 95, 111 / 103, 138 / 133; 1024 (of 2048 k) at 2500, 4096, 6000, 8190 48 / 49, 71 / 73, 112 / 104, 140 / 130; 1536 at 3000, 4096 74 / 68, 91 / 86; 512 at 2500, 4096, 8190,
// 16000 15.5 / 16.4, 18.3 / 24.2, 49 / 35, 76 / 64; 256 at 5000, 16000 11.4 / 15.6, 44 / 32; 65 - 700 rows of any 5 - 70 % slower.  (It follows the rounds no closer than that: over 125 products the
// line leaves 1.2 % to the better of the two, at most 20.)
struct TallGroups {
    int n, tiles, narrow;        // products; 32-column tiles of the image to each but the last, which has the rest; blocks of a narrow last product
    int64_t x_group, out_group;  // elements between their operands, their outputs
};
template <typename T, int BMR, int TW, bool NARROW>
__global__ __launch_bounds__(256, 2) void dense_tall_groups_kernel(DTallArgs a, TallGroups g) {
    const bool narrow = NARROW && (int)blockIdx.x < g.narrow;
    const int each = (a.M + 32 * BMR - 1) / (32 * BMR) * a.col_blocks;
    const int tile = narrow ? blockIdx.x : xcd_run(blockIdx.x - g.narrow, gridDim.x - g.narrow);
    const int i = narrow ? g.n - 1 : min(tile / each, g.n - 1), first = i * g.tiles;
    a.x = reinterpret_cast<const T*>(a.x) + i * g.x_group;
    a.out = reinterpret_cast<T*>(a.out) + i * g.out_group;
    a.prep += (int64_t)first * (a.K >> 6) * 4096;
    a.N = i + 1 < g.n ? g.tiles * 32 : a.N - first * 32;
    a.NT = (a.N + 31) >> 5;
    if (NARROW && narrow) {
        a.col_blocks = 1;
        dense_tall_tile<T, 2, 0, 1>(a, tile, 0);
    } else {
        a.col_blocks = (a.NT + 4 * TW - 1) / (4 * TW);
        dense_tall_tile<T, BMR, 0, TW>(a, tile - i * each, 0);
    }
}

template <typename T, int BM, int BN, int ACT>
__global__ __launch_bounds__(256) void dense_tall_finish_kernel(DTallArgs a) {
    constexpr int PER_ROW = ACT == 2 ? BN / 8 : BN / 4;
    const int idx = blockIdx.x * 256 + threadIdx.x;
    const int m = idx / PER_ROW, g = idx % PER_ROW;
    int row_block, col_block;
    tile_at(a.tile0 + blockIdx.y, (a.M + BM - 1) / BM, a.col_blocks, row_block, col_block);
    const int row = row_block * BM + m;
    if (m >= BM || row >= a.M) return;
    const float* src = a.scratch + (int64_t)blockIdx.y * a.S * (BM * BN) + m * BN;
    auto part_sum = [&](int col) {
        f32x4 v = {0, 0, 0, 0};
        for (int s = 0; s < a.S; ++s) v += *reinterpret_cast<const f32x4*>(src + (int64_t)s * (BM * BN) + col);
        return v;
    };
    const T* bias = reinterpret_cast<const T*>(a.bias);
    T* out = reinterpret_cast<T*>(a.out) + (int64_t)row * a.ldo;
    if (ACT == 2) {
        const int t = g >> 2, c = (g & 3) * 4, j = (col_block * (BN / 32) + t) * 16 + c, half = a.N >> 1;
        if (j >= half) return;
        const f32x4 gate = part_sum(t * 32 + c), up = part_sum(t * 32 + 16 + c);
#pragma unroll
        for (int e = 0; e < 4; ++e)
            out[j + e] = from_f32<T>(act2_of<T>(a, to_f32(from_f32<T>(gate[e] + (bias ? to_f32(bias[j + e]) : 0.f))),
                                                to_f32(from_f32<T>(up[e] + (bias ? to_f32(bias[half + j + e]) : 0.f)))));
    } else {
        const int n = col_block * BN + g * 4;
        const f32x4 v = part_sum(g * 4);
        if (a.out_f32) {
            float* sums = reinterpret_cast<float*>(a.out) + (int64_t)row * a.ldo;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n + e < a.N) sums[n + e] = v[e] + (bias ? to_f32(bias[n + e]) : 0.f);
            return;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (n + e < a.N) out[n + e] = dense::finish_out<T>(v[e] + (bias ? to_f32(bias[n + e]) : 0.f), a.gelu);
    }
}

constexpr int CUS = 256;

struct TallPlan {
    int BMR, TW;            // 32-row blocks and 32-column tiles per wave: a tile of 32 BMR x 128 TW
    int col_blocks, tiles;
    int whole;              // tiles of the unsplit launch; the rest is split S ways, `per` k64-steps each
    int S, per;
    double us;
};
// us per k64-step of a block that has its CU to itself, and of a CU's share of a full chip.  These and the constants of walk_us, launch_us and the two
// plan makers are fitted to 280 products of 65 to 8000 rows and 1024 x 1024 to 57344 x 8192, each with up to 48 plans, weights cold (the copies of
// a matrix that take turns are more than the caches hold): the estimates are 5 % off, the plans that they pick 0.9 % behind the best, at most 9.  (Of the 32x32x16 form; with 16x16x32
// they are 13 % off, mostly above, and the plans still 1.0 % behind the best of 57 products, at most 13.)
struct TallCost {
    double alone, busy;
};
constexpr TallCost TALL_COST[3][2] = {{{0.262, 0.356}, {0.609, 0.599}}, {{0.347, 0.411}, {0.659, 0.705}}, {{0.420, 0.508}, {0.692, 0.853}}};
// Blocks that walk `per` steps each: a last round that is not full costs more than three quarters of a whole one
double walk_us(int64_t blocks, int64_t per, const TallCost& c) {
    const int64_t rounds = blocks / CUS, rest = blocks % CUS;
    const double alone = per * c.alone, busy = per * c.busy, share = (double)rest / CUS;
    if (rounds == 0) return alone + std::max(0.0, busy - alone) * share;
    return std::max(alone, rounds * busy + (rest ? busy * (0.77 + 0.23 * share) : 0.0));
}
// ... with the weights' way from HBM, which hides behind the walk as far as one of the two is short
double launch_us(double walk, int64_t K, int64_t N) { return 5.55 + std::hypot(walk, 2.0 * K * N / 6.33e6); }
constexpr int MAX_PARTS = 384;  // blocks of the split launch: 48 MiB of fp32 tiles

// Rows x columns of a tile, and whether the tiles past the last whole round of 256 are split over k: 256 rows of 24576 x 6144 are 48 tiles of 128 x
// 256 that walk 384 steps each (264 us; 95 split in four), 765 rows of 2048 x 11264 352 tiles of 96 x 128 (44 us; 52 in tiles of 128 x 128).
// GELU: in the unsplit launch each thread evaluates it 16 BMR TW times, one behind the other, GELU_NS each (erf 180, a call; tanh 40): the finish launch has a thread
// for every four (1024 x 1024 at 65 - 256 rows, tiles of 64 x 128, 128 x 256: erf +6.4, +25 us, tanh +1.3, +5; behind a split +0.9).
template <int GELU_NS>
TallPlan make_plan_tall(int64_t M, int64_t K, int64_t N) {
    const int64_t steps = K / 64, NT = cdiv64(N, 32);
    TallPlan best{};
    double best_us = 1e30;
    for (int BMR = 2; BMR <= 4; ++BMR)
        for (int TW = 1; TW <= 2; ++TW) {
            const TallCost c = TALL_COST[BMR - 2][TW - 1];
            const int64_t cb = cdiv64(NT, 4 * TW), tiles = cb * cdiv64(M, 32 * BMR), rounds = tiles / CUS, rest = tiles % CUS;
            for (int S = 1; S <= 12; ++S) {
                const int64_t per = cdiv64(steps, S);
                if (S > 1 && (rest == 0 || rest * S > MAX_PARTS || per < 4)) break;
                if ((S - 1) * per >= steps) continue;
                double us;
                if (S > 1) {  // the finish launch and the partial tiles; behind whole rounds, a launch of its own
                    us = launch_us(rounds * steps * c.busy + walk_us(rest * S, per, c), K, N) + 1.0 + 0.27 * (S - 1) + (rounds ? 6.7 : 0.0) +
                         2.0 * rest * S * (32 * BMR) * (128 * TW) * 4 / 8.9e6;
                } else {
                    us = launch_us(walk_us(tiles, steps, c), K, N);
                }
                if (GELU_NS && (S == 1 || rounds)) us += GELU_NS * 1e-3 * 16 * BMR * TW;
                if (us < best_us) {
                    best_us = us;
                    best = {BMR, TW, (int)cb, (int)tiles, (int)(S > 1 ? tiles - rest : tiles), S, (int)per, us};
                }
            }
        }
    return best;
}

// ... where the consumer adds the parts: every tile in the same number of them, and no launch behind: completions of two prompts of 54 tokens, 8 hybrid layers
// of 2048, 2360 -> 2250 us (2145 with the plans kept, below).  Past a whole round of 256 blocks the rest costs what it costs in make_plan_tall: priced
// by its share alone, 257 - 320 blocks looked best and were the slower way.  us with the norm behind, the passes of 64 rows / by the share / now: 6144 x
// 6144 at 100, 128 rows 33.8 / 35.9 / 26.0, 34.6 / 38.2 / 30.2; 24576 x 6144 at 65, 160 119 / 90 / 69, 203 / 126 / 87; 11008 x 4096 at 256 55 / 60 / 41; 28672 x
// 8192 at 128 120 / 134 / 108; 13824 x 5120 at 193 119 / 65 / 50; 8192 x 10240 in front of a q / k norm at 192 66 / 74 / 58.
TallPlan make_plan_parts(int64_t M, int64_t K, int64_t N) {
    const int64_t steps = K / 64, NT = cdiv64(N, 32);
    TallPlan best{};
    double best_us = 1e30;
    for (int BMR = 2; BMR <= 4; ++BMR)
        for (int TW = 1; TW <= 2; ++TW) {
            const TallCost c = TALL_COST[BMR - 2][TW - 1];
            const int64_t cb = cdiv64(NT, 4 * TW), tiles = cb * cdiv64(M, 32 * BMR);
            for (int S = 1; S <= 8; ++S) {
                const int64_t per = cdiv64(steps, S);
                if (S > 1 && per < 4) break;
                if ((S - 1) * per >= steps) continue;
                const double us = launch_us(walk_us(tiles * S, per, c), K, N) + 0.06 * (S - 1) + 2.0 * S * M * N * 4 / 4.8e6;
                if (us < best_us) {
                    best_us = us;
                    best = {BMR, TW, (int)cb, (int)tiles, 0, S, (int)per, us};
                }
            }
        }
    return best;
}

// TGIS_DTALL_PLAN=BMR,TW,S: this plan for every product that it fits
bool plan_from_env(int64_t M, int64_t K, int64_t N, bool parts, TallPlan& p) {
    const char* e = getenv("TGIS_DTALL_PLAN");
    int b = 0, t = 0, S = 0;
    if (!e || sscanf(e, "%d,%d,%d", &b, &t, &S) != 3 || b < 2 || b > 4 || t < 1 || t > 2 || S < 1 || S > 16) return false;
    const int64_t steps = K / 64, cb = cdiv64(cdiv64(N, 32), 4 * t), tiles = cb * cdiv64(M, 32 * b), per = cdiv64(steps, S);
    if ((S - 1) * per >= steps || (!parts && S > 1 && tiles % CUS * S > MAX_PARTS)) return false;
    p = {b, t, (int)cb, (int)tiles, (int)(parts ? 0 : S > 1 ? tiles - tiles % CUS : tiles), S, (int)per, 0.0};
    return true;
}

// A plan takes 1 - 2 us to make, a short prompt's launch 4 to prepare: each thread keeps those of the sizes that it asked for last.
template <TallPlan (*MAKE)(int64_t, int64_t, int64_t)>
TallPlan kept_plan(int64_t M, int64_t K, int64_t N) {
    struct Entry {
        int64_t M, K, N;
        TallPlan plan;
    };
    thread_local Entry kept[64] = {};
    Entry& e = kept[(M * 5 + K / 64 * 3 + N / 32) % 64];
    if (e.M != M || e.K != K || e.N != N) e = {M, K, N, MAKE(M, K, N)};
    return e.plan;
}

TallPlan plan_tall(int64_t M, int64_t K, int64_t N, int act) {
    TallPlan p;
    if (plan_from_env(M, K, N, false, p)) return p;
    return act == 4 ? kept_plan<make_plan_tall<180>>(M, K, N) : act == 5 ? kept_plan<make_plan_tall<40>>(M, K, N) : kept_plan<make_plan_tall<0>>(M, K, N);
}

TallPlan plan_parts(int64_t M, int64_t K, int64_t N) {
    TallPlan p;
    return plan_from_env(M, K, N, true, p) ? p : kept_plan<make_plan_parts>(M, K, N);
}

int64_t plan_scratch(const TallPlan& p) {
    return p.whole < p.tiles ? (int64_t)(p.tiles - p.whole) * p.S * (32 * p.BMR) * (128 * p.TW) * 4 : 0;
}

template <typename T, int BMR, int ACT, int TW>
int launch_blocks(const DTallArgs& a, int tiles, int S, hipStream_t st) {
    constexpr size_t ring = (size_t)X_RING * (32 * BMR) * 128, rows = (size_t)(32 * BMR) * ((ACT == 2 ? 64 : 128) * TW + 8) * 2;
    constexpr size_t lds = ring > rows ? ring : rows;
    static const hipError_t attr = hipFuncSetAttribute((const void*)dense_tall_kernel<T, BMR, ACT, TW>,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    TGIS_CHECK_HIP(attr);
    hipLaunchKernelGGL((dense_tall_kernel<T, BMR, ACT, TW>), dim3((unsigned)tiles, (unsigned)S), dim3(256), lds, st, a);
    TGIS_CHECK_LAUNCH();
    return TGIS_OK;
}

template <typename T, int ACT>
int launch_shape(const TallPlan& p, const DTallArgs& a, int tiles, int S, hipStream_t st) {
    switch (p.BMR * 10 + p.TW) {
        case 21: return launch_blocks<T, 2, ACT, 1>(a, tiles, S, st);
        case 22: return launch_blocks<T, 2, ACT, 2>(a, tiles, S, st);
        case 31: return launch_blocks<T, 3, ACT, 1>(a, tiles, S, st);
        case 32: return launch_blocks<T, 3, ACT, 2>(a, tiles, S, st);
        case 41: return launch_blocks<T, 4, ACT, 1>(a, tiles, S, st);
        default: return launch_blocks<T, 4, ACT, 2>(a, tiles, S, st);
    }
}

template <typename T, int ACT>
int launch_finish(const TallPlan& p, const DTallArgs& a, int tiles, hipStream_t st) {
#define TGIS_TALL_FINISH(B, W)                                                                                                         \
    hipLaunchKernelGGL((dense_tall_finish_kernel<T, 32 * B, 128 * W, ACT>),                                                            \
                       dim3((unsigned)cdiv64((int64_t)32 * B * (128 * W) / (ACT == 2 ? 8 : 4), 256), (unsigned)tiles), dim3(256), 0, st, a)
    switch (p.BMR * 10 + p.TW) {
        case 21: TGIS_TALL_FINISH(2, 1); break;
        case 22: TGIS_TALL_FINISH(2, 2); break;
        case 31: TGIS_TALL_FINISH(3, 1); break;
        case 32: TGIS_TALL_FINISH(3, 2); break;
        case 41: TGIS_TALL_FINISH(4, 1); break;
        default: TGIS_TALL_FINISH(4, 2); break;
    }
#undef TGIS_TALL_FINISH
    TGIS_CHECK_LAUNCH();
    return TGIS_OK;
}

template <typename T>
int run_tall(const TallPlan& p, DTallArgs& a, int act, hipStream_t st) {
    a.per = a.K / 64;
    a.S = 1;
    if (p.whole > 0) {
        const int rc = act == 2 ? launch_shape<T, 2>(p, a, p.whole, 1, st) : launch_shape<T, 0>(p, a, p.whole, 1, st);
        if (rc != TGIS_OK) return rc;
    }
    if (p.whole < p.tiles) {
        a.tile0 = p.whole;
        a.per = p.per;
        a.S = p.S;
        a.part = 1;
        const int rc = launch_shape<T, 0>(p, a, p.tiles - p.whole, p.S, st);
        if (rc != TGIS_OK) return rc;
        return act == 2 ? launch_finish<T, 2>(p, a, p.tiles - p.whole, st) : launch_finish<T, 0>(p, a, p.tiles - p.whole, st);
    }
    return TGIS_OK;
}
}  // namespace

// Is this kernel the faster way?  us, the alternative / this kernel, weights cold, launches back to back; of 480 products on either side of 256 rows the
// choice is 0.5 and 2.6 % behind the better of the two, with GELU 0.4 and 0.6, as parts 0.3, with SiLU 0.3 and 0.9.
// Up to 256 rows the alternative is the weight-streaming kernel, which goes over the weights once per 64 rows (a product below 65 rows stays there):
//   65 / 128 / 192 / 256 rows: 4096 x 4096 17.1 / 14.9, 17.8 / 16.1, 24.6 / 18.3, 25.4 / 21; 5632 x 2048 15.3 / 14.8, 15.4 / 15.0, 20.2 / 16.1, 20.8 / 17.5; 4096 x
//   12288 37.6 / 28.4, 33.2 / 31.1, 60.5 / 38, 64.5 / 42; 6144 x 24576 106 / 68, 113 / 78, 166 / 95, 198 / 100; 24576 x 6144 120 / 68, 115 / 73, 218 / 87, 216 /
//   95; with SiLU 1024 x 5632 9.5 / 8.9, 9.8 / 10, 17 / 10, 17 / 10; 2048 x 11264 21 / 17, 21 / 19, 34 / 23, 40 / 25
// It stays where its passes are one round of two-tile blocks of up to 1024 k that split k: 2048 x 2048 10.1 / 10.2, 10.9 / 11.3, 12.0 / 12.6, 12.5 / 13.9; 1536
// x 1536 8.9 / 9.4, 9.3 / 10.0, 10.1 / 10.8, 11.7 / 10.8; 2048 x 1024 8.9 / 9.6, 9.3 / 10.2, 9.8 / 10.6, 10.5 / 10.9; as parts in front of a norm from 128 such
// blocks of up to 2560 k on (2048 x 2048 9.7 / 9.8, 10.7 / 11.2, 11.9 / 12.3, 12.5 / 13.1; but 1024 x 1024 7.9 / 7.5, 8.0 / 7.8 and 4096 x 1024 10.9 / 9.9,
// 11.1 / 11.2).  GELU of fewer than eight steps, which have no split: 320 x 1280 10.1 / 11.2.
// Above, it is the library, with a launch of its own for the activation.
//   act 0 / GELU: it wins where its tiles of 128 x 256 fill more than half the chip (4096 x 6144 at 800, 1024 rows 47 / 56, 52 / 61; 3072 x 5120 at 900, 1400 40 / 44,
//   49 / 50; 28672 x 8192 at 600 259 / 346; layers of 3072, 8192 at 1390 rows 394 / 371 us with it, of 4096, 14336 at 900 494 / 467), but not on narrow products of
//   long k (11008 x 4096 at 1024, 1400 rows 102 / 85, 133 / 124; 13824 x 5120 at 1200 1.7), nor past k of 16384 (below).  Between k of 9600 and 16384 more rows give as much as they take
//   (1700 rows: 11008 x 4096 152 / 135, 10240 x 2560 104 / 114, 14336 x 7168 246 / 298).  Below that the two are close (300, 512, 1024 rows: 2048 x
//   2560 13.3 / 14.8, 15.3 / 16.6, 22.9 / 19.7; 4096 x 4096 26.2 / 25.6, 30 / 31, 41.9 / 42.7; 5632 x 2048 26 / 22.5, 26.7 / 23.6, 40 / 35; 6144 x 6400 44.7 / 43.5,
//   67 / 60, 91 / 88), and inside a model this kernel is the faster one also where it is not alone: 22 layers of 2048, 5632 at 257, 400 rows 2781 / 2466,
//   2810 / 2669 us, both launched one by one
//   act 2: up to 32 Mi weights always (300, 1024, 4096, 8192 rows: 1024 x 5632 0.60, 0.77, 0.91, 0.82 of the library and the activation; 2048 x 11264 0.86, 0.93,
//   0.94, 0.83); larger ones from 513 rows on, but for widths of whole 4096s, on which the library is at its best (600, 1400, 2048, 8192 rows: 4096 x 22016
//   0.90, 0.79, 0.82, 0.99; 5120 x 27648 0.98, 0.92, 0.94, 0.98; 3072 x 16384 1.14, 0.97, 1.06, 1.07; 4096 x 28672 0.95, 0.99, 1.03, 1.11; 8192 x 57344 0.97,
//   1.08, 1.16, 1.16)
// Narrow and shallow ones stay where they were: 2048 x 512 at 128 / 300 rows 8.6 / 9.2, 8.2 / 9.0; 64 x 2048 at 600, 1400 rows 4.4 / 5.1, 5.2 / 6.8.
static bool passes_in_a_round(int64_t M, int64_t K, int64_t N, int64_t from_blocks) {
    const dense::DensePlan pass = dense::plan_dense(K, N, M);
    const int64_t blocks = cdiv64(cdiv64(N, 32), pass.TN) * cdiv64(M, 64) * pass.S;
    return pass.TN == 2 && pass.S > 1 && pass.KR <= 1024 && blocks >= from_blocks && blocks <= CUS;
}
// Past k of 16384, up to 2048 rows and 7168 columns.  The library's time goes in steps of up to twice, by a choice of kernels that follows no rule of sizes; drawn here
// is where it was the longer one, of 1938 products (k 16448 - 36864, 1024 - 7168 columns, 900 - 2048 rows; this kernel takes 0.70 of its time) but for one in 140.  us, library / this:
//   up to 4096 columns  24576 x 4096 at 1408, 1700, 2048 rows 420 / 274, 428 / 315, 490 / 350; 18432 x 3584 219 / 204 - 336 / 239; 16448 x 1024 169 / 64 (18496 x 3456 at 1760 208 / 246); past k of
//                       24576 up to 2048 (28672 x 2048 at 2048 325 / 205, but x 4096 at 1408 298 / 323, x 3072 at 2048 293 / 397, 34944 x 2304 at 1969 308 / 374)
//   up to 6144 columns  as far as 8.9 M outputs: 24576 x 5120 at 1280, 1700 403 / 330, 616 / 378; x 6144 at 1152, 1393 373 / 355, 628 / 375; but at 1464, 1536 385 / 400, 388 / 416, x 5120 at 1792 382 /
//                       394, x 5723 at 1676 395 / 434.  From 1601 rows of 24 columns of 256 tiles on again: 24576 x 6144 at 1650, 1700 669 / 444, 675 / 459 (23424 x 6144 at 1599 367 / 398)
//   up to 7168          as far as 7.4 M: 28672 x 7168 at 900, 1024 485 / 391, 503 / 393, but at 1152, 1344, 1408 413 / 438, 463 / 505, 466 / 525 (at 1280 738 / 465); x 8128 at 850 369 / 438
// 8 layers of 6144, 24576 at 1300, 1700 rows 9.39 -> 7.65, 10.90 -> 9.23 ms.
static bool pays_past_16k(int64_t M, int64_t K, int64_t N) {
    if (K <= 16384 || M > 2048) return false;
    if (N <= (K <= 24576 ? 4096 : 2048)) return true;
    if (N > 7168 || M > 1792 || (K > 24576 && N <= 4096)) return false;
    return M * N <= (N <= 6144 ? 8900000 : 7400000) || (M > 1600 && N > 23 * 256 && N <= 6144 && M * N <= 10500000);
}
static bool dense_tall_pays(int64_t M, int64_t K, int64_t N, int act, bool parts) {
    if (M < TGIS_DENSE_TALL_MIN_M || K < 64 || K % 64 != 0 || N < 1024) return false;
    TallPlan forced;
    if (plan_from_env(M, K, N, parts, forced)) return true;
    const bool gelu = act == 4 || act == 5;
    if (parts) return M <= 256 && !(K <= 2560 && passes_in_a_round(M, K, N, 128));
    if (M <= 256) return act == 2 || (!passes_in_a_round(M, K, N, 0) && !(gelu && K < 512));
    if (act == 2) return M <= 8192 && (K * N <= (32 << 20) || (M > 512 && N % 4096 != 0));
    if (pays_past_16k(M, K, N)) return true;
    if (M > 1400 || K < 512 || M * N > std::min<int64_t>(1500 * K, 6300000)) return false;
    return cdiv64(M, 128) * cdiv64(N, 256) <= CUS / 2 || (K > 9600 && N < 8192);
}

// Bytes of scratch of tgis_dense_tall where it is the faster way to this product, -1 where it is not.
extern "C" int64_t tgis_dense_tall_bytes(int64_t M, int64_t K, int64_t N, int act) {
    if (!(act == 0 || act == 2 || act == 4 || act == 5) || !dense_tall_pays(M, K, N, act, false)) return -1;
    return plan_scratch(plan_tall(M, K, N, act));
}

static bool rows_ok(const void* x, int64_t ldx, int64_t K) {  // (a tile's rows are addressed with 31 bits)
    return ldx >= K && ldx % 8 == 0 && (uintptr_t)x % 16 == 0 && ldx < (1ll << 22);
}

static DTallArgs tall_args(const void* x, int64_t ldx, const void* prepared, int64_t M, int64_t K, int64_t N, void* scratch) {
    DTallArgs a{};
    a.x = x;
    a.ldx = ldx;
    a.prep = (const uint8_t*)prepared;
    a.M = (int)M;
    a.K = (int)K;
    a.N = (int)N;
    a.NT = (int)cdiv64(N, 32);
    a.scratch = (float*)scratch;
    return a;
}

// out = act(x @ w^T + bias) in the model dtype, or (act 0) in fp32.  act 0; 4 / 5: GELU (erf / tanh) of the rounded sum; 2: SiLU(gate) * up of a gate | up image
// (out [M, N / 2]), or with glu_limit > 0 the clamped unit (DenseArgs::glu_limit).
extern "C" int tgis_dense_tall(const void* x, int64_t ldx, const void* prepared, const void* bias, void* out, int64_t ldo, int64_t M, int64_t K,
                               int64_t N, int dtype, int out_f32, int act, float glu_alpha, float glu_limit, void* workspace,
                               int64_t workspace_bytes, void* stream) {
    TGIS_CHECK_ARG(x && prepared && out && M >= 0 && K >= 64 && K % 64 == 0 && N >= 1, "tgis_dense_tall: bad arguments");
    TGIS_CHECK_ARG((dtype == TGIS_F16 || dtype == TGIS_BF16) && (act == 0 || act == 2 || act == 4 || act == 5), "tgis_dense_tall: bad dtype or act");
    TGIS_CHECK_ARG(!out_f32 || act == 0, "tgis_dense_tall: activations are written in the model dtype");
    TGIS_CHECK_ARG(act != 2 || N % 32 == 0, "tgis_dense_tall: act 2 needs a gate|up image (N / 2 a multiple of 16)");
    TGIS_CHECK_ARG(rows_ok(x, ldx, K), "tgis_dense_tall: x rows must be 16-byte aligned and less than 2^22 elements apart");
    if (M == 0) return TGIS_OK;
    const TallPlan p = plan_tall(M, K, N, act);
    TGIS_CHECK_ARG(plan_scratch(p) == 0 || (workspace && workspace_bytes >= plan_scratch(p)), "tgis_dense_tall: workspace too small");
    DTallArgs a = tall_args(x, ldx, prepared, M, K, N, workspace);
    a.bias = bias;
    a.out = out;
    a.ldo = ldo;
    a.gelu = act == 4 ? 1 : act == 5 ? 2 : 0;
    a.glu_alpha = glu_alpha;
    a.glu_limit = glu_limit;
    a.out_f32 = out_f32;
    a.vec = ldo % 8 == 0 && (uintptr_t)out % 16 == 0;
    a.col_blocks = p.col_blocks;
    const hipStream_t st = (hipStream_t)stream;
    TgisTimedScope timed(TGIS_OP_DENSE_GEMM, st);
    return dtype == TGIS_F16 ? run_tall<f16>(p, a, act == 2 ? 2 : 0, st) : run_tall<bf16>(p, a, act == 2 ? 2 : 0, st);
}

// Several products in one launch (TallGroups), unsplit: the tile of the least walk.
struct GroupsPlan {
    int BMR, TW, col_blocks, tiles, narrow;
};
static GroupsPlan plan_groups(int64_t M, int64_t K, int64_t N_group, int64_t N, int64_t groups) {
    const int64_t last = N - (groups - 1) * N_group;
    const bool narrow = groups > 1 && last <= 128 && (M > 5000 || M * N_group > 6000000);
    GroupsPlan best{};
    double best_us = 1e30;
    TallPlan forced;
    const bool fixed = plan_from_env(M, K, N, false, forced);
    for (int BMR = 2; BMR <= 4; ++BMR)
        for (int TW = narrow ? 2 : 1; TW <= 2; ++TW) {
            if (fixed && (BMR != forced.BMR || TW != std::max(forced.TW, narrow ? 2 : 1))) continue;
            const int64_t cb = cdiv64(N_group, 128 * TW);
            const int64_t tiles = cdiv64(M, 32 * BMR) * (cb * (groups - 1) + (narrow ? 0 : cdiv64(last, 128 * TW)));
            const double us = launch_us(walk_us(tiles, K / 64, TALL_COST[BMR - 2][TW - 1]), K, N);
            if (us < best_us) {
                best_us = us;
                best = {BMR, TW, (int)cb, (int)tiles, narrow ? (int)cdiv64(M, 64) : 0};
            }
        }
    return best;
}

template <typename T, int BMR, int TW, bool NARROW> static int launch_groups(const GroupsPlan& p, const DTallArgs& a, const TallGroups& g, hipStream_t st) {
    constexpr size_t ring = (size_t)X_RING * (32 * BMR) * 128, rows = (size_t)(32 * BMR) * (128 * TW + 8) * 2;
    constexpr size_t lds = ring > rows ? ring : rows;
    static const hipError_t attr = hipFuncSetAttribute((const void*)dense_tall_groups_kernel<T, BMR, TW, NARROW>,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    TGIS_CHECK_HIP(attr);
    hipLaunchKernelGGL((dense_tall_groups_kernel<T, BMR, TW, NARROW>), dim3((unsigned)(p.narrow + p.tiles)), dim3(256), lds, st, a, g);
    TGIS_CHECK_LAUNCH();
    return TGIS_OK;
}
template <typename T> static int launch_groups_shape(const GroupsPlan& p, const DTallArgs& a, const TallGroups& g, hipStream_t st) {
    switch (p.BMR * 10 + p.TW + (p.narrow ? 100 : 0)) {
        case 21: return launch_groups<T, 2, 1, false>(p, a, g, st);
        case 22: return launch_groups<T, 2, 2, false>(p, a, g, st);
        case 31: return launch_groups<T, 3, 1, false>(p, a, g, st);
        case 32: return launch_groups<T, 3, 2, false>(p, a, g, st);
        case 41: return launch_groups<T, 4, 1, false>(p, a, g, st);
        case 42: return launch_groups<T, 4, 2, false>(p, a, g, st);
        case 122: return launch_groups<T, 2, 2, true>(p, a, g, st);
        case 132: return launch_groups<T, 3, 2, true>(p, a, g, st);
        default: return launch_groups<T, 4, 2, true>(p, a, g, st);
    }
}

// Is one launch the faster way than the products one by one?  Up to where 256 x 256 tiles of one of them fill half the chip, which is where the library's begin to
// be ahead by more than four launches' ends.  Four products and a narrow one, bf16, weights cold, us, one by one / together:
//   2048 x 2048, 64: 65 rows 54 / 17, 300 68 / 23, 1024 77 / 47, 1393 92 / 57, 2045 109 / 77, 3000 128 / 110, 4096 152 / 140 (128 tiles; 6000 194 / 198, 8190 224 / 271)
//   4096 x 4096, 128: 65 72 / 39, 512 132 / 98, 1024 182 / 143, 2045 265 / 261 (128 tiles; 3000 358 / 380, 4096 414 / 508)
//   2560 x 2560, 160: 300 72 / 30, 1393 129 / 82, 3000 184 / 162 (120 tiles; 4096 235 / 214, 6000 267 / 308);  1024 x 1024, 64: 8190 105 / 85 (128 tiles)
// Prompts through 8 layers of 2048 of which every other takes such a launch: 1 x 70 tokens 1144 / 937 us, 2 x 150 1163 / 978, 4 x 333 ragged 1862 / 1714, 4 x 1024 4402 /
// 4370; 24 prompts and eight tokens each 6978 / 6845.
extern "C" int tgis_dense_tall_groups_pays(int64_t M, int64_t K, int64_t N_group, int64_t N, int64_t groups) {
    if (M < TGIS_DENSE_TALL_MIN_M || K < 64 || K % 64 != 0 || N_group <= 0 || N_group % 32 != 0 || groups < 2 || N <= (groups - 1) * N_group || N > groups * N_group)
        return 0;
    return cdiv64(M, 256) * cdiv64(N_group, 256) <= CUS / 2 ? 1 : 0;
}

extern "C" int tgis_dense_tall_groups(const void* x, int64_t ldx, int64_t x_group, const void* prepared, void* out, int64_t ldo, int64_t out_group,
                                      int64_t M, int64_t K, int64_t N_group, int64_t N, int64_t groups, int dtype, void* stream) {
    TGIS_CHECK_ARG(x && prepared && out && M >= 0 && K >= 64 && K % 64 == 0, "tgis_dense_tall_groups: bad arguments");
    TGIS_CHECK_ARG(dtype == TGIS_F16 || dtype == TGIS_BF16, "tgis_dense_tall_groups: bad dtype");
    TGIS_CHECK_ARG(rows_ok(x, ldx, K) && x_group % 8 == 0, "tgis_dense_tall_groups: x rows must be 16-byte aligned and less than 2^22 elements apart");
    TGIS_CHECK_ARG(N_group > 0 && N_group % 32 == 0 && groups >= 1 && N > (groups - 1) * N_group && N <= groups * N_group && ldo >= std::min(N, N_group),
                   "tgis_dense_tall_groups: %ld columns do not make %ld groups of up to %ld", (long)N, (long)groups, (long)N_group);
    TGIS_CHECK_ARG(cdiv64(M, 64) * (cdiv64(N, 128) + groups) <= 2147483647LL, "tgis_dense_tall_groups: too many tiles");
    if (M == 0) return TGIS_OK;
    const GroupsPlan p = plan_groups(M, K, N_group, N, groups);
    DTallArgs a = tall_args(x, ldx, prepared, M, K, N, nullptr);
    a.out = out;
    a.ldo = ldo;
    a.vec = ldo % 8 == 0 && (uintptr_t)out % 16 == 0 && out_group % 8 == 0;
    a.col_blocks = p.col_blocks;
    a.per = (int)(K / 64);
    a.S = 1;
    const TallGroups g{(int)groups, (int)(N_group / 32), p.narrow, x_group, out_group};
    const hipStream_t st = (hipStream_t)stream;
    TgisTimedScope timed(TGIS_OP_DENSE_GEMM, st);
    return dtype == TGIS_F16 ? launch_groups_shape<f16>(p, a, g, st) : launch_groups_shape<bf16>(p, a, g, st);
}

// The product as fp32 partial sums for the consumers of tgis_dense_gemm_partial's, in the same layout; up to 256 rows.
extern "C" int64_t tgis_dense_tall_partial_bytes(int64_t M, int64_t K, int64_t N) {
    if (!dense_tall_pays(M, K, N, 0, true)) return -1;
    return cdiv64(M, 32) * 32 * cdiv64(N, 32) * 32 * 4 * plan_parts(M, K, N).S;
}

extern "C" int tgis_dense_tall_partial(const void* x, int64_t ldx, const void* prepared, int64_t M, int64_t K, int64_t N, int dtype, float* slabs,
                                       int64_t slabs_bytes, int* num_slabs, int64_t* slab_ld, void* stream) {
    TGIS_CHECK_ARG(x && prepared && slabs && M >= 1 && M <= 256 && K >= 64 && K % 64 == 0 && N >= 1, "tgis_dense_tall_partial: bad arguments");
    TGIS_CHECK_ARG(dtype == TGIS_F16 || dtype == TGIS_BF16, "tgis_dense_tall_partial: bad dtype");
    TGIS_CHECK_ARG(rows_ok(x, ldx, K), "tgis_dense_tall_partial: x rows must be 16-byte aligned and less than 2^22 elements apart");
    const TallPlan p = plan_parts(M, K, N);
    TGIS_CHECK_ARG(slabs_bytes >= cdiv64(M, 32) * 32 * cdiv64(N, 32) * 32 * 4 * p.S, "tgis_dense_tall_partial: slab buffer too small");
    if (num_slabs) *num_slabs = p.S;
    if (slab_ld) *slab_ld = cdiv64(N, 32) * 32;
    DTallArgs a = tall_args(x, ldx, prepared, M, K, N, slabs);
    a.col_blocks = p.col_blocks;
    a.per = p.per;
    a.S = p.S;
    a.part = 2;
    const hipStream_t st = (hipStream_t)stream;
    TgisTimedScope timed(TGIS_OP_DENSE_GEMM, st);
    return dtype == TGIS_F16 ? launch_shape<f16, 0>(p, a, p.tiles, p.S, st) : launch_shape<bf16, 0>(p, a, p.tiles, p.S, st);
}
