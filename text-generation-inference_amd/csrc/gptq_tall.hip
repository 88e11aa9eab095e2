// The int4 GEMM at prefill sizes: more rows than the streaming kernels of gptq_gemm_body.h / gptq_wide_body.h take in one pass.
//
// Those re-stream and re-dequantise the weights once per 32 (64) rows; the library path (dequantise the whole matrix to a scratch copy,
// then hipBLASLt) pays for the copy.  In between, one block keeps BM = 32 BMR rows of x in LDS and each of its four waves owns TW
// 32-column tiles: a wave loads 1 KiB of the prepared image per k64-step and tile, dequantises it ONCE into four MFMA B fragments and
// applies them to all BMR row blocks.  No scratch copy of W, no second pass over the weights, SiLU * up in the epilogue.
//
// Rows of x go to LDS by direct loads, 64 k at a time, three steps ahead, into a ring of four buffers: no registers, no stores, and one
// barrier per step, behind which the NEXT step's x is complete too, so that its first fragments are read
// before the barrier.  A buffer row is 128 bytes; its 16-byte pieces are stored at piece ^ (row / 2 & 7) (each lane of the load asks for the
// piece that belongs at its place), so that fragment reads of 16 rows meet no bank twice.  Inside a step the slices are
// pipelined: while one is multiplied, the next is dequantised and its A fragments are read.
//
// Bound: the matrix cores, which this card's power holds to 1.7 (32x32x16) and 1.95 PFLOP/s (16x16x32) on random data in a bare loop, and
// the dequantisation's share of that power.  A 128 x 256 tile of 4096 k takes 45 us alone on a CU, 56 on a full chip (1.2 PFLOP/s); several
// blocks on a CU only share its matrix cores, so that the plan below weighs whole rounds of 256 CUs.  7B layer, 765 rows, us, with the loop in whole turns of its
// ring (below) / and the 16x16x32 form: qkv 79 -> 77 -> 73, o 36 -> 32, gate_up 145 -> 138 -> 130, down 81 -> 74; 300 rows 41 -> 38, 28 -> 23, 72 -> 68, 45 -> 42.
#include <stdlib.h>
#include <algorithm>
#include <type_traits>
#include "common.h"
#include "gptq_gemm_body.h"
#include "gptq_tall.h"
#include "tall_ring.h"

namespace {

using gptq::PrepLayout;
using gptq::prep_layout;

struct TallArgs {
    const f16* x;
    int64_t ldx;
    const uint8_t* prep;
    int64_t offB;
    const f16* bias;
    f16* out;
    int64_t ldo;
    int M, K, N, NT, KS, G, spg_shift;
    int tile0, col_blocks;  // this launch: tiles tile0 + 0 .. gridDim.x - 1 in the order of tile_at
    int per, S;             // k64-steps per split, splits (blockIdx.y)
    int part;               // 1: fp32 tiles [blockIdx.x][split][BM][BN] in `scratch` instead of the finished output
    int vec;                // rows of `out` take 16-byte stores
    float* scratch;
};

constexpr int TALL_RING = tall::RING;  // buffers of x

// The order of tiles (tall_ring.h).  us, columns fastest over the whole chip / this: 4096 x 22016 with SiLU at 300, 765, 6000 rows 74.9 / 69.4, 148.6 /
// 146.2, 989 / 961; 8192 x 57344 with SiLU at 300, 3000 rows 345 / 324, 2611 / 2456; 11008 x 4096 at 140, 300, 765 rows 33.3 / 30.3, 41.3 / 42.6,
// 79.4 / 79.1; 4096 x 4096 at 433 25.3 / 25.9.  (Groups of 4: alike, 69, 145, 955; 327, 2432; 30.2, 44.4, 78.0; 26.8.)
using tall::tile_at;
using tall::xcd_run;

// A wave's sums, 32 BMR rows of TW tiles, as the two shapes of the matrix instruction leave them in its lanes.  each: f(row, column of the tile, sum); pairs: the
// same of a gate | up tile, f(row, j, rounded gate, rounded up) of its columns j and 16 + j, given their biases.
template <int BMR, int TW> struct Sums16 {
    f32x4 v[TW][2][2 * BMR];  // 16x16x32: [tile][its left, right columns][rows 16 i .. + 15]
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int t = 0; t < TW; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int rf = 0; rf < 2 * BMR; ++rf) v[t][h][rf] = f32x4{0, 0, 0, 0};
    }
    template <typename F> __device__ __forceinline__ void each(int t, int lane, F f) const {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int rf = 0; rf < 2 * BMR; ++rf)
#pragma unroll
                for (int r = 0; r < 4; ++r) f(rf * 16 + 4 * (lane >> 4) + r, h * 16 + (lane & 15), v[t][h][rf][r]);
    }
    template <typename F> __device__ __forceinline__ void pairs(int t, int lane, float bias_gate, float bias_up, F f) const {
#pragma unroll
        for (int rf = 0; rf < 2 * BMR; ++rf)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                f(rf * 16 + 4 * (lane >> 4) + r, lane & 15, (float)(f16)(v[t][0][rf][r] + bias_gate), (float)(f16)(v[t][1][rf][r] + bias_up));
    }
};
template <int BMR, int TW> struct Sums32 {
    f32x16 v[TW][BMR];  // 32x32x16: [tile][rows 32 i .. + 31]
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int t = 0; t < TW; ++t)
#pragma unroll
            for (int rb = 0; rb < BMR; ++rb) v[t][rb] = f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    }
    static __device__ __forceinline__ int row_of(int lane, int rb, int r) { return rb * 32 + (r & 3) + 8 * (r >> 2) + 4 * (lane >> 5); }
    template <typename F> __device__ __forceinline__ void each(int t, int lane, F f) const {
#pragma unroll
        for (int rb = 0; rb < BMR; ++rb)
#pragma unroll
            for (int r = 0; r < 16; ++r) f(row_of(lane, rb, r), lane & 31, v[t][rb][r]);
    }
    // Lanes 0 - 15 of a half wave hold gate columns, 16 - 31 the matching up columns.  Swapping those rows of lanes between two
    // accumulator rows gives every lane a (gate, up) pair: the lower lanes that of row r, the upper ones that of row r + 1.
    template <typename F> __device__ __forceinline__ void pairs(int t, int lane, float bias_gate, float bias_up, F f) const {
        const int c = lane & 31;
        const float bv = c < 16 ? bias_gate : bias_up;
#pragma unroll
        for (int rb = 0; rb < BMR; ++rb)
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const uint32_t v0 = __builtin_bit_cast(uint32_t, (float)(f16)(v[t][rb][r] + bv));
                const uint32_t v1 = __builtin_bit_cast(uint32_t, (float)(f16)(v[t][rb][r + 1] + bv));
                const auto p = __builtin_amdgcn_permlane16_swap(v0, v1, false, false);
                const uint32_t g0 = p[0], u0 = p[1];  // (a bit cast of a vector's element itself reads element 0)
                f(row_of(lane, rb, r) + (c >> 4), c & 15, __builtin_bit_cast(float, g0), __builtin_bit_cast(float, u0));
            }
    }
};

// M16: products by the 16x16x32 instruction instead of 32x32x16.  Under the card's power limit it does more: bare loops on random f16 1.95 against 1.71 PFLOP/s
// (bf16 2.10, 1.77).  Where a SIMD has one wave it is the slower one: twice the products to issue, and 19 TW register moves between the lanes' halves a step.
// us, 32x32x16 / 16x16x32, tiles of 96 x 128, 96 x 256, 128 x 256: 4096 x 22016 with SiLU at 2045 rows 370 / 352, 362 / 339, 340 / 316; 4096 x 12288 at 1500 152 /
// 146, 143 / 139, 161 / 155; of up to 256 blocks 4096 x 4096 at 763 33.1 / 34.2, 41.5 / 49.6, 46.7 / 57.1; 11008 x 4096 at 2045 (128 x 256) 164 / 172.
// Tiles of 64 rows have too few products to a dequantised fragment for either to matter (4096 x 12288 at 763 rows 92 / 91, 94 / 94).
template <int BMR, int ACT, int TW, bool M16>
__global__ __launch_bounds__(256, 2) void gptq_gemm_tall_kernel(TallArgs a) {
    constexpr int BM = 32 * BMR;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];  // [TALL_RING][BM][128 bytes]
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    int row_block, col_block;
    tile_at(a.tile0 + xcd_run(blockIdx.x, gridDim.x), (a.M + BM - 1) / BM, a.col_blocks, row_block, col_block);
    const int m0 = row_block * BM;
    const int mrows = min(BM, a.M - m0);
    const int split = blockIdx.y;
    const int nt_raw0 = (col_block * 4 + w) * TW;
    const int ksteps = a.K >> 6;                                         // K % 64 == 0 (host)
    const int ks0 = split * a.per, n = min(ksteps, ks0 + a.per) - ks0;   // n >= 1 (host)

    const uint8_t *wtile[TW], *sztile[TW];
#pragma unroll
    for (int t = 0; t < TW; ++t) {
        const int nt = min(nt_raw0 + t, a.NT - 1);
        wtile[t] = a.prep + (int64_t)nt * a.KS * 1024;
        sztile[t] = a.prep + a.offB + (int64_t)nt * a.G * 128;
    }
    const uint32_t woff = lane * 16, szoff = (lane & 31) * 4;
    // (M16 has no registers to spare for addresses; where a wave is waited for, the loads that need none are the slower ones: 4096 x 4096 at 300 rows in tiles of
    // 64 x 128 24.2 / 25.8 us.  There the offset is one 64-bit shift: extended from 32 bits it keeps the scalar unit in front of each step's last products, 2048 x
    // 2048 at 300 rows 13.1 / 13.4, 4096 x 4096 at 400 23.3 / 23.9.)
    auto sz_at = [&](int t, int ks) -> uint32_t {
        const int g = min(ks >> a.spg_shift, a.G - 1);
        if constexpr (M16) {
            return tall::buffer_word(sztile[t], a.G * 128, szoff, g * 128);
        } else {
            const uint8_t* p = sztile[t] + (int64_t)g * 128;
            PIN_SGPR(p);
            return *(const GLOBAL_AS uint32_t*)(p + szoff);
        }
    };
    auto w_at = [&](int t, int ks) -> u32x4 {
        const int k = min(ks, ksteps - 1);
        if constexpr (M16) {
            return __builtin_bit_cast(u32x4, tall::buffer_piece<2>(wtile[t], a.KS * 1024, woff, k * 1024));
        } else {
            const uint8_t* p = wtile[t] + (int64_t)k * 1024;
            PIN_SGPR(p);
            return __builtin_nontemporal_load((const GLOBAL_AS u32x4*)(p + woff));
        }
    };

    // x: load j of wave w brings rows 8 (4 j + w) .. + 7 (rows past M: the last one, never stored)
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
    uint32_t rowoff[BMR];
#pragma unroll
    for (int j = 0; j < BMR; ++j)
        rowoff[j] = (uint32_t)(min(8 * (4 * j + w) + (lane >> 3), mrows - 1) * (int)a.ldx * 2 + ((lane & 7) ^ (4 * (w & 1) + (lane >> 4))) * 16);
    const char* xbase = reinterpret_cast<const char*>(a.x + (int64_t)m0 * a.ldx);
    auto x_load = [&](int step, int buf) {
        const char* xb = xbase + (int64_t)min(ks0 + step, ksteps - 1) * 128;
        PIN_SGPR(xb);
#pragma unroll
        for (int j = 0; j < BMR; ++j)
            kib_to_lds(xb, rowoff[j], __builtin_amdgcn_readfirstlane(lds0 + buf * (BM * 128) + (4 * j + w) * 1024));
    };

    uint32_t EXr = 0x64006400u, M0r = 0x000F000Fu, M1r = 0x00F000F0u;
    asm volatile("" : "+v"(EXr));
    asm volatile("" : "+s"(M0r), "+s"(M1r));
    std::conditional_t<M16, Sums16<BMR, TW>, Sums32<BMR, TW>> acc;
    acc.clear();
    // A fragments.  M16: lane (c, q) has row c of its sixteen, and of the 32 k of slice m the step's piece 4 (q / 2) + 2 m + q % 2, as the swap in `halves` leaves
    // those of the weights.  Else: slice i, row lane % 32, piece i + 4 (lane / 32).
    const int c = lane & 15, q = lane >> 4;
    constexpr int SLICES = M16 ? 2 : 4, FRAGS = M16 ? 2 * BMR : BMR;
    uint32_t apos[SLICES];
#pragma unroll
    for (int i = 0; i < SLICES; ++i) {
        const int row = M16 ? c : lane & 31, piece = M16 ? (q >> 1) * 4 + i * 2 + (q & 1) : i + 4 * (lane >> 5);
        apos[i] = (uint32_t)(row * 128 + (piece ^ ((row >> 1) & 7)) * 16);
    }

    x_load(0, 0);
    x_load(1, 1);
    x_load(2, 2);
    // k64-steps of weights in flight per wave, slices of x in registers: the 16x16x32 form of the larger tiles has room for less
    constexpr bool LEAN = M16 && TW == 2;
    constexpr int WR = LEAN && BMR == 4 ? 2 : 4, AS = LEAN ? 1 : 2;
    u32x4 wq[WR][TW];
    uint32_t szr[WR][TW];
#pragma unroll
    for (int s = 0; s < WR; ++s)
#pragma unroll
        for (int t = 0; t < TW; ++t) {
            szr[s][t] = sz_at(t, ks0 + s);
            wq[s][t] = w_at(t, ks0 + s);
        }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();

    f16x8 b[2][TW], av[AS][FRAGS];
    uint32_t scale[TW][2];
    // A register of the image holds a tile's left columns in the first and third row of lanes, its right ones in the others: swapping the second row of one
    // with the first of the next, and the fourth with the third, leaves the left columns of both in one register, the right ones in the other.
    auto halves = [&](uint32_t& l, uint32_t& r) {
        const auto p = __builtin_amdgcn_permlane16_swap(l, r, false, false);
        l = p[0];
        r = p[1];
    };
    auto words = [&](u32x4 (&wr)[TW], int t, int m) {
        if (!M16) return;
        uint32_t l = wr[t][2 * m], r = wr[t][2 * m + 1];
        halves(l, r);
        wr[t][2 * m] = l;
        wr[t][2 * m + 1] = r;
    };
    auto scales = [&](const uint32_t (&sz)[TW], int t) {
        scale[t][0] = scale[t][1] = sz[t];
        if (M16) halves(scale[t][0], scale[t][1]);
    };
    auto dequant = [&](f16x8& dst, const u32x4 (&wr)[TW], int t, int u) {  // word u of a step: M16 half u % 2 of slice u / 2, else slice u
        const f16x2 szh = __builtin_bit_cast(f16x2, scale[t][M16 ? u & 1 : 0]);
        const f16 zd1 = (f16)960.f - szh[1];
        dst = gptq::dequant8(wr[t][u], f16x2{szh[1], szh[1]}, f16x2{zd1, zd1}, f16x2{szh[0], szh[0]}, EXr, M0r, M1r);
    };
    auto read_a = [&](int rf, int buf, int i) { av[i % AS][rf] = ld16<f16x8>(smem + buf * (BM * 128) + rf * (BM * 128 / FRAGS) + apos[i]); };
#pragma unroll
    for (int rf = 0; rf < FRAGS; ++rf) read_a(rf, 0, 0);
#pragma unroll
    for (int t = 0; t < TW; ++t) {
        scales(szr[0], t);
        words(wq[0], t, 0);
        dequant(b[0][t], wq[0], t, 0);
    }
    auto step = [&](int s, auto slot_, auto tail_) {
        constexpr int SL = decltype(slot_)::value;
        constexpr bool TAIL = decltype(tail_)::value;  // (at most RING - 1 steps, the first at slot 0)
        constexpr int NX = (SL + 1) % TALL_RING, WS = SL % WR, WN = (SL + 1) % WR;
        constexpr bool REFILL = !TAIL || SL + WR < TALL_RING - 1;
        if constexpr (!TAIL) x_load(s + 3, (SL + 3) % TALL_RING);  // everyone is done with that buffer since the barrier of the step before
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            __builtin_amdgcn_sched_barrier(0);
            auto refill = [&]() {
                if constexpr (REFILL) {
                    if (u < 3) return;
#pragma unroll
                    for (int t = 0; t < TW; ++t) {
                        wq[WS][t] = w_at(t, ks0 + s + WR);
                        szr[WS][t] = sz_at(t, ks0 + s + WR);
                    }
                }
            };
            auto dequant_next = [&](int t) {
                if (u == 3) scales(szr[WN], t);
                if (u & 1) words(wq[u == 3 ? WN : WS], t, u == 1);
                dequant(b[(u + 1) & 1][t], wq[u == 3 ? WN : WS], t, (u + 1) & 3);
            };
            if constexpr (LEAN) {
                refill();
                // rows in turn, in this order: a slice's are read again, for the next slice, behind their last product, and the next fragment of each tile is
                // dequantised between two of them
#pragma unroll
                for (int rf = 0; rf < 2 * BMR; ++rf) {
#pragma unroll
                    for (int t = 0; t < TW; ++t) acc.v[t][u & 1][rf] = mfma16(av[0][rf], b[u & 1][t], acc.v[t][u & 1][rf]);
                    if (u & 1) read_a(rf, u == 1 ? SL : NX, (u >> 1) ^ 1);
#pragma unroll
                    for (int t = 0; t < TW; ++t)
                        if (rf == (2 * BMR * t) / TW) dequant_next(t);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                if (!M16 || !(u & 1)) {
                    const int next = M16 ? (u >> 1) ^ 1 : (u + 1) & 3;
#pragma unroll
                    for (int rf = 0; rf < FRAGS; ++rf) read_a(rf, next ? SL : NX, next);
                    __builtin_amdgcn_sched_barrier(0);
                }
                refill();
#pragma unroll
                for (int t = 0; t < TW; ++t) dequant_next(t);
#pragma unroll
                for (int rf = 0; rf < FRAGS; ++rf)
#pragma unroll
                    for (int t = 0; t < TW; ++t) {
                        if constexpr (M16)
                            acc.v[t][u & 1][rf] = mfma16(av[u >> 1][rf], b[u & 1][t], acc.v[t][u & 1][rf]);
                        else
                            acc.v[t][rf] = mfma32(av[u & 1][rf], b[u & 1][t], acc.v[t][rf]);
                    }
                // the dequantisation's 13 TW instructions, and the swaps in front, between the products
                constexpr int PRODUCTS = FRAGS * TW;
#pragma unroll
                for (int g = 0; g < PRODUCTS; ++g) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, ((M16 ? 16 : 13) * TW + PRODUCTS - 1) / PRODUCTS, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // the x loads of step s + 2 were issued a step ago: behind them this wave has asked for that step's 2 TW weights and scales
        // and, in whole turns, for everything of this step
        tall::meet<TAIL ? 0 : BMR + 4 * TW>();
    };
    tall::ring_steps(n, step);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no direct load may still be on its way to LDS when the block ends

    constexpr int BN = 128 * TW;
    if (a.part) {
        float* dst = a.scratch + ((int64_t)xcd_run(blockIdx.x, gridDim.x) * a.S + split) * (BM * BN) + w * (32 * TW);
#pragma unroll
        for (int t = 0; t < TW; ++t) acc.each(t, lane, [&](int row, int col, float sum) { dst[(int64_t)row * BN + t * 32 + col] = sum; });
        return;
    }
    // finished: the tile goes through LDS so that rows leave in 16-byte pieces, 512 (256 with SiLU * up) contiguous bytes a row
    constexpr int BO = ACT == 2 ? BN / 2 : BN, OS = BO + 8;
    const int n_out = ACT == 2 ? a.N >> 1 : a.N, n0 = col_block * BO;
    __syncthreads();
    f16* tile_out = reinterpret_cast<f16*>(smem);  // [BM][OS]
#pragma unroll
    for (int t = 0; t < TW; ++t) {
        const int nt = min(nt_raw0 + t, a.NT - 1);
        if (ACT == 2) {
            const int j = nt * 16 + c;
            acc.pairs(t, lane, a.bias ? (float)a.bias[j] : 0.f, a.bias ? (float)a.bias[(a.N >> 1) + j] : 0.f, [&](int row, int col, float gate, float up) {
                const float sl = gate / (1.f + __expf(-gate));
                tile_out[row * OS + (w * TW + t) * 16 + col] = (f16)((float)(f16)sl * up);
            });
        } else {
            const float left = a.bias ? (float)a.bias[nt * 32 + (M16 ? c : lane & 31)] : 0.f, right = M16 && a.bias ? (float)a.bias[nt * 32 + 16 + c] : left;
            acc.each(t, lane, [&](int row, int col, float sum) {
                tile_out[row * OS + (w * TW + t) * 32 + col] = (f16)(sum + (M16 && col >= 16 ? right : left));
            });
        }
    }
    __syncthreads();
    constexpr int PIECES = BO / 8;
    for (int p = tid; p < mrows * PIECES; p += 256) {
        const int m = p / PIECES, col = (p % PIECES) * 8;
        if (n0 + col >= n_out) continue;  // (outputs come in whole groups of 16 columns)
        const f16x8 v = *reinterpret_cast<const f16x8*>(tile_out + m * OS + col);
        f16* o = a.out + (int64_t)(m0 + m) * a.ldo + n0 + col;
        if (a.vec) {
            st16(o, v);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = v[e];
        }
    }
}

// The tiles that were split over k: sum of a tile's S fp32 parts in fixed order, then what the kernel above does with an unsplit tile.
// grid (four-column groups of a tile / 256, tiles); ACT 2: four (gate, up) pairs.
template <int BM, int BN, int ACT>
__global__ __launch_bounds__(256) void tall_finish_kernel(TallArgs a) {
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
    if (ACT == 2) {
        const int t = g >> 2, c = (g & 3) * 4, j = (col_block * (BN / 32) + t) * 16 + c, half = a.N >> 1;
        if (j >= half) return;
        const f32x4 gate = part_sum(t * 32 + c), up = part_sum(t * 32 + 16 + c);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float mine = (float)(f16)(gate[e] + (a.bias ? (float)a.bias[j + e] : 0.f));
            const float other = (float)(f16)(up[e] + (a.bias ? (float)a.bias[half + j + e] : 0.f));
            a.out[(int64_t)row * a.ldo + j + e] = (f16)((float)(f16)(mine / (1.f + __expf(-mine))) * other);
        }
    } else {
        const int n = col_block * BN + g * 4;
        if (n >= a.N) return;
        const f32x4 v = part_sum(g * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) a.out[(int64_t)row * a.ldo + n + e] = (f16)(v[e] + (a.bias ? (float)a.bias[n + e] : 0.f));
    }
}

// ---- how a GEMM is cut ----------------------------------------------------------------------------------------------------------
constexpr int CUS = 256;

struct TallPlan {
    int BMR, TW;
    int col_blocks, tiles;  // tiles of BM x 128 TW
    int whole;              // leading tiles that are not split
    int S, per;             // the others: splits, k64-steps per split
    double us;              // what the model below expects
};

// us per k64-step of a block that has its CU to itself, and of a CU's share of a full chip (several blocks on each; clocks drop under
// the matrix cores' load).  Fitted to launches of 23 - 400 us at the 7B shapes; over 21 matrices and 16 row counts from 65 to 6000, weights
// cold, the plans that the model picks are 1.1 % up to 256 rows, 0.6 above behind the best of up to 48 that were timed at each size (with the 16x16x32 form 0.5 %
// over 53 products, at most 9).
struct TallCost {
    double alone, busy;
};
constexpr TallCost TALL_COST[3][2] = {{{0.33, 0.286}, {0.42, 0.50}}, {{0.41, 0.367}, {0.52, 0.70}}, {{0.45, 0.472}, {0.63, 0.85}}};

// Rows x columns of a tile, and whether the tiles past the last whole round of 256 are split over k.  One size does not do: 765 rows of
// a 7B gate_up are 516 tiles of 128 x 256, two rounds and four tiles, which take a third round (187 us; 161 with the four split in
// eight); a 7B qkv at that size is 768 tiles of 96 x 128, three whole rounds (86 us against 101 for 288 of 128 x 256).  (With 12 us for a split
// behind no whole round, where it costs 7, 3072 x 3072 at 129 - 192 rows was 96 unsplit tiles of 18.6 us, 14.7 in three parts; 5120 x 5120 at 256
// 30.6 / 26.7, 8192 x 3072 at 600 51 / 47, 5632 x 2048 at 765 34 / 30.)
TallPlan plan_tall(int64_t M, int64_t K, int64_t N) {
    const int64_t steps = K / 64, NT = cdiv64(N, 32);
    TallPlan best{};
    double best_us = 1e30;
    for (int BMR = 2; BMR <= 4; ++BMR)
        for (int TW = 1; TW <= 2; ++TW) {
            const TallCost c = TALL_COST[BMR - 2][TW - 1];
            const int64_t cb = cdiv64(NT, 4 * TW), tiles = cb * cdiv64(M, 32 * BMR), rounds = tiles / CUS, rest = tiles % CUS;
            const double alone = 4.0 + steps * c.alone, busy = 1.5 + steps * c.busy, share = (double)rest / CUS;
            for (int S = 1; S <= 16; ++S) {
                const int64_t per = cdiv64(steps, S);
                if (S > 1 && (rest == 0 || rest * S > CUS || per < 4)) break;
                if ((S - 1) * per >= steps) continue;  // an empty last split
                double us = rounds * busy;
                if (S > 1)  // the splits, their fp32 tiles written and read, and the launch that adds them; behind whole rounds, a launch of its own
                    us += 7.0 + (rounds ? 5.0 : 0.0) + per * c.alone + 2.0 * rest * S * (32 * BMR) * (128 * TW) * 4 / 4e6;
                else if (rounds == 0)
                    us = alone + std::max(0.0, busy - alone) * share;
                else
                    us = std::max(alone, us + (rest ? busy * (0.55 + 0.45 * share) : 0.0));
                if (us < best_us) {
                    best_us = us;
                    best = {BMR, TW, (int)cb, (int)tiles, (int)(S > 1 ? tiles - rest : tiles), S, (int)per, us};
                }
            }
        }
    if (const char* e = getenv("TGIS_TALL_PLAN")) {  // tuning hook: "BMR,TW,S" (S splits all tiles past the last whole round)
        int b = 0, t = 0, S = 0;
        if (sscanf(e, "%d,%d,%d", &b, &t, &S) == 3 && b >= 2 && b <= 4 && t >= 1 && t <= 2 && S >= 1 && S <= 16) {
            const int64_t cb = cdiv64(NT, 4 * t), tiles = cb * cdiv64(M, 32 * b), per = cdiv64(steps, S);
            if ((S - 1) * per < steps) best = {b, t, (int)cb, (int)tiles, (int)(S > 1 ? tiles - tiles % CUS : tiles), S, (int)per, 0.0};
        }
    }
    return best;
}

int64_t plan_scratch(const TallPlan& p) {
    return p.whole < p.tiles ? (int64_t)(p.tiles - p.whole) * p.S * (32 * p.BMR) * (128 * p.TW) * 4 : 0;
}

template <int BMR, int ACT, int TW, bool M16>
int launch_form(const TallArgs& a, int tiles, int S, hipStream_t st) {
    constexpr size_t ring = (size_t)TALL_RING * (32 * BMR) * 128, rows = (size_t)(32 * BMR) * ((ACT == 2 ? 64 : 128) * TW + 8) * 2;
    constexpr size_t lds = ring > rows ? ring : rows;
    static const hipError_t attr = hipFuncSetAttribute((const void*)gptq_gemm_tall_kernel<BMR, ACT, TW, M16>,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    TGIS_CHECK_HIP(attr);
    hipLaunchKernelGGL((gptq_gemm_tall_kernel<BMR, ACT, TW, M16>), dim3((unsigned)tiles, (unsigned)S), dim3(256), lds, st, a);
    TGIS_CHECK_LAUNCH();
    return TGIS_OK;
}
// (M16: where CUs have two blocks, and tiles of more than 64 rows)
template <int BMR, int ACT, int TW>
int launch_blocks(const TallArgs& a, int tiles, int S, hipStream_t st) {
    if constexpr (BMR > 2)
        if ((int64_t)tiles * S > CUS) return launch_form<BMR, ACT, TW, true>(a, tiles, S, st);
    return launch_form<BMR, ACT, TW, false>(a, tiles, S, st);
}
template <int ACT>
int launch_shape(const TallPlan& p, const TallArgs& a, int tiles, int S, hipStream_t st) {
    switch (p.BMR * 10 + p.TW) {
        case 21: return launch_blocks<2, ACT, 1>(a, tiles, S, st);
        case 22: return launch_blocks<2, ACT, 2>(a, tiles, S, st);
        case 31: return launch_blocks<3, ACT, 1>(a, tiles, S, st);
        case 32: return launch_blocks<3, ACT, 2>(a, tiles, S, st);
        case 41: return launch_blocks<4, ACT, 1>(a, tiles, S, st);
        default: return launch_blocks<4, ACT, 2>(a, tiles, S, st);
    }
}

template <int ACT>
int launch_finish(const TallPlan& p, const TallArgs& a, int tiles, hipStream_t st) {
#define TGIS_TALL_FINISH(B, W)                                                                                                         \
    hipLaunchKernelGGL((tall_finish_kernel<32 * B, 128 * W, ACT>),                                                                     \
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

TallArgs tall_args(const void* x, int64_t ldx, const void* prepared, int64_t M, int64_t K, int64_t N, int64_t groups, float* scratch) {
    const PrepLayout p = prep_layout(K, N, groups);
    const int64_t spg = K / groups / 64;
    TallArgs a{};
    a.x = (const f16*)x;
    a.ldx = ldx;
    a.prep = (const uint8_t*)prepared;
    a.offB = p.offB;
    a.M = (int)M;
    a.K = (int)K;
    a.N = (int)N;
    a.NT = (int)p.NT;
    a.KS = (int)p.KS;
    a.G = (int)groups;
    a.spg_shift = 30;
    if (groups > 1)
        for (a.spg_shift = 0; (1 << a.spg_shift) < spg; ++a.spg_shift) {}
    a.scratch = scratch;
    return a;
}

}  // namespace

// Rows from which it may replace the 64-row streaming passes, and up to which it replaces dequantise + library GEMM: (library with its
// dequantisation / tall, us, the four GEMMs of a 7B layer) 4096 rows 1428 / 1360, 6000 rows 2169 / 2011, 8190 rows 2595 / 2693; at 16128 rows
// hipBLASLt's 256 x 256 tiles, free of dequantisation, run at 1.4 PFLOP/s against 1.2 - 1.25.
int64_t gptq::tall_min_m(int act) {
    static const int64_t v = getenv("TGIS_TALL_MIN_M") ? atoll(getenv("TGIS_TALL_MIN_M")) : 0;
    return v ? v : act == 2 ? 65 : 129;
}
int64_t gptq::tall_max_m() {
    static const int64_t v = getenv("TGIS_TALL_MAX_M") ? atoll(getenv("TGIS_TALL_MAX_M")) : 8192;
    return v;
}
bool gptq::tall_serves(int64_t K, int64_t groups, bool act_order, int act) {
    if (act_order || act == 1 || K % 64 != 0 || groups <= 0) return false;
    const int64_t gs = K / groups, spg = gs / 64;
    return groups == 1 || (gs % 64 == 0 && (spg & (spg - 1)) == 0);
}
// Between 3072 and tall_max_m() rows it depends on the library's 256 x 256 tiles: whether they fill their rounds of 256, and each block has as many of them (rounds that
// do not divide the tiles, up to ten, send the library to kernels that take 1.2 to 1.5 times as long).  act 0, us, dequantise ([N][K]) and library / this kernel, weights cold:
//   93 % full and dealt evenly:  5120 x 15360 at 4096, 6000, 8190 481 / 529, 704 / 769, 936 / 1021; 11008 x 4096 at 4096, 7476, 8190 262 / 299, 476 / 545, 498 / 587; 8192 x 10240 at 4376, 6000,
//                        8190 544 / 602, 729 / 806, 933 / 1072; 4096 x 12288 at 4096, 5225, 8190 297 / 332, 401 / 430, 572 / 656; 7168 x 7168 at 6711 (756 tiles) 486 / 554; 13824 x 5120 at 6264
//                        (500) 620 / 697
//   93 % full, not evenly:  8192 x 10240 at 4728 (760 tiles) 827 / 614; 8192 x 8192 at 5683 (736) 758 / 604; 7168 x 7168 at 6409 (728) 684 / 530; 17920 x 6656 at 7206 (754) 1687 / 1368; 5120 x
//                        15360 at 7203 (1740) 972 / 884.  Of 1640 drawn products this kernel takes 0.86 of the time, at three rounds 0.78, and 79 are more than 2 % behind, at most 10
//   two rounds 93 - 95 % full past k of 13056:  13824 x 5120 at 6000 976 / 681; 14336 x 4096 at 7459 1028 / 714; 28672 x 8192 at 3625 1728 / 1404 (291 drawn: 0.75)
//   less:                4096 x 12288 at 6000 580 / 482; 11008 x 4096 at 5225 672 / 402; 8192 x 10240 at 3500, 4096, 5225 623 / 490, 716 / 530, 813 / 714; 13824 x 5120 at 3500, 5225, 8190 772 /
//                        417, 891 / 601, 1060 / 898; 28672 x 8192 at 5225, 7168 2499 / 1964, 3247 / 2706; but also 4096 x 12288 at 3500 279 / 306, 4096 x 4096 at 7168 183 / 206, 8192 x 8192 at 5225,
//                        7168 537 / 572, 705 / 746, which are dealt evenly too (672, 448, 672, 896 tiles)
//   one round, from three fifths on, of long k:  11008 x 4096 at 3500 245 / 273; 8192 x 3072 at 4096, 5000 169 / 199, 180 / 207 (5632 x 2048 at 4096,
//                        half a round, 86 / 87)
// With SiLU * up this kernel is in front of the library and its activation launch (4096 x 22016 at 4096, 8190 rows 740 / 611, 1291 / 1207; 2048 x
// 11264 198 / 178, 421 / 333; 8192 x 57344 at 2045, 3500 1598 / 1514, 2666 / 2662, but at 4096, 8190 2889 / 3027, 5632 / 6084).
bool gptq::tall_before_library(int64_t M, int64_t K, int64_t N, int act) {
    if (M <= 3072 || act == 2 || getenv("TGIS_TALL_MAX_M")) return M <= tall_max_m();
    const int64_t tiles = cdiv64(M, 256) * cdiv64(N, 256), slots = cdiv64(tiles, CUS) * CUS;
    const int64_t rounds = slots / CUS;
    const bool evenly = (tiles % rounds == 0 || rounds > 10) && !(rounds == 2 && 100 * tiles < 95 * slots && K > 13056);
    const bool long_round = tiles <= CUS && 10 * tiles > 6 * CUS && K >= 5120;
    return M <= tall_max_m() && !(evenly && 100 * tiles >= 93 * slots) && !long_round;
}
// Up to 256 rows the passes take k in parallel (k-parts, splits) where a tile here walks it alone, so it depends on the matrix which of
// the two is done first.  us, the passes with the launch that adds their slabs / this kernel with a norm behind it (act 2: either alone):
//   act 0:  2048 x 2560 at 129 / 256 rows 16.2 / 17.3, 16.7 / 17.2; 3072 x 5120 21.0 / 23.5, 34.4 / 24.6; 4096 x 4096 23.2 / 20.8, 24.7 /
//           27.8; 2048 x 6144 25.5 / 18.3, 27.5 / 19.4; 4096 x 12288 51.8 / 37.5, 52.4 / 42.4; 11008 x 4096 44.5 / 30.9, 46.6 / 36.9; 8192 x
//           10240 49.1 / 45.5, 88.9 / 56.2; 28672 x 8192 146 / 98, 162 / 126
//   act 2:  2048 x 11264 at 65 / 128 / 129 / 256 rows 15.1 / 15.8, 15.1 / 13.7, 26.1 / 17.7, 28.3 / 19.7; 4096 x 22016 45.5 / 31.0, 46.7 / 34.9,
//           67.5 / 44.9, 74.0 / 55.7; 8192 x 57344 185 / 92, 185 / 121, 272 / 177, 348 / 225; 1024 x 8192 11.9 / 11.4, 13.6 / 9.2, 10.7 / 8.7, 11.3 / 9.0
// The passes' time is that of their rounds of 256 blocks, each its chunks of 256 k per k-part (fitted to 30 shapes, within 8 %).
static bool pays_below_257_rows(int64_t M, int64_t K, int64_t N, int act) {
    const gptq::GemmPlan pass = gptq::plan_gemm(K, N, act, M);
    const double rounds = (double)cdiv64(cdiv64(cdiv64(N, 32), pass.TN) * cdiv64(M, 64) * pass.S, CUS), chunks = pass.KR / 256 / pass.WK;
    const double passes = act == 2 ? 2.0 + rounds * (2.0 + chunks * (pass.TN == 4 ? 2.65 : 1.9))
                                   : 5.0 + rounds * (3.0 + chunks * (pass.TN == 4 ? 2.45 : 1.65));
    const TallPlan p = plan_tall(M, K, N);
    return (act == 2 ? 1.1 * p.us - 1.0 : 1.1 * p.us + 1.0) <= passes;
}
bool gptq::tall_ok(int64_t M, int64_t K, int64_t N, int64_t groups, bool act_order, int act) {
    if (M < tall_min_m(act) || !tall_serves(K, groups, act_order, act)) return false;
    return M > 256 || getenv("TGIS_TALL_MIN_M") || getenv("TGIS_TALL_PLAN") || pays_below_257_rows(M, K, N, act);
}
int64_t gptq::tall_workspace_bytes(int64_t M, int64_t K, int64_t N) { return plan_scratch(plan_tall(M, K, N)); }

int gptq::launch_tall(const void* x, int64_t ldx, const void* prepared, const void* bias, void* out, int64_t ldo, int64_t M, int64_t K,
                      int64_t N, int64_t groups, int act, float* scratch, hipStream_t st) {
    const TallPlan p = plan_tall(M, K, N);
    TallArgs a = tall_args(x, ldx, prepared, M, K, N, groups, scratch);
    a.bias = (const f16*)bias;
    a.out = (f16*)out;
    a.ldo = ldo;
    a.vec = ldo % 8 == 0 && (uintptr_t)out % 16 == 0;
    a.col_blocks = p.col_blocks;
    a.per = (int)(K / 64);
    a.S = 1;
    if (p.whole > 0) {
        const int rc = act == 2 ? launch_shape<2>(p, a, p.whole, 1, st) : launch_shape<0>(p, a, p.whole, 1, st);
        if (rc != TGIS_OK) return rc;
    }
    if (p.whole < p.tiles) {
        a.tile0 = p.whole;
        a.per = p.per;
        a.S = p.S;
        a.part = 1;
        const int rc = launch_shape<0>(p, a, p.tiles - p.whole, p.S, st);  // (fp32 tiles: the same for both activations)
        if (rc != TGIS_OK) return rc;
        return act == 2 ? launch_finish<2>(p, a, p.tiles - p.whole, st) : launch_finish<0>(p, a, p.tiles - p.whole, st);
    }
    return TGIS_OK;
}
