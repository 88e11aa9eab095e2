// The dense decode GEMM with everything a block needs asked for at once.
//
// dense_gemm_unit (dense_gemm_body.h) keeps two k64-steps of weights in flight per wave and passes x through LDS 256 k at a time, so that
// a narrow projection is a chain of three to five dependent trips to memory: 5 - 11 us for 8 - 46 MB.  Here
//   * the 8 waves of a block split the k range step by step (wave w: steps w, w + 8, ...; the block reads its tiles' weights as
//     dense runs) and each has WIDE_DEPTH steps of TN tiles on their way to its registers from the first instruction on;
//   * x goes to LDS by direct loads, 512 Q k at a time (a PHASE, one buffer; two buffers where there are several phases): at the widths
//     of small models the whole k range is one phase, and a wave waits for memory once;
//   * the k-parts meet once, in LDS laid out [wave][tile][register][lane] (every access 64 consecutive words), and wave w finishes
//     registers 2 w, 2 w + 1 of every tile (R16, up to 16 rows: register w).
// x in LDS: [256-k chunk][row][512 bytes], piece p (16 bytes) of row m at p ^ (m & 7), so that the fragment reads of 32 (16) rows meet no
// bank twice; each lane of a direct load asks for the piece that belongs at its place.  Only the rows of the batch are loaded: what lies
// in the others never reaches an output that is stored.
#pragma once
#include "dense_gemm_body.h"

namespace dense {

constexpr int WIDE_WAVES = 8;
constexpr int WIDE_DEPTH = 4;  // k64-steps in flight per wave

// Q (1, 2 or 4): k64-steps per wave and phase.  A block takes the whole k range and all rows.  rows_lds: rows of x in LDS, even.
template <typename T, int TN, int ACT, int MR, bool R16, int Q>
__device__ __forceinline__ void dense_wide_unit(const DenseArgs& a, const int ntg, const int rows_lds, unsigned char* smem) {
    static_assert(!R16 || MR == 1, "16-row staging is for single 32-row passes");
    static_assert(WIDE_DEPTH % Q == 0, "phases and the ring stay in step");
    using V8 = typename VecT<T>::x8;
    constexpr int W = WIDE_WAVES, CHUNKS = 2 * Q;  // 256-k chunks per phase
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int mrows = min(R16 ? 16 : 32 * MR, a.M);
    const int n = a.K >> 6;                // k64-steps; K % 64 == 0, n >= 1 (host)
    const int mine = (n - w + W - 1) / W;  // steps of this wave
    const int phases = (n + W * Q - 1) / (W * Q);
    const int buf_bytes = CHUNKS * rows_lds * 512;

    // x: one load brings two rows of a chunk
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
    const char* xbase = reinterpret_cast<const char*>(a.x);
    const int pairs = rows_lds >> 1;
    auto x_phase = [&](int p) {
        for (int l = w; l < CHUNKS * pairs; l += W) {
            const int chunk = l / pairs, pair = l - chunk * pairs, m = 2 * pair + (lane >> 5);
            const int k = min((p * CHUNKS + chunk) * 256 + ((lane & 31) ^ (m & 7)) * 8, a.K - 8);  // (past the range: never read)
            const char* xb = xbase;
            PIN_SGPR(xb);
            kib_to_lds(xb, (uint32_t)(min(m, mrows - 1) * (int)a.ldx * 2 + k * 2),
                          __builtin_amdgcn_readfirstlane(lds0 + (p & 1) * buf_bytes + (chunk * rows_lds + 2 * pair) * 512));
        }
    };

    const char* wtile[TN];
#pragma unroll
    for (int t = 0; t < TN; ++t)
        wtile[t] = reinterpret_cast<const char*>(a.prep) + (int64_t)min(ntg * TN + t, a.NT - 1) * a.KS * 4096;
    const uint32_t woff = lane * 16;
    V8 wq[WIDE_DEPTH][TN][4];
    auto w_load = [&](int i_, V8 (&dst)[TN][4]) {
        const int64_t off = (int64_t)min(i_ * W + w, n - 1) * 4096;
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            const char* p = wtile[t] + off;
            PIN_SGPR(p);
#pragma unroll
            for (int i = 0; i < 4; ++i) dst[t][i] = __builtin_nontemporal_load((const GLOBAL_AS V8*)(p + i * 1024 + woff));
        }
    };

    // ACT 3: cache slot and rotary position of the rows this wave will finish
    constexpr int NR = R16 ? 1 : 2, NREG = NR * W;
    int32_t rpos[ACT == 3 ? MR : 1][ACT == 3 ? NR : 1], rslot[ACT == 3 ? MR : 1][ACT == 3 ? NR : 1];
    if (ACT == 3) {
#pragma unroll
        for (int mr = 0; mr < MR; ++mr)
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                const int r = w * NR + j;
                const int m = min(mr * 32 + (r & 3) + 8 * (r >> 2) + 4 * (lane >> 5), mrows - 1);
                rpos[mr][j] = a.positions[m];
                rslot[mr][j] = a.slots[m];
            }
    }

    x_phase(0);
#pragma unroll
    for (int d = 0; d < WIDE_DEPTH; ++d) w_load(d, wq[d]);

    f32x16 acc[TN][MR];
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int mr = 0; mr < MR; ++mr) acc[t][mr] = f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const int arow = lane & (R16 ? 15 : 31);
    for (int i0 = 0; i0 < phases * Q; i0 += WIDE_DEPTH) {
#pragma unroll
        for (int d = 0; d < WIDE_DEPTH; ++d) {
            const int i_ = i0 + d;  // this wave's i_-th step, in ring slot d
            if (d % Q == 0) {
                const int p = i_ / Q;
                if (p >= phases) break;
                // this wave's part of the phase's x has arrived: behind its loads the wave has asked for WIDE_DEPTH steps of weights
                // (first phase) or refilled Q of them (later ones, unless its range is about to end)
                if (p == 0)
                    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(WIDE_DEPTH * TN * 4) : "memory");
                else if (i_ - 1 + WIDE_DEPTH < mine)
                    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(Q * TN * 4) : "memory");
                else
                    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                if (p + 1 < phases) x_phase(p + 1);  // everyone is done with that buffer since this barrier
            }
            if (i_ < mine) {
                const int s = (d % Q) * W + w;  // k64-step within the phase
                const unsigned char* xb = smem + ((i_ / Q) & 1) * buf_bytes + (s >> 2) * rows_lds * 512;
                const int piece0 = (s & 3) * 8 + (lane >> 5) * 4;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    V8 av[MR];
#pragma unroll
                    for (int mr = 0; mr < MR; ++mr) {
                        const int m = min(mr * 32 + arow, rows_lds - 1);
                        av[mr] = ld16<V8>(xb + m * 512 + (((piece0 + i) ^ (m & 7)) << 4));
                    }
#pragma unroll
                    for (int t = 0; t < TN; ++t)
#pragma unroll
                        for (int mr = 0; mr < MR; ++mr) acc[t][mr] = mfma32(av[mr], wq[d][t][i], acc[t][mr]);
                }
                if (i_ + WIDE_DEPTH < mine) w_load(i_ + WIDE_DEPTH, wq[d]);
            }
        }
    }

    // ACT 3: the cos / sin entries of the rows this wave will finish, asked for before the exchange
    T rcos[TN][ACT == 3 ? MR : 1][ACT == 3 ? NR : 1], rsin[TN][ACT == 3 ? MR : 1][ACT == 3 ? NR : 1];
    if (ACT == 3) {
        const int per = a.rD >> 5;
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            const int nt = min(ntg * TN + t, a.NT - 1), tt = nt - (nt / per) * per, dr = 16 * tt + (lane & 15);
            const bool roth = nt / per < a.rH + a.rHkv;
#pragma unroll
            for (int mr = 0; mr < MR; ++mr)
#pragma unroll
                for (int j = 0; j < NR; ++j) {
                    rcos[t][mr][j] = roth ? reinterpret_cast<const T*>(a.cosb)[(int64_t)rpos[mr][j] * (a.rD >> 1) + dr] : (T)1.f;
                    rsin[t][mr][j] = roth ? reinterpret_cast<const T*>(a.sinb)[(int64_t)rpos[mr][j] * (a.rD >> 1) + dr] : (T)0.f;
                }
        }
    }
    __syncthreads();  // everyone is done with x
    float* red = reinterpret_cast<float*>(smem) + lane;  // [wave][tile][row block][register][lane]
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int mr = 0; mr < MR; ++mr)
#pragma unroll
            for (int r = 0; r < NREG; ++r) red[(((w * TN + t) * MR + mr) * NREG + r) * 64] = acc[t][mr][r];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < TN; ++t) {
        if (ntg * TN + t >= a.NT) return;
        float fin[MR][NR];
#pragma unroll
        for (int mr = 0; mr < MR; ++mr)
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                float v = red[((t * MR + mr) * NREG + w * NR + j) * 64];
#pragma unroll
                for (int k = 1; k < W; ++k) v += red[(((k * TN + t) * MR + mr) * NREG + w * NR + j) * 64];
                fin[mr][j] = v;
            }
        dense_finish<T, ACT, MR, NR>(a, fin, w * NR, ntg * TN + t, 0, 0, 0, mrows, lane, rslot, rcos[t], rsin[t]);
    }
}

// rows of a batch whose x is staged `rows_lds` (even) rows high, and the LDS of a block
static inline int wide_rows_lds(int64_t M, int MR) { return (int)(std::min<int64_t>(M, 32 * MR) + 1) / 2 * 2; }
static inline size_t wide_lds_bytes(int64_t M, int64_t K, int TN, int MR, bool R16, int Q) {
    const int64_t phases = cdiv64(K, 512 * Q);
    const size_t x = (size_t)std::min<int64_t>(phases, 2) * (2 * Q) * wide_rows_lds(M, MR) * 512;
    return std::max(x, (size_t)WIDE_WAVES * TN * MR * (R16 ? 8 : 16) * 256);
}

}  // namespace dense
