// Prefill attention over the paged cache (gfx950, MFMA 16x16x32): the many-q-rows counterpart of attn_paged_kernel.
// Same mathematics, page layouts and column convention (a column = one (q token, q head of the GQA group) pair);
// what changes is who reads K/V.  In attn_paged_kernel every wave loads the fragments of a page for its own 16
// columns, which is right for decode (one pass over the cache) and wasteful for prefill, where the same page is needed
// by every q tile of the sequence: measured 100-180 TFLOP/s, bound by L1 fragment traffic.  Here a block of 4 waves
// owns 128 columns (32 per wave, two 16-column groups; half of that where prompts are few), brings each 32-token page to LDS once and every wave takes its
// K / V^T fragments from there, each fragment read feeding two MFMAs.
//
// Pages go to LDS by direct loads, three ahead of the one that is multiplied, in a ring of four: no registers, no
// stores, one barrier per page; their numbers are read a page earlier still.  (One page ahead through registers, its
// number looked up on the way, a block waited for two dependent trips to memory per page.)
// LDS images of a page: K as in global memory ([tile][D/8][16 tokens][8]: a fragment is one contiguous KiB, lane l
// reads piece l); V^T regrouped to [D/16][4 chunks][16 rows][8 token columns] so that lane (row l&15, chunk l>>4) again
// reads piece l of a contiguous KiB — each lane of a direct load asks for the piece that belongs at its place.
//
// The scores of the next page are multiplied while the exponentials of this one run, and this page's values while the
// next one's maxima are found: a wave has work for the matrix cores and the vector units at the same time.
// us before / now: 16 x 1008 tokens, 32 heads of 128: 415 / 299; 1 x 4096: 352 / 204; 2 x 4093, 48 heads on one cached:
// 626 / 530; 8 x 1024, 64 on 8: 310 / 224; 4 x 1024, 32 on 4, D 64: 60 / 44.  What is left is shared out between vector
// units, matrix cores and L2 (without the page loads 245, 166, 447 us; without the exponentials 269, 178, 483).
// Softmax: the running maximum is kept scaled; a score costs one maximum, one fma, one exp2 and half a conversion.  The
// normaliser is the sum of the ROUNDED probabilities, as flash-attention's, and comes from the matrix cores (a row block
// of ones beside V^T): 32 additions and conversions a page less.
#include <stdlib.h>
#include <algorithm>
#include <type_traits>
#include "common.h"
#include "attention_args.h"

#define PIN_SGPR(p) asm volatile("" : "+s"(p))

namespace {

// maximum over the four 16-lane rows of a wave, in every lane
__device__ __forceinline__ float max_over_rows(float v) {
    const auto h = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
    const uint32_t h0 = h[0], h1 = h[1];
    v = fmaxf(__builtin_bit_cast(float, h0), __builtin_bit_cast(float, h1));
    const auto q = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
    const uint32_t q0 = q[0], q1 = q[1];
    return fmaxf(__builtin_bit_cast(float, q0), __builtin_bit_cast(float, q1));
}

constexpr int PREFILL_RING = 4;  // pages in LDS

// ROWS: the "rows" pages of attn_varlen.hip (keys token-major, values channel-major) instead of those of kv_layout.h.  There the token
// that a score row stands for is chosen so that the probabilities a lane holds are eight neighbours of a value row.
// CG: 16-column groups per wave (2; 1 where that leaves the chip idle, see the launcher).
template <typename T, int D, bool ROWS, int CG>
__global__ __launch_bounds__(256, 2) void attn_prefill_kernel(AttnPrefillArgs a) {
    using V8 = typename VecT<T>::x8;
    constexpr int KS = D / 32;  // k-steps of the QK^T MFMA
    constexpr int NB = D / 16;  // 16-row blocks of O^T
    constexpr int PAGE_ELEMS = 32 * D;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    T* lds = reinterpret_cast<T*>(smem);  // [PREFILL_RING][K page | V page]
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, c = lane >> 4;
    // long (late) tiles first: the causal triangle's tail is short ones.  The tiles of a (sequence, kv head, chunk) read the same pages:
    // where those groups come in eights (xcd_remap), each keeps to one XCD (blocks are dealt to the eight in turn), whose L2 then holds them.
    int qt = blockIdx.x, head_block = blockIdx.y, b = blockIdx.z;
    if (a.xcd_remap) {
        const int tiles = gridDim.x, heads = gridDim.y, id = blockIdx.x + tiles * (blockIdx.y + heads * blockIdx.z);
        const int group = (id >> 3) / tiles * 8 + (id & 7);
        qt = (id >> 3) % tiles;
        head_block = group % heads;
        b = group / heads;
    }
    qt = gridDim.x - 1 - qt;
    const int hk = head_block / a.HC, hc = head_block % a.HC;

    const int q0 = a.cu_q[b], q_len = a.cu_q[b + 1] - q0;
    const int TQB = a.TQ * 4 * CG;  // q tokens of the block's tile (64 CG columns)
    const int t0 = qt * TQB;
    if (t0 >= q_len) return;
    const int ctx = a.ctx_lens[b];
    const int g = col & (a.Gp - 1);
    const int head = hk * a.G + hc * 16 + g;
    int tq[CG], kmax[CG];
    bool col_valid[CG];
    int wave_kmax = 0, wave_kmin = 0x7fffffff;
#pragma unroll
    for (int cg = 0; cg < CG; ++cg) {
        tq[cg] = ((w * CG + cg) * 16 + col) >> a.Gp_shift;
        col_valid[cg] = (g < a.Gc) && (hc * 16 + g < a.G) && (t0 + tq[cg] < q_len);
        kmax[cg] = col_valid[cg] ? (ctx - q_len + t0 + tq[cg] + 1) : 0;  // this column attends to positions < kmax
        wave_kmax = max(wave_kmax, kmax[cg]);
        if (col_valid[cg]) wave_kmin = min(wave_kmin, kmax[cg]);  // invalid columns (q = 0, never stored) need no mask
    }
    // wave-uniform bound: pages at or past it are fully masked for this wave and skipped
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        wave_kmax = max(wave_kmax, __shfl_xor(wave_kmax, o, 64));
        wave_kmin = min(wave_kmin, __shfl_xor(wave_kmin, o, 64));
    }
    wave_kmax = __builtin_amdgcn_readfirstlane(wave_kmax);
    wave_kmin = __builtin_amdgcn_readfirstlane(wave_kmin);
    const int kend = ctx - q_len + min(q_len, t0 + TQB);  // keys needed by any column of the block
    const int pages = (kend + 31) >> 5;

    // Q^T fragments (B operand): lane supplies Q[col][ks*32 + c*8 .. +8]; a negative scale is Q's sign, so that the largest score stays it
    // (and with it the masked ones the smallest); a scale of zero is a Q of zeros
    const float scale = a.scale_log2 == 0.f ? 1.f : __builtin_fabsf(a.scale_log2);
    V8 qf[CG][KS];
#pragma unroll
    for (int cg = 0; cg < CG; ++cg) {
        const T* qp = reinterpret_cast<const T*>(a.q) + (int64_t)(q0 + t0 + tq[cg]) * a.ld_q + (int64_t)head * D + c * 8;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            if (col_valid[cg] && a.scale_log2 != 0.f) {
                qf[cg][ks] = ld16<V8>(qp + ks * 32);
                if (a.scale_log2 < 0.f) qf[cg][ks] = -qf[cg][ks];
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) qf[cg][ks][e] = (T)0.f;
            }
        }
    }

    // Rotary embedding of q: a lane holds both halves of its pairs.  (A pass of its own read and wrote q: 16128 rows of 32 heads of 128 72 us, 763 rows 5.8.  Whole
    // prompts, by a pass / here: 16 x 1008 tokens through 32 layers of 4096 171.8 / 170.0 ms, 3 of 763 in all 11.80 / 11.61, 2 x 1400 through 22 layers of 2048 6.87 / 6.68.)
    if (!ROWS && a.cosb) {
#pragma unroll
        for (int cg = 0; cg < CG; ++cg) {
            if (!col_valid[cg]) continue;
            const int64_t at = (int64_t)a.positions[q0 + t0 + tq[cg]] * (D / 2) + c * 8;
#pragma unroll
            for (int ks = 0; ks < KS / 2; ++ks) {
                const V8 cv = ld16<V8>(reinterpret_cast<const T*>(a.cosb) + at + ks * 32), sv = ld16<V8>(reinterpret_cast<const T*>(a.sinb) + at + ks * 32);
                V8& lo = qf[cg][ks];
                V8& hi = qf[cg][ks + KS / 2];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float x1 = to_f32(lo[e]), x2 = to_f32(hi[e]), cf = to_f32(cv[e]), sf = to_f32(sv[e]);
                    lo[e] = from_f32<T>(x1 * cf - x2 * sf);
                    hi[e] = from_f32<T>(x1 * sf + x2 * cf);
                }
            }
        }
    }

    f32x4 o[CG][NB], total[CG];  // total: the normaliser, alike in all four rows
    float ms[CG];                // running maximum times scale_log2
#pragma unroll
    for (int cg = 0; cg < CG; ++cg) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) o[cg][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
        total[cg] = f32x4{0.f, 0.f, 0.f, 0.f};
        ms[cg] = NEG_BIG;
    }
    V8 ones;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = (T)1.f;

    // ---- pages on their way to LDS: a KiB of K and one of V^T per load pair, NL pairs per wave and page -------------
    constexpr int NL = D / 64;
    const auto* btrow = (const __attribute__((address_space(4))) int32_t*)(uintptr_t)(a.bt + (int64_t)b * a.max_pages);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
    uint32_t koff[NL], voff[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        const int blk = i * 4 + w;  // KiB of the page: K as it lies; V^T: rows 16 blk .. + 15
        const int row = lane & 15, chunk = lane >> 4;
        koff[i] = blk * 1024 + lane * 16;
        voff[i] = (chunk * D + blk * 16 + row) * 16;
        if (ROWS) {
            koff[i] = (((row >> 2) * 8 + blk / KS * 4 + (row & 3)) * D + (blk % KS * 4 + chunk) * 8) * 2;
            voff[i] = ((blk * 16 + row) * 32 + chunk * 8) * 2;
        }
    }
    auto page_number = [&](int p) { return btrow[max(min(p, pages - 1), 0)]; };
    auto page_load = [&](int pg, int buf) {
        const int64_t at = ((int64_t)pg * a.Hkv + hk) * (PAGE_ELEMS * 2);
        const char* kp = reinterpret_cast<const char*>(a.kpool) + at;
        const char* vp = reinterpret_cast<const char*>(a.vpool) + at;
        PIN_SGPR(kp);
        PIN_SGPR(vp);
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + buf * (PAGE_ELEMS * 4) + (i * 4 + w) * 1024);
            kib_to_lds(kp, koff[i], dst);
            kib_to_lds(vp, voff[i], dst + PAGE_ELEMS * 2);
        }
    };
    page_load(page_number(0), 0);
    if (pages > 1) page_load(page_number(1), 1);
    if (pages > 2) page_load(page_number(2), 2);
    int next = page_number(3);

    auto page_barrier = [&](auto later_) {  // all of this wave's loads but the last `later` pages', and after it everyone's
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(later_)::value * 2 * NL) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto scores = [&](int p, f32x4 (&s)[CG][2]) {
        const T* kl = lds + (p & 3) * 2 * PAGE_ELEMS + lane * 8;
#pragma unroll
        for (int cg = 0; cg < CG; ++cg)
#pragma unroll
            for (int t = 0; t < 2; ++t) s[cg][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const V8 kf = ld16<V8>(kl + t * (16 * D) + ks * 512);
#pragma unroll
                for (int cg = 0; cg < CG; ++cg) s[cg][t] = mfma16(kf, qf[cg][ks], s[cg][t]);
            }
    };
    // masked scores of page p become -inf; the columns' new maxima; alpha: what moves the sums so far to them
    float alpha[CG];
    auto maxima = [&](int p, f32x4 (&s)[CG][2], auto masked_tag) {
#pragma unroll
        for (int cg = 0; cg < CG; ++cg) {
            if (decltype(masked_tag)::value) {
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[cg][t][r] = (p * 32 + c * (ROWS ? 8 : 4) + t * (ROWS ? 4 : 16) + r < kmax[cg]) ? s[cg][t][r] : -__builtin_inff();
            }
            const float top = max_over_rows(fmaxf(fmaxf(fmaxf(s[cg][0][0], s[cg][0][1]), fmaxf(s[cg][0][2], s[cg][0][3])),
                                                  fmaxf(fmaxf(s[cg][1][0], s[cg][1][1]), fmaxf(s[cg][1][2], s[cg][1][3]))));
            const float m_new = fmaxf(ms[cg], top * scale);
            alpha[cg] = __builtin_amdgcn_exp2f(ms[cg] - m_new);
            ms[cg] = m_new;
        }
    };
    // One page: its probabilities and products, and the scores and maxima of the next, so that each of the two chains has the matrix
    // cores while the other has the vector units.
    auto attend = [&](int p, f32x4 (&s)[CG][2], f32x4 (&sn)[CG][2], auto masked_tag) {
        scores(p + 1, sn);
        V8 pf[CG], vf[NB];
#pragma unroll
        for (int cg = 0; cg < CG; ++cg)
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    pf[cg][t * 4 + r] = from_f32<T>(__builtin_amdgcn_exp2f(__builtin_fmaf(s[cg][t][r], scale, -ms[cg])));
        const T* vl = lds + (p & 3) * 2 * PAGE_ELEMS + PAGE_ELEMS + lane * 8;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) vf[nb] = ld16<V8>(vl + nb * 512);
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * KS, 0);  // K's fragments, then products of scores among the exponentials
        __builtin_amdgcn_sched_group_barrier(0x402, 8, 0);
#pragma unroll
        for (int g = 0; g < 2 * CG * KS; ++g) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x402, 20 / KS, 0);
            if (g >= 2 * (CG - 1) * KS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int cg = 0; cg < CG; ++cg) o[cg][nb] = mfma16(vf[nb], pf[cg], o[cg][nb]);
#pragma unroll
        for (int cg = 0; cg < CG; ++cg) total[cg] = mfma16(ones, pf[cg], total[cg]);
        maxima(p + 1, sn, masked_tag);
#pragma unroll
        for (int g = 0; g < CG * (NB + 1); ++g) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x402, 4, 0);
        }
        // the running maximum moves rarely once a few pages are in: rescale O only when some column's did
        if (__builtin_amdgcn_ballot_w64(alpha[0] != 1.f || alpha[CG - 1] != 1.f) != 0) {
#pragma unroll
            for (int cg = 0; cg < CG; ++cg) {
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) o[cg][nb] *= alpha[cg];
                total[cg] *= alpha[cg];
            }
        }
    };
    f32x4 s0[CG][2], s1[CG][2];
    if (pages > 2)
        page_barrier(std::integral_constant<int, 2>{});
    else if (pages > 1)
        page_barrier(std::integral_constant<int, 1>{});
    else
        page_barrier(std::integral_constant<int, 0>{});
    scores(0, s0);
    maxima(0, s0, std::true_type{});  // (nothing to rescale yet)
    auto arrive = [&](int p) {
        page_barrier(std::integral_constant<int, 1>{});  // page p + 1 is there, the buffer of page p - 1 free
        page_load(next, (p + 3) & 3);
        next = page_number(p + 4);
    };
    // Interior pages (every key of the next one visible to every column of the wave) take the mask-free form, two at a time; a wave
    // meets at most ceil(32 columns / 32) + 1 diagonal pages per tile.  (Loops of their own: the waves of a block only have to meet at
    // the same number of barriers.)
    int p = 0;
    for (const int interior = min(wave_kmin >> 5, pages) - 2; p < interior; p += 2) {
        arrive(p);
        attend(p, s0, s1, std::false_type{});
        arrive(p + 1);
        attend(p + 1, s1, s0, std::false_type{});
    }
    for (const int own_pages = (wave_kmax + 31) >> 5; p < pages; ++p) {
        if (p + 2 < pages)  // (past the last page nothing is asked for: a short context has few pages to hide that behind)
            page_barrier(std::integral_constant<int, 1>{});
        else
            page_barrier(std::integral_constant<int, 0>{});
        if (p + 3 < pages) {
            page_load(next, (p + 3) & 3);
            next = page_number(p + 4);
        }
        if (p >= own_pages) continue;
        attend(p, s0, s1, std::true_type{});
#pragma unroll
        for (int cg = 0; cg < CG; ++cg)
#pragma unroll
            for (int t = 0; t < 2; ++t) s0[cg][t] = s1[cg][t];
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no direct load may still be on its way to LDS when the block ends

    // ---- epilogue: O^T[d][col] -> out[token][head][d]: a lane has four neighbours of a row, four lanes 32 bytes of it -----------------
    // (through LDS for 16-byte pieces: 3 - 5 % slower)
    using V4 = typename VecT<T>::x4;
#pragma unroll
    for (int cg = 0; cg < CG; ++cg) {
        if (!col_valid[cg]) continue;
        const float ls = total[cg][0];  // every lane of a column holds the column's normaliser
        const float inv = ls > 0.f ? 1.f / ls : 0.f;
        const int64_t tok = q0 + t0 + tq[cg];
        T* dst = reinterpret_cast<T*>(a.out) + tok * a.ld_out + head * D + c * 4;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            V4 v;
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = from_f32<T>(o[cg][nb][r] * inv);
            if (a.out_frag)
                *reinterpret_cast<V4*>(reinterpret_cast<T*>(a.out) + xf_off(tok, head * D + c * 4 + nb * 16, a.ld_out)) = v;
            else
                *reinterpret_cast<V4*>(dst + nb * 16) = v;
        }
    }
}

}  // namespace

int tgis_launch_attn_prefill(const AttnArgs& a, int64_t B, int Hkv, int D, int64_t max_q_len, int dtype, bool rows, hipStream_t st, const void* cos,
                             const void* sin, const int32_t* positions) {
    TGIS_CHECK_ARG(cdiv64(max_q_len, a.TQ * 4) <= 2147483647LL && (int64_t)Hkv * a.HC <= 65535 && B <= 65535, "tgis_attn_paged: grid too large");
    const int64_t groups = (int64_t)Hkv * a.HC * B;
    // Tiles of 128 columns, or of 64 where those would leave part of the chip idle: of the 512 blocks that are resident at once a quarter may
    // be missing at D 128 (us, 128 / 64).  D 128: 1 x 100 tokens, 32 heads 8.5 / 6.3; 1 x 1000 30.8 / 27.7; 1 x 512, 64 heads on 8 19.1 / 15.7;
    // 375 tiles, 1 x 1000, 48 on 1 43.7 / 31.5; from 384 on 12 x 65, 32 heads 9.6 / 10.8; 48 x 20, 32 on 8 8.0 / 9.6; 12 x 100, 48 on 1 12.9 /
    // 14.8; 32 x 33 10.7 / 11.1; 8 x 100, 64 on 8 12.8 / 13.8 (4 x 300, 32 heads 18.5 / 16.9; 24 x 20, 64 on 8 9.6 / 8.9); 16 x 1008 300 / 337.
    // D 64: 1 x 1500, 32 on 4 40 / 30; 24 x 33 6.6 / 5.0; 384 tiles, 32 x 33 6.7 / 5.6; 512, 64 x 33, 16 on 8 6.1 / 6.5.
    int cg = groups * cdiv64(max_q_len, a.TQ * 8) < (D == 128 ? 384 : 512) ? 1 : 2;
    if (const char* e = getenv("TGIS_PREFILL_CG")) cg = atoi(e) == 1 ? 1 : 2;  // tuning and test hook
    const int64_t q_tiles = cdiv64(max_q_len, a.TQ * 4 * cg);
    AttnPrefillArgs dealt{a, cos, sin, positions};
    dealt.xcd_remap = groups % 8 == 0 && (double)q_tiles * groups <= 2147483647.0;
    dim3 grid((unsigned)q_tiles, (unsigned)(Hkv * a.HC), (unsigned)B);
    const size_t lds = (size_t)PREFILL_RING * 2 * 32 * D * 2;  // buffers of (K page + V page)
#define TGIS_PREFILL_LAUNCH(T, DD, R)                                                                             \
    do {                                                                                                          \
        if (cg == 1)                                                                                              \
            hipLaunchKernelGGL((attn_prefill_kernel<T, DD, R, 1>), grid, dim3(256), lds, st, dealt);              \
        else                                                                                                      \
            hipLaunchKernelGGL((attn_prefill_kernel<T, DD, R, 2>), grid, dim3(256), lds, st, dealt);              \
    } while (0)
#define TGIS_PREFILL_WIDTH(T, R) do { if (D == 128) TGIS_PREFILL_LAUNCH(T, 128, R); else TGIS_PREFILL_LAUNCH(T, 64, R); } while (0)
    if (dtype == TGIS_F16) {
        if (rows) TGIS_PREFILL_WIDTH(f16, true); else TGIS_PREFILL_WIDTH(f16, false);
    } else {
        if (rows) TGIS_PREFILL_WIDTH(bf16, true); else TGIS_PREFILL_WIDTH(bf16, false);
    }
#undef TGIS_PREFILL_WIDTH
#undef TGIS_PREFILL_LAUNCH
    TGIS_CHECK_LAUNCH();
    return TGIS_OK;
}
