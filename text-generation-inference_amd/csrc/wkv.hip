// Linear-recurrence ("wkv", RWKV-style) time mixing with state slots:
//   token shift   mix_s[t] = h[t] + (h[t-1] - h[t]) * mu_s           (h[-1] of a step's first token comes from the slot)
//   decay         log w[t] = -exp(w0 + W2 tanh(a[t]))                 (a = the rank-reduced projection of mix_w, done by a GEMM)
//   recurrence    o[t] = (S + diag(u) k[t] v[t]^T)^T r[t];   S <- diag(w[t]) S + k[t] v[t]^T      per head, S in fp32
//   output        o / rms(o) per head, * gain * silu(gate)
// State per slot: S[head][key channel][value channel] (fp32) and the last token's mixer input (fp32).  A sequence whose
// step starts at position 0 starts from zeros whatever its slot held before: slots need no clearing when they change hands.
#include "common.h"
#include <algorithm>
#include <type_traits>
#include "wave_dpp.h"

namespace {

template <typename T> __device__ __forceinline__ float ldf(const T* p) { return (float)*p; }

__device__ __forceinline__ int seq_of_token(const int32_t* __restrict__ cu_q, int B, int t) {
    int lo = 0, hi = B;
    while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if (cu_q[mid] <= t) lo = mid; else hi = mid;
    }
    return lo;
}

// grid (token, block of 256 x VEC columns); out[s][t][c], s < NM.  Bound by its writes (one fp32 row in, NM two-byte rows out): VEC 4
// stores 8 or 16 bytes per thread (4096 x 2048, five mixes: 47 -> 29 us), 1 is for widths that are not multiples of 4 and for small steps,
// where it is more workgroups (us, VEC 1 / 4: 1 x 2048 2.8 / 3.0, 64 x 2048 2.9 / 3.1, 128 x 2048 3.4 / 3.3, 300 x 2048 5.4 / 4.7).
template <typename T, int VEC>
__global__ __launch_bounds__(256) void token_shift_mix_kernel(const float* __restrict__ h, const float* __restrict__ shift_state,
                                                              const int32_t* __restrict__ state_slots, const int32_t* __restrict__ cu_q,
                                                              const int32_t* __restrict__ positions, int B, const float* __restrict__ mu,
                                                              int NM, T* __restrict__ out, int64_t Ttot, int64_t W) {
    typedef float F __attribute__((ext_vector_type(VEC)));
    typedef T TV __attribute__((ext_vector_type(VEC)));
    const int t = blockIdx.x;
    const int64_t c = ((int64_t)blockIdx.y * blockDim.x + threadIdx.x) * VEC;
    if (c >= W) return;
    const int b = seq_of_token(cu_q, B, t);
    const bool first = t == cu_q[b];
    const bool fresh = first && positions[t] == 0;
    const float* prev = first ? shift_state + (int64_t)state_slots[b] * W : h + (int64_t)(t - 1) * W;
    const F x = *reinterpret_cast<const F*>(h + (int64_t)t * W + c);
    F d = *reinterpret_cast<const F*>(prev + c);
    if (fresh) d = F(0.f);
    d -= x;
    for (int s = 0; s < NM; ++s) {
        const F m = x + d * *reinterpret_cast<const F*>(mu + (int64_t)s * W + c);
        TV o;
#pragma unroll
        for (int e = 0; e < VEC; ++e) o[e] = (T)m[e];
        *reinterpret_cast<TV*>(out + ((int64_t)s * Ttot + t) * W + c) = o;
    }
}

// grid (TB tokens, 256-channel block): logw[t][c] = -exp(w0[c] + sum_r tanh(a[t][r]) * w2t[r][c])
// TB tokens share a read of w2t's columns: with one token per workgroup a 4 x 1024-token step reads the 512 KiB matrix 4096 times from
// L2 (rank 64, 4096 x 2048: 79 -> 39 us).  TB 8 from 1024 tokens on where that leaves a workgroup per CU (1024 x 512, rank 64: 7.1 / 7.0; 1024 x
// 256 5.5 / 6.8); else single tokens keep the chip filled.
template <typename T, int TB>
__global__ __launch_bounds__(256) void wkv_decay_kernel(const T* __restrict__ a, int64_t ld_a, const float* __restrict__ w2t,
                                                        const float* __restrict__ w0, float* __restrict__ logw, int R, int64_t C,
                                                        int64_t Ttot) {
    extern __shared__ float th[];  // [R][TB]
    const int64_t t0 = (int64_t)blockIdx.x * TB;
    const int n = (int)min((int64_t)TB, Ttot - t0);
    for (int i = threadIdx.x; i < R * TB; i += blockDim.x) {
        const int t = TB == 1 ? 0 : i / R, rr = i - t * R;
        th[rr * TB + t] = t < n ? tanhf(ldf(a + (t0 + t) * ld_a + rr)) : 0.f;
    }
    __syncthreads();
    const int64_t c = (int64_t)blockIdx.y * blockDim.x + threadIdx.x;
    if (c >= C) return;
    float z[TB];
    const float z0 = w0[c];
#pragma unroll
    for (int t = 0; t < TB; ++t) z[t] = z0;
#pragma unroll (TB == 1 ? 8 : 16)
    for (int rr = 0; rr < R; ++rr) {
        const float w = w2t[(int64_t)rr * C + c];
#pragma unroll
        for (int t = 0; t < TB; ++t) z[t] += th[rr * TB + t] * w;
    }
#pragma unroll
    for (int t = 0; t < TB; ++t)
        if (t < n) logw[(t0 + t) * C + c] = -expf(z[t]);
}

// The same for long steps as a product on the fp32 matrix instruction (16x16x4): a workgroup has 64 tokens x 256 channels, wave w its
// channels 32 w .. + 31; 64 ranks at a time, w2t's rows go straight to the B operand and are on their way while tanh(a) is staged in LDS.
// Eight tokens per read of w2t's columns were bound by those reads from L2 (4096 x 2048, rank 64: 41 us; 23 in this form, of which the
// matrix instruction needs 7 and the tanh of each of the eight column blocks 2).  Two workgroups a CU: 25 us with one.
constexpr int DECAY_TOKENS = 64, DECAY_COLS = 256, DECAY_RANKS = 64;

template <typename T>
__global__ __launch_bounds__(512, 4) void wkv_decay_tiles_kernel(const T* __restrict__ a, int64_t ld_a, const float* __restrict__ w2t,
                                                              const float* __restrict__ w0, float* __restrict__ logw, int R, int64_t C,
                                                              int64_t Ttot) {
    __shared__ float th[DECAY_TOKENS][DECAY_RANKS + 4];
    constexpr int STEPS = DECAY_RANKS / 4, PER = DECAY_TOKENS / 8;
    const int64_t t0 = (int64_t)blockIdx.x * DECAY_TOKENS;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lq = lane >> 4, lc = lane & 15;
    const int64_t c0 = (int64_t)blockIdx.y * DECAY_COLS + wave * 32 + lc;
    bool in[2];
    f32x4 z[4][2];
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
        in[ct] = c0 + 16 * ct < C;
        const float z0 = in[ct] ? w0[c0 + 16 * ct] : 0.f;
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) z[rt][ct] = f32x4{z0, z0, z0, z0};
    }
    for (int r0 = 0; r0 < R; r0 += DECAY_RANKS) {
        float x[PER], b[STEPS][2];
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int64_t t = t0 + wave + 8 * i;
            x[i] = (r0 + lane < R && t < Ttot) ? ldf(a + t * ld_a + r0 + lane) : 0.f;
        }
#pragma unroll
        for (int k = 0; k < STEPS; ++k)
#pragma unroll
            for (int ct = 0; ct < 2; ++ct)
                b[k][ct] = (in[ct] && r0 + 4 * k + lq < R) ? w2t[(int64_t)(r0 + 4 * k + lq) * C + c0 + 16 * ct] : 0.f;
#pragma unroll
        for (int i = 0; i < PER; ++i) th[wave + 8 * i][lane] = tanhf(x[i]);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < STEPS; ++k) {
            if (r0 + 4 * k >= R) break;
#pragma unroll
            for (int rt = 0; rt < 4; ++rt) {
                const float y = th[16 * rt + lc][4 * k + lq];
#pragma unroll
                for (int ct = 0; ct < 2; ++ct) z[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(y, b[k][ct], z[rt][ct], 0, 0, 0);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int64_t t = t0 + 16 * rt + 4 * lq + e;
#pragma unroll
            for (int ct = 0; ct < 2; ++ct)
                if (t < Ttot && in[ct]) logw[t * C + c0 + 16 * ct] = -expf(z[rt][ct][e]);
        }
}

// One workgroup per (sequence, head) = four thread groups: thread (q, j) owns value channel j and keeps the rows
// i in [q DQ, (q + 1) DQ) of column j of S in registers (rows of S evolve independently of each other, so the four groups
// never have to meet inside a token: each leaves its part of o in LDS and the parts are added once per chunk).  Tokens are
// staged through LDS CH at a time; all threads of a wave read the same r / k / w element at the same time (LDS broadcast).
// The next chunk's r, k, v, gate and log-decay are fetched into registers while the current one is computed.
constexpr int CH = 16;
constexpr int IS = 4;  // row groups

template <typename T, int DMAX>
__global__ __launch_bounds__((DMAX < 64 ? 64 : DMAX) * IS) void wkv_scan_kernel(
    const T* __restrict__ r, const T* __restrict__ k, const T* __restrict__ v, const T* __restrict__ gate, int64_t ld,
    const float* __restrict__ logw, const float* __restrict__ u, const float* __restrict__ gain, float* __restrict__ state,
    float* __restrict__ shift_state, const float* __restrict__ h, int64_t W, const int32_t* __restrict__ state_slots,
    const int32_t* __restrict__ cu_q, const int32_t* __restrict__ positions, T* __restrict__ out, int64_t ld_out, int H, int d,
    float eps) {
    constexpr int NJ = DMAX < 64 ? 64 : DMAX;  // threads per row group (whole waves)
    constexpr int NT = NJ * IS;
    constexpr int DQ = DMAX / IS;
    constexpr int PER = (CH * DMAX + NT - 1) / NT;
    __shared__ float rr[CH][DMAX], kk[CH][DMAX], ww[CH][DMAX], vv[CH][DMAX], gg[CH][DMAX], oo[IS][CH][DMAX], us[DMAX];
    const int b = blockIdx.x, head = blockIdx.y;
    const int tid = threadIdx.x;
    const int q = tid / NJ, j = tid % NJ;
    const int t0 = cu_q[b], t1 = cu_q[b + 1];
    if (t1 <= t0) return;
    const int64_t slot = state_slots[b];
    const bool fresh = positions[t0] == 0;
    float* Sg = state + ((slot * H + head) * d) * (int64_t)d;  // [i][j]
    float S[DQ];
#pragma unroll
    for (int ii = 0; ii < DQ; ++ii) {
        const int i = q * DQ + ii;
        S[ii] = (!fresh && i < d && j < d) ? Sg[(int64_t)i * d + j] : 0.f;
    }
    if (tid < DMAX) us[tid] = tid < d ? u[head * d + tid] : 0.f;
    const int64_t col0 = (int64_t)head * d;
    const int64_t C = (int64_t)H * d;
    float pr[PER], pk[PER], pv[PER], pg[PER], pw[PER];
    auto fetch = [&](int tc) {
        const int n = min(CH, t1 - tc);
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int idx = tid + e * NT, tt = idx / DMAX, i = idx % DMAX;
            const bool ok = tt < n && i < d;
            const int64_t at = (int64_t)(tc + tt) * ld + col0 + i;
            pr[e] = ok ? ldf(r + at) : 0.f;
            pk[e] = ok ? ldf(k + at) : 0.f;
            pv[e] = ok ? ldf(v + at) : 0.f;
            pg[e] = ok ? ldf(gate + at) : 0.f;
            pw[e] = ok ? logw[(int64_t)(tc + tt) * C + col0 + i] : 0.f;
        }
    };
    fetch(t0);
    for (int tc = t0; tc < t1; tc += CH) {
        const int n = min(CH, t1 - tc);
        __syncthreads();  // the previous chunk is consumed
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int idx = tid + e * NT, tt = idx / DMAX, i = idx % DMAX;
            if (tt < CH) {
                rr[tt][i] = pr[e];
                kk[tt][i] = pk[e];
                vv[tt][i] = pv[e];
                gg[tt][i] = pg[e];
                ww[tt][i] = expf(pw[e]);
            }
        }
        __syncthreads();
        if (tc + CH < t1) fetch(tc + CH);
        const int jj = j < DMAX ? j : 0;
        for (int tt = 0; tt < n; ++tt) {
            const float vj = vv[tt][jj];
            float a = 0.f, bonus = 0.f;
#pragma unroll
            for (int ii = 0; ii < DQ; ++ii) {
                const int i = q * DQ + ii;
                const float ri = rr[tt][i], ki = kk[tt][i];
                a += ri * S[ii];
                bonus += ri * us[i] * ki;
                S[ii] = ww[tt][i] * S[ii] + ki * vj;
            }
            if (j < DMAX) oo[q][tt][j] = a + bonus * vj;
        }
        __syncthreads();
        // the row groups' parts are added; per-head unit norm, gain, gate: one wave per token
        const int wave = tid >> 6, lane = tid & 63, nw = NT >> 6;
        for (int tt = wave; tt < n; tt += nw) {
            float ov[(DMAX + 63) / 64];
            float ss = 0.f;
#pragma unroll
            for (int cc = 0; cc < (DMAX + 63) / 64; ++cc) {
                const int c = lane + 64 * cc;
                float o = 0.f;
                if (c < d) {
#pragma unroll
                    for (int g4 = 0; g4 < IS; ++g4) o += oo[g4][tt][c];
                }
                ov[cc] = o;
                ss += o * o;
            }
            ss = wave_sum(ss);
            const float rinv = 1.0f / sqrtf(ss / (float)d + eps);
#pragma unroll
            for (int cc = 0; cc < (DMAX + 63) / 64; ++cc) {
                const int c = lane + 64 * cc;
                if (c < d) {
                    const float gt = gg[tt][c];
                    out[(int64_t)(tc + tt) * ld_out + col0 + c] = (T)(ov[cc] * rinv * gain[col0 + c] * (gt / (1.f + expf(-gt))));
                }
            }
        }
    }
    if (j < d) {
#pragma unroll
        for (int ii = 0; ii < DQ; ++ii) {
            const int i = q * DQ + ii;
            if (i < d) Sg[(int64_t)i * d + j] = S[ii];
        }
    }
    if (head == 0) {
        const float* last = h + (int64_t)(t1 - 1) * W;
        float* dst = shift_state + slot * W;
        for (int64_t c = tid; c < W; c += NT) dst[c] = last[c];
    }
}

// The same recurrence 16 tokens at a time, for head widths that are multiples of 4 and rows of aligned groups of four elements.
//
// A token-by-token scan is a serial chain of 0.7 us per token at d = 64 (LDS round trips and 80 dependent-ish vector instructions), on
// one workgroup per (sequence, head).  Over a chunk the state is only needed twice,
//   O = R' S0 + A V          R'_t = r_t * prod_{x < t} w_x          A[t][s] = sum_i r_t[i] k_s[i] prod_{s < x < t} w_x[i], A[t][t] = r u k
//   S = diag(E) S0 + K'^T V  E = prod_x w_x                         K'_s = k_s * prod_{x > s} w_x
// four products that go through the fp32 matrix instruction (16x16x4), 36 of them per wave and chunk at d = 64.
//   * Half of the waves ("makers") stage chunk c + 1 and form its A, R', K' and E while the other half ("holders") run chunk c's
//     products and finish its output: only the holders' part is a chain from chunk to chunk.
//   * The state stays in the holders' accumulators from chunk to chunk: holder w has columns 16 w .. 16 w + 15, register r of tile
//     `it` in lane l is row 16 it + 4 (l / 16) + r, which is also the B operand of a k-step over the rows {16 it + 4 q + r, q = 0 .. 3}.
//   * Decays are only ever multiplied, in the order of time (a thread per (token, four channels) walks the chunk and keeps its key's
//     decayed value), never divided or formed as differences of logarithms: products that underflow do so as in the scan, and the
//     error is the scan's.  A's sums over channels are a reduce-scatter over the token's lanes, 15 moves for 16 sums.
// A sequence that brings fewer than TOKENWISE tokens (decode) is bound by reading and writing its state: it is walked token by token
// with the state spread over all threads in 16-byte pieces.
// 4 x 1024 tokens, 32 heads of 64, bf16: 697 us for the token-by-token scan, 409 us with one set of waves doing both halves' work, 162 us
// in this form (2.5 us per chunk: the makers' walk through the chunk, 21 vector instructions per token, is the longer half), 84 us in segments.
constexpr int CHUNK = 16;
constexpr int TOKENWISE = 5;

// Long runs on few (sequence, head) pairs are a chain of 2.5 us per 16 tokens on a part of the chip (4 x 1024 tokens, 32 heads: 128 blocks).
// They are cut into segments that are walked side by side: wkv_segment_kernel forms what each segment
// but the last adds to the state and the product of its decays, and a segment of wkv_chunk_kernel takes its state from the records of the
// segments in front of it.  Record 0 of a pair is the state in front of the step (the last segment overwrites its slot), record x + 1 is
// segment x's: [D][D] and [D] floats.  The last segment of the grid takes all that is left of a run.
constexpr __host__ __device__ int record_floats(int D) { return D * D + D; }
__device__ __forceinline__ int segments_of(int tokens, int seg_len, int most) { return min((tokens + seg_len - 1) / seg_len, most); }

// grid (sequence, head, segment): S = sum_s (k_s prod_{x > s} w_x) v_s^T over the segment's tokens, E = prod_x w_x.  SUB tokens at a time,
// from the last to the first: a thread has one channel of SUB / 4 of them, decays its keys behind each other, and the four groups of a
// channel meet in LDS; then wave w adds its 16 columns on the fp32 matrix instruction.  Decays are multiplied, as in the chunks.
template <typename T, int D>
__global__ __launch_bounds__(4 * D) void wkv_segment_kernel(
    const T* __restrict__ k, const T* __restrict__ v, int64_t ld, const float* __restrict__ logw, const float* __restrict__ state,
    const int32_t* __restrict__ state_slots, const int32_t* __restrict__ cu_q, const int32_t* __restrict__ positions, int H, int d,
    float* __restrict__ records, int seg_len) {
    constexpr int SUB = D > 64 ? 32 : 64, PT = SUB / 4, NI = D / 16, SV = D + 16;
    __shared__ float kd[SUB][SV], vv[SUB][SV], through[4][D];
    const int b = blockIdx.x, head = blockIdx.y, seg = blockIdx.z;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int run0 = cu_q[b], run1 = cu_q[b + 1];
    const int most = gridDim.z + 1;
    if (seg + 1 >= segments_of(run1 - run0, seg_len, most)) return;
    float* rec = records + (((int64_t)b * H + head) * most + seg + 1) * record_floats(D);
    const int64_t col0 = (int64_t)head * d, C = (int64_t)H * d;
    if (seg == 0) {
        const float* Sg = state + ((state_slots[b] * (int64_t)H + head) * d) * (int64_t)d;
        const bool fresh = positions[run0] == 0;
        for (int x = tid; x < D * D; x += 4 * D) {
            const int i = x / D, j = x % D;
            rec[x - record_floats(D)] = (!fresh && i < d && j < d) ? Sg[(int64_t)i * d + j] : 0.f;
        }
    }
    const int t0 = run0 + seg * seg_len;
    const int ch = tid % D, group = tid / D;
    const bool mine = ch < d;
    T pk[PT], pv[PT];
    float pw[PT];
    auto fetch = [&](int sub) {
#pragma unroll
        for (int x = 0; x < PT; ++x) {
            const int64_t t = t0 + sub * SUB + group * PT + x;
            pk[x] = mine ? k[t * ld + col0 + ch] : (T)0.f;
            pv[x] = mine ? v[t * ld + col0 + ch] : (T)0.f;
            pw[x] = mine ? logw[t * C + col0 + ch] : 0.f;
        }
    };
    const int lq = lane >> 4, lc = lane & 15, j = 16 * wave + lc;
    f32x4 S[NI];
#pragma unroll
    for (int it = 0; it < NI; ++it) S[it] = f32x4{0.f, 0.f, 0.f, 0.f};
    float behind = 1.f;  // the decays of everything behind this part
    fetch(seg_len / SUB - 1);
    for (int sub = seg_len / SUB - 1; sub >= 0; --sub) {
        float key[PT], y = 1.f;
#pragma unroll
        for (int x = PT - 1; x >= 0; --x) {
            key[x] = (float)pk[x] * y;
            y *= expf(pw[x]);
        }
        through[group][ch] = y;
#pragma unroll
        for (int x = 0; x < PT; ++x) vv[group * PT + x][ch] = (float)pv[x];
        __syncthreads();
        if (sub > 0) fetch(sub - 1);
        float later = behind;
#pragma unroll
        for (int g = 3; g >= 0; --g) {
            const float z = through[g][ch];
            if (g > group) later *= z;
            behind *= z;
        }
#pragma unroll
        for (int x = 0; x < PT; ++x) kd[group * PT + x][ch] = key[x] * later;
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < SUB / 4; ++ks) {
            const float vb = vv[4 * ks + lq][j];
#pragma unroll
            for (int it = 0; it < NI; ++it) S[it] = __builtin_amdgcn_mfma_f32_16x16x4f32(kd[4 * ks + lq][16 * it + lc], vb, S[it], 0, 0, 0);
        }
        __syncthreads();
    }
#pragma unroll
    for (int it = 0; it < NI; ++it)
#pragma unroll
        for (int e = 0; e < 4; ++e) rec[(16 * it + 4 * lq + e) * D + j] = S[it][e];
    if (group == 0) rec[D * D + ch] = behind;
}

template <typename T, int D, bool SEGMENTS>
__global__ __launch_bounds__(8 * D, SEGMENTS && D == 64 ? 4 : 1) void wkv_chunk_kernel(
    const T* __restrict__ r, const T* __restrict__ k, const T* __restrict__ v, const T* __restrict__ gate, int64_t ld,
    const float* __restrict__ logw, const float* __restrict__ u, const float* __restrict__ gain, float* __restrict__ state,
    float* __restrict__ shift_state, const float* __restrict__ h, int64_t W, const int32_t* __restrict__ state_slots,
    const int32_t* __restrict__ cu_q, const int32_t* __restrict__ positions, T* __restrict__ out, int64_t ld_out, int H, int d,
    float eps, const float* __restrict__ records, int seg_len) {
    typedef T T4 __attribute__((ext_vector_type(4)));
    constexpr int NT = 8 * D, NH = NT / 2;  // threads, threads per half
    constexpr int L = D / 4;     // lanes per token
    constexpr int NI = D / 16;   // row tiles of the state
    constexpr int PRE = D > 64 || (SEGMENTS && D == 64) ? 2 : 8;  // (1024 threads on a CU have half the registers)
    constexpr int SV = D + 16;   // row stride of operands read as [4 rows][16 columns]: four rows cover the 64 banks
    constexpr int SR = D + 4;    // row stride of operands read as [16 rows][4 columns]
    __shared__ __attribute__((aligned(16))) float rr[CHUNK][D], ww[CHUNK][D], oo[CHUNK][SR];
    struct Operands {
        float vv[2][CHUNK][SV], kd[2][CHUNK][SV], rp[2][CHUNK][SR], aa[2][CHUNK][CHUNK + 4], ee[2][D];
    };
    __shared__ __attribute__((aligned(16))) Operands sm;
    auto &vv = sm.vv, &kd = sm.kd;
    auto &rp = sm.rp;
    auto &aa = sm.aa;
    auto &ee = sm.ee;
    const int b = blockIdx.x, head = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63;
    int t0 = cu_q[b], t1 = cu_q[b + 1];
    if (t1 <= t0) return;
    const int64_t slot = state_slots[b];
    const bool fresh = positions[t0] == 0;
    const int segs = SEGMENTS ? segments_of(t1 - t0, seg_len, gridDim.z) : 1, seg = SEGMENTS ? blockIdx.z : 0;
    if (seg >= segs) return;
    t0 += seg * seg_len;
    if (seg + 1 < segs) t1 = t0 + seg_len;
    const float* rec = SEGMENTS ? records + ((int64_t)b * H + head) * gridDim.z * record_floats(D) : nullptr;
    const int64_t col0 = (int64_t)head * d, C = (int64_t)H * d;
    float* Sg = state + ((slot * H + head) * d) * (int64_t)d;  // [i][j]
    const int half_tid = tid % NH;
    const int s = half_tid / L, c4 = (half_tid % L) * 4;  // token s of a chunk, channels c4 .. c4 + 3
    const bool mine = c4 < d;
    const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};
    auto raw4 = [&](const T* p, int t) -> T4 { return *reinterpret_cast<const T4*>(p + (int64_t)t * ld + col0 + c4); };
    auto wide4 = [](T4 x) -> f32x4 { return f32x4{(float)x[0], (float)x[1], (float)x[2], (float)x[3]}; };
    auto row4 = [&](const T* p, int t) -> f32x4 { return wide4(raw4(p, t)); };
    T4 none;
#pragma unroll
    for (int e = 0; e < 4; ++e) none[e] = (T)0.f;
    f32x4 g4 = zero4;
    if (mine) g4 = *reinterpret_cast<const f32x4*>(gain + col0 + c4);
    // per-head unit norm, gain, gate of token t (o4: its four channels; threads of the token's lanes together)
    auto finish = [&](f32x4 o4, f32x4 gt, int t, bool live) {
        float ss = o4[0] * o4[0] + o4[1] * o4[1] + o4[2] * o4[2] + o4[3] * o4[3];
        ss = sum_neighbours<(L < 16 ? L : 16)>(live ? ss : 0.f);
        if (L > 16) ss += __shfl_xor(ss, 16, 64);
        if (live && mine) {
            const float rinv = 1.0f / sqrtf(ss / (float)d + eps);
            T4 res;
#pragma unroll
            for (int e = 0; e < 4; ++e) res[e] = (T)(o4[e] * rinv * g4[e] * (gt[e] / (1.f + expf(-gt[e]))));
            *reinterpret_cast<T4*>(out + (int64_t)t * ld_out + col0 + c4) = res;
        }
    };
    if (head == 0 && seg + 1 == segs) {
        const float* last = h + (int64_t)(t1 - 1) * W;
        float* dst = shift_state + slot * W;
        for (int64_t c = tid; c < W; c += NT) dst[c] = last[c];
    }

    if (!SEGMENTS && t1 - t0 < TOKENWISE) {
        constexpr int RG = NT / L, RPT = D / RG;  // row groups, rows per thread: rows rg, rg + RG, ...
        const int n = t1 - t0, rg = tid / L;
        float(*parts)[TOKENWISE - 1][D] = reinterpret_cast<float(*)[TOKENWISE - 1][D]>(&sm);  // [waves][token][column]
        static_assert(sizeof(float) * (NT / 64) * (TOKENWISE - 1) * D <= sizeof(sm.vv) + sizeof(sm.kd), "the waves' parts of the output");
        f32x4 St[RPT];
#pragma unroll
        for (int x = 0; x < RPT; ++x) {
            const int i = rg + x * RG;
            St[x] = (!fresh && mine && i < d) ? *reinterpret_cast<const f32x4*>(Sg + (int64_t)i * d + c4) : zero4;
        }
        const f32x4 u4 = mine ? *reinterpret_cast<const f32x4*>(u + col0 + c4) : zero4;
        f32x4 vt[TOKENWISE - 1];
#pragma unroll
        for (int t = 0; t < TOKENWISE - 1; ++t) vt[t] = (mine && t < n) ? row4(v, t0 + t) : zero4;
        f32x4 gt = zero4;
        if (tid < NH && s < n && mine) gt = row4(gate, t0 + s);
        if (tid < NH && s < n) {
            f32x4 rc = zero4, kc = zero4, wc = zero4;
            if (mine) {
                rc = row4(r, t0 + s);
                kc = row4(k, t0 + s);
                wc = *reinterpret_cast<const f32x4*>(logw + (int64_t)(t0 + s) * C + col0 + c4);
            }
            float diag = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                diag += rc[e] * u4[e] * kc[e];
                wc[e] = expf(wc[e]);
            }
            *reinterpret_cast<f32x4*>(&rr[s][c4]) = rc;
            *reinterpret_cast<f32x4*>(&ww[s][c4]) = wc;
            *reinterpret_cast<f32x4*>(&rp[0][s][c4]) = kc;
            diag = sum_neighbours<(L < 16 ? L : 16)>(diag);
            if (L > 16) diag += __shfl_xor(diag, 16, 64);
            if (half_tid % L == 0) aa[0][s][0] = diag;
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < TOKENWISE - 1; ++t) {
            if (t >= n) break;
            f32x4 o4 = zero4;
#pragma unroll
            for (int x = 0; x < RPT; ++x) {
                const int i = rg + x * RG;
                const float ri = rr[t][i], wi = ww[t][i], ki = rp[0][t][i];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    o4[e] += ri * St[x][e];
                    St[x][e] = wi * St[x][e] + ki * vt[t][e];
                }
            }
            // the wave's row groups, then (below) the waves
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (L <= 8) o4[e] += __shfl_xor(o4[e], 8, 64);
                if (L <= 16) o4[e] += __shfl_xor(o4[e], 16, 64);
                o4[e] += __shfl_xor(o4[e], 32, 64);
            }
            if (lane < L) *reinterpret_cast<f32x4*>(&parts[tid >> 6][t][c4]) = o4;
        }
#pragma unroll
        for (int x = 0; x < RPT; ++x) {
            const int i = rg + x * RG;
            if (mine && i < d) *reinterpret_cast<f32x4*>(Sg + (int64_t)i * d + c4) = St[x];
        }
        __syncthreads();
        if (tid < NH) {
            f32x4 o4 = zero4;
            if (s < n && mine) {
                const f32x4 vs = row4(v, t0 + s);
                const float diag = aa[0][s][0];
#pragma unroll
                for (int w = 0; w < NT / 64; ++w) o4 += *reinterpret_cast<const f32x4*>(&parts[w][s][c4]);
#pragma unroll
                for (int e = 0; e < 4; ++e) o4[e] += diag * vs[e];
            }
            finish(o4, gt, t0 + s, s < n);
        }
        return;
    }

    const int wave = __builtin_amdgcn_readfirstlane(half_tid >> 6);
    const int chunks = (t1 - t0 + CHUNK - 1) / CHUNK;
    if (tid < NH) {  // ---- makers ----
        const int s_lo = wave * (64 / L), s_hi = s_lo + 64 / L - 1;
        const f32x4 u4 = mine ? *reinterpret_cast<const f32x4*>(u + col0 + c4) : zero4;
        T4 pr, pk, pv;  // as loaded: widening them here would wait for them here
        f32x4 pw;
        auto fetch = [&](int c) {
            const int t = t0 + c * CHUNK + s;
            pr = pk = pv = none;  // tokens past the end and padded channels: no key, no decay
            pw = zero4;
            if (mine && t < t1) {
                pr = raw4(r, t);
                pk = raw4(k, t);
                pv = raw4(v, t);
                pw = *reinterpret_cast<const f32x4*>(logw + (int64_t)t * C + col0 + c4);
            }
        };
        fetch(0);
        for (int c = 0; c <= chunks; ++c) {  // holders are one chunk behind
            const int buf = c & 1;
            const f32x4 rc = wide4(pr), kc = wide4(pk);
            float diag = 0.f;
            if (c < chunks) {
                f32x4 wc;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    wc[e] = expf(pw[e]);
                    diag += rc[e] * u4[e] * kc[e];
                }
                *reinterpret_cast<f32x4*>(&rr[s][c4]) = rc;
                *reinterpret_cast<f32x4*>(&ww[s][c4]) = wc;
                *reinterpret_cast<f32x4*>(&vv[buf][s][c4]) = wide4(pv);
            }
            __syncthreads();
            if (c < chunks) {
                if (c + 1 < chunks) fetch(c + 1);
                int own = s;  // (opaque: sixteen hoisted comparison masks would not fit the scalar registers)
                asm volatile("" : "+v"(own));
                float p[CHUNK];
                f32x4 x = zero4, y = {1.f, 1.f, 1.f, 1.f}, rd = zero4;
#pragma unroll
                for (int th = 0; th < CHUNK; th += PRE) {
                    f32x4 w4[PRE], r4[PRE];  // all LDS reads of PRE tokens in flight together
#pragma unroll
                    for (int t = 0; t < PRE; ++t) {
                        w4[t] = *reinterpret_cast<const f32x4*>(&ww[th + t][c4]);
                        r4[t] = *reinterpret_cast<const f32x4*>(&rr[th + t][c4]);
                    }
#pragma unroll
                    for (int t = 0; t < PRE; ++t) {
                        const int tt = th + t;
                        p[tt] = 0.f;
                        if (tt > s_hi) {  // x: the key of token s as token tt sees it
                            p[tt] = r4[t][0] * x[0] + r4[t][1] * x[1] + r4[t][2] * x[2] + r4[t][3] * x[3];
#pragma unroll
                            for (int e = 0; e < 4; ++e) x[e] *= w4[t][e];
                        } else {          // y: the decay of everything in front of token tt
                            if (tt >= s_lo) {
                                const bool at = tt == own;
                                const float q = r4[t][0] * x[0] + r4[t][1] * x[1] + r4[t][2] * x[2] + r4[t][3] * x[3];
                                p[tt] = at ? diag : q;
#pragma unroll
                                for (int e = 0; e < 4; ++e) {
                                    x[e] = at ? kc[e] : x[e] * w4[t][e];
                                    rd[e] = at ? rc[e] * y[e] : rd[e];
                                }
                            }
#pragma unroll
                            for (int e = 0; e < 4; ++e) y[e] *= w4[t][e];
                        }
                    }
                }
                if (s == CHUNK - 1) *reinterpret_cast<f32x4*>(&ee[buf][c4]) = y;
                *reinterpret_cast<f32x4*>(&rp[buf][s][c4]) = rd;
                *reinterpret_cast<f32x4*>(&kd[buf][s][c4]) = x;
                // sums over the token's lanes: a lane passes on the half of its sums that its partner keeps
                auto halve = [&](auto ctrl, auto width_, int bit) {
                    constexpr int width = decltype(width_)::value;
                    const bool upper = (lane & bit) != 0;
#pragma unroll
                    for (int i = 0; i < width; ++i) {
                        const float keep = upper ? p[width + i] : p[i], pass = upper ? p[i] : p[width + i];
                        p[i] = keep + moved<decltype(ctrl)::value>(0.f, pass);
                    }
                };
                constexpr int W0 = L >= 16 ? 8 : 16;
                using std::integral_constant;
                if constexpr (L >= 16) halve(integral_constant<int, 0x140>{}, integral_constant<int, 8>{}, 8);  // lane 15 - i of the row
                halve(integral_constant<int, 0x141>{}, integral_constant<int, W0 / 2>{}, 4);                    // lane 7 - i of the half row
                halve(integral_constant<int, 0x1B>{}, integral_constant<int, W0 / 4>{}, 2);                     // lane 3 - i of the quad
                halve(integral_constant<int, 0xB1>{}, integral_constant<int, W0 / 8>{}, 1);                     // lane ^ 1
                if (L > 16) p[0] += __shfl_xor(p[0], 16, 64);
                if (L >= 16) {
                    aa[buf][lane & 15][s] = p[0];
                } else {
                    aa[buf][2 * (lane & 7)][s] = p[0];
                    aa[buf][2 * (lane & 7) + 1][s] = p[1];
                }
            }
            __syncthreads();
        }
        return;
    }

    // ---- holders ----
    const int lq = lane >> 4, lc = lane & 15, j = 16 * wave + lc;
    f32x4 S[NI];
#pragma unroll
    for (int it = 0; it < NI; ++it)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int i = 16 * it + 4 * lq + e;
            if (SEGMENTS && segs > 1)
                S[it][e] = rec[i * D + j];
            else
                S[it][e] = (!fresh && i < d && j < d) ? Sg[(int64_t)i * d + j] : 0.f;
        }
    if (SEGMENTS) {
        for (int x = 1; x <= seg; ++x) {  // what the segments in front of this one make of the state
            rec += record_floats(D);
#pragma unroll
            for (int it = 0; it < NI; ++it) {
                const f32x4 e4 = *reinterpret_cast<const f32x4*>(rec + D * D + 16 * it + 4 * lq);
#pragma unroll
                for (int e = 0; e < 4; ++e) S[it][e] = e4[e] * S[it][e] + rec[(16 * it + 4 * lq + e) * D + j];
            }
        }
    }
    __syncthreads();
    __syncthreads();  // the makers' first chunk
    for (int c = 0; c < chunks; ++c) {
        const int buf = c & 1, t = t0 + c * CHUNK + s;
        T4 gt = none;
        if (mine && t < t1) gt = raw4(gate, t);
        float vb[4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) vb[ks] = vv[buf][4 * ks + lq][j];
        f32x4 s0 = zero4, s1 = zero4;
#pragma unroll
        for (int it = 0; it < NI; ++it) {
            const f32x4 a4 = *reinterpret_cast<const f32x4*>(&rp[buf][lc][16 * it + 4 * lq]);
            s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[0], S[it][0], s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[1], S[it][1], s1, 0, 0, 0);
            s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[2], S[it][2], s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[3], S[it][3], s1, 0, 0, 0);
        }
        f32x4 o0 = s0, o1 = s1;
#pragma unroll
        for (int ks = 0; ks < 4; ks += 2) {
            o0 = __builtin_amdgcn_mfma_f32_16x16x4f32(aa[buf][lc][4 * ks + lq], vb[ks], o0, 0, 0, 0);
            o1 = __builtin_amdgcn_mfma_f32_16x16x4f32(aa[buf][lc][4 * ks + 4 + lq], vb[ks + 1], o1, 0, 0, 0);
        }
        // A is zero past its diagonal, but 0 times a value that is not finite is no zero: such a value shows in every row of its column.
        // Then each token adds up only the values that it sees, and those in front of it stay what they are token by token.
        if (__builtin_amdgcn_ballot_w64(!(fabsf(o0[0] + o1[0]) < __builtin_inff())) != 0) {
            o0 = s0;
            o1 = s1;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                for (int x = 0; x <= 4 * lq + e; ++x) o0[e] += aa[buf][4 * lq + e][x] * vv[buf][x][j];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) oo[4 * lq + e][j] = o0[e] + o1[e];
        __syncthreads();
#pragma unroll
        for (int it = 0; it < NI; ++it) {
            S[it] *= *reinterpret_cast<const f32x4*>(&ee[buf][16 * it + 4 * lq]);
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
                S[it] = __builtin_amdgcn_mfma_f32_16x16x4f32(kd[buf][4 * ks + lq][16 * it + lc], vb[ks], S[it], 0, 0, 0);
        }
        finish(*reinterpret_cast<const f32x4*>(&oo[s][c4]), wide4(gt), t, t < t1);
        __syncthreads();
    }
    if (seg + 1 < segs) return;
#pragma unroll
    for (int it = 0; it < NI; ++it)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int i = 16 * it + 4 * lq + e;
            if (i < d && j < d) Sg[(int64_t)i * d + j] = S[it][e];
        }
}

// A decode step: the log-decay's second factor and the recurrence of the few tokens a sequence brings, in one launch.
//
// Bound by a chain of trips to memory (which sequence, its state and its rows, their answers) and the state's bytes; in the chunk kernel
// above a single token paid for that kernel's size, 52 KiB of LDS and eight waves with three barriers' worth of staging, and the decay for
// a launch of its own.  Here the state, the token's rows and the decay's weights are asked for together, each thread loads the rows of
// r, k and u that its state rows need, and the waves meet three times.  24 sequences, 32 heads of 64, rank 64, us: 18.0 + 4.9 / 10.5.
constexpr int STEP_THREADS = 256, STEP_WAVES = STEP_THREADS / 64, STEP_MAX_RANK = 1024;

template <typename T, int D>
__global__ __launch_bounds__(STEP_THREADS) void wkv_step_kernel(
    const T* __restrict__ r, const T* __restrict__ k, const T* __restrict__ v, const T* __restrict__ gate, const T* __restrict__ low,
    int64_t ld, int64_t ld_low, const float* __restrict__ w2t, const float* __restrict__ w0, int R, const float* __restrict__ u,
    const float* __restrict__ gain, float* __restrict__ state, float* __restrict__ shift_state, const float* __restrict__ h, int64_t W,
    const int32_t* __restrict__ state_slots, const int32_t* __restrict__ cu_q, const int32_t* __restrict__ positions, T* __restrict__ out,
    int64_t ld_out, int H, int d, float eps) {
    typedef T T4 __attribute__((ext_vector_type(4)));
    constexpr int L = D / 4, RG = STEP_THREADS / L, RPT = D / RG;  // lanes per state row, row groups, (neighbouring) rows per thread
    constexpr int P = STEP_THREADS / D, EARLY = 16;                // parts of the decay's sum; weights a thread asks for at once
    static_assert(RPT % 4 == 0, "rows of a thread come in fours");
    __shared__ float th[STEP_MAX_RANK], part[P][D], bonus_of[STEP_WAVES];
    __shared__ __attribute__((aligned(16))) float ww[D], o_of[STEP_WAVES][D];
    const int b = blockIdx.x, head = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int t0 = cu_q[b], t1 = cu_q[b + 1];
    const int64_t slot = state_slots[b];
    if (t1 <= t0) return;
    const int64_t col0 = (int64_t)head * d, C = (int64_t)H * d;
    float* Sg = state + ((slot * H + head) * d) * (int64_t)d;  // [i][j]
    const int c4 = (tid % L) * 4, i0 = tid / L * RPT;
    const bool mine = c4 < d;
    const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};
    f32x4 St[RPT], u4[RPT / 4], r4[RPT / 4], k4[RPT / 4];
#pragma unroll
    for (int x = 0; x < RPT; ++x) St[x] = (mine && i0 + x < d) ? *reinterpret_cast<const f32x4*>(Sg + (int64_t)(i0 + x) * d + c4) : zero4;
    auto wide4 = [](T4 x) -> f32x4 { return f32x4{(float)x[0], (float)x[1], (float)x[2], (float)x[3]}; };
    auto rows4 = [&](const T* p, int t, f32x4 (&dst)[RPT / 4]) {
#pragma unroll
        for (int y = 0; y < RPT / 4; ++y)
            dst[y] = i0 + 4 * y < d ? wide4(*reinterpret_cast<const T4*>(p + (int64_t)t * ld + col0 + i0 + 4 * y)) : zero4;
    };
#pragma unroll
    for (int y = 0; y < RPT / 4; ++y) u4[y] = i0 + 4 * y < d ? *reinterpret_cast<const f32x4*>(u + col0 + i0 + 4 * y) : zero4;
    const f32x4 g4 = mine ? *reinterpret_cast<const f32x4*>(gain + col0 + c4) : zero4;
    const int zc = tid % D, zp = tid / D, per = (R + P - 1) / P, za = zp * per, ze = min(R, za + per);  // this thread's part of the decay
    float wz[EARLY];
#pragma unroll
    for (int e = 0; e < EARLY; ++e) wz[e] = (zc < d && za + e < ze) ? w2t[(int64_t)(za + e) * C + col0 + zc] : 0.f;
    const float z0 = zc < d ? w0[col0 + zc] : 0.f;
    if (positions[t0] == 0) {
#pragma unroll
        for (int x = 0; x < RPT; ++x) St[x] = zero4;
    }
    for (int t = t0; t < t1; ++t) {
        rows4(r, t, r4);
        rows4(k, t, k4);
        f32x4 v4 = zero4, gt = zero4;
        if (mine) {
            v4 = wide4(*reinterpret_cast<const T4*>(v + (int64_t)t * ld + col0 + c4));
            gt = wide4(*reinterpret_cast<const T4*>(gate + (int64_t)t * ld + col0 + c4));
        }
        for (int i = tid; i < R; i += STEP_THREADS) th[i] = tanhf((float)low[(int64_t)t * ld_low + i]);
        __syncthreads();
        float z = 0.f;
#pragma unroll
        for (int e = 0; e < EARLY; ++e) z += (za + e < ze ? th[za + e] : 0.f) * wz[e];
        for (int i = za + EARLY; i < ze; ++i) z += zc < d ? th[i] * w2t[(int64_t)i * C + col0 + zc] : 0.f;
        part[zp][zc] = z;
        __syncthreads();
        if (zp == 0) {
            z = z0;
#pragma unroll
            for (int p = 0; p < P; ++p) z += part[p][zc];
            ww[zc] = expf(-expf(z));
        }
        __syncthreads();
        f32x4 o = zero4;
        float bonus = 0.f;
#pragma unroll
        for (int y = 0; y < RPT / 4; ++y) {
            const f32x4 w4 = *reinterpret_cast<const f32x4*>(&ww[i0 + 4 * y]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                f32x4& S = St[4 * y + e];
                bonus += r4[y][e] * u4[y][e] * k4[y][e];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    o[c] += r4[y][e] * S[c];
                    S[c] = w4[e] * S[c] + k4[y][e] * v4[c];
                }
            }
        }
#pragma unroll
        for (int far = L; far < 64; far *= 2) {
            bonus += __shfl_xor(bonus, far, 64);
#pragma unroll
            for (int c = 0; c < 4; ++c) o[c] += __shfl_xor(o[c], far, 64);
        }
        if (lane < L) *reinterpret_cast<f32x4*>(&o_of[wave][c4]) = o;
        if (lane == 0) bonus_of[wave] = bonus;
        __syncthreads();
        if (wave == 0) {  // (its lanes past the first L repeat them)
            o = zero4;
            bonus = 0.f;
#pragma unroll
            for (int p = 0; p < STEP_WAVES; ++p) {
                o += *reinterpret_cast<const f32x4*>(&o_of[p][c4]);
                bonus += bonus_of[p];
            }
            float ss = 0.f;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                o[c] += bonus * v4[c];
                ss += o[c] * o[c];
            }
            ss = sum_neighbours<16>(ss);
            if (L > 16) ss += __shfl_xor(ss, 16, 64);
            if (lane < L && mine) {
                const float rinv = 1.0f / sqrtf(ss / (float)d + eps);
                T4 res;
#pragma unroll
                for (int e = 0; e < 4; ++e) res[e] = (T)(o[e] * rinv * g4[e] * (gt[e] / (1.f + expf(-gt[e]))));
                *reinterpret_cast<T4*>(out + (int64_t)t * ld_out + col0 + c4) = res;
            }
        }
    }
    if (mine) {
#pragma unroll
        for (int x = 0; x < RPT; ++x)
            if (i0 + x < d) *reinterpret_cast<f32x4*>(Sg + (int64_t)(i0 + x) * d + c4) = St[x];
    }
    if (head == 0) {
        const float* last = h + (int64_t)(t1 - 1) * W;
        float* dst = shift_state + slot * W;
        for (int64_t c = tid; c < W; c += STEP_THREADS) dst[c] = last[c];
    }
}

// Steps whose longest run has a few tokens, or a few more than a chunk, with more blocks than a CU holds at once (its registers let it hold
// one of the chunk kernel up to d = 64, two up to 32; four of the token-by-token one), walk their tokens one by one.  us, token by token /
// chunks, d 64: 24 sequences x 32 heads of 1, 5, 8, 12, 16, 17, 20 tokens 9.9 / 12.2, 12.3 / 17.7, 13.9 / 17.8, 17.5 / 18.0, 20.9 / 19.1, 22.6 /
// 25.1, 24.6 / 25.2; 32 x 64 heads of 5 29.0 / 41.6; but 8 x 32 heads of 5 9.1 / 8.0.  d 32: 24 x 32 heads of 5, 12, 16, 17, 20 8.1 / 12.2, 11.2 /
// 12.4, 13.0 / 12.4, 14.2 / 17.1, 15.3 / 16.9; 16 x 32 of 5 7.5 / 7.6.  d 128, 32 x 16 heads of 5: by 1.15 in chunks.
bool runs_by_token(int64_t blocks, int d, int64_t max_q_len) {
    if (max_q_len < 1 || d > 64 || blocks <= (d <= 32 ? 512 : 256)) return false;
    return max_q_len <= CHUNK ? max_q_len <= (d <= 32 ? 12 : 10) : max_q_len <= (d <= 32 ? 20 : 17);
}

struct Segments {
    int count, tokens;
};
// As many segments as the chip takes blocks of the chunk kernel at once (two a CU up to d = 64, held to 128 registers there; one above), none
// shorter than what a block needs to come up.  us, one block per (sequence, head) / segments, bf16: d 64, 32 heads: 4 x 1024 tokens 162 / 84
// (4 segments; 6 of them 95), 1 x 1024 147 / 37, 1 x 4093 618 / 87, 1 x 256 41 / 25, 4 x 256 42 / 34, 8 x 512 82 / 80, 8 x 1024 160 / 143, 6 x 700
// 110 / 99; d 32: 4 x 1024, 32 heads 150 / 60; d 128, 16 heads: 4 x 1024 262 / 136 (8 segments 171), 1 x 2048 515 / 162, 8 x 1024 266 / 211.
Segments segments_for(int64_t blocks, int d, int64_t max_q_len) {
    const int64_t room = d <= 64 ? 512 : 256, least = d <= 64 ? 64 : 256;
    const int64_t most = std::min(std::min(room / blocks, max_q_len / least), (int64_t)16);
    if (most < 2) return {1, 0};
    const int64_t tokens = cdiv64(cdiv64(max_q_len, most), 64) * 64;
    return {(int)cdiv64(max_q_len, tokens), (int)tokens};
}

template <typename T>
int launch_scan(const void* r, const void* k, const void* v, const void* gate, int64_t ld, const float* logw, const float* u,
                const float* gain, float* state, float* shift_state, const float* h, int64_t W, const int32_t* slots,
                const int32_t* cu_q, const int32_t* positions, void* out, int64_t ld_out, int B, int H, int d, float eps,
                int64_t max_q_len, void* ws, hipStream_t st) {
    // the chunked form takes rows in groups of four elements (any head width that is a multiple of 4, aligned tensors)
    const size_t quad = 4 * sizeof(T);
    auto rows_of_four = [&](const void* p, int64_t stride) { return (uintptr_t)p % quad == 0 && stride % 4 == 0; };
    if (!runs_by_token((int64_t)B * H, d, max_q_len) && d % 4 == 0 && rows_of_four(r, ld) && rows_of_four(k, ld) && rows_of_four(v, ld) && rows_of_four(gate, ld) &&
        rows_of_four(out, ld_out) && (uintptr_t)logw % 16 == 0 && (uintptr_t)u % 16 == 0 && (uintptr_t)gain % 16 == 0 &&
        (uintptr_t)state % 16 == 0) {
        const Segments cut = segments_for((int64_t)B * H, d, max_q_len);
        float* records = cut.count > 1 ? (float*)ws : nullptr;
#define TGIS_WKV_CHUNKS(DM)                                                                                                       \
    do {                                                                                                                          \
        if (records) {                                                                                                            \
            hipLaunchKernelGGL((wkv_segment_kernel<T, DM>), dim3((unsigned)B, (unsigned)H, (unsigned)cut.count - 1), dim3(4 * DM), 0, st, \
                               (const T*)k, (const T*)v, ld, logw, state, slots, cu_q, positions, H, d, records, cut.tokens);    \
            hipLaunchKernelGGL((wkv_chunk_kernel<T, DM, true>), dim3((unsigned)B, (unsigned)H, (unsigned)cut.count), dim3(8 * DM), 0, st, \
                               (const T*)r, (const T*)k, (const T*)v, (const T*)gate, ld, logw, u, gain, state, shift_state, h, W, \
                               slots, cu_q, positions, (T*)out, ld_out, H, d, eps, records, cut.tokens);                         \
        } else {                                                                                                                  \
            hipLaunchKernelGGL((wkv_chunk_kernel<T, DM, false>), dim3((unsigned)B, (unsigned)H), dim3(8 * DM), 0, st, (const T*)r, \
                               (const T*)k, (const T*)v, (const T*)gate, ld, logw, u, gain, state, shift_state, h, W, slots, cu_q, \
                               positions, (T*)out, ld_out, H, d, eps, nullptr, 0);                                               \
        }                                                                                                                         \
    } while (0)
        if (d <= 32)
            TGIS_WKV_CHUNKS(32);
        else if (d <= 64)
            TGIS_WKV_CHUNKS(64);
        else
            TGIS_WKV_CHUNKS(128);
#undef TGIS_WKV_CHUNKS
        return 0;
    }
#define TGIS_WKV_LAUNCH(DM)                                                                                               \
    hipLaunchKernelGGL((wkv_scan_kernel<T, DM>), dim3((unsigned)B, (unsigned)H), dim3((DM < 64 ? 64 : DM) * IS), 0, st, (const T*)r, \
                       (const T*)k, (const T*)v, (const T*)gate, ld, logw, u, gain, state, shift_state, h, W, slots, cu_q,    \
                       positions, (T*)out, ld_out, H, d, eps)
    if (d <= 32)
        TGIS_WKV_LAUNCH(32);
    else if (d <= 64)
        TGIS_WKV_LAUNCH(64);
    else
        TGIS_WKV_LAUNCH(128);
#undef TGIS_WKV_LAUNCH
    return 0;
}

}  // namespace

static bool dtype3(int d) { return d == TGIS_F16 || d == TGIS_BF16 || d == TGIS_F32; }

extern "C" int tgis_token_shift_mix(const float* h, const float* shift_state, const int32_t* state_slots, const int32_t* cu_seqlens_q,
                                    const int32_t* positions, int64_t B, const float* mu, int num_mixes, void* out, int64_t T,
                                    int64_t W, int dtype, void* stream) {
    TGIS_CHECK_ARG(h && shift_state && state_slots && cu_seqlens_q && positions && mu && out, "tgis_token_shift_mix: null tensor");
    TGIS_CHECK_ARG(B >= 1 && num_mixes >= 1 && W >= 1 && dtype3(dtype), "tgis_token_shift_mix: bad arguments");
    if (T == 0) return TGIS_OK;
    hipStream_t st = (hipStream_t)stream;
    const bool vec = T * W >= 196608 && W % 4 == 0 && (uintptr_t)h % 16 == 0 && (uintptr_t)shift_state % 16 == 0 && (uintptr_t)mu % 16 == 0 &&
                     (uintptr_t)out % (dtype == TGIS_F32 ? 16 : 8) == 0;
    const dim3 grid((unsigned)T, (unsigned)cdiv64(W, vec ? 1024 : 256));
#define TGIS_SHIFT(TT)                                                                                                             \
    do {                                                                                                                           \
        if (vec)                                                                                                                   \
            hipLaunchKernelGGL((token_shift_mix_kernel<TT, 4>), grid, dim3(256), 0, st, h, shift_state, state_slots, cu_seqlens_q, \
                               positions, (int)B, mu, num_mixes, (TT*)out, T, W);                                                  \
        else                                                                                                                       \
            hipLaunchKernelGGL((token_shift_mix_kernel<TT, 1>), grid, dim3(256), 0, st, h, shift_state, state_slots, cu_seqlens_q, \
                               positions, (int)B, mu, num_mixes, (TT*)out, T, W);                                                  \
    } while (0)
    if (dtype == TGIS_F16)
        TGIS_SHIFT(f16);
    else if (dtype == TGIS_BF16)
        TGIS_SHIFT(bf16);
    else
        TGIS_SHIFT(float);
#undef TGIS_SHIFT
    TGIS_CHECK_LAUNCH();
    return TGIS_OK;
}

extern "C" int tgis_wkv_decay(const void* a, int64_t ld_a, const float* w2t, const float* w0, float* logw, int64_t T, int rank,
                              int64_t C, int dtype, void* stream) {
    TGIS_CHECK_ARG(a && w2t && w0 && logw && rank >= 1 && rank <= 8192 && C >= 1 && C <= 65535 * 256 && ld_a >= rank && dtype3(dtype), "tgis_wkv_decay: bad arguments");
    if (T == 0) return TGIS_OK;
    hipStream_t st = (hipStream_t)stream;
    const int64_t tiles = cdiv64(T, DECAY_TOKENS) * cdiv64(C, DECAY_COLS);
    // us, the forms without tiles / tiles: rank 64, 2048 channels: 512 tokens 13.4 / 12.3, 1024 12.7 / 13.4, 2048 22 / 14.9, 4096 41 / 23, 8192 78 /
    // 42; 512 x 4096 22 / 13; 4096 x 256 8.3 / 12.4; rank 128: 256 x 4096 23 / 19.5, 1024 x 2048 22 / 20.5; rank 256, 4096 x 2048 138 / 60; rank 16,
    // 4096 x 4096 26 / 29.  (Below 1024 tokens the other form is a token per workgroup.)
    if (rank >= 64 && tiles >= (T < 1024 ? 64 : 192) && C <= (int64_t)65535 * DECAY_COLS) {
        const dim3 cut((unsigned)cdiv64(T, DECAY_TOKENS), (unsigned)cdiv64(C, DECAY_COLS));
#define TGIS_DECAY(TT) hipLaunchKernelGGL(wkv_decay_tiles_kernel<TT>, cut, dim3(512), 0, st, (const TT*)a, ld_a, w2t, w0, logw, rank, C, T)
        if (dtype == TGIS_F16)
            TGIS_DECAY(f16);
        else if (dtype == TGIS_BF16)
            TGIS_DECAY(bf16);
        else
            TGIS_DECAY(float);
#undef TGIS_DECAY
        TGIS_CHECK_LAUNCH();
        return TGIS_OK;
    }
    const int tb = T >= 1024 && rank <= 512 && cdiv64(T, 8) * cdiv64(C, 256) >= 256 ? 8 : 1;
    const size_t lds = (size_t)rank * tb * sizeof(float);
    const dim3 grid((unsigned)cdiv64(T, tb), (unsigned)cdiv64(C, 256));
#define TGIS_DECAY(TT)                                                                                                              \
    do {                                                                                                                            \
        if (tb == 8)                                                                                                                \
            hipLaunchKernelGGL((wkv_decay_kernel<TT, 8>), grid, dim3(256), lds, st, (const TT*)a, ld_a, w2t, w0, logw, rank, C, T); \
        else                                                                                                                        \
            hipLaunchKernelGGL((wkv_decay_kernel<TT, 1>), grid, dim3(256), lds, st, (const TT*)a, ld_a, w2t, w0, logw, rank, C, T); \
    } while (0)
    if (dtype == TGIS_F16)
        TGIS_DECAY(f16);
    else if (dtype == TGIS_BF16)
        TGIS_DECAY(bf16);
    else
        TGIS_DECAY(float);
#undef TGIS_DECAY
    TGIS_CHECK_LAUNCH();
    return TGIS_OK;
}

extern "C" int64_t tgis_wkv_scan_workspace(int64_t B, int H, int d, int64_t max_q_len) {
    if (B < 1 || H < 1 || d < 1 || d > 128) return 0;
    const Segments cut = segments_for(B * H, d, max_q_len);
    return cut.count > 1 ? B * H * cut.count * record_floats(d <= 32 ? 32 : d <= 64 ? 64 : 128) * (int64_t)sizeof(float) : 0;
}

extern "C" int tgis_wkv_scan_segments(const void* r, const void* k, const void* v, const void* gate, int64_t ld, const float* logw,
                                      const float* u, const float* gain, float* state, float* shift_state, const float* h, int64_t W,
                                      const int32_t* state_slots, const int32_t* cu_seqlens_q, const int32_t* positions, void* out,
                                      int64_t ld_out, int64_t B, int H, int d, float eps, int64_t max_q_len, void* workspace,
                                      int64_t workspace_bytes, int dtype, void* stream) {
    TGIS_CHECK_ARG(r && k && v && gate && logw && u && gain && state && shift_state && h && state_slots && cu_seqlens_q &&
                       positions && out,
                   "tgis_wkv_scan: null tensor");
    TGIS_CHECK_ARG(B >= 1 && H >= 1 && d >= 1 && d <= 128, "tgis_wkv_scan: head width %d (1 .. 128 supported)", d);
    TGIS_CHECK_ARG(ld >= (int64_t)H * d && ld_out >= (int64_t)H * d && W >= 1 && dtype3(dtype), "tgis_wkv_scan: bad strides or dtype");
    TGIS_CHECK_ARG(!workspace || ((uintptr_t)workspace % 16 == 0 && workspace_bytes >= tgis_wkv_scan_workspace(B, H, d, max_q_len)),
                   "tgis_wkv_scan: the workspace must be 16-byte aligned and of tgis_wkv_scan_workspace bytes");
    hipStream_t st = (hipStream_t)stream;
    TgisTimedScope timed(TGIS_OP_SCAN, st);
#define TGIS_SCAN(TT)                                                                                                                    \
    launch_scan<TT>(r, k, v, gate, ld, logw, u, gain, state, shift_state, h, W, state_slots, cu_seqlens_q, positions, out, ld_out, (int)B, H, \
                    d, eps, max_q_len, workspace, st)
    if (dtype == TGIS_F16)
        TGIS_SCAN(f16);
    else if (dtype == TGIS_BF16)
        TGIS_SCAN(bf16);
    else
        TGIS_SCAN(float);
#undef TGIS_SCAN
    TGIS_CHECK_LAUNCH();
    return TGIS_OK;
}

extern "C" int tgis_wkv_scan_runs(const void* r, const void* k, const void* v, const void* gate, int64_t ld, const float* logw,
                                  const float* u, const float* gain, float* state, float* shift_state, const float* h, int64_t W,
                                  const int32_t* state_slots, const int32_t* cu_seqlens_q, const int32_t* positions, void* out,
                                  int64_t ld_out, int64_t B, int H, int d, float eps, int64_t max_q_len, int dtype, void* stream) {
    return tgis_wkv_scan_segments(r, k, v, gate, ld, logw, u, gain, state, shift_state, h, W, state_slots, cu_seqlens_q, positions, out,
                                  ld_out, B, H, d, eps, max_q_len, nullptr, 0, dtype, stream);
}

extern "C" int tgis_wkv_scan(const void* r, const void* k, const void* v, const void* gate, int64_t ld, const float* logw,
                             const float* u, const float* gain, float* state, float* shift_state, const float* h, int64_t W,
                             const int32_t* state_slots, const int32_t* cu_seqlens_q, const int32_t* positions, void* out,
                             int64_t ld_out, int64_t B, int H, int d, float eps, int dtype, void* stream) {
    return tgis_wkv_scan_segments(r, k, v, gate, ld, logw, u, gain, state, shift_state, h, W, state_slots, cu_seqlens_q, positions, out,
                                  ld_out, B, H, d, eps, 0, nullptr, 0, dtype, stream);
}

// rows of groups of four aligned elements, as the chunk form wants them; d <= 128, rank <= STEP_MAX_RANK
extern "C" int tgis_wkv_step(const void* r, const void* k, const void* v, const void* gate, const void* low, int64_t ld, int64_t ld_low,
                             const float* w2t, const float* w0, int rank, const float* u, const float* gain, float* state,
                             float* shift_state, const float* h, int64_t W, const int32_t* state_slots, const int32_t* cu_seqlens_q,
                             const int32_t* positions, void* out, int64_t ld_out, int64_t B, int H, int d, float eps, int dtype,
                             void* stream) {
    TGIS_CHECK_ARG(r && k && v && gate && low && w2t && w0 && u && gain && state && shift_state && h && state_slots && cu_seqlens_q &&
                       positions && out,
                   "tgis_wkv_step: null tensor");
    TGIS_CHECK_ARG(B >= 1 && H >= 1 && H <= 65535 && d >= 4 && d <= 128 && d % 4 == 0 && rank >= 1 && rank <= STEP_MAX_RANK,
                   "tgis_wkv_step: head width %d (multiples of 4 up to 128), rank %d (up to %d)", d, rank, STEP_MAX_RANK);
    const uintptr_t four = dtype == TGIS_F32 ? 16 : 8;
    TGIS_CHECK_ARG(dtype3(dtype) && ld >= (int64_t)H * d && ld_out >= (int64_t)H * d && ld_low >= rank && ld % 4 == 0 && ld_out % 4 == 0 &&
                       ((uintptr_t)r | (uintptr_t)k | (uintptr_t)v | (uintptr_t)gate | (uintptr_t)out) % four == 0 &&
                       ((uintptr_t)u | (uintptr_t)gain | (uintptr_t)state) % 16 == 0 && W >= 1,
                   "tgis_wkv_step: rows must be groups of four aligned elements");
    hipStream_t st = (hipStream_t)stream;
    TgisTimedScope timed(TGIS_OP_SCAN, st);
#define TGIS_STEP(TT, DM)                                                                                                             \
    hipLaunchKernelGGL((wkv_step_kernel<TT, DM>), dim3((unsigned)B, (unsigned)H), dim3(STEP_THREADS), 0, st, (const TT*)r, (const TT*)k, \
                       (const TT*)v, (const TT*)gate, (const TT*)low, ld, ld_low, w2t, w0, rank, u, gain, state, shift_state, h, W,     \
                       state_slots, cu_seqlens_q, positions, (TT*)out, ld_out, H, d, eps)
#define TGIS_STEP_WIDTH(TT) do { if (d <= 64) TGIS_STEP(TT, 64); else TGIS_STEP(TT, 128); } while (0)
    if (dtype == TGIS_F16)
        TGIS_STEP_WIDTH(f16);
    else if (dtype == TGIS_BF16)
        TGIS_STEP_WIDTH(bf16);
    else
        TGIS_STEP_WIDTH(float);
#undef TGIS_STEP_WIDTH
#undef TGIS_STEP
    TGIS_CHECK_LAUNCH();
    return TGIS_OK;
}
