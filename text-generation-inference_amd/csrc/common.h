// Shared helpers for the gfx950 kernels of libtgis_hip.so (CDNA4 only: wave64, MFMA, 160 KiB LDS).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include "../../include/tgis_hip.h"

typedef _Float16 f16;
typedef __bf16 bf16;
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// ---- error plumbing (host) ---------------------------------------------------------------------
void tgis_set_error(const char* fmt, ...);
#define TGIS_CHECK_ARG(cond, ...)          \
    do {                                   \
        if (!(cond)) {                     \
            tgis_set_error(__VA_ARGS__);   \
            return TGIS_EINVAL;            \
        }                                  \
    } while (0)
#define TGIS_CHECK_HIP(expr)                                                              \
    do {                                                                                  \
        hipError_t _e = (expr);                                                           \
        if (_e != hipSuccess) {                                                           \
            tgis_set_error("%s failed: %s (%s:%d)", #expr, hipGetErrorString(_e), __FILE__, \
                           __LINE__);                                                     \
            return TGIS_EHIP;                                                             \
        }                                                                                 \
    } while (0)
#define TGIS_CHECK_LAUNCH() TGIS_CHECK_HIP(hipGetLastError())

// Optional event timing around an op's launches (see tgis_timing_* in tgis_hip.h).
struct TgisTimedScope {
    int op;
    hipStream_t stream;
    void* slot;
    TgisTimedScope(int op, hipStream_t s);
    ~TgisTimedScope();
};

// ---- dtype traits (device) ---------------------------------------------------------------------
template <typename T> struct VecT;
template <> struct VecT<f16> { using x2 = f16x2; using x4 = f16x4; using x8 = f16x8; };
template <> struct VecT<bf16> { using x2 = bf16x2; using x4 = bf16x4; using x8 = bf16x8; };

__device__ __forceinline__ float to_f32(f16 v) { return (float)v; }
__device__ __forceinline__ float to_f32(bf16 v) { return (float)v; }
template <typename T> __device__ __forceinline__ T from_f32(float v);
template <> __device__ __forceinline__ f16 from_f32<f16>(float v) { return (f16)v; }
template <> __device__ __forceinline__ bf16 from_f32<bf16>(float v) { return (bf16)v; }

__device__ __forceinline__ f32x4 mfma16(f16x8 a, f16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma32(f16x8 a, f16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// 16-byte global load/store of 8 two-byte elements.
template <typename V> __device__ __forceinline__ V ld16(const void* p) {
    return *reinterpret_cast<const V*>(p);
}
template <typename V> __device__ __forceinline__ void st16(void* p, V v) {
    *reinterpret_cast<V*>(p) = v;
}

// 1 KiB by a direct load: lane l's 16 bytes at base + off go to LDS byte `lds` + 16 l.  The wave waits for it by its vector memory count.
__device__ __forceinline__ void kib_to_lds(const char* base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds) : "memory", "m0");
}

// Sum / maximum over the 64 lanes of a wave, in every lane: v (+) v of lane ^ 32, ^ 16, ^ 8, ^ 4, ^ 2, ^ 1, by register moves (six trips
// through LDS with __shfl_xor, the same bits).  Lane ^ 4 is a rotation of the row by 4: lanes l and l ^ 8 are alike by then.
template <int CTRL> __device__ __forceinline__ float row_moved(float v) {
    const int x = __builtin_bit_cast(int, v);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(x, x, CTRL, 0xF, 0xF, false));
}
template <typename F> __device__ __forceinline__ float wave_reduce(float v, F op) {
    const uint32_t x = __builtin_bit_cast(uint32_t, v);
    const auto h = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    const uint32_t h0 = h[0], h1 = h[1];
    v = op(__builtin_bit_cast(float, h0), __builtin_bit_cast(float, h1));
    const uint32_t y = __builtin_bit_cast(uint32_t, v);
    const auto q = __builtin_amdgcn_permlane16_swap(y, y, false, false);
    const uint32_t q0 = q[0], q1 = q[1];
    v = op(__builtin_bit_cast(float, q0), __builtin_bit_cast(float, q1));
    v = op(v, row_moved<0x128>(v));  // rotated by 8
    v = op(v, row_moved<0x124>(v));  // by 4
    v = op(v, row_moved<0x4E>(v));   // lane ^ 2
    return op(v, row_moved<0xB1>(v));
}
__device__ __forceinline__ float wave_max(float v) {
    return wave_reduce(v, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float wave_sum(float v) {
    return wave_reduce(v, [](float a, float b) { return a + b; });
}

// Sum of S split-K slabs for 8 consecutive columns: all loads of a bucket are issued before the first add (a
// runtime-trip loop would serialise one L2 round trip per slab).  stride = elements between slabs.
template <int SB>
__device__ __forceinline__ void sum_slabs_bucket(const float* sp, int64_t stride, int S, f32x4& lo, f32x4& hi) {
    f32x4 l[SB], h[SB];
#pragma unroll
    for (int s = 0; s < SB; ++s) {
        const float* q = sp + (int64_t)min(s, S - 1) * stride;
        l[s] = *reinterpret_cast<const f32x4*>(q);
        h[s] = *reinterpret_cast<const f32x4*>(q + 4);
    }
    lo = l[0];
    hi = h[0];
#pragma unroll
    for (int s = 1; s < SB; ++s) {
        if (s < S) {
            lo += l[s];
            hi += h[s];
        }
    }
    for (int s = SB; s < S; ++s) {
        lo += *reinterpret_cast<const f32x4*>(sp + (int64_t)s * stride);
        hi += *reinterpret_cast<const f32x4*>(sp + (int64_t)s * stride + 4);
    }
}
__device__ __forceinline__ void sum_slabs8(const float* sp, int64_t stride, int S, f32x4& lo, f32x4& hi) {
    if (S <= 1)
        sum_slabs_bucket<1>(sp, stride, S, lo, hi);
    else if (S <= 2)
        sum_slabs_bucket<2>(sp, stride, S, lo, hi);
    else if (S <= 4)
        sum_slabs_bucket<4>(sp, stride, S, lo, hi);
    else
        sum_slabs_bucket<8>(sp, stride, S, lo, hi);
}

static inline int64_t cdiv64(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Element (row m, column k) of a [rows, K] activation stored in 32-row MFMA-FRAGMENT ORDER (TGIS_LD_FRAGMENTS in
// include/tgis_hip.h; K % 64 == 0): [row block m / 32][k64-step k / 64][i = k / 8 % 4][lane = 32 (k / 32 % 2) + m % 32][k % 8].
// One k64-step of a row block is four contiguous KiB, each the A operand of one v_mfma_f32_32x32x16 (lane l holds row l % 32,
// k-slots 8 (l / 32) ..+8) in the k order of the prepared weight images; 8 consecutive columns stay 16 contiguous bytes.
__host__ __device__ __forceinline__ int64_t xf_off(int64_t m, int64_t k, int64_t K) {
    return (m >> 5) * 32 * K + ((((k >> 6) << 2) + ((k >> 3) & 3)) * 64 + ((k >> 5) & 1) * 32 + (m & 31)) * 8 + (k & 7);
}

// GELU on an fp32 value (exact erf form, or the tanh approximation): ONE function for tgis_gelu and for the GEMM epilogues
// that apply it to their rounded output, which leave the same bits.
// The erf form is not inlined: inside a caller the compiler contracts the expression (and the library's polynomial) with whatever surrounds it, and the two then
// differ in the last bit.
__device__ __attribute__((noinline)) inline float gelu_erf_f32(float f) { return 0.5f * f * (1.f + erff(f * 0.7071067811865476f)); }
// f (1 + tanh u) / 2 = f / (1 + e^-2u), u = sqrt(2 / pi) (f + 0.044715 f^3): an exponential and a reciprocal of the hardware's, in operations that leave nothing
// to contract.  Against float64 no worse than with the library's tanh, whose 1 + tanh u loses its digits below zero (largest error over the values of bf16 in
// -8 .. 8, of the value: 4e-6, before the value itself).  us, the library's tanh / this: 8186 x 24576 bf16 through tgis_gelu 178 / 131; at the end of a launch of
// tiles of 128 x 256 +23 / +5.
__device__ __forceinline__ float gelu_tanh_f32(float f) {
    constexpr float K = -2.302208198f;  // -2 sqrt(2 / pi) log2 e
    const float e = __builtin_amdgcn_exp2f(f * __builtin_fmaf(f * f, 0.044715f * K, K));
    return f * __builtin_amdgcn_rcpf(1.f + e);
}
__device__ __forceinline__ float gelu_f32(float f, bool tanh_approx) { return tanh_approx ? gelu_tanh_f32(f) : gelu_erf_f32(f); }
