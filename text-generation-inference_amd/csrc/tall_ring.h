// What the GEMMs of prefills (gptq_tall.hip, dense_tall.hip) share: the order of their tiles, and their k loop over a ring of four LDS buffers of x,
// filled by direct loads three steps ahead.
#pragma once
#include <hip/hip_runtime.h>
#include <type_traits>

namespace tall {

// Tiles are walked in groups of GROUP_ROWS row blocks, each XCD its own run of them, so that its L2 serves a tile of weights to 8 blocks.
constexpr int GROUP_ROWS = 8;
// Block bid of a launch of n -> its tile: XCD x (blocks x, x + 8, ...) takes a run of neighbouring tiles
__device__ __forceinline__ int xcd_run(int bid, int n) {
    const int x = bid & 7, q = n >> 3, rem = n & 7;
    return x * q + min(x, rem) + (bid >> 3);
}
// Tile t of rows x cols blocks: groups of GROUP_ROWS row blocks, rows fastest
__device__ __forceinline__ void tile_at(int t, int rows, int cols, int& row, int& col) {
    const int per = GROUP_ROWS * cols, g = t / per, in = t - g * per, h = min(GROUP_ROWS, rows - g * GROUP_ROWS);
    row = g * GROUP_ROWS + in % h;
    col = in / h;
}

// 16 (4) bytes at base + at + off, base and at the same for the wave: the buffer form, which takes no 64-bit address per lane.  bytes: the range past which it reads
// zeros.  NT: 2 for a line that is read once.
template <int NT> __device__ __forceinline__ auto buffer_piece(const uint8_t* base, int bytes, uint32_t off, int at) {
    return __builtin_amdgcn_raw_buffer_load_b128(__builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base), 0, bytes, 0x00020000), off, at, NT);
}
__device__ __forceinline__ uint32_t buffer_word(const uint8_t* base, int bytes, uint32_t off, int at) {
    return __builtin_amdgcn_raw_buffer_load_b32(__builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base), 0, bytes, 0x00020000), off, at, 0);
}

constexpr int RING = 4;

// The end of a step: the buffer that step s + 2 reads is whole for every wave, with BEHIND vector loads issued behind its own.  The count holds
// only where each of these loads is sure to be issued: a load that nothing reads any more is dropped by the compiler, and the count then lets
// the one that it is meant for through.
template <int BEHIND> __device__ __forceinline__ void meet() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(BEHIND) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// step(s, slot s % RING, tail) for s = 0 .. n - 1: whole turns of the ring, then what is left: with a way out behind every step the compiler sees
// ways back to the first one from each of them, and waits there for every load there is.  In the tail nothing is fetched that no step
// is left to read, and a step ends with meet<0>, which counts on no load.
template <typename F> __device__ __forceinline__ void ring_steps(int n, F&& step) {
    using std::integral_constant;
    using std::false_type;
    using std::true_type;
    int s = 0;
    for (; s + RING <= n; s += RING) {
        step(s, integral_constant<int, 0>{}, false_type{});
        step(s + 1, integral_constant<int, 1>{}, false_type{});
        step(s + 2, integral_constant<int, 2>{}, false_type{});
        step(s + 3, integral_constant<int, 3>{}, false_type{});
    }
    if (s < n) {
        step(s, integral_constant<int, 0>{}, true_type{});
        if (s + 1 < n) {
            step(s + 1, integral_constant<int, 1>{}, true_type{});
            if (s + 2 < n) step(s + 2, integral_constant<int, 2>{}, true_type{});
        }
    }
}

}  // namespace tall
