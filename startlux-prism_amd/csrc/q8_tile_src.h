// Where a thread of the packed Q8_0 tile kernel (w8a8_packed.hip) loads its operands: one 64-bit base per operand, which
// the kernel puts in a buffer resource, and 32-bit offsets from it.  Every byte addressed lies inside the operand: rows
// past M are the last row again and 16-row tiles past N the last tile again (loaded, never stored).  The buffer's record
// count is no substitute for that: the range check is on voffset against the count minus soffset, which wraps where
// soffset alone exceeds the count, as a whole tile's offset does past N.
#pragma once

#include <stdint.h>

namespace prism {

template <int NT>
struct Q8TileSrc {
    int64_t a_base;                                  // activations: bytes to the wave's first row
    uint32_t a_v;                                    //   the lane's bytes of block bi, stage st: + 128 st + 32 bi (panels:
                                                     //   4096 st + 1024 bi)
    int64_t w_base;                                  // weights: bytes to the workgroup's first 16-row tile
    uint32_t w_v, w_s[NT];                           //   load i: + 2048 st; w_s is the same in a wave
    int64_t s_base;                                  // block scales: the same tile's
    uint32_t s_v;                                    //   + 128 st
};

// m0, n0: the workgroup's first row and column (both inside the matrix); wv: the wave (0..3), lane: 0..63.
// PAN: activations in the panel copy, whose rows go up to a multiple of 128.
template <bool PAN, int NT>
__host__ __device__ __forceinline__ Q8TileSrc<NT> q8_tile_src(int m0, int n0, int wv, int lane, int M, int N, int K) {
    auto lo = [](int a, int b) { return a < b ? a : b; };
    Q8TileSrc<NT> s;
    const int KP = K / 64, tid = 64 * wv + lane;
    const int mw = m0 + 32 * wv, row = PAN ? mw : lo(mw, M - 1);
    s.a_base = (int64_t)row * K;
    // the lane's 16 bytes of a block are row lane % 32, inputs 16 (lane / 32) .. + 15
    s.a_v = PAN ? 16 * lane : (uint32_t)(lo(mw + (lane & 31), M - 1) - row) * K + 16 * (lane >> 5);
    const int nt0 = n0 / 16, last = N / 16 - nt0 - 1;
    // load i of a stage: thread -> tile 2 i + tid / 128, 16 bytes (tid % 128) of its 2 KB run
    s.w_base = (int64_t)nt0 * KP * 1024;
    s.w_v = (tid & 127) * 16;
#pragma unroll
    for (int i = 0; i < NT; i++) s.w_s[i] = (uint32_t)lo(2 * i + (wv >> 1), last) * KP * 1024;
    // thread -> tile tid / 32 (past the 2 NT: not used), pair (tid / 16) % 2, row tid % 16: both blocks' fp16
    s.s_base = (int64_t)nt0 * KP * 64;
    s.s_v = (uint32_t)lo(tid >> 5, last) * KP * 64 + (tid & 31) * 4;
    return s;
}

}  // namespace prism
