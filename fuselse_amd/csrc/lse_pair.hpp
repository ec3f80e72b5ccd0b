// The IntLSE pair operations (Q16.16 and Q10.6), shared by the row kernels
// and the latency measurement.  Both are commutative (symmetric in a, b) and
// follow the reference's integer arithmetic (intlse/gpu/lse_kernel.cu:46-57,
// lse_kernel_q10_6.cu:35-43) with the shift count clamped as described in
// lse_int.hip.
#pragma once

#include <stdint.h>

namespace fl {

constexpr int kQNegInf = -0x3fffffff;

// Q16.16 values inside the folds are biased by 2^31, as unsigned: the order is
// the same, and |a - b| is one instruction on unsigned operands.
constexpr uint32_t kQBias = 0x80000000u;

// Q16.16 pair of biased values: max + M + LUT[(M >> 10) & 63] with
// M = (2^16 + ((lo - hi) & 0xFFFF)) >> ceil((hi - lo) / 2^16), the shift
// clamped to 31.  With t = |a - b| + 0xFFFF mod 2^32 (v_sad_u32) the shift is
// t >> 16, and 2^16 plus the low half of lo - hi is 2^16 plus the complement of
// t's low half, one bit select.  (Differences within 2^16 of 2^32, which only
// accumulators wrapped past the int32 limit reach, wrap t to a shift of 0, as
// the signed 32-bit difference does.)  Seven vector instructions and the table
// read, six of them in the chain with it; max, min, their difference, its
// halves and a two-instruction table offset took ten, eight in the chain.  The
// block-layout layer of 2048 x 32 nodes, 32 edges, batch 512, whose time this
// is, went from 472 to 421 us; rows of (16384, 1000) fp32 went from 20.1 to 18.9,
// of (65536, 256) from 62.9 to 59.9 (a block per row); (512, 128256), at its memory
// bound, did not change.
template <bool USE_LUT>
__device__ __forceinline__ uint32_t q16_pair(uint32_t a, uint32_t b, const int* __restrict__ lut) {
    const uint32_t hi = a > b ? a : b;
    uint32_t t, fr;
    asm("v_sad_u32 %0, %1, %2, %3" : "=v"(t) : "v"(a), "v"(b), "s"(0xFFFFu));
    const uint32_t th = t >> 16;
    const uint32_t sh = th < 31u ? th : 31u;
    asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(fr) : "v"(t), "v"(0x10000u), "s"(0x1FFFFu));
    const uint32_t m = fr >> sh;
    if constexpr (USE_LUT) {
        // table offset (m >> 8) & 0xFC: byte 1 of m, masked
        uint32_t off;
        asm("v_and_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_1 src1_sel:DWORD"
            : "=v"(off)
            : "v"(m), "s"(0xFCu));
        return hi + m + (uint32_t)*reinterpret_cast<const int*>(reinterpret_cast<const char*>(lut) + off);
    } else {
        return hi + m;
    }
}

// Q10.6 pair through the gap table: max(a, b) + g[min(|a - b|, 385)],
// g[385] = 0.  Every table entry is at most 69, so the table is bytes and the
// clamped gap is the LDS address itself; the clamp is one v_med3_i32 of
// (a - b, b - a, 385), the median being min(|a - b|, 385).  The differences
// cannot overflow: inputs are int16, an accumulator exceeds the largest input
// by at most 64 * log2(N), and the identity -0x3fffffff stays below 2^30 in
// magnitude after any number of pair steps.  Measured 18% shorter per pair
// step than max/min, subtract, clamp and a word address.
__device__ __forceinline__ int q10_pair(int a, int b, const uint8_t* __restrict__ g) {
    const int hi = a > b ? a : b;
    const int u = a - b, nu = b - a;
    int d;
    asm("v_med3_i32 %0, %1, %2, %3" : "=v"(d) : "v"(u), "v"(nu), "s"(385));
    return hi + (int)g[d];
}

}  // namespace fl
