#pragma once
// The digit planes of fixed-point values, for every kernel that slices, and the fast rounding of the
// convolution kernels that slice inside the contraction.
#include "rg_internal.h"
#include "rg_mfma.h"

namespace rg {

// 1.5 * 2^23: for |v| < 2^22, v + ROUND_MAGIC rounds v to an integer (nearest-even) and leaves it
// in the sum's low mantissa bits: bits(sum) = 0x4B400000 + X, whose bits 0..21 are those of X.
constexpr float ROUND_MAGIC = 12582912.0f;

// The base-128 digits of a fixed-point value X (|X| <= 127 * 128^(S-1)), most significant first:
// X = sum_p d[p] 128^(S-1-p) with a signed top digit d[0] = floor(X / 128^(S-1)) in [-127, 127] and
// unsigned lower digits d[p] in [0, 127] (the bit fields of X). Any digit split with these weights
// gives the same exact products; this one keeps the lower digits' sign bits clear, which lowers the
// matrix cores' switching power (about 2% more int8 MFMA throughput measured on MI355X with N(0,1)
// digit planes than balanced digits in [-64, 63]).
//
// Word w of the digit planes of 16 fixed-point values: values t[0..3] (positions 4 w .. 4 w + 3),
// each given by its bits 0 .. 7 S (two's complement; the bits above are ignored); plane p's 16 bytes
// are d[p], most significant digit first. Two values share a register from the first step on
// (v_perm_b32 takes the two bytes each digit lies in), so a value costs 3.25 instructions at S = 3
// against 6.25 for its digits one by one and their packing (256^3 7.70 -> 7.49 us, 512^3 10.28 ->
// 9.90, 768x768x8192 62.8 -> 62.3, 8192x768x768 47.8 -> 47.4).
template <int S>
__device__ __forceinline__ void pack_word(const int (&t)[4], v4i (&d)[S], int w) {
    const uint32_t a = (uint32_t)t[0], b = (uint32_t)t[1], c = (uint32_t)t[2], e = (uint32_t)t[3];
    const uint32_t lo0 = __builtin_amdgcn_perm(b, a, 0x05040100u);  // bits 0..15 of a, b
    const uint32_t lo1 = __builtin_amdgcn_perm(e, c, 0x05040100u);
    if constexpr (S == 1) {
        d[0][w] = (int)__builtin_amdgcn_perm(lo1, lo0, 0x06040200u);
    } else {
        d[S - 1][w] = (int)(__builtin_amdgcn_perm(lo1, lo0, 0x06040200u) & 0x7F7F7F7Fu);
        const uint32_t mid = __builtin_amdgcn_perm(lo1 >> 7, lo0 >> 7, 0x06040200u);
        if constexpr (S == 2) {
            d[0][w] = (int)mid;
        } else {
            d[1][w] = (int)(mid & 0x7F7F7F7Fu);
            const uint32_t hi0 = __builtin_amdgcn_perm(b, a, 0x06050201u);  // bits 8..23
            const uint32_t hi1 = __builtin_amdgcn_perm(e, c, 0x06050201u);
            d[0][w] = (int)__builtin_amdgcn_perm(hi1 >> 6, hi0 >> 6, 0x06040200u);
        }
    }
}

template <int S>
__device__ __forceinline__ void pack16(const int (&t)[16], v4i (&d)[S]) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const int x[4] = {t[4 * w], t[4 * w + 1], t[4 * w + 2], t[4 * w + 3]};
        pack_word<S>(x, d, w);
    }
}

// Largest magnitude bits over a wavefront, in every lane.
__device__ __forceinline__ uint32_t wave_umax(uint32_t m) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, off, 64));
    return m;
}

}  // namespace rg
