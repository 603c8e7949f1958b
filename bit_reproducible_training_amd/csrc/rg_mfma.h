#pragma once
// What the MFMA kernels share: the exact rounding of their level sums, the operand vector types,
// and the waits and LDS pointer casts of their pipelines.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "repro_gemm_math.h"

namespace rg {

// round_to_float for the rare inputs the binary64 paths hand over (|T| near or above 2^53),
// kept out of line so the epilogue's common path stays short.
static __device__ __noinline__ float round_to_float_rare(int64_t T, int E) {
    return repro_gemm::round_to_float(T, E);
}

// T = sum_l lv[l] * 2^(7 (L-1-l)) as an exact int64.
template <int L>
__device__ __forceinline__ int64_t combine_levels(const int (&lv)[L]) {
    int64_t t = 0;
#pragma unroll
    for (int l = 0; l < L; ++l) t += (int64_t)lv[l] * ((int64_t)1 << (7 * (L - 1 - l)));
    return t;
}

// round_to_float(T, E) for T = combine_levels(lv), with the levels combined in binary64:
// Horner steps h = 128 h + lv[l] over int32 levels stay below 2^53 in magnitude up to the
// next-to-last level (|h| < 2^31 (1 + 2^7 + 2^14 + 2^21) < 2^53 for L = 5), so they are
// exact; the last step is exact when the next-to-last |h| < 2^45 (then |T| < 2^52 + 2^31).
// Scaling by 2^E is exact in binary64 when f64_scale_exact(E) (every exponent the slicing
// produces is: |E| <= 2 * 149 + 28), and the conversion to binary32 is the one IEEE rounding
// (nearest-even, subnormals, -0.0, overflow to infinity). *ok = false when a condition fails;
// the value is then meaningless and round_to_float(combine_levels(lv), E) is the result.
template <int L>
__device__ __forceinline__ float round_levels_try(const int (&lv)[L], int E, bool* ok) {
    double h = (double)lv[0];
#pragma unroll
    for (int l = 1; l + 1 < L; ++l) h = __builtin_fma(h, 128.0, (double)lv[l]);
    bool exact = repro_gemm::f64_scale_exact(E);
    if (L > 1) {
        exact = exact && __builtin_fabs(h) < 0x1p45;
        h = __builtin_fma(h, 128.0, (double)lv[L - 1]);
    }
    *ok = exact;
    return (float)__builtin_ldexp(h, E);
}

// round_levels_try without its checks, where both always hold: E is a sum of two slicing exponents
// (each in [-149, 128]) less at most 28, well inside f64_scale_exact, and horner_exact(S, K) bounds
// the next-to-last Horner value.
template <int L>
__device__ __forceinline__ float round_levels_exact(const int (&lv)[L], int E) {
    double h = (double)lv[0];
#pragma unroll
    for (int l = 1; l < L; ++l) h = __builtin_fma(h, 128.0, (double)lv[l]);
    return (float)__builtin_ldexp(h, E);
}

// Whether every sum over K values of k keeps the next-to-last Horner value below 2^45 in magnitude.
// A digit product is at most 127 * 127, and level l < S has l + 1 of them per k, level S .. 2S-3 one
// fewer each: at S = 3 the first four levels reach K * 16129 (2^21 + 2 * 2^14 + 3 * 2^7 + 2)
// = K * 3.4360e10, below 2^45 = 3.5184e13 for K <= 1023; at S = 2, K * 16129 (2^7 + 2), for K below
// 2^24 (the int32 level sums end earlier); at S = 1 there is no such step.
__host__ __device__ constexpr bool horner_exact(int S, int K) { return S < 3 || K <= 1023; }

template <int L>
__device__ __forceinline__ float round_levels(const int (&lv)[L], int E) {
    bool ok;
    const float r = round_levels_try<L>(lv, E, &ok);
    return __builtin_expect(ok, 1) ? r : round_to_float_rare(combine_levels<L>(lv), E);
}

// round_to_float(T, E) for an int64 T: repro_gemm::round_to_float_f64 with its rare
// fallback out of line.
__device__ __forceinline__ float round_output(int64_t T, int E) {
    bool ok;
    const float r = repro_gemm::round_to_float_f64_try(T, E, &ok);
    return __builtin_expect(ok, 1) ? r : round_to_float_rare(T, E);
}

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// s_waitcnt on vector-memory operations only: wait until at most n are outstanding.
#define RG_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (((n) >> 4) << 14) | (7 << 4) | (15 << 8))
// s_waitcnt on LDS (and scalar memory) operations only: wait until none is outstanding.
#define RG_WAIT_LGKMCNT0() __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4) | (0 << 8))
// Lambdas of the kernels hold references to register arrays: they must be inlined, or the
// arrays would move to scratch memory.
#define RG_INLINE __attribute__((always_inline))
#define RG_LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))

}  // namespace rg
