// Exact, order-independent float32 sums (bias gradients, loss means) and the non-finite
// scan, for the layers built on the reproducible GEMM.
//
// Accumulation: a thread adds its values in binary64 while that is exact. Values whose magnitudes
// lie in [2^l, 2^(h+1)) are integers times 2^(l-23), so n of them sum to at most n 2^(h+1-l+23) such
// units, and every partial sum is exact while h - l + ceil(log2 n) <= 29: a thread keeps the largest
// magnitude and the smallest non-zero one of what its binary64 sum holds (16 values at a time), and
// when the next 16 would break the bound it moves the sum into its superaccumulator and starts
// again; 16 values that break it by themselves go into the superaccumulator, and the binary64 sum
// stays. N(0, 1) data hardly does either within a thread's share: a value costs about five vector
// instructions (widening, addition, the two bounds). Gradients of a softmax cross-entropy do both all
// the time (probabilities down to 1e-9 next to one near 1), so the superaccumulator's additions have
// no branch and return nothing: about 14 vector instructions and one LDS addition a value.
//
// The superaccumulator is exact for every float: 10 limbs per thread in LDS (limb l of thread t at
// acc[l][t], radix 2^32, limb l weighing 2^(32 l - 149)), cleared when a thread first needs it. A
// finite float is one wide term v < 2^55 at limb idx = (biased exponent - 1) / 32
// (repro_sum::wide_term); at most 252 wide adds land between carry resolutions, which keeps every
// limb below 2^32 + 252 * 2^55 < 2^63. Threads, waves, blocks and chunks are merged by integer
// addition of normalised limbs (exact and associative), and one thread per output divides exactly
// (for a mean) and rounds once (repro_sum::finalize). A wave whose lanes' sums still satisfy the
// bound together adds them in binary64 and, where the output has no other chunk and no division,
// rounds that one exact sum.
//
// Kernels by layout of x = [A][B][C]:
//   C == 1   columns: a 256-thread block covers 64 outputs x 4 row phases; a wave reads
//            64 consecutive floats of one row (bias gradient of a Linear layer).
//   C >  1   segments: one wave per (output, chunk) walks the output's values, runs of C contiguous
//            floats (conv bias gradient, loss mean, row sums), by 16-byte loads where they allow it.
// With more than one chunk per output, the chunks' limbs go to the workspace and a third
// kernel merges and rounds them.
//
// Measured on MI355X against the LDS accumulation of every value (us, whole sum): 256 x 64 x 3136
// 87 -> 37 (5.6 TB/s), 8192 x 4096 rows 45 -> 25 (5.3 TB/s) and columns 56 -> 28, 16384 rows of 1024
// 34 -> 14.5, 65536 rows of 128 86 -> 27, 1000 x 33 x 7 27 -> 5, one sum of 2^24 values 38 -> 23 (the
// merge of its 2048 chunks is one block's). The large ones run at the rate of a copy's reads; small
// ones are two launches. That is N(0, 1) data; values over a wide range (a softmax gradient, and
// uniform exponents in +-20): 8192 x 3072 columns 49 -> 43 and 49 -> 38, 256 x 64 x 3136 87 -> 58 and
// 87 -> 52. (One by one, with their history moved out first, the values that do not fit took 94, 82,
// 177 and 146.)
#include "rg_fastdiv.h"
#include "rg_internal.h"
#include "repro_sum.h"
#include "repro_sum_math.h"

#include <algorithm>
#include <climits>
#include <type_traits>

namespace rg {
namespace {

using repro_sum::LIMBS;

constexpr int SUM_THREADS = 256;
constexpr int BATCH = 16;         // values a thread loads and adds together
constexpr int FLUSH_AT = 252;     // wide adds per limb between carry resolutions
constexpr size_t SUM_ALIGN = 256;

size_t align_up(size_t x) { return (x + SUM_ALIGN - 1) / SUM_ALIGN * SUM_ALIGN; }

// Thread-private superaccumulator in LDS: limb l at p[l * SUM_THREADS].
struct LdsAcc {
    int64_t* p;

    __device__ void clear() {
#pragma unroll
        for (int l = 0; l < LIMBS; ++l) p[l * SUM_THREADS] = 0;
    }
    // One value, by an LDS addition that returns nothing (nobody else touches the address, so it is
    // atomic for free and nothing waits for it): p[idx] += +-significand << s. The exponent of a NaN
    // or an infinity is 255, which the caller looks for in the largest one (top_e); what it adds is
    // in bounds and never used.
    __device__ __forceinline__ void add(float x, uint32_t& top_e) {
        const uint32_t b = __float_as_uint(x), e = (b >> 23) & 0xFFu;
        top_e = max(top_e, e);
        const uint32_t sig = (b & 0x7FFFFFu) | (min(e, 1u) << 23), sh = max(e, 1u) - 1u;
        const int32_t sign = (int32_t)b >> 31;  // 0 or -1
        const int64_t v = ((int32_t)sig ^ sign) - sign;
        bump(sh >> 5, (int64_t)((uint64_t)v << (sh & 31u)));
    }
    __device__ __forceinline__ void bump(uint32_t limb, int64_t v) {
        __hip_atomic_fetch_add(p + limb * SUM_THREADS, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    // An exact sum of floats held in binary64 (a multiple of 2^-149 below 2^159): its 53-bit
    // significand, shifted to a limb boundary, is three 32-bit terms.
    __device__ void add_double(double x, int& nonfinite) {
        const uint64_t b = (uint64_t)__double_as_longlong(x);
        const int e = (int)(b >> 52) & 0x7FF;
        if (e == 0x7FF) {
            nonfinite = 1;
            return;
        }
        if (e == 0) return;  // zero: the smallest non-zero sum, 2^-149, is a normal binary64
        uint64_t m = (b & 0xFFFFFFFFFFFFFull) | 0x10000000000000ull;
        int sh = e - 1075 + 149;  // |x| = m 2^(sh - 149)
        if (sh < 0) {  // (the bits shifted out are zeros)
            m >>= -sh;
            sh = 0;
        }
        const int idx = sh >> 5, s = sh & 31;
        const int64_t t0 = (int64_t)(uint32_t)(m << s);
        const int64_t t1 = (int64_t)(uint32_t)(m >> (32 - s)), t2 = s ? (int64_t)(m >> (64 - s)) : 0;
        const int64_t sign = (int64_t)b >> 63;  // 0 or -1
        bump(idx, (t0 ^ sign) - sign);
        bump(idx + 1, (t1 ^ sign) - sign);
        bump(idx + 2, (t2 ^ sign) - sign);
    }
    // Carries: limbs 0..LIMBS-2 into [0, 2^32), the top limb keeps the sign.
    __device__ void carry() {
        int64_t c = 0;
#pragma unroll
        for (int l = 0; l < LIMBS; ++l) {
            int64_t t = p[l * SUM_THREADS] + c;
            if (l + 1 < LIMBS) {
                c = t >> 32;
                t -= c * ((int64_t)1 << 32);
            }
            p[l * SUM_THREADS] = t;
        }
    }
};

// ceil(log2(n)) for n >= 1.
__device__ __forceinline__ int log2_up(uint32_t n) { return 32 - __clz((int)(n - 1)); }

// Whether n values with largest magnitude `top` and smallest non-zero one `low` sum exactly in
// binary64 in any order: h - l + ceil(log2 n) <= 29. low is kept as 2 * bits - 1 without the sign
// (zeros map to the largest key, so they never are the smallest); a subnormal counts as the smallest
// normal exponent, whose last bit is its unit. An infinity may pass the bound (with magnitudes near
// 2^100 and above beside it), and a NaN is in neither: the binary64 sum is not finite then, which every
// use of it checks.
__device__ __forceinline__ bool sums_exactly(float top, uint32_t low, int log2n) {
    const int h = (int)(__float_as_uint(top) >> 23), l = max(1, (int)(low >> 24));
    return max(h, 1) - l + log2n <= 29;
}

// A thread's sum: binary64 while exact, the superaccumulator otherwise.
struct ThreadSum {
    LdsAcc limbs;
    double acc0 = 0.0, acc1 = 0.0;
    float top = 0.0f;            // of what acc0 + acc1 hold
    uint32_t low = 0xFFFFFFFFu;
    uint32_t count = 0;
    int since = 0;               // additions to the limbs since their carries
    bool used = false;           // the limbs hold something (and were cleared)
    int nonfinite = 0;

    __device__ void spill() {    // binary64 -> limbs
        use();
        limbs.add_double(acc0 + acc1, nonfinite);
        ++since;
        acc0 = acc1 = 0.0;
        top = 0.0f;
        low = 0xFFFFFFFFu;
        count = 0;
    }
    __device__ void use() {
        if (!used) {
            limbs.clear();
            used = true;
        }
    }
    // Adds v; the values from `live` on (the same for the whole wave) are zeros.
    template <int N>
    __device__ __forceinline__ void add(const float (&v)[N], int live = N) {
        // A NaN is in neither bound; it makes the binary64 sum a NaN, which spill() and the final
        // steps see.
        float m = 0.0f;
        uint32_t k = 0xFFFFFFFFu;
#pragma unroll
        for (int i = 0; i < N; ++i) m = fmaxf(m, __builtin_fabsf(v[i]));
#pragma unroll
        for (int i = 0; i < N; ++i) k = min(k, 2u * __float_as_uint(v[i]) - 1u);
        const float m_all = fmaxf(top, m);
        const uint32_t k_all = min(low, k);
        if (__builtin_expect(!sums_exactly(m_all, k_all, log2_up(count + N)), 0)) {
            const bool alone = sums_exactly(m, k, log2_up(N));
            if (alone) {
                spill();
                top = m;
                low = k;
            } else {  // (what the binary64 sum holds stays there)
                use();
                uint32_t top_e = 0;
#pragma unroll
                for (int g = 0; g < N; g += 4) {
                    if (g >= live) break;
#pragma unroll
                    for (int i = g; i < N && i < g + 4; ++i) limbs.add(v[i], top_e);
                }
                nonfinite |= top_e == 0xFFu;
                since += N;
            }
            if (since >= FLUSH_AT - BATCH) {
                limbs.carry();
                since = 0;
            }
            if (!alone) return;
        } else {
            top = m_all;
            low = k_all;
        }
        count += N;
#pragma unroll
        for (int i = 0; i < N; i += 2) {
            acc0 += (double)v[i];
            if (i + 1 < N) acc1 += (double)v[i + 1];
        }
    }
    // Everything into normalised limbs.
    __device__ void finish() {
        if (count > 0) spill();
        else use();
        limbs.carry();
    }
};

// Lowers flag[0] to op_id if any of the wave's lanes holds `bad`: one atomic per such wave.
__device__ inline void report(bool bad, int* flag, int op_id) {
    const unsigned long long votes = __ballot(bad);
    if (votes != 0 && (threadIdx.x & 63) == (unsigned)(__ffsll((long long)votes) - 1))
        atomicMin(flag, op_id);
}

// watch (in both kernels below): the pass that reads the values also reports a NaN or an
// infinity among them, as scan_nonfinite does (watch.flag null: no report). A bias gradient and the
// check of the incoming gradient are then one read of it: 8192 x 3072, 17 us of scan saved.
struct Watch {
    int* flag;
    int op_id;
};

// C == 1. Block = 64 outputs (lanes) x 4 row phases (waves); chunk = blockIdx.y covers rows
// [a0, a1), phase w takes rows a0 + w, a0 + w + 4, ...
__global__ void __launch_bounds__(SUM_THREADS)
sum_columns(const float* __restrict__ x, int A, int B, int rows_per_chunk, int chunks,
            uint32_t divisor, float* __restrict__ out, int64_t* __restrict__ part,
            int* __restrict__ part_nf, Watch watch) {
    __shared__ int64_t acc[LIMBS * SUM_THREADS];
    __shared__ int nf_sh[SUM_THREADS];
    const int t = threadIdx.x, col = t & 63, phase = t >> 6;
    const int b = blockIdx.x * 64 + col;
    const int chunk = blockIdx.y;
    const int a0 = chunk * rows_per_chunk;
    const int a1 = min(A, a0 + rows_per_chunk);
    ThreadSum sum{LdsAcc{acc + t}};
    if (b < B) {
        // A few rows, as every bias gradient of a small batch has, go in a batch of four: in one of 16,
        // mostly zeros, 11 x 1000000 values took 43 us, of a wide range 66, against 38 and 46.
        auto rows = [&](int a, auto N) {
            float v[decltype(N)::value];
#pragma unroll
            for (int g = 0; g < decltype(N)::value; ++g) {
                const int r = a + 4 * g;
                v[g] = r < a1 ? x[(size_t)r * B + b] : 0.0f;
            }
            sum.add<decltype(N)::value>(v, (a1 - a + 3) / 4);
        };
        int a = a0 + phase;
        for (; a + 16 < a1; a += 4 * BATCH) rows(a, std::integral_constant<int, BATCH>());
        if (a < a1) rows(a, std::integral_constant<int, 4>());
    }
    sum.finish();
    if (watch.flag != nullptr) report(sum.nonfinite != 0, watch.flag, watch.op_id);
    nf_sh[t] = sum.nonfinite;
    __syncthreads();
    // The four phases' limbs: thread t adds limb (t >> 6) + 4 i of output t & 63.
#pragma unroll
    for (int l = phase; l < LIMBS; l += 4) {
        int64_t s = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) s += acc[l * SUM_THREADS + col + 64 * w];
        if (chunks > 1) {
            if (b < B) part[((size_t)chunk * LIMBS + l) * B + b] = s;
        } else {
            acc[l * SUM_THREADS + col] = s;  // (only this thread reads the four)
        }
    }
    const int nf = nf_sh[col] | nf_sh[col + 64] | nf_sh[col + 128] | nf_sh[col + 192];
    if (chunks > 1) {
        if (phase == 0 && b < B) part_nf[(size_t)chunk * B + b] = nf;
        return;
    }
    __syncthreads();
    if (phase == 0 && b < B) out[b] = repro_sum::finalize(acc + col, SUM_THREADS, divisor, nf);
}

// C > 1. Wave w of block x handles item 4 x + w of the B * chunks (output, chunk) items,
// output b = item / chunks, chunk item % chunks: summands [i0, i1) of the A*C values of b, in
// order a-major (VEC: in fours, C a multiple of four and x 16-byte aligned). Every wave of a block
// has work when B * chunks fills the grid, however small B is.
template <bool VEC>
__global__ void __launch_bounds__(SUM_THREADS)
sum_segments(const float* __restrict__ x, int A, int B, int C, FastDiv dC, int chunks, uint32_t divisor,
             float* __restrict__ out, int64_t* __restrict__ part, int* __restrict__ part_nf,
             Watch watch) {
    __shared__ int64_t acc[LIMBS * SUM_THREADS];
    __shared__ int64_t merged[4][LIMBS];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const long long item = (long long)blockIdx.x * 4 + w;
    if (item >= (long long)B * chunks) return;  // (no block barrier below)
    const int b = (int)(item / chunks), chunk = (int)(item - (long long)b * chunks);
    ThreadSum sum{LdsAcc{acc + t}};
    constexpr int V = VEC ? 4 : 1;
    const long long units = (long long)A * C / V;
    const uint32_t u0 = (uint32_t)(units * chunk / chunks), u1 = (uint32_t)(units * (chunk + 1) / chunks);
    auto load = [&](uint32_t ug, float* v) {
        const uint32_t i = min(ug, u1 - 1) * V;
        const uint32_t a = fdiv(i, dC);
        const float* p = x + ((size_t)a * B + b) * C + (i - a * (uint32_t)C);
        if (VEC) {
            float4 q = *reinterpret_cast<const float4*>(p);
            if (ug >= u1) q = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            v[0] = q.x;
            v[1] = q.y;
            v[2] = q.z;
            v[3] = q.w;
        } else {
            v[0] = ug < u1 ? *p : 0.0f;
        }
    };
    constexpr int G = BATCH / V;  // loads of a batch; a short rest (or row) goes one load at a time
    uint32_t u = u0 + lane;
    for (; u - lane + 64 * (G / 4) < u1; u += 64 * G) {
        float v[BATCH];
#pragma unroll
        for (int g = 0; g < G; ++g) load(u + 64 * g, v + V * g);
        sum.add<BATCH>(v);
    }
    for (; u - lane < u1; u += 64) {
        float v[V];
        load(u, v);
        sum.add<V>(v);
    }
    // The wave's lanes in binary64 where that is exact (a NaN or an infinity makes the sum one).
    float top = sum.top;
    uint32_t low = sum.low;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        top = fmaxf(top, __shfl_xor(top, off, 64));
        low = min(low, (uint32_t)__shfl_xor((int)low, off, 64));
    }
    const uint32_t total = (u1 - u0) * V + 64u * BATCH;  // at least what the lanes added
    const bool exact = __ballot(sum.used) == 0 && sums_exactly(top, low, log2_up(total));
    if (exact && chunks == 1 && divisor == 1) {
        double s = sum.acc0 + sum.acc1;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
        if (lane == 0) {
            // A zero sum is +0.0; a NaN among the values gives the NaN of repro_sum::finalize.
            const bool nan = !(__builtin_fabs(s) < __builtin_inf());
            out[b] = nan ? __uint_as_float(0x7FC00000u) : (s == 0.0 ? 0.0f : (float)s);
            if (nan && watch.flag != nullptr) atomicMin(watch.flag, watch.op_id);
        }
        return;
    }
    sum.finish();
    const int nf = __ballot(sum.nonfinite != 0) != 0;
    if (nf && lane == 0 && watch.flag != nullptr) atomicMin(watch.flag, watch.op_id);
    // Limb l of the wave: four lanes add 16 threads' limbs each. (A wave's LDS operations are in
    // order, and only this wave's threads' limbs are read.)
    __builtin_amdgcn_wave_barrier();
    int64_t s = 0;
    if (lane < 4 * LIMBS) {
#pragma unroll
        for (int j = 0; j < 16; ++j) s += acc[(lane >> 2) * SUM_THREADS + 64 * w + 16 * (lane & 3) + j];  // < 2^38
    }
    s += __shfl_xor(s, 1, 64);
    s += __shfl_xor(s, 2, 64);
    if (chunks > 1) {
        if (lane < 4 * LIMBS && (lane & 3) == 0) part[((size_t)chunk * LIMBS + (lane >> 2)) * B + b] = s;
        if (lane == 0) part_nf[(size_t)chunk * B + b] = nf;
        return;
    }
    if (lane < 4 * LIMBS && (lane & 3) == 0) merged[w][lane >> 2] = s;
    __builtin_amdgcn_wave_barrier();
    if (lane == 0) out[b] = repro_sum::finalize(merged[w], 1, divisor, nf);
}

// Merges the chunks of each output and rounds once. Few chunks: 32 outputs a block, eight threads
// each (consecutive threads take consecutive outputs; thread s adds chunks s, s + 8, ...); many: a
// block per output, thread t adding chunks t, t + 256, ... Either way the block adds its threads'
// sums in LDS; the normalised limbs (each < 2^32) of at most 65535 chunks sum below 2^48 in int64.
constexpr int MERGE_BLOCK_FROM = 64;

__global__ void __launch_bounds__(SUM_THREADS)
sum_merge_groups(const int64_t* __restrict__ part, const int* __restrict__ part_nf, int B,
                 int chunks, uint32_t divisor, float* __restrict__ out) {
    __shared__ int64_t red[LIMBS][SUM_THREADS];
    __shared__ int nf_sh[SUM_THREADS];
    const int t = threadIdx.x, o = t & 31, sub = t >> 5;
    const int b = blockIdx.x * 32 + o;
    int64_t tot[LIMBS];
#pragma unroll
    for (int l = 0; l < LIMBS; ++l) tot[l] = 0;
    int nf = 0;
    if (b < B) {
        for (int k = sub; k < chunks; k += 16) {  // two chunks' loads together
            const int k2 = k + 8 < chunks ? k + 8 : k;
            int64_t v[2][LIMBS];
#pragma unroll
            for (int l = 0; l < LIMBS; ++l) {
                v[0][l] = part[((size_t)k * LIMBS + l) * B + b];
                v[1][l] = part[((size_t)k2 * LIMBS + l) * B + b];
            }
            nf |= part_nf[(size_t)k * B + b] | part_nf[(size_t)k2 * B + b];
#pragma unroll
            for (int l = 0; l < LIMBS; ++l) tot[l] += v[0][l] + (k2 == k ? 0 : v[1][l]);
        }
    }
#pragma unroll
    for (int l = 0; l < LIMBS; ++l) red[l][t] = tot[l];
    nf_sh[t] = nf;
    __syncthreads();
    // Thread (o, sub) adds limbs sub and sub + 8 of output o; its own column is no other's.
    for (int l = sub; l < LIMBS; l += 8) {
        int64_t s = 0;
#pragma unroll
        for (int g = 0; g < 8; ++g) s += red[l][o + 32 * g];
        red[l][o] = s;
    }
    __syncthreads();
    if (sub == 0 && b < B) {
#pragma unroll
        for (int g = 1; g < 8; ++g) nf |= nf_sh[o + 32 * g];
        out[b] = repro_sum::finalize(&red[0][o], SUM_THREADS, divisor, nf);
    }
}

__global__ void __launch_bounds__(SUM_THREADS)
sum_merge(const int64_t* __restrict__ part, const int* __restrict__ part_nf, int B, int chunks,
          uint32_t divisor, float* __restrict__ out) {
    __shared__ int64_t red[LIMBS][SUM_THREADS];
    __shared__ int nf_sh[SUM_THREADS];
    const int b = blockIdx.x, t = threadIdx.x;
    int64_t tot[LIMBS];
#pragma unroll
    for (int l = 0; l < LIMBS; ++l) tot[l] = 0;
    int nf = 0;
    for (int k = t; k < chunks; k += SUM_THREADS) {
#pragma unroll
        for (int l = 0; l < LIMBS; ++l) tot[l] += part[((size_t)k * LIMBS + l) * B + b];
        nf |= part_nf[(size_t)k * B + b];
    }
#pragma unroll
    for (int l = 0; l < LIMBS; ++l) red[l][t] = tot[l];
    nf_sh[t] = nf;
    __syncthreads();
    for (int s = SUM_THREADS / 2; s > 0; s >>= 1) {
        if (t < s) {
#pragma unroll
            for (int l = 0; l < LIMBS; ++l) red[l][t] += red[l][t + s];
            nf_sh[t] |= nf_sh[t + s];
        }
        __syncthreads();
    }
    if (t == 0) {
        int64_t lim[LIMBS];
#pragma unroll
        for (int l = 0; l < LIMBS; ++l) lim[l] = red[l][0];
        out[b] = repro_sum::finalize(lim, 1, divisor, nf_sh[0]);
    }
}

// Non-finite scan (repro_torch/src/kernels.cu:8-20): one vote per wave, one atomic min per
// wave that saw a NaN or infinity. Grid-stride over 16-byte vectors when x is aligned.
__device__ inline bool is_nonfinite(float v) {
    return (repro_gemm::float_to_bits(v) & 0x7F800000u) == 0x7F800000u;
}

// The n floats at x, op_id the number reported for them, by `blocks` blocks of a scan.
struct ScanPart {
    const float* x;
    size_t n;
    int vec;
    int op_id;
    unsigned blocks;
};

// Two arrays' scans in one launch (the second may be empty, with no blocks): a layer checks its
// input and its weight with one launch instead of two.
__global__ void __launch_bounds__(SUM_THREADS)
scan_nonfinite(ScanPart p0, ScanPart p1, int* flag) {
    const bool second = blockIdx.x >= p0.blocks;
    const float* __restrict__ x = second ? p1.x : p0.x;
    const size_t n = second ? p1.n : p0.n;
    const size_t tid = (size_t)(blockIdx.x - (second ? p0.blocks : 0)) * SUM_THREADS + threadIdx.x;
    const size_t stride = (size_t)(second ? p1.blocks : p0.blocks) * SUM_THREADS;
    bool bad = false;
    size_t tail = 0;
    if (second ? p1.vec : p0.vec) {
        const size_t n4 = n / 4;
        const float4* x4 = reinterpret_cast<const float4*>(x);
        for (size_t i = tid; i < n4; i += stride) {
            const float4 v = x4[i];
            bad = bad || is_nonfinite(v.x) || is_nonfinite(v.y) || is_nonfinite(v.z) ||
                  is_nonfinite(v.w);
        }
        tail = 4 * n4;
    }
    for (size_t i = tail + tid; i < n; i += stride) bad = bad || is_nonfinite(x[i]);
    report(bad, flag, second ? p1.op_id : p0.op_id);
}

ScanPart scan_part(const float* x, size_t n, int op_id) {
    ScanPart p{x, n, (reinterpret_cast<uintptr_t>(x) & 15) == 0, op_id, 0};
    const size_t per_block = (size_t)SUM_THREADS * (p.vec ? 16 : 4);
    p.blocks = (unsigned)std::min<size_t>((n + per_block - 1) / per_block, 4096);
    return p;
}

struct SumLayout {
    bool columns;
    int chunks;
    int rows_per_chunk;   // columns kind
    size_t nf_offset, total;
};

int sum_layout(int A, int B, int C, const rg_sum_config* cfg, int num_cus, SumLayout* Lp) {
    if (!cfg || A <= 0 || B <= 0 || C <= 0 || cfg->chunks < 0) return hipErrorInvalidValue;
    if ((long long)A * C > INT_MAX) return hipErrorInvalidValue;
    SumLayout L{};
    L.columns = C == 1;
    const long long count = (long long)A * C;
    const int max_chunks = (int)std::min<long long>(65535, L.columns ? A : count);
    int chunks = cfg->chunks;
    if (chunks == 0) {
        const int target_blocks = 2 * std::max(1, num_cus);
        if (L.columns) {
            const int bx = (B + 63) / 64;
            chunks = (target_blocks + bx - 1) / bx;
            chunks = std::min(chunks, std::max(1, A / 64));     // >= 64 rows per chunk
        } else {
            const long long target_waves = 4LL * target_blocks;      // (output, chunk) items
            chunks = (int)std::min<long long>((target_waves + B - 1) / B, 65535);
            chunks = (int)std::min<long long>(chunks, std::max(1LL, count / 2048));
        }
    }
    chunks = std::max(1, std::min(chunks, max_chunks));
    if (L.columns) {
        L.rows_per_chunk = (A + chunks - 1) / chunks;
        chunks = (A + L.rows_per_chunk - 1) / L.rows_per_chunk;  // no empty chunk
    }
    L.chunks = chunks;
    const size_t slots = chunks > 1 ? (size_t)chunks * B : 0;
    L.nf_offset = align_up(slots * LIMBS * sizeof(int64_t));
    L.total = slots ? L.nf_offset + align_up(slots * sizeof(int)) : 0;
    *Lp = L;
    return hipSuccess;
}

int sum_layout_current(int A, int B, int C, const rg_sum_config* cfg, SumLayout* L) {
    if (!cfg) return hipErrorInvalidValue;
    DeviceInfo dev{false, 1};
    if (cfg->chunks == 0) {
        const int e = query_device(&dev);
        if (e != hipSuccess) return e;
    }
    return sum_layout(A, B, C, cfg, dev.num_cus, L);
}

}  // namespace
}  // namespace rg

extern "C" {

void rg_sum_config_init(rg_sum_config* cfg) {
    if (!cfg) return;
    cfg->chunks = 0;
    cfg->mean = 0;
}

int rg_make_sum_plan(int A, int B, int C, const rg_sum_config* cfg, rg_sum_plan* plan) {
    if (!plan) return hipErrorInvalidValue;
    rg::SumLayout L;
    const int e = rg::sum_layout_current(A, B, C, cfg, &L);
    if (e != hipSuccess) return e;
    plan->chunks = L.chunks;
    plan->workspace_bytes = L.total;
    return hipSuccess;
}

int rg_sum_plan_for_device(int A, int B, int C, const rg_sum_config* cfg, int num_cus,
                           rg_sum_plan* plan) {
    if (!plan) return hipErrorInvalidValue;
    rg::SumLayout L;
    const int e = rg::sum_layout(A, B, C, cfg, num_cus, &L);
    if (e != hipSuccess) return e;
    plan->chunks = L.chunks;
    plan->workspace_bytes = L.total;
    return hipSuccess;
}

int rg_sum_fp32_ws(const float* x, float* out, int A, int B, int C, const rg_sum_config* cfg,
                   void* workspace, size_t workspace_bytes, void* stream) {
    return rg_sum_watch_fp32_ws(x, out, A, B, C, cfg, workspace, workspace_bytes, nullptr, 0, stream);
}

int rg_sum_watch_fp32_ws(const float* x, float* out, int A, int B, int C, const rg_sum_config* cfg,
                         void* workspace, size_t workspace_bytes, int* flag, int op_id,
                         void* stream_) {
    if (!x || !out) return hipErrorInvalidValue;
    rg::SumLayout L;
    const int e = rg::sum_layout_current(A, B, C, cfg, &L);
    if (e != hipSuccess) return e;
    if (L.total && (!workspace || workspace_bytes < L.total)) return hipErrorInvalidValue;
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    const uint32_t divisor = cfg->mean ? (uint32_t)((long long)A * C) : 1u;
    const rg::Watch watch{flag, op_id};
    int64_t* part = L.total ? static_cast<int64_t*>(workspace) : nullptr;
    int* part_nf = L.total ? reinterpret_cast<int*>(static_cast<char*>(workspace) + L.nf_offset)
                           : nullptr;
    if (L.columns) {
        dim3 grid((B + 63) / 64, L.chunks);
        hipLaunchKernelGGL(rg::sum_columns, grid, dim3(rg::SUM_THREADS), 0, stream, x, A, B,
                           L.rows_per_chunk, L.chunks, divisor, out, part, part_nf, watch);
    } else {
        const long long items = (long long)B * L.chunks;
        if ((items + 3) / 4 > INT_MAX) return hipErrorInvalidValue;
        const bool vec = C % 4 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0;
        const auto segments = vec ? rg::sum_segments<true> : rg::sum_segments<false>;
        hipLaunchKernelGGL(segments, dim3((unsigned)((items + 3) / 4)), dim3(rg::SUM_THREADS), 0, stream,
                           x, A, B, C, rg::make_fastdiv((uint32_t)C), L.chunks, divisor, out, part, part_nf,
                           watch);
    }
    if (L.chunks > 1) {
        if (L.chunks < rg::MERGE_BLOCK_FROM)
            hipLaunchKernelGGL(rg::sum_merge_groups, dim3((B + 31) / 32), dim3(rg::SUM_THREADS), 0, stream,
                               part, part_nf, B, L.chunks, divisor, out);
        else
            hipLaunchKernelGGL(rg::sum_merge, dim3((unsigned)B), dim3(rg::SUM_THREADS), 0, stream,
                               part, part_nf, B, L.chunks, divisor, out);
    }
    return hipGetLastError();
}

int rg_sum_fp32(const float* x, float* out, int A, int B, int C, const rg_sum_config* cfg,
                void* stream) {
    rg_sum_plan plan;
    int e = rg_make_sum_plan(A, B, C, cfg, &plan);
    if (e != hipSuccess) return e;
    void* ws = nullptr;
    if (plan.workspace_bytes && (e = hipMalloc(&ws, plan.workspace_bytes)) != hipSuccess) return e;
    e = rg_sum_fp32_ws(x, out, A, B, C, cfg, ws, plan.workspace_bytes, stream);
    if (e == hipSuccess) e = hipStreamSynchronize(static_cast<hipStream_t>(stream));
    if (ws) (void)hipFree(ws);
    return e;
}

int rg_scan_finite(const float* x, int* flag, size_t n, int op_id, void* stream) {
    return rg_scan_finite_pair(x, n, op_id, nullptr, 0, 0, flag, stream);
}

int rg_scan_finite_pair(const float* x, size_t nx, int op_x, const float* y, size_t ny, int op_y,
                        int* flag, void* stream_) {
    if (nx == 0 && ny == 0) return hipSuccess;
    if ((nx && !x) || (ny && !y) || !flag) return hipErrorInvalidValue;
    const rg::ScanPart p0 = rg::scan_part(x, nx, op_x), p1 = rg::scan_part(y, ny, op_y);
    hipLaunchKernelGGL(rg::scan_nonfinite, dim3(p0.blocks + p1.blocks), dim3(rg::SUM_THREADS), 0,
                       static_cast<hipStream_t>(stream_), p0, p1, flag);
    return hipGetLastError();
}

}  // extern "C"
