// The convolution's forward pass and input gradient as one implicit GEMM on the int8 matrix
// cores, quantising the gathered values inside the contraction.
//
// Definition (repro_conv_cuda/repro_conv_math.cuh:1-18): the forward pass scales every window by
// its own maximum and every filter by its own; the input gradient scales dY by one exponent per
// image and the weights by one for all, and adds a pixel's terms over windows and filters. With
// the scales known before the contraction, neither pass needs its window matrix in memory:
//   1. maxima: forward, the largest magnitude over the channels of every pixel of x (a window's
//      maximum is the largest of its pixels'); input gradient, the largest of every image of dY
//      and of the weights.
//   2. the weights' digit panels (in the first launch for the forward pass, whose filters' scales
//      are local; a launch of its own for the input gradient).
//   3. the contraction: output channels x output positions, k running over (16 channels, tap,
//      channel): a block gathers the source values of its positions, one tap and channel per
//      load instruction with 64 neighbouring positions along the lanes, rounds them to fixed
//      point, writes their digits into LDS in the MFMA's operand layout, contracts them with the
//      weights' panels (copied global -> LDS) and rounds every output once.
// The integer sums are the definition's whatever the order of k, so are the bits.
//
// The gather replaces a digit matrix of S bytes per (position, k) written to and read back from
// HBM (173 MB each way for 32 x 64 x 56 x 56, 3x3, S = 3) and the NCHW transposes around the GEMM:
// positions are the MFMA's columns, so a wavefront stores 32 neighbouring output pixels per row.
// A strided input gradient splits the pixels into the residues (y mod SY, x mod SX), each of
// which is a stride-1 gather over its own subset of taps.
//
// Measured on MI355X (us per pass, GEMM pipeline -> here, S = 3): 32 x 64 x 56 x 56, 64 filters 3x3,
// padding 1: forward 137-146 -> 59 (maxima and weights 9, contraction 47), input gradient 283 -> 57;
// 64 -> 256 filters 1x1: 114 -> 74 and 177 -> 58; 8 x 32 x 56 x 56, 48 filters 5x5: 55 -> 32 and
// 93 -> 38; 32 x 512 x 7 x 7, 512 filters 3x3 (parts along k): 81 -> 66 and 228 -> 66. Bounds at the
// first shape: the matrix instructions take 15 us of the contraction at 2.1 GHz; a block's time is
// 9k cycles before its first stage, 3.4k a stage (two blocks' matrix instructions 2.3k, rounding
// 1.1k) and 6k in the epilogue, and 784 blocks are 1.5 rounds of the 512 that fit.
#include "rg_conv_fused.h"

#include <algorithm>
#include <climits>
#include <cstring>
#include <type_traits>

#include "repro_gemm_math.h"
#include "rg_conv_cost.h"
#include "rg_digits.h"
#include "rg_internal.h"
#include "rg_mfma.h"

namespace rg {
namespace {

constexpr int THREADS = 256;
constexpr size_t ALIGN = 256;
size_t align_up(size_t x) { return (x + ALIGN - 1) / ALIGN * ALIGN; }
int ceil_div(long long a, long long b) { return (int)((a + b - 1) / b); }
__host__ __device__ inline int ceil16(int c) { return (c + 15) / 16; }

// Units (output channel, 16 k) of a block of the weights' slicing; longer rows are cut into chunks.
constexpr int QCHUNK = 1024;

// Digit panels of 8 output channels (panel rows r0 .. r0 + 7) of one class, chunk `chunk` of k: [row / 32][k / 32][S]
// panels of 1 KiB. FORWARD: one scale per row, from the row's own maximum; otherwise the common
// scale of the maximum `wmax`. Small next to the contraction: 64 x 576 weights take a few us.
template <int S, bool FORWARD>
__device__ __forceinline__ void slice_weights(const FusedPlan& p, const FusedClass& c,
                                              const float* __restrict__ w, char* ws, int strip,
                                              int chunk, uint32_t wmax) {
    const int t = threadIdx.x;
    const int r0 = strip * 8;
    __shared__ int sexp[8];
    if (FORWARD) {
        const int r = r0 + (t >> 5);
        float m = 0.0f;
        if (r < p.F) {
            const float* row = w + (size_t)r * p.wrow;
            int k = t & 31;
            for (; k + 7 * 32 < p.wrow; k += 8 * 32) {
                float v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] = row[k + 32 * j];
#pragma unroll
                for (int j = 0; j < 8; ++j) m = fmaxf(m, fabsf(v[j]));
            }
            for (; k < p.wrow; k += 32) m = fmaxf(m, fabsf(row[k]));
        }
#pragma unroll
        for (int off = 16; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
        if ((t & 31) == 0) sexp[t >> 5] = repro_gemm::scale_exponent(m);
    } else if (t < 8) {
        sexp[t] = repro_gemm::scale_exponent(__uint_as_float(wmax));
    }
    __syncthreads();
    int* ef = reinterpret_cast<int*>(ws + p.ef);
    if (t < 8) ef[r0 + t] = sexp[t];
    char* q = ws + p.q + c.qoff;
    const int kpanels = 2 * c.stages;
    const int units = 8 * 4 * c.stages, u1 = min(units, (chunk + 1) * QCHUNK);
    for (int u = chunk * QCHUNK + t; u < u1; u += THREADS) {
        const int r = r0 + (u & 7), g = u >> 3;
        const int cg = (int)fdiv((uint32_t)g, c.dT), tap = g - cg * c.T;
        const int ty = (int)fdiv((uint32_t)tap, c.dTW), tx = tap - ty * c.TW;
        const RowScale rs = row_scale<S>(sexp[u & 7]);
        const bool live = r < p.F && g < c.groups;
        const float* src = w + (size_t)(live ? r : 0) * p.wrs + (c.wt0 + ty * c.wt1 + tx * c.wtx);
        float v[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int ch = cg * 16 + i;
            v[i] = live && ch < p.C ? src[(size_t)ch * p.wcs] : 0.0f;
        }
        int x[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = round_fixed(v[i], rs);
        v4i d[S];
        pack16<S>(x, d);
        v4i* out = reinterpret_cast<v4i*>(q) +
                   ((size_t)(r >> 5) * kpanels + (g >> 1)) * S * 64 + (r & 31) + 32 * (g & 1);
#pragma unroll
        for (int s = 0; s < S; ++s) out[s * 64] = d[s];
    }
}

// Forward, first launch: the weights' panels (blocks [0, qblocks)) and every pixel's largest
// magnitude bits over the channels (64 pixels x 4 channel phases a block; a NaN's bits are larger
// than any number's, so a NaN wins, as in the definition's window maxima).
template <int S>
__global__ void __launch_bounds__(THREADS)
fused_fwd_prepare(FusedPlan p, const float* __restrict__ x, const float* __restrict__ w, char* ws) {
    if ((int)blockIdx.x < p.qblocks) {
        const int strip = (int)blockIdx.x / p.cls[0].qchunks;
        slice_weights<S, true>(p, p.cls[0], w, ws, strip, blockIdx.x - strip * p.cls[0].qchunks, 0u);
        return;
    }
    __shared__ uint32_t red[4][64];
    const int lane = threadIdx.x & 63, ph = threadIdx.x >> 6;
    // The pixels of the window tiles that the contraction gives to an XCD are read on that XCD
    // (qblocks is a multiple of 8, or the order is only a little less local), so that x's lines are
    // in its L2 when the contraction copies them.
    const int blk = xcd_order(blockIdx.x - p.qblocks, p.maxima_blocks, 128);
    const uint32_t i = (uint32_t)blk * 64u + lane;
    const uint32_t HW = p.H * p.W, total = (uint32_t)p.N * HW;
    uint32_t m = 0;
    if (i < total) {
        const uint32_t n = fdiv(i, p.dHW);
        const float* s = x + (size_t)n * p.C * HW + (i - n * HW);
        int c = ph;
        for (; c + 28 < p.C; c += 32) {
            uint32_t v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = __float_as_uint(s[(size_t)(c + 4 * j) * HW]) & 0x7FFFFFFFu;
#pragma unroll
            for (int j = 0; j < 8; ++j) m = max(m, v[j]);
        }
        for (; c < p.C; c += 4) m = max(m, __float_as_uint(s[(size_t)c * HW]) & 0x7FFFFFFFu);
    }
    red[ph][lane] = m;
    __syncthreads();
    if (ph == 0 && i < total)
        reinterpret_cast<uint32_t*>(ws + p.maxima)[i] =
            max(max(red[0][lane], red[1][lane]), max(red[2][lane], red[3][lane]));
}

// Input gradient, first launch: partial maxima of every image of dY (img_parts each) and of the
// weights (w_parts): the largest magnitude skipping NaN, and the largest bits (which tell whether
// a NaN or an infinity is present). Entry e at maxima[2 e], maxima[2 e + 1].
__global__ void __launch_bounds__(THREADS)
fused_dx_maxima(FusedPlan p, const float* __restrict__ dy, const float* __restrict__ w, char* ws) {
    const int images = p.N * p.img_parts;
    const float* src;
    long long count;
    int part, parts;
    // (an XCD takes the images whose positions the contraction gives to it, or nearly)
    const int b = (int)blockIdx.x < images ? xcd_order(blockIdx.x, images, p.img_chunk) : (int)blockIdx.x;
    if (b < images) {
        const int n = b / p.img_parts;
        part = b - n * p.img_parts;
        parts = p.img_parts;
        count = (long long)p.C * p.H * p.W;
        src = dy + (size_t)n * count;
    } else {
        part = b - images;
        parts = p.w_parts;
        count = p.wcount;
        src = w;
    }
    const long long i0 = count * part / parts, i1 = count * (part + 1) / parts;
    uint32_t key = 0, raw = 0;
    long long i = i0 + threadIdx.x;
    for (; i + 7 * THREADS < i1; i += 8 * THREADS) {
        uint32_t v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = __float_as_uint(src[i + j * THREADS]) & 0x7FFFFFFFu;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            raw = max(raw, v[j]);
            key = max(key, v[j] > 0x7F800000u ? 0u : v[j]);
        }
    }
    for (; i < i1; i += THREADS) {
        const uint32_t v = __float_as_uint(src[i]) & 0x7FFFFFFFu;
        raw = max(raw, v);
        key = max(key, v > 0x7F800000u ? 0u : v);
    }
    __shared__ uint32_t red[2][THREADS / 64];
    key = wave_umax(key);
    raw = wave_umax(raw);
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = key;
        red[1][threadIdx.x >> 6] = raw;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        uint32_t m = 0;
#pragma unroll
        for (int k = 0; k < THREADS / 64; ++k) m = max(m, red[threadIdx.x][k]);
        reinterpret_cast<uint32_t*>(ws + p.maxima)[2 * (size_t)b + threadIdx.x] = m;
    }
}

// Input gradient, second launch: the weights' panels of every class with the common scale (blocks
// [0, qblocks)), and every image's maxima from its parts (a wavefront per image).
template <int S>
__global__ void __launch_bounds__(THREADS)
fused_dx_weights(FusedPlan p, const float* __restrict__ w, char* ws) {
    const uint2* parts = reinterpret_cast<const uint2*>(ws + p.maxima);
    const int lane = threadIdx.x & 63;
    if ((int)blockIdx.x >= p.qblocks) {
        const int n = ((int)blockIdx.x - p.qblocks) * (THREADS / 64) + (threadIdx.x >> 6);
        if (n >= p.N) return;
        uint32_t key = 0, raw = 0;
        for (int k = lane; k < p.img_parts; k += 64) {
            const uint2 m = parts[(size_t)n * p.img_parts + k];
            key = max(key, m.x);
            raw = max(raw, m.y);
        }
        key = wave_umax(key);
        raw = wave_umax(raw);
        if (lane == 0) reinterpret_cast<uint2*>(ws + p.imax)[n] = make_uint2(key, raw);
        return;
    }
    __shared__ uint32_t red;
    if (threadIdx.x < 64) {
        uint32_t key = 0;
        for (int k = lane; k < p.w_parts; k += 64) key = max(key, parts[(size_t)p.N * p.img_parts + k].x);
        key = wave_umax(key);
        if (lane == 0) red = key;
    }
    __syncthreads();
    int c = 0;
    while (c + 1 < p.nclass && (int)blockIdx.x >= p.cls[c + 1].qblock0) ++c;
    const int b = blockIdx.x - p.cls[c].qblock0, strip = b / p.cls[c].qchunks;
    slice_weights<S, false>(p, p.cls[c], w, ws, strip, b - strip * p.cls[c].qchunks, red);
}

// The outputs from image n0 on (the range ends before the offsets of positions that are not stored),
// or the int64 sums of one part of k (FusedPlan::split > 1), laid out like them.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t output_rsrc(const FusedPlan& p, float* out, const char* ws,
                                                              int part, int n0) {
    const size_t image = (size_t)p.F * p.OPL * (p.split > 1 ? 8u : 4u), tail = (size_t)(p.N - n0) * image;
    char* base = p.split > 1 ? const_cast<char*>(ws) + p.part + (size_t)part * p.N * image : reinterpret_cast<char*>(out);
    return __builtin_amdgcn_make_buffer_rsrc((void*)(base + (size_t)n0 * image), (short)0,
                                             (int)(tail > 0x7FFFFFFFu ? 0x7FFFFFFFu : (uint32_t)tail), 0x00020000);
}

// Rounds and stores a wavefront's TF tiles of 32 channels x 32 positions: register e of a tile
// holds channel 8 (e / 4) + 4 (lane / 32) + e % 4, position lane % 32. sef: the tiles' channel
// exponents (less 14 (S - 1)); f0: the first channel; er: the lane's position's exponent; o: its
// output at channel 0 (bytes from the block's first image, whose resource is orsrc; an offset past
// its range for a position that is not stored). exact: horner_exact, uniform. sbias: the tiles'
// channel biases, added to the rounded outputs, or null.
template <int S, int TF>
__device__ __forceinline__ void store_tiles(const v16i (&acc)[2 * S - 1][TF], const int* sef, int f0, int F,
                                            uint32_t plane4, int er, __amdgpu_buffer_rsrc_t orsrc,
                                            uint32_t o, bool exact, bool partial, const float* sbias) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int L = 2 * S - 1;
    const int lane = threadIdx.x & 63;
    const uint32_t oh = o == 0x80000000u ? o : o + (uint32_t)(4 * (lane >> 5)) * plane4;
    if (partial) {  // one part of k: the exact integers, at twice the outputs' offsets
        typedef int v2i __attribute__((ext_vector_type(2)));
        const uint32_t oh2 = oh == 0x80000000u ? oh : 2u * oh;
#pragma unroll
        for (int ti = 0; ti < TF; ++ti) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                int lv[L];
#pragma unroll
                for (int l = 0; l < L; ++l) lv[l] = acc[l][ti][e];
                const int64_t sum = combine_levels<L>(lv);
                const int f = f0 + ti * 32 + 8 * (e >> 2) + (e & 3);
                const v2i w = {(int)(uint32_t)sum, (int)(sum >> 32)};
                if (f + 4 * (lane >> 5) < F)
                    __builtin_amdgcn_raw_buffer_store_b64(w, orsrc, oh2, 2u * (uint32_t)f * plane4, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        return;
    }
#pragma unroll
    for (int ti = 0; ti < TF; ++ti) {
        const int fl = ti * 32 + 4 * (lane >> 5);
        const bool inside = f0 + ti * 32 + 32 <= F;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float val[4];
            bool all_ok = true;
            if (exact) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    int lv[L];
#pragma unroll
                    for (int l = 0; l < L; ++l) lv[l] = acc[l][ti][4 * q + i];
                    val[i] = round_levels_exact<L>(lv, er + sef[fl + 8 * q + i]);
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    int lv[L];
#pragma unroll
                    for (int l = 0; l < L; ++l) lv[l] = acc[l][ti][4 * q + i];
                    bool ok;
                    val[i] = round_levels_try<L>(lv, er + sef[fl + 8 * q + i], &ok);
                    all_ok = all_ok && ok;
                }
                if (__builtin_expect(!all_ok, 0)) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        int lv[L];
#pragma unroll
                        for (int l = 0; l < L; ++l) lv[l] = acc[l][ti][4 * q + i];
                        val[i] = round_to_float_rare(combine_levels<L>(lv), er + sef[fl + 8 * q + i]);
                    }
                }
            }
            if (sbias != nullptr) {  // uniform
#pragma unroll
                for (int i = 0; i < 4; ++i) val[i] += sbias[fl + 8 * q + i];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t so = (uint32_t)(f0 + ti * 32 + 8 * q + i) * plane4;
                if (inside || f0 + fl + 8 * q + i < F)
                    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(val[i]), orsrc, oh, so, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#endif
}

// The contraction. Block: NWW x NWF wavefronts, wavefront (ww, wf) computes the 32 positions of
// window group ww for TF * 32 output channels. Each stage holds 64 values of k (4 groups of 16):
// the digits of the block's 32 NWW positions, quantised by all wavefronts (a task: 64 positions x
// one group; the lane is the position, so every load instruction reads 64 neighbouring positions
// of one channel and tap), and the channels' digit panels, copied by direct global -> LDS loads.
// Two LDS slots: while the matrix cores contract stage s, the source values of stage s + 1 are in
// registers (their loads were issued a stage earlier) and are rounded into the other slot.
// Two blocks share a compute unit at TF * NWF <= 2, so one block's rounding runs under the other's
// matrix work. It serves one tap (nothing to share between taps), strided classes with few taps and
// images too wide to patch; where taps overlap, its fetches (one per value and tap, nine cache
// accesses per load instruction) made it 8-25% slower than fused_patch.
template <int S, int TF, int NWW, int NWF, bool FORWARD>
__global__ void __launch_bounds__(64 * NWW * NWF, 2)
fused_contract(FusedPlan p, const float* __restrict__ src, const char* __restrict__ ws,
               float* __restrict__ out, const float* __restrict__ bias) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int L = 2 * S - 1;
    constexpr int NW = NWW * NWF;
    constexpr int BW = 32 * NWW;                   // positions per block
    constexpr int WG = NWW / 2;                    // 64-position groups
    constexpr int TPW = 4 * WG / NW;               // quantising tasks per wavefront and stage
    static_assert(TPW * NW == 4 * WG, "tasks split evenly");
    constexpr int PQ = TF * NWF * 2 * S;           // channel panels per stage
    constexpr int PP = NWW * 2 * S;                // position panels per stage
    // One array: with several, the compiler orders every read of the copied panels after all
    // outstanding loads. [slot][PP position panels, PQ channel panels], then the positions'
    // and the channels' exponents and, per wavefront, 1 when all positions whose exponents it
    // took have the fast rounding.
    constexpr int BF = 32 * TF * NWF;              // output channels per block
    __shared__ v4i lds[2 * (PP + PQ) + 2][64];
    static_assert(BW + 2 * BF + NW <= 512, "exponents, flags and biases fit two panels");
    int* sexp = reinterpret_cast<int*>(lds[2 * (PP + PQ)]);
    int* sef = sexp + BW;
    int* sfast = sef + BF;
    float* sbias = reinterpret_cast<float*>(sfast + NW);

    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int ww = wave % NWW, wf = wave / NWW;

    int ci = 0;
    const int lin = xcd_order(blockIdx.x, gridDim.x, 64);
    const int part = (int)fdiv((uint32_t)lin, p.dblocks), item = lin - part * p.blocks;
    while (ci + 1 < p.nclass && item >= p.cls[ci + 1].block0) ++ci;
    const FusedClass& c = p.cls[ci];
    const int local = item - c.block0;
    const int tile = local / p.ftiles, ft = local - tile * p.ftiles;
    const int r0 = tile * BW;
    const int HW = p.H * p.W;
    const uint32_t chw4 = (uint32_t)(p.C * HW) * 4u;
    const int n0 = (int)fdiv((uint32_t)r0, c.dP);

    // Source: a buffer resource from the block's first image on (less padoff), so that offsets are
    // 32-bit; lanes without a source value (zero padding, positions past the end) use an offset
    // past the range, which reads zero.
    const size_t tail = ((size_t)(p.N - n0)) * chw4 + (size_t)c.padoff;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(reinterpret_cast<const char*>(src) + (size_t)n0 * chw4 - c.padoff), (short)0,
        (int)(tail > 0x7FFFFFFFu ? 0x7FFFFFFFu : (uint32_t)tail), 0x00020000);
    constexpr uint32_t NOWHERE = 0x80000000u;

    // This wavefront's tasks: positions wg * 64 + lane, groups q0 + j of every stage.
    const int wg = wave % WG, q0 = (wave / WG) * TPW;
    uint32_t voff;
    uint32_t ymask, xmask;  // taps whose source row / column exists
    {
        const int r = r0 + wg * 64 + lane;
        const int rr = min(r, c.rows - 1);
        const int n = (int)fdiv((uint32_t)rr, c.dP);
        const int g = rr - n * c.P;
        const int gy = (int)fdiv((uint32_t)g, c.dGW), gx = g - gy * c.GW;
        const int y = gy * p.sy + c.y0, x = gx * p.sx + c.x0;
        voff = (uint32_t)(n - n0) * chw4 + (uint32_t)((y * p.W + x) * 4 + c.padoff);
        auto mask = [](int v, int taps, int size) RG_INLINE {
            const int lo = max(0, -v), hi = min(taps, size - v);
            return hi > lo ? ((1u << hi) - 1u) & ~((1u << lo) - 1u) : 0u;
        };
        ymask = r < c.rows ? mask(y, c.TH, p.H) : 0u;
        xmask = mask(x, c.TW, p.W);
    }
    float v[TPW][16];
    const uint32_t plane4 = (uint32_t)HW * 4u;
    auto load_task = [&](int s, int j) RG_INLINE {
        const int g = 4 * s + q0 + j;
        const int cg = (int)fdiv((uint32_t)g, c.dT), tap = g - cg * c.T;
        const int ty = (int)fdiv((uint32_t)tap, c.dTW), tx = tap - ty * c.TW;
        const uint32_t vo = ((ymask >> ty) & (xmask >> tx) & 1u) ? voff : NOWHERE;
        // (the clamp changes no lane that reads: it keeps a tap beyond every source row in range)
        const uint32_t so = min((uint32_t)(ty * p.W + tx) * 4u, plane4 - 4u + (uint32_t)c.padoff);
        // Channels past the last read the last one's values: their weights' digits are 0.
        const uint32_t last = so + (uint32_t)(p.C - 1) * plane4;
#pragma unroll
        for (int i = 0; i < 16; ++i)
            v[j][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                rsrc, vo, min(so + (uint32_t)(cg * 16 + i) * plane4, last), 0));
    };
    auto load = [&](int s) RG_INLINE {
#pragma unroll
        for (int j = 0; j < TPW; ++j) load_task(s, j);
    };

    // Channels' panels of a stage, NW wavefronts in turn.
    const __amdgpu_buffer_rsrc_t qrsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(ws + p.q), (short)0, (int)p.qbytes, 0x00020000);
    const uint32_t qrow = (uint32_t)c.stages * (2u * S * PANEL_BYTES);  // bytes per 32 channels
    auto copy = [&](v4i (*slot)[64], int s) RG_INLINE {
#pragma unroll
        for (int i = 0; i < (PQ + NW - 1) / NW; ++i) {
            const int pi = wave + NW * i;
            if (PQ % NW == 0 || pi < PQ) {
                const int fp = pi / (2 * S), o = pi - fp * (2 * S);
                const uint32_t off = c.qoff + (uint32_t)(ft * (TF * NWF) + fp) * qrow +
                                     (uint32_t)s * (2u * S * PANEL_BYTES) + (uint32_t)o * PANEL_BYTES;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(qrsrc, RG_LDS_PTR(&slot[pi][0]), 16,
                                                         (uint32_t)lane * 16u, off, 0, 0);
            }
        }
    };

    const int s0 = c.stages * part / p.split, stages = c.stages * (part + 1) / p.split - s0;  // this part's
    if (stages > 0) {
        copy(lds + PP, s0);
        __builtin_amdgcn_sched_barrier(0);
        load(s0);
    }

    // The positions' exponents, SUB threads each (they share a window's taps). A position takes the
    // fast rounding (one fused multiply-add) when all its values are finite and its scale 2^n is
    // one normal float.
    constexpr int SUB = 64 * NW / BW;
    {
        const int pos = t / SUB, sub = t % SUB;
        const int r = r0 + pos;
        const bool live = r < c.rows;
        const int rr = live ? r : c.rows - 1;
        const int n = (int)fdiv((uint32_t)rr, c.dP);
        uint32_t key = 0, raw = 0;
        if (FORWARD) {
            const int g = rr - n * c.P;
            const int gy = (int)fdiv((uint32_t)g, c.dGW), gx = g - gy * c.GW;
            const int y = gy * p.sy + c.y0, x = gx * p.sx + c.x0;
            const uint32_t* m = reinterpret_cast<const uint32_t*>(ws + p.maxima) + (size_t)n * HW;
            for (int k0 = sub; k0 < c.T; k0 += 8 * SUB) {
                uint32_t v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {  // every load is issued: a missing tap reads pixel 0
                    const int k = min(k0 + j * SUB, c.T - 1);
                    const int ty = (int)fdiv((uint32_t)k, c.dTW), tx = k - ty * c.TW;
                    const bool in = (unsigned)(y + ty) < (unsigned)p.H && (unsigned)(x + tx) < (unsigned)p.W;
                    v[j] = m[in ? (y + ty) * p.W + x + tx : 0];
                    v[j] = in ? v[j] : 0u;
                }
#pragma unroll
                for (int j = 0; j < 8; ++j) key = max(key, v[j]);
            }
#pragma unroll
            for (int off = 1; off < SUB; off <<= 1) key = max(key, (uint32_t)__shfl_xor((int)key, off, 64));
            raw = key;
        } else {
            const uint2 m = reinterpret_cast<const uint2*>(ws + p.imax)[n];
            key = m.x;
            raw = m.y;
        }
        const int se = repro_gemm::scale_exponent(__uint_as_float(key));
        const int n2 = 7 * (S - 1) - se;
        if (sub == 0) sexp[pos] = se;
        const bool slow = live && !(raw < 0x7F800000u && n2 >= -126 && n2 <= 127);
        const bool any_slow = __ballot(slow) != 0;
        if (lane == 0) sfast[wave] = !any_slow;
        const int* ef = reinterpret_cast<const int*>(ws + p.ef) + ft * BF;
        if (t < BF) {
            sef[t] = ef[t] - 14 * (S - 1);
            if (bias != nullptr) sbias[t] = ft * BF + t < p.F ? bias[ft * BF + t] : 0.0f;
        }
    }
    __syncthreads();
    int allfast = 1;  // the SUB wavefronts that took this group's exponents
#pragma unroll
    for (int i = 0; i < SUB; ++i) allfast &= sfast[wg * SUB + i];
    const bool fast = __builtin_amdgcn_readfirstlane(allfast) != 0;
    const int se = sexp[wg * 64 + lane];
    const RowScale rs = row_scale<S>(se);
    const float scale = __uint_as_float((uint32_t)(7 * (S - 1) - se + 127) << 23);  // if fast
    // Task j's digits into a slot. FAST (a std::integral_constant): the fast rounding.
    auto quantise_task = [&](v4i (*slot)[64], int j, auto FAST) RG_INLINE {
        const int q = q0 + j;
        int x[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            if constexpr (decltype(FAST)::value) x[i] = __float_as_int(__builtin_fmaf(v[j][i], scale, ROUND_MAGIC));
            else x[i] = round_fixed(v[j][i], rs);
        }
        v4i d[S];
        pack16<S>(x, d);
#pragma unroll
        for (int s = 0; s < S; ++s)
            slot[((wg * 2 + (lane >> 5)) * 2 + (q >> 1)) * S + s][(lane & 31) + 32 * (q & 1)] = d[s];
    };

    v16i acc[L][TF];
#pragma unroll
    for (int l = 0; l < L; ++l)
#pragma unroll
        for (int ti = 0; ti < TF; ++ti)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[l][ti][e] = 0;
    auto contract = [&](v4i (*cur)[64]) RG_INLINE {
        v4i (*sq)[64] = cur + PP;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            v4i fa[S][TF], fb[S];
#pragma unroll
            for (int q = 0; q < S; ++q) {
                fb[q] = cur[(ww * 2 + kk) * S + q][lane];
#pragma unroll
                for (int ti = 0; ti < TF; ++ti) fa[q][ti] = sq[((wf * TF + ti) * 2 + kk) * S + q][lane];
            }
#pragma unroll
            for (int a = 0; a < S; ++a)
#pragma unroll
                for (int b = 0; b < S; ++b)
#pragma unroll
                    for (int ti = 0; ti < TF; ++ti)
                        acc[a + b][ti] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[a][ti], fb[b], acc[a + b][ti], 0, 0, 0);
        }
    };
    // Everything written to a slot is visible after this: this wavefront's copies have landed
    // (`loads` younger source loads may stay in flight), its LDS writes are done, all have arrived.
    auto publish = [&](bool loads) RG_INLINE {
        __builtin_amdgcn_sched_barrier(0);
        if (loads) RG_WAIT_VMCNT(16 * TPW);
        else RG_WAIT_VMCNT(0);
        RG_WAIT_LGKMCNT0();
        asm volatile("s_barrier" ::: "memory");
    };
    auto quantise = [&](v4i (*slot)[64]) RG_INLINE {
#pragma unroll
        for (int j = 0; j < TPW; ++j) {
            if (fast) quantise_task(slot, j, std::true_type());
            else quantise_task(slot, j, std::false_type());
        }
    };
    if (stages > 0) {
        quantise(lds);
        if (stages > 1) load(s0 + 1);
        publish(stages > 1);
        v4i (*cur)[64] = lds, (*next)[64] = lds + PP + PQ;
        for (int s = 0; s + 1 < stages; ++s) {
            copy(next + PP, s0 + s + 1);
            __builtin_amdgcn_sched_barrier(0);
            contract(cur);
            quantise(next);
            if (s + 2 < stages) load(s0 + s + 2);
            publish(s + 2 < stages);
            v4i (*freed)[64] = cur;
            cur = next;
            next = freed;
        }
        contract(cur);
    }

    const int r = r0 + ww * 32 + (lane & 31);
    const int rr = min(r, c.rows - 1);
    const int n = (int)fdiv((uint32_t)rr, c.dP);
    const int g = rr - n * c.P;
    const int gy = (int)fdiv((uint32_t)g, c.dGW), gx = g - gy * c.GW;
    const uint32_t oplane4 = (uint32_t)p.OPL * 4u;
    const uint32_t o = r < c.rows ? (uint32_t)(n - n0) * ((uint32_t)p.F * oplane4) +
                                        (uint32_t)((gy * p.osy + c.oy) * p.OW + gx * p.osx + c.ox) * 4u
                                  : NOWHERE;
    if (FORWARD && p.split > 1 && part == 0 && ft == 0 && wf == 0 && lane < 32 && r < c.rows)
        reinterpret_cast<int*>(const_cast<char*>(ws) + p.ew)[(size_t)n * p.OPL + gy * p.OW + gx] = sexp[ww * 32 + lane];
    store_tiles<S, TF>(acc, sef + wf * TF * 32, ft * BF + wf * TF * 32, p.F, oplane4,
                       sexp[ww * 32 + (lane & 31)], output_rsrc(p, out, ws, part, n0), o, p.exact != 0, p.split > 1,
                       bias != nullptr ? sbias + wf * TF * 32 : nullptr);
#endif
}

// The contraction for taps that overlap (stride 1, four or at least six taps): the source values of
// the block's positions are copied once per 16 channels into LDS, as a patch of padded source rows
// (zero padding written out by the copy's range check), and every tap reads its values from there:
// through the vector cache each value was fetched once per tap, and those fetches bounded the
// gathering kernel. A wavefront rounds the values of its own 32 positions straight into the
// MFMA's operand registers (lane l: position l % 32, the 16 channels of k group 2 i + l / 32), so
// the digits never go through LDS. Positions run over (image, column strip, row, column): strips
// narrow wide images until a block's patch fits PX values per channel.
// Patch slots: channel group cg in slot cg % 2, copied as patch_first and patch_due say.
// LDS: 2 x 16 x 384 x 4 B of patches and two stages of 64 output channels' panels, 74 KB: two
// blocks of 4 wavefronts share a compute unit.
template <int S, int TF, bool FORWARD>
__global__ void __launch_bounds__(256, 2)
fused_patch(FusedPlan p, const float* __restrict__ src, const char* __restrict__ ws,
            float* __restrict__ out, const float* __restrict__ bias) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int L = 2 * S - 1;
    constexpr int NW = 4, BW = 32 * NW, BF = 32 * TF;
    constexpr int PX = FUSED_PATCH_PX, NG = PX / 64;
    constexpr int PQ = TF * 2 * S;                 // channel panels per stage
    // One array (with several, the compiler would order every read of a copied region after all
    // outstanding copies): patches, channel panels, positions' exponents, channels' exponents and
    // the positions' slow flags.
    constexpr int PATCH4 = 16 * PX / 4;            // v4i per patch slot
    __shared__ v4i lds[2 * PATCH4 + 2 * PQ * 64 + (2 * BW + 2 * BF) / 4];
    float* patch = reinterpret_cast<float*>(lds);
    v4i* panels = lds + 2 * PATCH4;
    int* sexp = reinterpret_cast<int*>(panels + 2 * PQ * 64);
    int* sslow = sexp + BW;
    int* sef = sslow + BW;
    float* sbias = reinterpret_cast<float*>(sef + BF);

    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const FusedClass& c = p.cls[0];
    const int lin = xcd_order(blockIdx.x, gridDim.x, 64);
    const int part = (int)fdiv((uint32_t)lin, p.dblocks), item = lin - part * p.blocks;
    const int tile = item / p.ftiles, ft = item - tile * p.ftiles;
    const int r0 = tile * BW;
    const int HW = p.H * p.W;
    const uint32_t plane4 = (uint32_t)HW * 4u, chw4 = (uint32_t)p.C * plane4;
    const int PH = c.GH + c.TH - 1, PW = c.GW + c.TW - 1;  // padded rows per strip, their length
    const int img0 = (int)fdiv((uint32_t)r0, c.dP);
    const int n0 = (int)fdiv((uint32_t)img0, c.dNS);

    // (img, padded row, column) of a position: img counts the strips of all images.
    auto locate = [&](int r, int* img, int* gy, int* gx) RG_INLINE {
        *img = (int)fdiv((uint32_t)r, c.dP);
        const int g = r - *img * c.P;
        *gy = (int)fdiv((uint32_t)g, c.dGW);
        *gx = g - *gy * c.GW;
    };
    int base_row;  // padded row of the block's first position
    {
        int img, gy, gx;
        locate(r0, &img, &gy, &gx);
        base_row = img * PH + gy;
    }
    const size_t tail = (size_t)(p.N - n0) * chw4;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(reinterpret_cast<const char*>(src) + (size_t)n0 * chw4), (short)0,
        (int)(tail > 0x7FFFFFFFu ? 0x7FFFFFFFu : (uint32_t)tail), 0x00020000);
    constexpr uint32_t NOWHERE = 0x80000000u;
    uint32_t voff[NG];  // source offsets of patch values 64 g + lane
    auto patch_offsets = [&]() RG_INLINE {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            if (g >= c.pxgroups) break;
            const int px = 64 * g + lane;
            const int pr = (int)fdiv((uint32_t)px, c.dPW), xx = px - pr * PW;
            const int row = base_row + pr;
            const int img = (int)fdiv((uint32_t)row, c.dPH);
            const int n = (int)fdiv((uint32_t)img, c.dNS), strip = img - n * c.NS;
            const int y = row - img * PH + c.y0, x = strip * c.GW + xx + c.x0;
            const bool in = n < p.N && (unsigned)y < (unsigned)p.H && (unsigned)x < (unsigned)p.W;
            voff[g] = in ? (uint32_t)(n - n0) * chw4 + (uint32_t)(y * p.W + x) * 4u : NOWHERE;
        }
    };
    // Copies channel group cg's patch into its slot: wavefront w takes channels 4 w .. 4 w + 3.
    // Channels past the last copy the last one's values: their weights' digits are 0.
    auto copy_patch = [&](int cg) RG_INLINE {
        float* slot = patch + (cg & 1) * (16 * PX);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int ch = wave * 4 + i;
            const uint32_t so = (uint32_t)min(cg * 16 + ch, p.C - 1) * plane4;
#pragma unroll
            for (int g = 0; g < NG; ++g)
                if (g < c.pxgroups)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, RG_LDS_PTR(slot + ch * PX + 64 * g), 4,
                                                             voff[g], so, 0, 0);
        }
    };
    const __amdgpu_buffer_rsrc_t qrsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(ws + p.q), (short)0, (int)p.qbytes, 0x00020000);
    const uint32_t qrow = (uint32_t)c.stages * (2u * S * PANEL_BYTES);  // bytes per 32 channels
    auto copy_panels = [&](int s) RG_INLINE {
        v4i* slot = panels + (s & 1) * (PQ * 64);
#pragma unroll
        for (int i = 0; i < (PQ + NW - 1) / NW; ++i) {
            const int pi = wave + NW * i;
            if (PQ % NW == 0 || pi < PQ) {
                const int fp = pi / (2 * S), o = pi - fp * (2 * S);
                const uint32_t off = (uint32_t)(ft * TF + fp) * qrow +
                                     (uint32_t)s * (2u * S * PANEL_BYTES) + (uint32_t)o * PANEL_BYTES;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(qrsrc, RG_LDS_PTR(slot + pi * 64), 16,
                                                         (uint32_t)lane * 16u, off, 0, 0);
            }
        }
    };
    // This part's stages and the channel groups they read.
    const int s0 = c.stages * part / p.split, s1 = c.stages * (part + 1) / p.split;
    const int cg0 = (int)fdiv((uint32_t)(4 * s0), c.dT);
    const int cgroups = min(ceil16(p.C), (int)fdiv((uint32_t)(4 * s1 - 1), c.dT) + 1);

    // Positions' exponents (two threads each; they share a window's taps) and the rounding they
    // take: the fast one (one fused multiply-add) when all values are finite and the scale 2^n is
    // one normal float.
    {
        const int pos = t >> 1, sub = t & 1;
        const int r = min(r0 + pos, c.rows - 1);
        int img, gy, gx;
        locate(r, &img, &gy, &gx);
        const int n = (int)fdiv((uint32_t)img, c.dNS), strip = img - n * c.NS;
        uint32_t key = 0, raw = 0;
        const int ef = t < BF ? reinterpret_cast<const int*>(ws + p.ef)[ft * BF + t] : 0;
        const float bv = bias != nullptr && t < BF && ft * BF + t < p.F ? bias[ft * BF + t] : 0.0f;
        auto first_copies = [&]() RG_INLINE {
            __builtin_amdgcn_sched_barrier(0);
            copy_panels(s0);
            patch_offsets();
            copy_patch(cg0);
            // (a part that starts in cg0's last groups reads the next group's patch at once)
            if (patch_first(s0) > 1 && cg0 + 1 < cgroups) copy_patch(cg0 + 1);
            __builtin_amdgcn_sched_barrier(0);
        };
        if (FORWARD) {
            const int y = gy + c.y0, x = strip * c.GW + gx + c.x0;
            const uint32_t* m = reinterpret_cast<const uint32_t*>(ws + p.maxima) + (size_t)n * HW;
            for (int k0 = sub; k0 < c.T; k0 += 16) {
                uint32_t v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {  // every load is issued: a missing tap reads pixel 0
                    const int k = min(k0 + 2 * j, c.T - 1);
                    const int ty = (int)fdiv((uint32_t)k, c.dTW), tx = k - ty * c.TW;
                    const bool in = (unsigned)(y + ty) < (unsigned)p.H && (unsigned)(x + tx) < (unsigned)p.W;
                    v[j] = m[in ? (y + ty) * p.W + x + tx : 0];
                    v[j] = in ? v[j] : 0u;
                }
                // The copies go out behind the first loads, so that these do not wait for them.
                if (k0 == sub) first_copies();
#pragma unroll
                for (int j = 0; j < 8; ++j) key = max(key, v[j]);
            }
            key = max(key, (uint32_t)__shfl_xor((int)key, 1, 64));
            raw = key;
        } else {
            const uint2 m = reinterpret_cast<const uint2*>(ws + p.imax)[n];
            first_copies();
            key = m.x;
            raw = m.y;
        }
        const int se = repro_gemm::scale_exponent(__uint_as_float(key));
        const int n2 = 7 * (S - 1) - se;
        if (sub == 0) {
            sexp[pos] = se;
            sslow[pos] = !(raw < 0x7F800000u && n2 >= -126 && n2 <= 127);
        }
        if (t < BF) {
            sef[t] = ef - 14 * (S - 1);
            if (bias != nullptr) sbias[t] = bv;
        }
    }

    v16i acc[L][TF];
#pragma unroll
    for (int l = 0; l < L; ++l)
#pragma unroll
        for (int ti = 0; ti < TF; ++ti)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[l][ti][e] = 0;
    // Everything copied or written so far is visible to the block after this.
    auto publish = [&]() RG_INLINE {
        __builtin_amdgcn_sched_barrier(0);
        RG_WAIT_VMCNT(0);
        RG_WAIT_LGKMCNT0();
        asm volatile("s_barrier" ::: "memory");
    };
    publish();

    const int pos = wave * 32 + (lane & 31);
    const int se = sexp[pos];
    const bool fast = __ballot(sslow[pos] != 0) == 0;
    const RowScale rs = row_scale<S>(se);
    const float scale = __uint_as_float((uint32_t)(7 * (S - 1) - se + 127) << 23);  // if fast
    int px0;  // patch value of this lane's position at tap (0, 0)
    {
        int img, gy, gx;
        locate(min(r0 + pos, c.rows - 1), &img, &gy, &gx);
        px0 = (img * PH + gy - base_row) * PW + gx;
    }
    // The 16 values of this lane's k group in step kk of stage s (groups 4 s + 2 kk and the next,
    // for the two lane halves; a group past the last reads any value, its weights' digits are 0).
    auto where = [&](int g) RG_INLINE {
        const int cg = (int)fdiv((uint32_t)g, c.dT), tap = g - cg * c.T;
        const int ty = (int)fdiv((uint32_t)tap, c.dTW), tx = tap - ty * c.TW;
        return (cg & 1) * (16 * PX) + ty * PW + tx;
    };
    auto read_values = [&](float (&v)[16], int s, int kk) RG_INLINE {
        const int g = 4 * s + 2 * kk;
        const int lo = where(g), hi = where(g + 1);
        const float* q = patch + px0 + (lane < 32 ? lo : hi);
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = q[i * PX];
    };
    auto digits_word = [&](const float (&v)[16], v4i (&d)[S], int w, auto FAST) RG_INLINE {
        int x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (decltype(FAST)::value) x[i] = __float_as_int(__builtin_fmaf(v[4 * w + i], scale, ROUND_MAGIC));
            else x[i] = round_fixed(v[4 * w + i], rs);
        }
        pack_word<S>(x, d, w);
    };
    auto read_panels = [&](v4i (&fa)[S][TF], int s, int kk) RG_INLINE {
        const v4i* q = panels + (s & 1) * (PQ * 64) + lane;
#pragma unroll
        for (int a = 0; a < S; ++a)
#pragma unroll
            for (int ti = 0; ti < TF; ++ti) fa[a][ti] = q[((ti * 2 + kk) * S + a) * 64];
    };
    // Digit product i = (a, b) of a step.
    auto product = [&](const v4i (&fa)[S][TF], const v4i (&fb)[S], int i) RG_INLINE {
        const int a = i / S, b = i % S;
#pragma unroll
        for (int ti = 0; ti < TF; ++ti)
            acc[a + b][ti] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[a][ti], fb[b], acc[a + b][ti], 0, 0, 0);
    };
    // The second step's rounding goes word by word between the first step's matrix instructions,
    // which run on their own (the fences keep that order).
    auto pipeline = [&](auto FAST) RG_INLINE {
        constexpr int EVERY = S == 3 ? 2 : 1;
        int next_cg = cg0 + patch_first(s0);
        for (int s = s0; s < s1; ++s) {
            float v[16], v1[16];
            v4i d0[S], d1[S], fa[S][TF];
            read_values(v, s, 0);
            read_panels(fa, s, 0);
            if (s + 1 < s1) copy_panels(s + 1);
            if (next_cg < cgroups && patch_due(next_cg, c.T, s)) {
                copy_patch(next_cg);
                ++next_cg;
            }
#pragma unroll
            for (int w = 0; w < 4; ++w) digits_word(v, d0, w, FAST);
            read_values(v1, s, 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < S * S; ++i) {
                product(fa, d0, i);
                if (i % EVERY == 0 && i / EVERY < 4) {
                    __builtin_amdgcn_sched_barrier(0);
                    digits_word(v1, d1, i / EVERY, FAST);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (S * S < 4) {
#pragma unroll
                for (int w = (S * S + EVERY - 1) / EVERY; w < 4; ++w) digits_word(v1, d1, w, FAST);
            }
            read_panels(fa, s, 1);
#pragma unroll
            for (int i = 0; i < S * S; ++i) product(fa, d1, i);
            publish();
        }
    };
    if (fast) pipeline(std::true_type());
    else pipeline(std::false_type());

    const int r = r0 + pos;
    int img, gy, gx;
    locate(min(r, c.rows - 1), &img, &gy, &gx);
    const int n = (int)fdiv((uint32_t)img, c.dNS), strip = img - n * c.NS;
    gx += strip * c.GW;
    const uint32_t oplane4 = (uint32_t)p.OPL * 4u;
    // (the last strip's columns past the image are not stored)
    const uint32_t o = r < c.rows && gx < p.OW
                           ? (uint32_t)(n - n0) * ((uint32_t)p.F * oplane4) + (uint32_t)(gy * p.OW + gx) * 4u
                           : NOWHERE;
    if (FORWARD && p.split > 1 && part == 0 && ft == 0 && lane < 32 && o != NOWHERE)
        reinterpret_cast<int*>(const_cast<char*>(ws) + p.ew)[(size_t)n * p.OPL + gy * p.OW + gx] = se;
    store_tiles<S, TF>(acc, sef, ft * BF, p.F, oplane4, se, output_rsrc(p, out, ws, part, n0), o, p.exact != 0,
                       p.split > 1, bias != nullptr ? sbias : nullptr);
#endif
}

// Adds the parts' exact sums and rounds once: out[n][f][pixel] (FusedPlan::split > 1).
template <bool FORWARD>
__global__ void __launch_bounds__(THREADS)
fused_reduce(FusedPlan p, const char* __restrict__ ws, float* __restrict__ out,
             const float* __restrict__ bias) {
    const uint32_t total = (uint32_t)p.N * p.F * p.OPL;
    const uint32_t i = blockIdx.x * THREADS + threadIdx.x;
    if (i >= total) return;
    const int64_t* part = reinterpret_cast<const int64_t*>(ws + p.part) + i;
    int64_t sum = 0;
    for (int k = 0; k < p.split; k += 4) {
        int64_t v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = k + j < p.split ? part[(size_t)(k + j) * total] : 0;
        sum += (v[0] + v[1]) + (v[2] + v[3]);
    }
    const uint32_t nf = fdiv(i, p.dOPL), pix = i - nf * (uint32_t)p.OPL;
    const uint32_t n = fdiv(nf, p.dF), f = nf - n * (uint32_t)p.F;
    const int ep = FORWARD ? reinterpret_cast<const int*>(ws + p.ew)[n * (uint32_t)p.OPL + pix]
                           : repro_gemm::scale_exponent(
                                 __uint_as_float(reinterpret_cast<const uint2*>(ws + p.imax)[n].x));
    const float v = round_output(sum, ep + reinterpret_cast<const int*>(ws + p.ef)[f] - 14 * (p.S - 1));
    out[i] = bias != nullptr ? v + bias[f] : v;
}

}  // namespace

bool fused_plan(int kind, const rg_conv_shape& s, int S, int num_cus, bool forced, FusedPlan* out) {
    FusedPlan p;
    std::memset(&p, 0, sizeof p);
    const int OH = (s.H + 2 * s.PY - s.KH) / s.SY + 1, OW = (s.W + 2 * s.PX - s.KW) / s.SX + 1;
    const bool dx = kind == RG_CONV_GRAD_INPUT;
    p.input_grad = dx;
    p.S = S;
    p.N = s.N;
    const int T = s.KH * s.KW;
    if (dx) {
        p.C = s.F; p.H = OH; p.W = OW; p.F = s.C;
        p.sy = p.sx = 1;
        p.OW = s.W; p.OPL = s.H * s.W; p.osy = s.SY; p.osx = s.SX;
        p.wrs = T; p.wcs = s.C * T;
        p.nclass = s.SY * s.SX;
    } else {
        p.C = s.C; p.H = s.H; p.W = s.W; p.F = s.F;
        p.sy = s.SY; p.sx = s.SX;
        p.OW = OW; p.OPL = OH * OW; p.osy = p.osx = 1;
        p.wrs = s.C * T; p.wcs = T;
        p.nclass = 1;
    }
    if (p.nclass > FUSED_MAX_CLASSES || s.KH > 31 || s.KW > 31) return false;
    p.wrow = s.C * T;
    p.wcount = (long long)s.F * s.C * T;
    p.tf = p.F > 32 ? 2 : 1;
    p.nwf = p.F > 64 ? 2 : 1;
    p.nww = 4;
    const int bw = 32 * p.nww;
    // The patch kernel: one class at stride 1 whose taps overlap enough (the slots' schedule needs
    // four taps or at least six), with strips narrow enough for a block's patch to fit.
    int strips = 1, strip_w = 0, pxgroups = 0;
    if (p.nclass == 1 && s.SY == 1 && s.SX == 1 && (T == 4 || T >= 6)) {
        const int gh = dx ? s.H : OH, gw = dx ? s.W : OW;
        // By widths from the widest that can fit, each with the fewest strips it takes (one strip count
        // after the other was 2-9 ms of host time a call on rows of 10^6 to 10^8 pixels).
        for (int w = std::min(gw, FUSED_PATCH_PX); w >= 1; --w) {
            const int ns = ceil_div(gw, w);
            w = ceil_div(gw, ns);
            const int vrows = (bw + w - 2) / w + 1, cross = (int)((bw + (long long)gh * w - 2) / ((long long)gh * w));
            const long long px = (long long)(vrows + (s.KH - 1) * (cross + 1)) * (w + s.KW - 1);
            if ((long long)ns * w * 4 > (long long)gw * 5) break;  // more than a quarter of dead columns
            if (px <= FUSED_PATCH_PX) {
                p.patch = 1;
                strips = ns;
                strip_w = w;
                pxgroups = ceil_div(px, 64);
                break;
            }
            // (nor with more strips of this width than it takes)
            if (w > 1 && (long long)(ceil_div(gw, w - 1) - 1) * w * 4 > (long long)gw * 5) break;
        }
    }
    if (p.patch) p.nwf = 1;
    const int bf = 32 * p.tf * p.nwf;
    p.ftiles = ceil_div(p.F, bf);
    const int Fp = p.ftiles * bf;
    int block0 = 0, qblock0 = 0;
    size_t q = 0;
    for (int i = 0; i < p.nclass; ++i) {
        FusedClass& c = p.cls[i];
        if (dx) {
            const int ry = i / s.SX, rx = i % s.SX;
            const int ky0 = (ry + s.PY) % s.SY, kx0 = (rx + s.PX) % s.SX;
            c.GH = ceil_div(s.H - ry, s.SY); c.GW = ceil_div(s.W - rx, s.SX);
            if (s.H <= ry) c.GH = 0;
            if (s.W <= rx) c.GW = 0;
            c.TH = s.KH > ky0 ? (s.KH - 1 - ky0) / s.SY + 1 : 0;
            c.TW = s.KW > kx0 ? (s.KW - 1 - kx0) / s.SX + 1 : 0;
            if (c.TH == 0 || c.TW == 0) c.TH = c.TW = 0;
            // Tap (ty, tx) is kernel position ky = ky0 + SY (TH - 1 - ty), whose window row is
            // oy = gy + (ry + PY - ky0) / SY - (TH - 1) + ty.
            c.y0 = (ry + s.PY - ky0) / s.SY - (c.TH - 1);
            c.x0 = (rx + s.PX - kx0) / s.SX - (c.TW - 1);
            c.oy = ry; c.ox = rx;
            c.wt0 = (ky0 + s.SY * (c.TH - 1)) * s.KW + kx0 + s.SX * (c.TW - 1);
            c.wt1 = -s.SY * s.KW;
            c.wtx = -s.SX;
        } else {
            c.GH = OH; c.GW = OW;
            c.TH = s.KH; c.TW = s.KW;
            c.y0 = -s.PY; c.x0 = -s.PX;
            c.wt0 = 0; c.wt1 = s.KW; c.wtx = 1;
        }
        c.NS = 1;
        if (p.patch) {
            c.NS = strips;
            c.GW = strip_w;
            c.pxgroups = pxgroups;
            c.dNS = make_fastdiv((uint32_t)strips);
            c.dPW = make_fastdiv((uint32_t)(c.GW + c.TW - 1));
            c.dPH = make_fastdiv((uint32_t)(c.GH + c.TH - 1));
        }
        c.P = c.GH * c.GW;
        const long long rows = (long long)p.N * c.NS * c.P;
        if (rows >= INT_MAX - 4096) return false;
        c.rows = (int)rows;
        c.T = c.TH * c.TW;
        c.groups = c.T * ceil_div(p.C, 16);
        c.stages = ceil_div(c.groups, 4);
        const long long pad = -((long long)c.y0 * p.W + c.x0) * 4;
        if (pad > (1 << 28)) return false;
        c.padoff = pad > 0 ? (int)pad : 0;
        c.tiles = c.rows > 0 ? ceil_div(c.rows, bw) : 0;
        c.dP = make_fastdiv((uint32_t)std::max(1, c.P));
        c.dGW = make_fastdiv((uint32_t)std::max(1, c.GW));
        c.dT = make_fastdiv((uint32_t)std::max(1, c.T));
        c.dTW = make_fastdiv((uint32_t)std::max(1, c.TW));
        c.block0 = block0;
        c.qblock0 = qblock0;
        if ((long long)block0 + (long long)c.tiles * p.ftiles > INT_MAX / 2) return false;
        block0 += c.tiles * p.ftiles;
        c.qchunks = std::max(1, ceil_div(8 * 4 * c.stages, QCHUNK));
        qblock0 += Fp / 8 * c.qchunks;
        c.qoff = (uint32_t)q;
        q += (size_t)Fp * c.stages * STEP_K * S;
        if (q >= (1u << 31)) return false;
        // Offsets of the block's images stay below 2^31 - 1 bytes.
        const double images = (double)bw / std::max(1, c.P) + 2.0;
        if (((images + 1.0) * p.C + 16.0) * p.H * p.W * 4.0 + c.padoff >= 2147483000.0) return false;
        if ((images + 1.0) * Fp * p.OPL * 8.0 >= 2147483000.0) return false;
        // Exact int32 level sums: at most (2^31 - 1) / 48387 values of k (S = 3; more at S < 3).
        if ((long long)c.stages * STEP_K > (S == 3 ? 44352 : S == 2 ? 66560 : 133120)) return false;
    }
    p.blocks = block0;
    p.qblocks = qblock0;
    p.qbytes = (uint32_t)q;
    p.dHW = make_fastdiv((uint32_t)(p.H * p.W));
    p.exact = horner_exact(S, T * p.C);
    if (p.blocks < 1) return false;
    int stages = 0;
    for (int i = 0; i < p.nclass; ++i) stages = std::max(stages, p.cls[i].stages);
    // Parts along k when the blocks leave the chip idle: each part writes its int64 sums, which a
    // further launch adds and rounds. Times in us: rounds of blocks (two per compute unit, one of
    // the 8-wavefront blocks) of a fixed 7 us plus 1.6 us a stage, the parts' traffic at 4 TB/s.
    const double outs = (double)p.N * p.F * p.OPL, slots = num_cus * (p.nwf == 2 ? 1.0 : 2.0);
    double best = 0.0;
    p.split = 1;
    for (int sp = 1; sp <= 32 && sp <= std::max(1, stages / 2); ++sp) {
        double t = std::ceil(p.blocks * (double)sp / slots) * (7.0 + 1.6 * ceil_div(stages, sp));
        if (sp > 1) t += 4.0 + outs * (16.0 * sp + 4.0) / 4.0e6;
        if (sp == 1 || t < 0.95 * best) {
            best = t;
            p.split = sp;
        }
    }
    if ((long long)p.blocks * p.split > INT_MAX / 2) p.split = 1;
    if (!forced) {
        // Against the GEMM pipeline (rg_conv_cost.h: how both were fitted, and what it replaced). Terms:
        // the launches, rounds of blocks and their steps (rounding, and S^2 matrix instructions per
        // tile; less where a compute unit has one block), the weights' slicing per unit of 16 k, the
        // maxima's read, the outputs' stores, the parts' sums, the length of a sum. (An input
        // gradient is mostly twice as fast here, and the pipeline's estimate the coarser one.)
        const bool lone = p.blocks * (double)p.split <= num_cus, wide = p.tf == 2;
        const double rounds = std::ceil(p.blocks * (double)p.split / slots), steps = rounds * ceil_div(stages, p.split);
        const double s9 = S * S / 9.0, units = q / (16.0 * S), source = (double)p.N * p.C * p.H * p.W, M = 1.0e6;
        double us;
        if (p.patch)
            us = 8.9 + 0.83 * dx + 2.6 * rounds +
                 (lone ? 0.38 + (wide ? 1.2 : 0.43) * s9 : 0.57 + (wide ? 1.2 : 0.7) * s9) * steps + 43.0 * units / M +
                 1.0 * source / M + 1.6 * outs / M + (p.split > 1 ? 2.9 + 4.9 * outs * p.split / M : 0.0) + 0.081 * stages;
        else
            us = 10.0 + 1.9 * dx + 1.2 * rounds +
                 (lone ? 0.75 + (wide ? 1.5 : 0.46) * s9 : 0.8 + (wide ? 1.4 : 1.1) * s9) * steps + 46.0 * units / M +
                 0.67 * source / M + 1.5 * outs / M + (p.split > 1 ? 3.0 + 4.7 * outs * p.split / M : 0.0) + 0.071 * stages;
        if (us > (dx ? 1.03 : 1.0) * conv_pipeline_us(kind, s, S, num_cus)) return false;
    }
    p.dblocks = make_fastdiv((uint32_t)p.blocks);
    p.dOPL = make_fastdiv((uint32_t)p.OPL);
    p.dF = make_fastdiv((uint32_t)p.F);
    size_t maxima;
    if (dx) {
        const long long per = (long long)p.C * p.H * p.W;
        p.img_parts = (int)std::max<long long>(1, std::min<long long>(ceil_div(1024, p.N), per / 4096));
        p.w_parts = (int)std::max<long long>(1, std::min<long long>(64, p.wcount / 4096));
        p.img_chunk = (int)std::max<long long>(1, std::min<long long>(p.N * p.img_parts / 8,
                                                                  64LL * bw * p.img_parts / std::max(1, p.OPL)));
        p.maxima_blocks = p.N * p.img_parts + p.w_parts;
        maxima = (size_t)p.maxima_blocks * 2 * sizeof(uint32_t);
    } else {
        const long long pixels = (long long)p.N * p.H * p.W;
        p.maxima_blocks = ceil_div(pixels, 64);
        maxima = (size_t)pixels * sizeof(uint32_t);
    }
    // A launch takes fewer than 2^32 work items, the pixels' maxima four a pixel. (The pipeline has no
    // pass over the pixels: from 2^30 of them on it still takes the strided passes, whose windows are few.)
    const double first = (double)p.maxima_blocks + (dx ? 0 : p.qblocks), contract = (double)p.blocks * p.split * p.nwf;
    if (std::max(first, contract) * THREADS >= 4294967296.0) return false;
    p.q = 0;
    p.ef = align_up(p.qbytes);
    p.maxima = p.ef + align_up((size_t)Fp * sizeof(int));
    p.imax = p.maxima + align_up(maxima);
    p.ew = p.imax + (dx ? align_up((size_t)p.N * 2 * sizeof(uint32_t)) : 0);
    p.part = p.ew + (!dx && p.split > 1 ? align_up((size_t)p.N * p.OPL * sizeof(int)) : 0);
    p.total = p.part + (p.split > 1 ? align_up((size_t)p.split * p.N * p.F * p.OPL * sizeof(int64_t)) : 0);
    *out = p;
    return true;
}

template <int S>
static void launch_s(const FusedPlan& p, const float* a, const float* w, const float* bias, float* out,
                     char* ws, hipStream_t stream) {
    if (p.input_grad) {
        fused_dx_maxima<<<(unsigned)p.maxima_blocks, THREADS, 0, stream>>>(p, a, w, ws);
        fused_dx_weights<S><<<(unsigned)(p.qblocks + ceil_div(p.N, THREADS / 64)), THREADS, 0, stream>>>(p, w, ws);
    } else {
        fused_fwd_prepare<S><<<(unsigned)(p.qblocks + p.maxima_blocks), THREADS, 0, stream>>>(p, a, w, ws);
    }
    if (p.patch) {
#define RG_PATCH(TF)                                                                             \
    (p.input_grad ? fused_patch<S, TF, false><<<(unsigned)(p.blocks * p.split), 256, 0, stream>>>(p, a, ws, out, bias) \
                  : fused_patch<S, TF, true><<<(unsigned)(p.blocks * p.split), 256, 0, stream>>>(p, a, ws, out, bias))
        if (p.tf == 2) RG_PATCH(2);
        else RG_PATCH(1);
#undef RG_PATCH
    } else {
#define RG_FUSED(TF, NWF)                                                                        \
    (p.input_grad                                                                                \
         ? fused_contract<S, TF, 4, NWF, false><<<(unsigned)(p.blocks * p.split), 256 * NWF, 0, stream>>>(p, a, ws, out, bias) \
         : fused_contract<S, TF, 4, NWF, true><<<(unsigned)(p.blocks * p.split), 256 * NWF, 0, stream>>>(p, a, ws, out, bias))
    if (p.nwf == 2) RG_FUSED(2, 2);
    else if (p.tf == 2) RG_FUSED(2, 1);
    else RG_FUSED(1, 1);
#undef RG_FUSED
    }
    if (p.split > 1) {
        const unsigned blocks = (unsigned)ceil_div((long long)p.N * p.F * p.OPL, THREADS);
        if (p.input_grad) fused_reduce<false><<<blocks, THREADS, 0, stream>>>(p, ws, out, bias);
        else fused_reduce<true><<<blocks, THREADS, 0, stream>>>(p, ws, out, bias);
    }
}

int fused_launch(const FusedPlan& p, const float* a, const float* w, const float* bias, float* out,
                 char* ws, hipStream_t stream) {
    switch (p.S) {
        case 1: launch_s<1>(p, a, w, bias, out, ws, stream); break;
        case 2: launch_s<2>(p, a, w, bias, out, ws, stream); break;
        case 3: launch_s<3>(p, a, w, bias, out, ws, stream); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace rg
