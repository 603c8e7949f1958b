// The convolution's weight gradient, dW[F][K] = dY^T[F][W] * im2col(x)[W][K] (K = C*KH*KW positions,
// W = N*OH*OW windows), as one contraction over the windows that rounds both operands itself.
//
// Definition (repro_conv_cuda/repro_conv_math.cuh:1-18): one scale per filter (its largest dY) and one
// per position (the largest value any window reads there). The scales need one pass over dY and x:
// the values that windows read at position (c, ky, kx) are a plane of x without some border, so the
// maxima of all KH*KW positions come from one running maximum per pixel over the images.
// Launches:
//   1. dw_maxima: partial maxima of every position and filter.
//   2. dw_contract: a block takes 32 TF filters x 128 positions over a range of output rows. The
//      source rows its windows read are copied into LDS once per chunk of rows, for the channels of
//      its positions; lane l of a wavefront holds position l % 32 and rounds the 16 values of k half
//      l / 32 from there straight into the MFMA operand (one scale per lane). dY's values are loaded
//      a stage ahead, rounded by the whole block and written to LDS as digit panels, which all four
//      wavefronts read. k runs over quads of four neighbouring windows of an output row (a row's last
//      quad is filled up with zero dY), so any order of rows and images is a legal order of k.
//   3. reduce_round adds the parts' int64 sums and rounds once.
// The integer sums are the definition's whatever the order of k, so are the bits.
//
// The GEMM pipeline's weight gradient instead writes the window matrix in fp32 (231 MB for
// 32 x 64 x 56 x 56, 3x3), reads it twice to slice it, writes its digits (173 MB) and reads them back.
//
// Measured on MI355X (us, GEMM pipeline -> here, S = 3): 32 x 64 x 56 x 56, 64 filters 3x3: 287 -> 95
// (maxima 17, contraction 75, reduction 6); 8 x 32 x 56 x 56, 48 filters 5x5: 101 -> 52; LeNet's 5x5
// layers at batch 100: 45 -> 26 and 42 -> 29. The contraction is bound by vector instruction issue:
// about ten per matrix instruction (six of them the rounding of the values, the rest offsets), where
// the matrix cores hide about five.
#include "rg_conv_dw.h"

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
constexpr int DW_POS = 128;          // positions per block
constexpr int DW_SLOT = 6144;        // source values per patch slot
constexpr int DW_GROUPS = 6;         // patch values per channel / 64, at most
constexpr int DW_STEPS = 16;         // k steps per chunk, at most
constexpr int DW_PIX = 1024;         // pixels per block of the position maxima
constexpr size_t ALIGN = 256;
size_t align_up(size_t x) { return (x + ALIGN - 1) / ALIGN * ALIGN; }
int ceil_div(long long a, long long b) { return (int)((a + b - 1) / b); }

// Taps along one axis whose windows read source coordinate v: bit k for (v + pad - k) = s * o, 0 <= o < n.
__device__ __forceinline__ uint32_t tap_mask(int v, int pad, int taps, int s, const FastDiv& ds, int n) {
    uint32_t m = 0;
    for (int k = 0; k < taps; ++k) {
        const int r = v + pad - k;
        if (r < 0) break;
        const int o = (int)fdiv((uint32_t)r, ds);
        if (o * s == r && o < n) m |= 1u << k;
    }
    return m;
}

// Blocks [0, C * xgroups * pgroups): channel c, a group of images, DW_PIX pixels: every thread keeps
// the largest magnitude bits (a NaN's are the largest) of its four pixels over the images, then each
// tap takes the maximum over the pixels its windows read: xmax[image group * pgroups + pixel group]
// [c * T + tap]. The rest: filter f, a group of images: dmax[group][f] = (largest magnitude skipping
// NaN, largest bits).
__global__ void __launch_bounds__(THREADS)
dw_maxima(DwPlan p, const float* __restrict__ x, const float* __restrict__ dy, char* ws) {
    __shared__ uint32_t red[2][THREADS / 64];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int xblocks = p.C * p.xgroups * p.pgroups;
    if ((int)blockIdx.x < xblocks) {
        const int HW = p.H * p.W;
        const int pg = blockIdx.x % p.pgroups, q = blockIdx.x / p.pgroups;
        const int c = q % p.C, xg = q / p.C;
        const int n0 = (int)((long long)p.N * xg / p.xgroups), n1 = (int)((long long)p.N * (xg + 1) / p.xgroups);
        uint32_t m[4] = {0, 0, 0, 0};
        int pix[4];  // this thread's pixels: four neighbours with 16-byte loads, else THREADS apart
#pragma unroll
        for (int j = 0; j < 4; ++j) pix[j] = pg * DW_PIX + (p.xvec ? 4 * t + j : j * THREADS + t);
        const float* s = x + ((size_t)n0 * p.C + c) * HW;
        const size_t image = (size_t)p.C * HW;
        if (p.xvec) {
            const float4* s4 = reinterpret_cast<const float4*>(s) + min(pix[0], HW - 4) / 4;
            for (int n = n0; n < n1; n += 4, s4 += image) {
                float4 v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = s4[(size_t)min(i, n1 - 1 - n) * (image / 4)];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    m[0] = max(m[0], __float_as_uint(v[i].x) & 0x7FFFFFFFu);
                    m[1] = max(m[1], __float_as_uint(v[i].y) & 0x7FFFFFFFu);
                    m[2] = max(m[2], __float_as_uint(v[i].z) & 0x7FFFFFFFu);
                    m[3] = max(m[3], __float_as_uint(v[i].w) & 0x7FFFFFFFu);
                }
            }
        } else {
            for (int n = n0; n < n1; n += 4, s += 4 * image) {
                uint32_t v[4][4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        v[i][j] = __float_as_uint(s[(size_t)min(i, n1 - 1 - n) * image + min(pix[j], HW - 1)]) & 0x7FFFFFFFu;
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) m[j] = max(m[j], v[i][j]);
            }
        }
        uint32_t ym[4], xm[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int y = (int)fdiv((uint32_t)pix[j], p.dW), xx = pix[j] - y * p.W;
            ym[j] = pix[j] < HW ? tap_mask(y, p.PY, p.TH, p.SY, p.dSY, p.OH) : 0u;
            xm[j] = tap_mask(xx, p.PX, p.TW, p.SX, p.dSX, p.OW);
        }
        __shared__ uint32_t taps[THREADS / 64][1024];
        // Four taps at a time, so that their cross-lane steps overlap.
        for (int k0 = 0; k0 < p.T; k0 += 4) {
            uint32_t v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int k = min(k0 + i, p.T - 1);
                const int ky = (int)fdiv((uint32_t)k, p.dTW), kx = k - ky * p.TW;
                v[i] = 0;
#pragma unroll
                for (int j = 0; j < 4; ++j) v[i] = max(v[i], ((ym[j] >> ky) & (xm[j] >> kx) & 1u) ? m[j] : 0u);
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = max(v[i], (uint32_t)__shfl_xor((int)v[i], off, 64));
            if (lane < 4 && k0 + lane < p.T) taps[wave][k0 + lane] = lane == 0 ? v[0] : lane == 1 ? v[1] : lane == 2 ? v[2] : v[3];
        }
        __syncthreads();
        uint32_t* out = reinterpret_cast<uint32_t*>(ws + p.xmax) + (size_t)(xg * p.pgroups + pg) * p.K + (size_t)c * p.T;
        for (int k = t; k < p.T; k += THREADS) out[k] = max(max(taps[0][k], taps[1][k]), max(taps[2][k], taps[3][k]));
        return;
    }
    const int b = blockIdx.x - xblocks;
    const int g = b / p.F, f = b - g * p.F;
    const int P = p.OH * p.OW;
    const int n0 = (int)((long long)p.N * g / p.dgroups), n1 = (int)((long long)p.N * (g + 1) / p.dgroups);
    uint32_t key = 0, raw = 0;
    for (int n = n0; n < n1; ++n) {
        const float* s = dy + ((size_t)n * p.F + f) * P;
        if (p.dvec) {
            const float4* s4 = reinterpret_cast<const float4*>(s);
            for (int i = t; i < P / 4; i += 4 * THREADS) {
                float4 v[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = s4[min(i + j * THREADS, P / 4 - 1)];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float w[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t b = __float_as_uint(w[e]) & 0x7FFFFFFFu;
                        raw = max(raw, b);
                        key = max(key, b > 0x7F800000u ? 0u : b);
                    }
                }
            }
            continue;
        }
        for (int i = t; i < P; i += 4 * THREADS) {
            uint32_t v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = __float_as_uint(s[min(i + j * THREADS, P - 1)]) & 0x7FFFFFFFu;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                raw = max(raw, v[j]);
                key = max(key, v[j] > 0x7F800000u ? 0u : v[j]);
            }
        }
    }
    key = wave_umax(key);
    raw = wave_umax(raw);
    if (lane == 0) {
        red[0][wave] = key;
        red[1][wave] = raw;
    }
    __syncthreads();
    if (t < 2)
        reinterpret_cast<uint32_t*>(ws + p.dmax)[2 * ((size_t)g * p.F + f) + t] =
            max(max(red[t][0], red[t][1]), max(red[t][2], red[t][3]));
}

// The contraction. Wavefront w: positions 32 w .. 32 w + 31 of the block's 128 x 32 TF filters, two k
// steps of 32 per stage. Chunk c of the part (its RC output rows' source rows) sits in patch slot
// c % 2, the first two copied before the first stage and the others as dw_due says. The quads' offsets
// (into dY and into the patch) are a table per chunk, in ring slot c % 4: table c + 2 is built when
// chunk c is copied (chunk c - 2, whose slot it takes, is done), at least a stage before dY's loads,
// which go out two stages ahead, look into it.
template <int S, int TF, int SXT>
__global__ void __launch_bounds__(256, 2)
dw_contract(DwPlan p, const float* __restrict__ dy, const float* __restrict__ x, char* __restrict__ ws) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int L = 2 * S - 1;
    constexpr int BF = 32 * TF;
    constexpr int PQ = TF * 2 * S;       // filter panels per stage
    constexpr int TASKS = 2 * TF;        // dY tasks (16 filters x 4 quads) per wavefront and stage
    constexpr int TABLE = 8 * DW_STEPS;  // quads per chunk, at most
    // One array (see rg_conv_fused.hip): patches, filter panels, quad tables (dY offsets, patch
    // offsets), the positions' and the filters' exponents and slow flags.
    __shared__ v4i lds[2 * DW_SLOT / 4 + 2 * PQ * 64 + 4 * 2 * TABLE / 4 + (2 * DW_POS + 2 * BF) / 4];
    float* patch = reinterpret_cast<float*>(lds);
    v4i* panels = lds + 2 * DW_SLOT / 4;
    int* tdy = reinterpret_cast<int*>(panels + 2 * PQ * 64);
    int* tx = tdy + 4 * TABLE;
    int* spos = tx + 4 * TABLE;
    int* sslow = spos + DW_POS;
    int* sfil = sslow + DW_POS;
    int* sfslow = sfil + BF;

    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int lin = xcd_order(blockIdx.x, gridDim.x, 64);
    const int tiles = p.ptiles * p.ftiles;
    const int part = lin / tiles, tile = lin - part * tiles;
    const int pt = tile / p.ftiles, ft = tile - pt * p.ftiles;
    const int chunk0 = part * p.per_part, nchunks = min(p.per_part, p.chunks - chunk0);
    const int nsteps = nchunks * p.KS, stages = (nsteps + 1) >> 1;
    const int p0 = pt * DW_POS;
    const int c0 = (int)fdiv((uint32_t)p0, p.dT);
    const int nch = (int)fdiv((uint32_t)min(p0 + DW_POS - 1, p.K - 1), p.dT) - c0 + 1;  // channels read
    const int HW = p.H * p.W, P = p.OH * p.OW;
    constexpr uint32_t NOWHERE = 0x80000000u;
    // (x and dY hold fewer than 2^29 values: dw_plan)
    const __amdgpu_buffer_rsrc_t xrsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)x, (short)0, (int)((uint32_t)p.N * p.C * HW * 4u), 0x00020000);
    const __amdgpu_buffer_rsrc_t drsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)dy, (short)0, (int)((uint32_t)p.N * p.F * P * 4u), 0x00020000);

    // Padded source row of the first tap of output row v = ((image, strip), oy).
    auto padded = [&](int v) RG_INLINE {
        const int img = (int)fdiv((uint32_t)v, p.dOH);
        return img * p.PH + (v - img * p.OH) * p.SY;
    };
    // Source rows of chunk c (of this part) into its slot: wavefront w takes channels w, w + 4, ...
    auto copy_patch = [&](int c) RG_INLINE {
        const int base = padded(min((chunk0 + c) * p.RC, p.vrows - 1));
        float* slot = patch + (c & 1) * DW_SLOT;
        uint32_t voff[DW_GROUPS];
#pragma unroll
        for (int g = 0; g < DW_GROUPS; ++g) {
            if (g >= p.pxgroups) break;
            const int px = 64 * g + lane;
            const int pr = (int)fdiv((uint32_t)px, p.dPW), xx = px - pr * p.PW;
            const int row = base + pr;
            const int img = (int)fdiv((uint32_t)row, p.dPH);
            const int n = (int)fdiv((uint32_t)img, p.dNS), strip = img - n * p.NS;
            const int y = row - img * p.PH - p.PY, xc = strip * p.SW * SXT + xx - p.PX;
            const bool in = n < p.N && (unsigned)y < (unsigned)p.H && (unsigned)xc < (unsigned)p.W;
            voff[g] = in ? (uint32_t)(n * p.C * HW + y * p.W + xc) * 4u : NOWHERE;
        }
        for (int ch = wave; ch < nch; ch += 4) {
            const uint32_t so = (uint32_t)((c0 + ch) * HW) * 4u;
#pragma unroll
            for (int g = 0; g < DW_GROUPS; ++g)
                if (g < p.pxgroups)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(xrsrc, RG_LDS_PTR(slot + ch * p.pxs + 64 * g), 4,
                                                             voff[g], so, 0, 0);
        }
    };
    // Quad table of chunk c: dY offset of the quad's first value for filter 0, with its number of
    // live columns less one in the low bits (a quad outside the part: NOWHERE), and its patch offset.
    auto build_table = [&](int c) RG_INLINE {
        for (int q = t; q < 8 * p.KS; q += 256) {
            const int r = (int)fdiv((uint32_t)q, p.dSQ), cq = q - r * p.SQ;
            const int v0 = (chunk0 + c) * p.RC, v = v0 + r;
            int off = (int)NOWHERE, xo = 0;
            if (c < nchunks && r < p.RC && v < p.vrows) {
                const int img = (int)fdiv((uint32_t)v, p.dOH), oy = v - img * p.OH;
                const int n = (int)fdiv((uint32_t)img, p.dNS), strip = img - n * p.NS;
                const int ox = strip * p.SW + 4 * cq;
                const int live = min(4, min(p.SW - 4 * cq, p.OW - ox));
                xo = (padded(v) - padded(v0)) * p.PW + 4 * cq * SXT;
                if (live > 0) off = (n * p.F * P + oy * p.OW + ox) * 4 + live - 1;
            }
            tdy[(c & 3) * TABLE + q] = off;
            tx[(c & 3) * TABLE + q] = xo;
        }
    };

    // First chunks and tables; the maxima's loads go out first.
    uint32_t key = 0, raw = 0;
    if (t < DW_POS) {
        const uint32_t* m = reinterpret_cast<const uint32_t*>(ws + p.xmax) + min(p0 + t, p.K - 1);
        const int n = p.xgroups * p.pgroups;
        for (int k = 0; k < n; k += 8) {
            uint32_t v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = m[(size_t)min(k + j, n - 1) * p.K];
#pragma unroll
            for (int j = 0; j < 8; ++j) key = max(key, v[j]);
        }
        raw = key;
    } else if (t < DW_POS + BF) {
        const int f = ft * BF + t - DW_POS;
        if (f < p.F) {
            const uint2* m = reinterpret_cast<const uint2*>(ws + p.dmax) + f;
            for (int k = 0; k < p.dgroups; k += 8) {
                uint2 v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] = m[(size_t)min(k + j, p.dgroups - 1) * p.F];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    key = max(key, v[j].x);
                    raw = max(raw, v[j].y);
                }
            }
        }
    }
    copy_patch(0);
    if (nchunks > 1) copy_patch(1);
    for (int c = 0; c < 4; ++c) build_table(c);
    {
        // The fast rounding: all values finite and the scale 2^n one normal float.
        const int se = repro_gemm::scale_exponent(__uint_as_float(key));
        const int n2 = 7 * (S - 1) - se;
        const int slow = !(raw < 0x7F800000u && n2 >= -126 && n2 <= 127);
        if (t < DW_POS) {
            spos[t] = se;
            sslow[t] = slow;
            if (part == 0 && ft == 0 && p0 + t < p.K) reinterpret_cast<int*>(ws + p.eb)[p0 + t] = se;
        } else if (t < DW_POS + BF) {
            sfil[t - DW_POS] = se;
            sfslow[t - DW_POS] = slow;
            if (part == 0 && pt == 0 && ft * BF + t - DW_POS < p.F)
                reinterpret_cast<int*>(ws + p.ea)[ft * BF + t - DW_POS] = se;
        }
    }
    v16i acc[L][TF];
#pragma unroll
    for (int l = 0; l < L; ++l)
#pragma unroll
        for (int ti = 0; ti < TF; ++ti)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[l][ti][e] = 0;
    __syncthreads();

    // This lane's position and filter.
    const int pos = p0 + wave * 32 + (lane & 31);
    const bool idle = p0 + wave * 32 >= p.K;  // uniform: none of the wavefront's positions exists
    const int pse = spos[wave * 32 + (lane & 31)];
    const RowScale prs = row_scale<S>(pse);
    const float pscale = __uint_as_float((uint32_t)(7 * (S - 1) - pse + 127) << 23);  // if fast
    int base;  // patch offset of the position's channel and tap
    {
        const int q = min(pos, p.K - 1);
        const int c = (int)fdiv((uint32_t)q, p.dT), tap = q - c * p.T;
        const int ky = (int)fdiv((uint32_t)tap, p.dTW), kx = tap - ky * p.TW;
        base = (c - c0) * p.pxs + ky * p.PW + kx;
    }
    // dY tasks: TF == 2: filters 16 w .. 16 w + 15, task j the quads 4 j .. 4 j + 3 of the stage's 16;
    // TF == 1: filters 16 (w % 2) .., quads 8 (w / 2) + 4 j ...
    const int fl = (TF == 2 ? wave : (wave & 1)) * 16 + (lane >> 2);  // filter within the block
    auto quads = [&](int j) RG_INLINE { return TF == 2 ? j : 2 * (wave >> 1) + j; };  // of 4 quads
    const int fse = sfil[fl];
    const RowScale frs = row_scale<S>(fse);
    const float fscale = __uint_as_float((uint32_t)(7 * (S - 1) - fse + 127) << 23);
    const bool fast = __ballot((!idle && sslow[wave * 32 + (lane & 31)] != 0) || sfslow[fl] != 0) == 0;
    const uint32_t frow = ft * BF + fl < p.F ? (uint32_t)((ft * BF + fl) * P) * 4u : NOWHERE;

    float d[TASKS][4];
    auto load_dy = [&](int s) RG_INLINE {
#pragma unroll
        for (int j = 0; j < TASKS; ++j) {
            const int qg = quads(j), step = 2 * s + (qg >> 1);
            const int c = (int)fdiv((uint32_t)step, p.dKS);
            const int e = tdy[(c & 3) * TABLE + (step - c * p.KS) * 8 + 4 * (qg & 1) + (lane & 3)];
            const bool live = e >= 0 && step < nsteps && frow != NOWHERE;
            const uint32_t off = live ? ((uint32_t)e & ~3u) + frow : NOWHERE;
            if (p.vec) {
                const v4i w = __builtin_amdgcn_raw_buffer_load_b128(drsrc, off, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) d[j][i] = __int_as_float(w[i]);
            } else {
                const int n = e & 3;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    d[j][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                        drsrc, i <= n ? off + 4u * i : NOWHERE, 0, 0));
            }
        }
    };
    auto round_word = [&](const float* v, float scale, const RowScale& rs, int (&xx)[4], auto FAST) RG_INLINE {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (decltype(FAST)::value) xx[i] = __float_as_int(__builtin_fmaf(v[i], scale, ROUND_MAGIC));
            else xx[i] = round_fixed(v[i], rs);
        }
    };
    // dY's digits of the held values into the panels of stage s: word j of filter fl's 16 bytes.
    auto write_dy = [&](int s, auto FAST) RG_INLINE {
        int* slot = reinterpret_cast<int*>(panels + (s & 1) * (PQ * 64));
#pragma unroll
        for (int j = 0; j < TASKS; ++j) {
            const int qg = quads(j);
            int xx[4];
            round_word(d[j], fscale, frs, xx, FAST);
            v4i w[S];
            pack_word<S>(xx, w, 0);
#pragma unroll
            for (int a = 0; a < S; ++a)
                slot[((((fl >> 5) * 2 + (qg >> 1)) * S + a) * 64 + (fl & 31) + 32 * (qg & 1)) * 4 + (lane & 3)] = w[a][0];
        }
    };
    // Patch offsets of this lane's four quads in a step, and one quad's values.
    auto x_quads = [&](int step) RG_INLINE {
        const int st = min(step, nsteps - 1);
        const int c = (int)fdiv((uint32_t)st, p.dKS);
        const v4i o = *reinterpret_cast<const v4i*>(tx + (c & 3) * TABLE + (st - c * p.KS) * 8 + 4 * (lane >> 5));
        return o + ((c & 1) * DW_SLOT + base);
    };
    auto read_quad = [&](float (&v)[4], int at) RG_INLINE {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = patch[at + i * SXT];
    };
    auto x_word = [&](const float (&v)[4], v4i (&b)[S], int w, auto FAST) RG_INLINE {
        int xx[4];
        round_word(v, pscale, prs, xx, FAST);
        pack_word<S>(xx, b, w);
    };
    // One step: digit a's panels are read while digit a - 1's products run; hook(i) goes between the
    // products, which run on their own (the fences keep that order).
    auto multiply = [&](const v4i (&fb)[S], int s, int kk, auto hook) RG_INLINE {
        const v4i* q = panels + (s & 1) * (PQ * 64) + lane;
        v4i fa[2][TF];
        auto read = [&](int a) RG_INLINE {
#pragma unroll
            for (int ti = 0; ti < TF; ++ti) fa[a & 1][ti] = q[((ti * 2 + kk) * S + a) * 64];
        };
        read(0);
#pragma unroll
        for (int a = 0; a < S; ++a) {
            if (a + 1 < S) read(a + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int b = 0; b < S; ++b) {
#pragma unroll
                for (int ti = 0; ti < TF; ++ti)
                    acc[a + b][ti] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[a & 1][ti], fb[b], acc[a + b][ti], 0, 0, 0);
                hook(a * S + b);
            }
        }
    };
    // Visible to the block after this: this wavefront's copies (dY loads issued since may stay in
    // flight) and LDS writes.
    auto publish = [&](bool loads) RG_INLINE {
        __builtin_amdgcn_sched_barrier(0);
        if (!loads) RG_WAIT_VMCNT(0);
        else if (p.vec) RG_WAIT_VMCNT(TASKS);
        else RG_WAIT_VMCNT(4 * TASKS);
        RG_WAIT_LGKMCNT0();
        asm volatile("s_barrier" ::: "memory");
    };
    auto pipeline = [&](auto FAST) RG_INLINE {
        constexpr int EVERY = S == 3 ? 2 : 1;
        load_dy(0);
        write_dy(0, FAST);
        if (stages > 1) load_dy(1);
        publish(stages > 1);
        int next = 2;
        for (int s = 0; s < stages; ++s) {
            if (next < nchunks && dw_due(next, p.KS, s)) {
                copy_patch(next);
                build_table(next + 2);
                ++next;
            }
            if (!idle) {
                v4i b0[S], b1[S];
                {
                    const v4i o = x_quads(2 * s);
                    float v[4][4];
#pragma unroll
                    for (int w = 0; w < 4; ++w) read_quad(v[w], o[w]);
#pragma unroll
                    for (int w = 0; w < 4; ++w) x_word(v[w], b0, w, FAST);
                }
                const v4i o = x_quads(2 * s + 1);
                float v[2][4];
                read_quad(v[0], o[0]);
                auto next_word = [&](int w) RG_INLINE {
                    if (w + 1 < 4) read_quad(v[(w + 1) & 1], o[w + 1]);
                    x_word(v[w & 1], b1, w, FAST);
                };
                multiply(b0, s, 0, [&](int i) RG_INLINE {
                    if (i % EVERY == 0 && i / EVERY < 4) {
                        __builtin_amdgcn_sched_barrier(0);
                        next_word(i / EVERY);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                });
                if (S * S < 4) {
#pragma unroll
                    for (int w = (S * S + EVERY - 1) / EVERY; w < 4; ++w) next_word(w);
                }
                multiply(b1, s, 1, [](int) RG_INLINE {});
            }
            if (s + 1 < stages) write_dy(s + 1, FAST);
            if (s + 2 < stages) load_dy(s + 2);
            publish(s + 2 < stages);
        }
    };
    if (fast) pipeline(std::true_type());
    else pipeline(std::false_type());

    // Exact sums of this part: register e of a tile holds filter 8 (e / 4) + 4 (lane / 32) + e % 4.
    if (idle || pos >= p.K) return;
    int64_t* out = reinterpret_cast<int64_t*>(ws + p.part) + (size_t)part * p.F * p.K + pos;
#pragma unroll
    for (int ti = 0; ti < TF; ++ti) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            int lv[L];
#pragma unroll
            for (int l = 0; l < L; ++l) lv[l] = acc[l][ti][e];
            const int f = ft * BF + ti * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
            if (f < p.F) out[(size_t)f * p.K] = combine_levels<L>(lv);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
#endif
}

template <int S>
void launch_s(const DwPlan& p, const float* dy, const float* x, char* ws, hipStream_t stream) {
    const unsigned blocks = (unsigned)(p.parts * p.ptiles * p.ftiles);
#define RG_DW(TF) \
    (p.SX == 1 ? dw_contract<S, TF, 1><<<blocks, 256, 0, stream>>>(p, dy, x, ws) \
               : dw_contract<S, TF, 2><<<blocks, 256, 0, stream>>>(p, dy, x, ws))
    if (p.tf == 2) RG_DW(2);
    else RG_DW(1);
#undef RG_DW
}

}  // namespace

bool dw_plan(const rg_conv_shape& s, int S, int num_cus, bool forced, DwPlan* out) {
    DwPlan p;
    std::memset(&p, 0, sizeof p);
    p.S = S; p.N = s.N; p.C = s.C; p.H = s.H; p.W = s.W; p.F = s.F;
    p.SY = s.SY; p.SX = s.SX; p.PY = s.PY; p.PX = s.PX;
    p.OH = (s.H + 2 * s.PY - s.KH) / s.SY + 1;
    p.OW = (s.W + 2 * s.PX - s.KW) / s.SX + 1;
    p.TH = s.KH; p.TW = s.KW; p.T = s.KH * s.KW; p.K = s.C * p.T;
    if (s.SX > 2 || s.KH > 31 || s.KW > 31) return false;
    // Offsets of x and dY in 32 bits.
    if ((double)p.N * p.C * p.H * p.W * 4.0 >= 2147483000.0) return false;
    if ((double)p.N * p.F * p.OH * p.OW * 4.0 >= 2147483000.0) return false;
    if ((double)p.F * p.K >= 1073741824.0) return false;
    // Channels of 128 neighbouring positions.
    const int nch = std::min(p.C, (DW_POS - 2 + p.T) / p.T + 1);
    // Strips and chunks: the widest strips whose patch fits with the fewest dead quads.
    double best = 0.0;
    for (int w = ceil_div(std::min(p.OW, 64 * DW_GROUPS), 4) * 4; w >= 4;) {
        // (width w from the widest that can fit, with the fewest strips it takes)
        const int ns = ceil_div(p.OW, w), sw = ceil_div(ceil_div(p.OW, ns), 4) * 4, sq = sw / 4;
        w = sw - 4;
        const double cols = (double)p.OW / ((double)ns * sw);
        const int pw = (sw - 1) * p.SX + p.TW;
        for (int rc = 1; rc <= 32; ++rc) {
            const int ks = std::max(2, ceil_div(rc * sq, 8));
            if (ks > DW_STEPS) break;
            const int cross = (rc + p.OH - 2) / p.OH;
            const long long nr = (long long)(rc - 1) * p.SY + p.TH + (long long)cross * std::max(0, p.TH - p.SY);
            const int groups = ceil_div(nr * pw, 64);
            const int pxs = 64 * groups + 20;  // (channels off the LDS banks of their neighbours)
            if (groups > DW_GROUPS || (long long)nch * pxs > DW_SLOT) break;
            // dead quads, and a little for source rows fetched again by the next chunk
            const double eff = cols * rc * sq / (8.0 * ks) - 0.01 * nr / (rc * p.SY);
            if (eff > best) {
                best = eff;
                p.NS = ns; p.SW = sw; p.SQ = sq; p.PW = pw; p.RC = rc; p.KS = ks;
                p.pxgroups = groups; p.pxs = pxs;
            }
        }
        if (p.NS && ns >= 2 * p.NS) break;
    }
    if (!p.NS) return false;
    p.PH = (p.OH - 1) * p.SY + p.TH;
    const double vrows = (double)p.N * p.NS * p.OH;
    if (vrows * (p.SY + p.TH) >= 1073741824.0) return false;
    p.vrows = (int)vrows;
    p.chunks = ceil_div(p.vrows, p.RC);
    p.tf = p.F > 32 ? 2 : 1;
    p.ptiles = ceil_div(p.K, DW_POS);
    p.ftiles = ceil_div(p.F, 32 * p.tf);
    p.vec = p.OW % 4 == 0 && p.SW % 4 == 0;
    // Parts along the windows: measured 1.45 us a k step for two blocks sharing a compute unit and
    // about 8 us a block besides; the parts' int64 sums are written and read at about 4 TB/s. At most
    // 2^31 / 48387 values of k a part (S = 3), so that every int32 level sum is exact.
    const int max_chunks = std::max(1, (S == 3 ? 44352 : S == 2 ? 66560 : 133120) / (32 * p.KS));
    const double tiles = (double)p.ptiles * p.ftiles, slots = 2.0 * num_cus, outs = (double)p.F * p.K;
    double cost = -1.0;
    // (Only the shortest part of each number of parts, until one round of blocks alone takes longer:
    // of all lengths 2-6 us of host time a call, of these 0.7-1.3.)
    for (int per = 1; per <= std::min(p.chunks, max_chunks);) {
        const int parts = ceil_div(p.chunks, per);
        const double round = 8.0 + 1.45 * per * p.KS;
        if (cost >= 0.0 && round >= cost) break;
        const double t = std::ceil(tiles * parts / slots) * round + outs * 16.0 * parts / 4.0e6;
        if (cost < 0.0 || t < cost) {
            cost = t;
            p.per_part = per;
            p.parts = parts;
        }
        if (parts == 1) break;
        per = ceil_div(p.chunks, parts - 1);
    }
    if (tiles * p.parts >= 1073741824.0) return false;
    // Maxima: enough blocks to keep the memory busy.
    p.pgroups = ceil_div((long long)p.H * p.W, DW_PIX);
    p.xgroups = (int)std::max<long long>(1, std::min<long long>(std::min(p.N, 64), ceil_div(2048, (long long)p.C * p.pgroups)));
    p.dgroups = (int)std::max<long long>(1, std::min<long long>(std::min(p.N, 64), ceil_div(1024, p.F)));
    if ((double)p.C * p.xgroups * p.pgroups + (double)p.F * p.dgroups >= 1073741824.0) return false;
    if (!forced) {
        // Against the GEMM pipeline (rg_conv_cost.h: how both were fitted, and what it replaced). With
        // many filters and few windows the pipeline is ahead, since it rounds every value once where
        // this kernel rounds it once per block of filters (32 x 512 x 7 x 7, 512 filters: 69 us against
        // 130 here). Terms: the launches, the k steps of the rounds of blocks (rounding, S^2 matrix
        // instructions per tile, dY by single values), the parts' sums, the maxima's reads and their
        // taps, the patches' copies, the maxima's groups, dY's reads by every position tile.
        const double steps = std::ceil(tiles * p.parts / slots) * p.per_part * p.KS, s9 = S * S / 9.0, M = 1.0e6;
        const double xs = (double)p.N * p.C * p.H * p.W, dys = (double)p.N * p.F * p.OH * p.OW;
        const double us = 12.0 + (0.25 + (p.tf == 2 ? 0.73 : 0.18) * s9 + (p.OW % 4 ? 0.26 : 0.0)) * steps +
                          5.0 * outs * p.parts / M + 1.2 * (xs + dys) / M +
                          0.017 * std::ceil(tiles * p.parts / slots) * p.per_part * p.pxgroups * nch +
                          300.0 * p.C * p.xgroups * p.pgroups * p.T / M + 0.2 * p.T + 0.065 * p.xgroups * p.pgroups +
                          0.29 * p.ptiles * dys / M;
        if (us > 0.97 * conv_pipeline_us(RG_CONV_GRAD_WEIGHT, s, S, num_cus)) return false;
    }
    p.dT = make_fastdiv((uint32_t)p.T);
    p.dTW = make_fastdiv((uint32_t)p.TW);
    p.dOH = make_fastdiv((uint32_t)p.OH);
    p.dPH = make_fastdiv((uint32_t)p.PH);
    p.dPW = make_fastdiv((uint32_t)p.PW);
    p.dSQ = make_fastdiv((uint32_t)p.SQ);
    p.dKS = make_fastdiv((uint32_t)p.KS);
    p.dNS = make_fastdiv((uint32_t)p.NS);
    p.dW = make_fastdiv((uint32_t)p.W);
    p.dSY = make_fastdiv((uint32_t)p.SY);
    p.dSX = make_fastdiv((uint32_t)p.SX);
    p.xmax = 0;
    p.dmax = align_up((size_t)p.xgroups * p.pgroups * p.K * sizeof(uint32_t));
    p.ea = p.dmax + align_up((size_t)p.dgroups * p.F * 2 * sizeof(uint32_t));
    p.eb = p.ea + align_up((size_t)p.F * sizeof(int));
    p.part = p.eb + align_up((size_t)p.K * sizeof(int));
    p.total = p.part + align_up((size_t)p.parts * p.F * p.K * sizeof(int64_t));
    *out = p;
    return true;
}

int dw_launch(const DwPlan& plan, const float* dy, const float* x, float* dw, char* ws, hipStream_t stream) {
    DwPlan p = plan;
    p.dvec = (reinterpret_cast<uintptr_t>(dy) & 15) == 0 && (p.OH * p.OW) % 4 == 0;
    p.xvec = (reinterpret_cast<uintptr_t>(x) & 15) == 0 && (p.H * p.W) % 4 == 0;
    p.vec = p.vec && p.dvec;
    dw_maxima<<<(unsigned)(p.C * p.xgroups * p.pgroups + p.F * p.dgroups), THREADS, 0, stream>>>(p, x, dy, ws);
    switch (p.S) {
        case 1: launch_s<1>(p, dy, x, ws, stream); break;
        case 2: launch_s<2>(p, dy, x, ws, stream); break;
        case 3: launch_s<3>(p, dy, x, ws, stream); break;
        default: return hipErrorInvalidValue;
    }
    Layout L;
    std::memset(&L, 0, sizeof L);
    L.S = p.S; L.M = p.F; L.N = p.K; L.batch = 1; L.split = p.parts; L.Mp = p.F; L.Np = p.K;
    launch_reduce_round(L, reinterpret_cast<const int64_t*>(ws + p.part), reinterpret_cast<const int*>(ws + p.ea),
                        reinterpret_cast<const int*>(ws + p.eb), dw, OutAddr{p.K, 0}, stream);
    return hipGetLastError();
}

}  // namespace rg
