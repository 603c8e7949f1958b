#pragma once
// The convolution's forward pass and input gradient as one implicit GEMM whose kernel quantises
// the gathered values itself (rg_conv_fused.hip). Internal to librepro_gemm.so.
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "repro_conv.h"
#include "rg_fastdiv.h"

namespace rg {

// One class of output positions that read the same taps: all of them (forward; input gradient
// at stride 1), or the pixels of one residue (y mod SY, x mod SX) of a strided input gradient.
// Grid position (gy, gx) of a class samples the source at (gy * sy + y0 + ty, gx * sx + x0 + tx)
// for its taps (ty, tx), and is the output pixel (gy * osy + oy, gx * osx + ox).
struct FusedClass {
    int GH, GW, P;         // grid, P = GH * GW positions per image
    int rows;              // N * P
    int y0, x0, TH, TW, T;
    int oy, ox;
    int groups, stages;    // k in groups of 16 channels of one tap; stages of 4 groups
    int padoff;            // bytes: keeps the lanes' offsets non-negative
    int wt0, wt1, wtx;     // weight of tap (ty, tx): offset wt0 + ty * wt1 + tx * wtx
    int tiles, qchunks;    // window tiles; chunks of a weight strip
    int block0, qblock0;   // first block of the class (contraction; weight slicing)
    uint32_t qoff;         // byte offset of its weight panels
    FastDiv dP, dGW, dT, dTW;
    // Patch kernel (FusedPlan::patch): the grid's columns are cut into NS strips of GW (P = GH * GW
    // positions a strip, rows = N * NS * P), and a block's patch takes pxgroups * 64 values.
    int NS, pxgroups;
    FastDiv dNS, dPW, dPH;
};

// Source values per channel that a block of the patch kernel holds in LDS.
constexpr int FUSED_PATCH_PX = 384;

constexpr int FUSED_MAX_CLASSES = 4;

struct FusedPlan {
    int input_grad, S;
    int N, C, H, W;        // source tensor (x, or dY with C = the layer's filters)
    int F;                 // output channels (filters, or the layer's input channels)
    int sy, sx;            // source coordinates per grid step
    int OW, OPL, osy, osx; // output plane: row length, pixels; output pixels per grid step
    int wrs, wcs;          // weight strides: output channel, source channel
    int wrow;              // weights per filter (forward: one scale per filter)
    long long wcount;      // all weights (input gradient: one scale for all)
    int patch;             // fused_patch (overlapping taps at stride 1) instead of fused_contract
    int nclass;
    FusedClass cls[FUSED_MAX_CLASSES];
    int tf, nwf, nww;      // block: 32 * nww windows x 32 * tf * nwf output channels
    int ftiles, blocks, qblocks;
    int maxima_blocks, img_parts, w_parts, img_chunk;
    int exact;             // horner_exact for every sum
    uint32_t qbytes;
    int split;             // parts along k
    FastDiv dHW, dblocks, dOPL, dF;
    size_t q, ef, maxima, imax, ew, part, total;  // workspace offsets
};

// Schedule of fused_patch's two patch slots (channel group cg in slot cg % 2), for a part of k from
// stage s0 on: how many groups, from the first it reads on, are copied before its first stage, and
// whether a later group cg is copied during stage s (at most one a stage): its slot is free, the last k
// group of cg - 2 lying before the stage. That comes a stage before cg's own first, floor(cg T / 4),
// for T = 4 and for every T >= 6 taps.
__host__ __device__ inline int patch_first(int s0) { return s0 > 0 ? 2 : 1; }
__host__ __device__ inline bool patch_due(int cg, int T, int s) { return cg < 2 || (cg - 1) * T <= 4 * s; }

// Fills *plan and returns true when the fused kernels take this pass (kind: RG_CONV_FORWARD or
// RG_CONV_GRAD_INPUT; the shape is valid): where they are faster than the GEMM pipeline, or with
// `forced` wherever they can.
bool fused_plan(int kind, const rg_conv_shape& s, int S, int num_cus, bool forced, FusedPlan* plan);

// a: x (forward) or dY; w: the layer's weights; bias: one float per output channel, added to the
// rounded outputs, or null; out: y or dX.
int fused_launch(const FusedPlan& p, const float* a, const float* w, const float* bias, float* out,
                 char* ws, hipStream_t stream);

}  // namespace rg
