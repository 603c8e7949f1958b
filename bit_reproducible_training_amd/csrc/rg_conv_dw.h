#pragma once
// The convolution's weight gradient as one contraction over the windows whose kernel rounds both
// operands itself (rg_conv_dw.hip). Internal to librepro_gemm.so.
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "repro_conv.h"
#include "rg_fastdiv.h"

namespace rg {

struct DwPlan {
    int S, N, C, H, W, F, SY, SX, PY, PX, OH, OW;
    int TH, TW, T, K;          // taps; K = C * T positions of a window
    int NS, SW, SQ;            // column strips of the output, their width, its quads (4 columns)
    int PH, PW;                // padded source rows of an (image, strip), their length
    int vrows;                 // N * NS * OH output rows
    int RC, KS;                // output rows per chunk, k steps (8 quads) per chunk
    int chunks, per_part, parts;
    int pxgroups, pxs;         // patch values per channel / 64, LDS distance of channels
    int tf, ptiles, ftiles;
    int vec;                   // rows of dY keep 16-byte quads (given an aligned base)
    int xvec, dvec;            // the maxima read x, dY by 16-byte loads
    // maxima
    int xgroups, pgroups, dgroups;  // image groups and pixel groups of x; image groups of dY
    FastDiv dT, dTW, dOH, dPH, dPW, dSQ, dKS, dNS, dW, dSY, dSX;
    size_t xmax, dmax, ea, eb, part, total;  // workspace offsets
};

// Schedule of dw_contract's two patch slots: whether chunk c >= 2 is copied (and table c + 2 built)
// during stage s, all KS steps of chunk c - 2 lying before it. That comes a stage before chunk c's own
// first, floor(c KS / 2), for KS >= 2.
__host__ __device__ inline bool dw_due(int c, int KS, int s) { return (c - 1) * KS <= 2 * s; }

// Fills *plan and returns true when the fused kernels take this weight gradient (a valid shape): where
// they are faster than the GEMM pipeline, or with `forced` wherever they can.
bool dw_plan(const rg_conv_shape& s, int S, int num_cus, bool forced, DwPlan* plan);

int dw_launch(const DwPlan& p, const float* dy, const float* x, float* dw, char* ws, hipStream_t stream);

}  // namespace rg
