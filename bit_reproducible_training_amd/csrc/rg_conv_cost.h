#pragma once
// Estimated GPU times (microseconds) of the convolution's GEMM pipeline, to weigh the implicit GEMMs
// of rg_conv_fused.hip and rg_conv_dw.hip against; any choice gives the same bits. Internal to
// librepro_gemm.so, host only.
//
// Fitted by non-negative least squares on relative errors to 76000 (shape, S) pairs measured on
// MI355X on both routes: 1-2048 channels and filters, 1-128 images of 1-112 pixels a side, kernels
// 1-11, strides 1 and 2, S = 1-3. Median error 5-6% for the forward pass and the weight gradient, 8%
// for the input gradient; the implicit GEMMs' own estimates (fused_plan, dw_plan) are 4-6% off.
// Choosing by them costs 0.3-0.8% over the faster route of every shape in the geometric mean, and is
// more than 20% slower than the pipeline on 0.2-0.3% of the shapes. Fixed limits on padding, parts,
// strides and window length were that on 10% of the forward passes (deep channels over few windows:
// 1x64x56x56 to 256 filters 3x3 28 us against 24, 22x828x8x8 to 51 filters 7x7 stride 2 119 against
// 42) and on 6% of the weight gradients, and missed forward passes that are faster here (32x64x56x56
// to 128 filters 3x3 stride 2 44 us against 56).
#include <algorithm>
#include <cmath>

#include "repro_conv.h"
#include "rg_internal.h"

namespace rg {

// The contraction of M x N outputs over K: the better of 128x128 and 64x64 tiles (the stage and block
// times of the GEMM planner), unsplit, split to fill one round of blocks, or split in eight.
inline double conv_contraction_us(double M, double N, double K, int S, int num_cus) {
    const double steps = std::ceil(K / STEP_K);
    double best = 0.0;
    for (int t = 2; t >= 1; --t) {
        const double stage = 0.1 + ((t == 2 ? 1.276 : 0.803) - 0.1) * (S * S / 9.0), block = t == 2 ? 8.5 : 3.0;
        const double tiles = std::ceil(M / (64 * t)) * std::ceil(N / (64 * t));
        const int lds = 12 * t * 2 * S * PANEL_BYTES;
        const double slots = (double)num_cus * std::max(1, std::min(2, 160 * 1024 / lds));
        const double splits[3] = {1.0, std::max(1.0, std::min(steps, std::floor(slots / tiles))), std::min(steps, 8.0)};
        for (const double sp : splits) {
            double us = std::ceil(tiles * sp / slots) * (std::ceil(steps / sp) * stage + block);
            if (sp > 1.0) us += 3.0 + M * N * (8.0 * (sp + 1.0) + 4.0) / 4.0e6;
            if (best == 0.0 || us < best) best = us;
        }
    }
    return best;
}

// Million values, thousands of windows: the units of the terms below.
inline double conv_pipeline_us(int pass, const rg_conv_shape& s, int S, int num_cus) {
    const double OH = (s.H + 2 * s.PY - s.KH) / s.SY + 1, OW = (s.W + 2 * s.PX - s.KW) / s.SX + 1;
    const double T = (double)s.KH * s.KW, K = s.C * T, win = s.N * OH * OW, F = s.F, M = 1.0e6;
    if (pass == RG_CONV_FORWARD) {
        // Slicing of windows and filters (gathered; past the one-pass slicing packed first), the
        // slicing's chain along K, the outputs' transpose.
        const double Kp = STEP_K * std::ceil(K / STEP_K), cols = win * Kp / M, outs = win * F / M;
        const double windows = Kp <= ONEPASS_MAX_K ? (0.77 + 0.23 * S) * cols + 1.5 * std::min(cols, 1.0) : 7.7 + 2.6 * cols;
        return 8.9 + 0.8 * conv_contraction_us(win, F, K, S, num_cus) + windows + 1.2 * F * Kp / M + 2.4 * outs +
               1.8 * std::min(outs, 0.5) + 2.2 * std::min(Kp, (double)ONEPASS_MAX_K) / 1e3 + 0.01 * win / 1e3;
    }
    if (pass == RG_CONV_GRAD_WEIGHT)  // packing and slicing of windows and dY
        return 15.0 + 0.83 * conv_contraction_us(F, K, win, S, num_cus) + 2.8 * win * K / M + 3.7 * win * F / M +
               0.22 * win / 1e3 + 0.62 * F * K / M + 1.7 * std::min(win, 4096.0) / 1e3 + (win > 4096.0 ? 1.5 : 0.0);
    // Input gradient: slicing of dY, the column slicing of the weights under one scale (slow already
    // for a million of them), the int64 products, and col2im's reads of them.
    const double pixels = (double)s.N * s.C * s.H * s.W;
    return 15.0 + 0.79 * conv_contraction_us(K, win, F, S, num_cus) + 0.95 * win * K / M + 4.5 * win * F / M +
           2.2 * pixels / M + 0.66 * pixels * T / M + 0.35 * T + 0.68 * F * K / M + 54.0 * std::min(F * K / M, 1.0) +
           0.014 * std::sqrt(F * K) + 0.23 * win / 1e3;
}

}  // namespace rg
