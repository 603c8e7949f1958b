"""The layers' fused forms against the operations they combine: the bias added where the outputs are
rounded, the gradient's check in the bias sum's read, two checks in one launch. Bits are equal."""
import ctypes

import pytest
import torch

import bit_reproducible_training_amd as rg
from bit_reproducible_training_amd import _lib
from bit_reproducible_training_amd._lib import _backend, lib
from test_conv_fused_plan import FWD, fused

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.contiguous().view(torch.int32)


def _bias(n):
    b = torch.randn(n, device="cuda")
    b[0] = 0.0
    b[-1] = -0.0
    if n > 3:
        b[1], b[2] = 3e38, 1e-41
    return b


# One output up to several tiles of each contraction: the one-launch kernel, the row band, the
# tiles with full and partial edges, and split reductions of each thread count.
GEMMS = [(1, 1, 1), (64, 64, 64), (33, 65, 100), (512, 96, 200), (4096, 100, 64), (2048, 768, 768),
         (1024, 2304, 768), (130, 129, 1000), (128, 128, 1024), (128, 128, 65536), (77, 33, 30000),
         (999, 1003, 513)]


@pytest.mark.parametrize("M,N,K", GEMMS)
@pytest.mark.parametrize("S", [1, 2, 3])
def test_linear_bias_is_one_addition_after_the_gemm(M, N, K, S):
    torch.manual_seed(M + N + K)
    x, w, b = torch.randn(M, K, device="cuda"), torch.randn(N, K, device="cuda"), _bias(N)
    x[0] = 0.0  # zero outputs: +0.0 + -0.0
    want = rg.gemm(x, w, M, N, K, False, True, S) + b
    assert torch.equal(_bits(_backend.linear(x, w, b, M, N, K, S)), _bits(want))
    # Biases the kernels do not read: another stride, a broadcast shape.
    strided = torch.empty(N, 2, device="cuda")[:, 0].copy_(b)
    assert torch.equal(_bits(_backend.linear(x, w, strided, M, N, K, S)), _bits(want))
    one = b.view(1, N)
    assert torch.equal(_bits(_backend.linear(x, w, one, M, N, K, S)), _bits(want))


def test_a_lazily_negated_bias_is_its_value():
    """A negated view's memory holds the opposite values; the layers' biases may be such views."""
    x, w, b = torch.randn(5, 40, device="cuda"), torch.randn(8, 40, device="cuda"), _bias(8)
    neg = torch._neg_view(b)
    assert neg.is_neg() and neg.is_contiguous()
    want = rg.gemm(x, w, 5, 8, 40, False, True, 3) + neg
    assert torch.equal(_bits(_backend.linear(x, w, neg, 5, 8, 40, 3)), _bits(want))
    xc, wc = torch.randn(2, 3, 6, 6, device="cuda"), torch.randn(8, 3, 3, 3, device="cuda")
    want = rg.conv2d(xc, wc, 1, 1, 0, 0, 3) + neg.view(1, -1, 1, 1)
    assert torch.equal(_bits(_backend.conv2d_bias(xc, wc, neg, 1, 1, 0, 0, 3)), _bits(want))


@pytest.mark.parametrize("algo", list(rg.Algo))
@pytest.mark.parametrize("split_k", [1, 3])
def test_bias_entry_point_over_algorithms(algo, split_k):
    M, N, K = 130, 70, 300
    A, B, b = torch.randn(M, K, device="cuda"), torch.randn(K, N, device="cuda"), _bias(N)
    cfg = rg.Config(algo=algo, split_k=split_k)
    want = rg.gemm(A, B, M, N, K, cfg=cfg) + b
    plan = rg.make_plan(M, N, K, cfg)
    ws = torch.empty(max(plan.workspace_bytes, 1), dtype=torch.uint8, device="cuda")
    C = torch.empty(M, N, device="cuda")
    c = cfg.to_c()
    stream = torch.cuda.current_stream().cuda_stream
    args = (C.data_ptr(), M, N, K, ctypes.byref(c), ws.data_ptr(), ws.numel(), stream)
    assert lib.rg_gemm_bias_fp32_ws(A.data_ptr(), B.data_ptr(), b.data_ptr(), *args) == 0
    assert torch.equal(_bits(C), _bits(want))
    assert lib.rg_gemm_bias_fp32_ws(A.data_ptr(), B.data_ptr(), None, *args) == 1


# (N, C, H, W, F, K, stride, padding): direct, window gather (1x1), patch, the GEMM pipeline, one output
# pixel, channel counts off the tiles. The route that each of CONV_ROUTES takes is asserted beside it.
CONVS = [(100, 6, 14, 14, 16, 5, 1, 0), (2, 3, 9, 9, 5, 3, 1, 1), (4, 64, 28, 28, 70, 1, 1, 0),
         (4, 64, 28, 28, 128, 3, 2, 1), (4, 64, 28, 28, 64, 3, 1, 1), (3, 40, 17, 19, 33, 3, 1, 1),
         (2, 512, 7, 7, 512, 3, 1, 1), (8, 256, 14, 14, 256, 3, 2, 0), (64, 16, 5, 5, 120, 5, 1, 0)]


@pytest.mark.parametrize("shape", CONVS)
@pytest.mark.parametrize("S", [1, 3])
def test_conv_bias_is_one_addition_after_the_convolution(shape, S):
    N, C, H, W, F, K, s, p = shape
    torch.manual_seed(sum(shape))
    x, w, b = torch.randn(N, C, H, W, device="cuda"), torch.randn(F, C, K, K, device="cuda"), _bias(F)
    want = rg.conv2d(x, w, s, s, p, p, S) + b.view(1, -1, 1, 1)
    assert torch.equal(_bits(_backend.conv2d_bias(x, w, b, s, s, p, p, S)), _bits(want))


# The same with its route: (holds patches, has parts along k, several taps), the window gather's and the
# patches' reductions of parts among them; None: the GEMM pipeline.
CONV_ROUTES = [((16, 64, 28, 28, 8, 2, 2, 1), (0, False, True)), ((8, 64, 28, 28, 33, 1, 1, 0), (0, False, False)),
               ((1, 4200, 3, 3, 33, 1, 2, 0), (0, True, False)), ((1, 512, 3, 3, 33, 3, 2, 1), (0, True, True)),
               ((8, 64, 28, 28, 33, 2, 1, 1), (1, False, True)), ((1, 1024, 3, 3, 33, 2, 1, 1), (1, True, True)),
               ((4, 64, 28, 28, 128, 3, 2, 1), None), ((1, 750, 8, 7, 200, 5, 2, 2), None)]


@pytest.mark.parametrize("shape,route", CONV_ROUTES)
@pytest.mark.parametrize("S", [1, 3])
def test_conv_bias_on_every_route(shape, route, S):
    N, C, H, W, F, K, s, p = shape
    plan = fused(FWD, (N, C, H, W, F, K, K, s, s, p, p))
    taken = (plan["patch"], plan["split"] > 1, plan["taps"] > 1) if plan["taken"] else None
    assert taken == route
    test_conv_bias_is_one_addition_after_the_convolution(shape, S)


# (A, B, C) of sums over A and C: columns and segments, one chunk and several, few and many.
SUMS = [(1, 1, 1), (7, 65, 1), (5000, 33, 1), (100000, 3, 1), (1, 9, 64), (3, 5, 7), (100, 16, 100),
        (64, 4, 3136), (2, 700, 13)]


@pytest.mark.parametrize("A,B,C", SUMS)
@pytest.mark.parametrize("bad", [None, float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("wide", [False, True])
def test_sum_watch_reports_what_the_scan_reports(A, B, C, bad, wide):
    torch.manual_seed(A + B + C)
    x = torch.randn(A, B, C, device="cuda")
    if wide:  # the superaccumulator's range
        x.view(-1)[::2] *= 1e30
        x.view(-1)[0] = 1e-38
    n = x.numel()
    for at in ({0, n // 2, n - 1} if bad is not None else {0}):
        y = x.clone()
        if bad is not None:
            y.view(-1)[at] = bad
        clean, flag = (torch.full((1,), 9, dtype=torch.int32, device="cuda") for _ in range(2))
        rg.scan_finite(y, clean, 4)
        out = _backend.exact_sum_watch(y, A, B, C, flag, 4)
        assert int(flag) == int(clean) == (9 if bad is None else 4)
        assert torch.equal(_bits(out), _bits(rg.exact_sum(y, A, B, C)))
        low = torch.full((1,), 2, dtype=torch.int32, device="cuda")
        _backend.exact_sum_watch(y, A, B, C, low, 4)
        assert int(low) == 2


@pytest.mark.parametrize("nx,ny", [(1, 1), (0, 5), (5, 0), (0, 0), (4096, 3), (70001, 5000), (3, 1 << 20)])
@pytest.mark.parametrize("offset", [0, 1])
def test_pair_scan_is_two_scans(nx, ny, offset):
    def check(bx, by, want):
        x, y = torch.ones(nx + 1, device="cuda")[offset:nx + offset], torch.ones(ny, device="cuda")
        if bx is not None:
            x[bx] = float("nan")
        if by is not None:
            y[by] = float("-inf")
        flag = torch.full((1,), 99, dtype=torch.int32, device="cuda")
        _backend.scan_finite_pair(x, 7, y, 3, flag)
        assert int(flag) == want
    check(None, None, 99)
    if nx:
        check(nx - 1, None, 7)
        check(0, None, 7)
    if ny:
        check(None, ny - 1, 3)
        check(None, 0, 3)
    if nx and ny:
        check(nx - 1, ny - 1, 3)


@pytest.mark.parametrize("frozen_bias", [False, True])
def test_a_bad_gradient_is_reported_with_and_without_its_bias_sum(frozen_bias):
    guard = rg.guard()
    guard.reset()
    for layer, x in ((rg.Linear(5, 3).cuda(), torch.randn(4, 5, device="cuda")),
                     (rg.Conv2d(2, 3, 3).cuda(), torch.randn(2, 2, 5, 5, device="cuda"))):
        layer.bias.requires_grad_(not frozen_bias)
        y = layer(x)
        g = torch.ones_like(y)
        g.view(-1)[1] = float("nan")
        y.backward(g)
        with pytest.raises(FloatingPointError, match="gradient"):
            guard.check()
        guard.reset()
