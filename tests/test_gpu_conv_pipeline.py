"""GPU parity of the convolution's GEMM pipeline (im2col, slicing, contraction, the input gradient's
int64 products and col2im), forced on shapes that the automatic choice may give to other kernels:
the oracle's bits. Its callers are the shapes that the implicit GEMMs cannot take, or take longer for."""
import numpy as np
import pytest

import bit_reproducible_training_amd as rg
from gpu_util import note
from oracle import oracle as O
from test_gpu_conv import DIRECT_SHAPES, LENET, RC, _oracle, _run_algo
from test_gpu_nonfinite import NAN_ROUTE_SHAPES, _plant_nonfinite
from test_nonfinite import conv_oracle

pytestmark = pytest.mark.gpu


def _inputs(shape, seed):
    N, C, H, W, F, KH, KW = shape[:7]
    OH, OW = O.conv_out_hw(shape)
    rng = np.random.default_rng(seed)
    x = (rng.standard_normal(N * C * H * W) * 2.0 ** rng.integers(-20, 20, N * C * H * W)).astype(np.float32)
    x[rng.random(x.size) < 0.1] = 0.0
    w = (rng.standard_normal(F * C * KH * KW) * 0.1).astype(np.float32)
    dy = (rng.standard_normal((N, F * OH * OW)) * 2.0 ** rng.integers(-30, 30, (N, 1))).astype(np.float32)
    return x, w, dy.ravel()


def _check(torch, shape, S, seed):
    x, w, dy = _inputs(shape, seed)
    for kind, a, b in (("fwd", x, w), ("dW", dy, x), ("dX", dy, w)):
        note("conv pipeline", kind, shape, "S=%d" % S)
        got = _run_algo(torch, kind, a, b, shape, S, RC.ALGO_PIPELINE).view(np.uint32).ravel()
        assert np.array_equal(got, _oracle(kind, a, b, shape, S).view(np.uint32).ravel()), (kind, shape, S)


@pytest.mark.parametrize("S", [1, 2, 3])
def test_pipeline_matches_oracle(torch_gpu, S):
    # Beside the direct kernels' shapes: windows of 4680 values, too long for the one-pass slicing, so
    # that the forward pass packs the im2col matrix; column stride 3; 5x5 and 1x1 col2im.
    shapes = [s for s in DIRECT_SHAPES if S == 3 or s not in LENET]
    shapes += [(1, 520, 5, 5, 3, 3, 3, 1, 1, 1, 1), (3, 9, 20, 19, 33, 3, 3, 3, 3, 1, 1),
               (2, 33, 12, 12, 40, 5, 5, 1, 1, 2, 2), (3, 32, 9, 13, 70, 1, 1, 1, 1, 0, 0)]
    for i, shape in enumerate(shapes):
        _check(torch_gpu, shape, S, 100 * S + i)


def test_pipeline_beyond_65535_images(torch_gpu):
    """More images than a grid's y dimension holds: the [N][F][P] <-> [N*P][F] reorders fall back from
    the tiled transposes to their element-wise kernels."""
    _check(torch_gpu, (65537, 2, 3, 2, 3, 2, 1, 1, 1, 0, 0), 3, 65537)


@pytest.mark.parametrize("S", [1, 3])
@pytest.mark.parametrize("algo", [RC.ALGO_PIPELINE, RC.ALGO_FUSED])
def test_nonfinite_routes(torch_gpu, S, algo):
    """NaN and infinities on every slicing route of the pipeline (gathered and packed windows, one
    read in parts, two passes), and on the implicit GEMMs at the same shapes."""
    for si, shape in enumerate(NAN_ROUTE_SHAPES):
        N, C, H, W, F, KH, KW = shape[:7]
        OH, OW = O.conv_out_hw(shape)
        rng = np.random.default_rng(170 + 7 * S + si)
        x = rng.standard_normal((N, C, H, W)).astype(np.float32)
        w = rng.standard_normal((F, C, KH, KW)).astype(np.float32)
        dy = rng.standard_normal((N, F, OH, OW)).astype(np.float32)
        _plant_nonfinite(rng, x, 3)
        for kind, a, b in (("fwd", x, w), ("dW", dy, x)):
            if algo == RC.ALGO_FUSED and kind == "fwd" and C * KH * KW > 44352:
                with pytest.raises(rg.ReproGemmError):  # past its int32 level sums
                    RC.conv2d_algo_workspace(RC.FORWARD, RC.ConvShape(*shape), S, algo)
                continue
            note("nonfinite conv", kind, shape, "S=%d algo=%d" % (S, algo))
            got = _run_algo(torch_gpu, kind, a.ravel(), b.ravel(), shape, S, algo).view(np.uint32).ravel()
            want = conv_oracle(kind, x, w, dy, shape, S).view(np.uint32).ravel()
            assert np.array_equal(got, want), (kind, shape, S, algo)


def test_what_the_implicit_gemms_cannot_take(torch_gpu):
    for p, shape in ((RC.GRAD_INPUT, (2, 8, 20, 20, 16, 5, 5, 3, 3, 2, 2)),    # nine residues
                     (RC.GRAD_WEIGHT, (2, 8, 20, 20, 16, 3, 3, 1, 3, 1, 1)),   # column stride 3
                     (RC.FORWARD, (1, 2, 40, 8, 4, 33, 3, 1, 1, 0, 0))):       # 33 rows of taps
        g = RC.ConvShape(*shape)
        with pytest.raises(rg.ReproGemmError) as e:
            RC.conv2d_algo_workspace(p, g, 3, RC.ALGO_FUSED)
        assert e.value.code == 801
        assert RC.conv2d_algo_workspace(p, g, 3, RC.ALGO_PIPELINE) == RC.conv2d_algo_workspace(p, g, 3, RC.ALGO_GEMM)
