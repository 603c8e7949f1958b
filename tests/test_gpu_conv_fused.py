"""GPU parity of the fused convolution kernels (forward pass and both gradients) with the oracle,
bit for bit, at the sizes where they can go wrong: blocks and patches that span images and column
strips, tiles cut by the last position and channel, channel counts off a group of 16, parts along
k, residue classes of a strided input gradient (some without taps), kernels larger than the image,
output rows that are not whole quads, scales past one normal float, NaN and infinities."""
import numpy as np
import pytest

from gpu_util import note
from oracle import oracle as O
from test_conv_fused_plan import DW, DX, FWD, fused
from test_gpu_conv import RC, _oracle, _run_algo

pytestmark = pytest.mark.gpu

# shape: (N, C, H, W, F, KH, KW, SY, SX, PY, PX)
SHAPES = [
    (2, 16, 8, 8, 16, 3, 3, 1, 1, 1, 1),        # one position past a block
    (9, 20, 7, 7, 40, 3, 3, 1, 1, 1, 1),        # blocks over several images
    (1, 16, 20, 112, 40, 3, 3, 1, 1, 1, 1),     # two column strips
    (1, 18, 9, 131, 16, 3, 3, 1, 1, 0, 1),      # strips with dead columns
    (1, 40, 30, 30, 24, 5, 5, 1, 1, 2, 2),
    (2, 33, 12, 12, 16, 2, 2, 1, 1, 0, 0),      # four taps
    (1, 50, 13, 40, 17, 7, 7, 1, 1, 3, 3),
    (1, 35, 16, 16, 70, 2, 3, 1, 1, 1, 0),      # six taps, 70 channels (a second tile, ragged)
    (3, 32, 40, 13, 130, 1, 1, 1, 1, 0, 0),     # one tap
    (1, 600, 6, 6, 65, 3, 3, 1, 1, 1, 1),       # parts along k
    (4, 20, 20, 20, 70, 5, 5, 2, 2, 2, 2),      # four residue classes
    (2, 17, 17, 19, 9, 3, 5, 2, 1, 0, 2),
    (2, 40, 11, 11, 24, 1, 1, 2, 2, 0, 0),      # classes without taps
    (1, 16, 3, 3, 16, 3, 3, 1, 1, 3, 3),        # padding wider than the image
    (2, 16, 3, 4, 20, 9, 9, 1, 1, 4, 4),        # kernel larger than the image
    (5, 16, 7, 7, 16, 4, 4, 1, 2, 3, 0),
    (40, 3, 28, 28, 6, 5, 5, 1, 1, 2, 2),       # weight gradient: one of four wavefronts has positions
    (2, 30, 56, 56, 40, 3, 3, 1, 1, 1, 1),      # three position tiles, the last ragged
    (1, 3, 50, 300, 20, 3, 3, 2, 2, 1, 1),      # column stride 2, strips
    (9, 20, 24, 22, 33, 3, 3, 3, 1, 0, 0),      # row stride 3, rows of 20 columns
]


# The window gather with several taps: strides, padding, one and several parts along k, channels off a
# group of 16, taps beyond every source row, 31 taps a side.
GATHERS = [
    (1, 256, 9, 9, 70, 7, 7, 2, 2, 3, 3),
    (1, 512, 7, 7, 40, 3, 3, 2, 2, 1, 1),
    (1, 4200, 5, 5, 33, 1, 1, 1, 1, 0, 0),
    (2, 20, 13, 17, 33, 5, 3, 3, 2, 2, 0),
    (3, 5, 11, 9, 12, 3, 3, 2, 1, 1, 1),
    (2, 16, 3, 40, 16, 31, 2, 1, 2, 15, 1),
    (1, 33, 2, 2, 130, 5, 5, 1, 2, 2, 2),
    (1, 18, 4, 140, 20, 1, 31, 1, 3, 0, 15),
]


def _inputs(shape, seed):
    N, C, H, W, F, KH, KW = shape[:7]
    OH, OW = O.conv_out_hw(shape)
    rng = np.random.default_rng(seed)
    x = (rng.standard_normal(N * C * H * W) * 2.0 ** rng.integers(-12, 12, N * C * H * W)).astype(np.float32)
    w = (rng.standard_normal(F * C * KH * KW) * 0.1).astype(np.float32)
    dy = (rng.standard_normal((N, F * OH * OW)) * 2.0 ** rng.integers(-30, 30, (N, 1))).astype(np.float32)
    return x, w, dy.ravel()


def _check(torch, shape, S, x, w, dy):
    for kind, a, b in (("fwd", x, w), ("dX", dy, w), ("dW", dy, x)):
        note("fused conv", kind, shape, "S=%d" % S)
        got = _run_algo(torch, kind, a, b, shape, S, RC.ALGO_FUSED).view(np.uint32).ravel()
        assert np.array_equal(got, _oracle(kind, a, b, shape, S).view(np.uint32).ravel()), (kind, shape, S)


@pytest.mark.parametrize("S", [1, 2, 3])
def test_fused_matches_oracle(torch_gpu, S):
    for i, shape in enumerate(SHAPES):
        _check(torch_gpu, shape, S, *_inputs(shape, 10 * S + i))


@pytest.mark.parametrize("S", [1, 2, 3])
def test_gathered_taps_match_oracle(torch_gpu, S):
    for i, shape in enumerate(GATHERS):
        x, w, dy = _inputs(shape, 1000 + 10 * S + i)
        if i % 2:
            x[np.random.default_rng(i).integers(0, x.size, 4)] = [np.nan, np.inf, -np.inf, 1e-40]
        note("fused gather", shape, "S=%d" % S)
        got = _run_algo(torch_gpu, "fwd", x, w, shape, S, RC.ALGO_FUSED).view(np.uint32).ravel()
        assert np.array_equal(got, _oracle("fwd", x, w, shape, S).view(np.uint32).ravel()), (shape, S)


# Planes and rows of whole quads, which the weight gradient reads by 16-byte loads from aligned bases.
QUADS = [(2, 16, 8, 8, 16, 3, 3, 1, 1, 1, 1), (3, 9, 12, 16, 40, 3, 3, 1, 1, 1, 1),
         (2, 17, 17, 32, 33, 3, 4, 2, 2, 1, 1), (1, 20, 4, 64, 6, 1, 1, 1, 1, 0, 0)]


@pytest.mark.parametrize("offset_a,offset_b", [(0, 0), (1, 0), (0, 1), (1, 3)])
def test_bases_off_16_bytes(torch_gpu, offset_a, offset_b):
    """Operands that start 0, 4 or 12 bytes past a 16-byte boundary: the loads by quads of either
    operand, or of both, give way to single ones."""
    torch = torch_gpu
    stream = torch.cuda.current_stream().cuda_stream
    assert any(fused(DW, s, forced=True)["taken"] and O.conv_out_hw(s)[1] % 4 == 0 for s in QUADS)
    for shape in QUADS:
        g = RC.ConvShape(*shape)
        x, w, dy = _inputs(shape, 31)
        for kind, p, a, b in (("fwd", RC.FORWARD, x, w), ("dW", RC.GRAD_WEIGHT, dy, x), ("dX", RC.GRAD_INPUT, dy, w)):
            want = _oracle(kind, a, b, shape, 3).view(np.uint32).ravel()
            da, db = (torch.empty(v.size + 4, device="cuda")[o:o + v.size].copy_(torch.from_numpy(v))
                      for v, o in ((a, offset_a), (b, offset_b)))
            assert da.data_ptr() % 16 == 4 * offset_a and db.data_ptr() % 16 == 4 * offset_b
            for algo in (RC.ALGO_FUSED, RC.ALGO_PIPELINE):
                note("conv bases", kind, shape, offset_a, offset_b, "algo=%d" % algo)
                out = torch.full((want.size,), float("nan"), device="cuda")
                ws = torch.empty(RC.conv2d_algo_workspace(p, g, 3, algo), dtype=torch.uint8, device="cuda")
                assert RC.repro_conv2d_algo_ws(p, da.data_ptr(), db.data_ptr(), out.data_ptr(), g, 3, algo,
                                               ws.data_ptr(), ws.numel(), stream) == 0
                assert np.array_equal(out.cpu().numpy().view(np.uint32), want), (kind, shape, algo)


def test_shapes_cover_the_routes():
    plans = [(p, fused(p, s, forced=True)) for s in SHAPES for p in (FWD, DX)]
    for pass_ in (FWD, DX):
        mine = [f for p, f in plans if p == pass_ and f["taken"]]
        assert any(f["patch"] and f["split"] == 1 for f in mine)
        assert any(f["split"] > 1 for f in mine)
        assert any(not f["patch"] for f in mine)
        assert any(f["strips"] > 1 for f in mine)
        assert {f["tf"] for f in mine} == {1, 2}
    mine = [(s, f) for s in SHAPES for f in [fused(DW, s, forced=True)] if f["taken"]]
    assert len(mine) >= 10 and any(f["strips"] > 1 for _, f in mine) and {f["tf"] for _, f in mine} == {1, 2}
    gathers = [fused(FWD, s, forced=True) for s in GATHERS]
    assert all(f["taken"] and not f["patch"] for f in gathers)
    for several_taps, parts in ((True, False), (True, True), (False, True)):
        assert any((f["taps"] > 1) == several_taps and (f["split"] > 1) == parts for f in gathers)
    assert {s[8] for s, _ in mine} == {1, 2} and any((s[3] + 2 * s[10] - s[6]) // s[8] % 4 != 3 for s, _ in mine)


@pytest.mark.parametrize("what", ["tiny", "huge", "nonfinite"])
def test_fused_slow_rounding(torch_gpu, what):
    """Rows whose scale is not one normal float (maxima below 2^-100 or near 2^127) and values
    that are not finite leave the one-multiply-add rounding."""
    for shape in (SHAPES[1], SHAPES[9], SHAPES[10], SHAPES[17]):
        x, w, dy = _inputs(shape, 77)
        rng = np.random.default_rng(5)
        for t in (x, dy):
            if what == "tiny":
                t *= np.float32(2.0 ** -125)
            elif what == "huge":
                hit = rng.random(t.size) < 0.3
                t[hit] = np.where(rng.random(hit.sum()) < 0.5, 3e38, -1e38)
            else:
                t[rng.integers(0, t.size, 3)] = np.nan
                t[rng.integers(0, t.size, 2)] = np.inf
        _check(torch_gpu, shape, 3, x, w, dy)
