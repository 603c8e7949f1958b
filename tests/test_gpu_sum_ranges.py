"""The exact sum's binary64 accumulation at the edges of its exactness bound, against the oracle bit
for bit: value ranges just inside and outside what a batch, a thread and a wave may add, ranges that
grow while a thread sums, zeros and subnormals, rows shorter than a wave, and NaN or infinities on
every path."""
import numpy as np
import pytest

import bit_reproducible_training_amd as rg
from gpu_util import bits, note, to_dev
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# (A, B, C): one row per wave, rows in fours and not, single and several chunks, columns, few rows of
# columns (a batch of four for each of the block's phases, of 16, rests of either)
SHAPES = [(1, 5, 3), (1, 3, 64), (1, 4, 260), (3, 5, 7), (7, 3, 1000), (2, 2, 20000), (1, 1, 300001),
          (70, 65, 1), (3000, 130, 1), (1, 1, 1), (5, 66, 1), (16, 64, 1), (17, 70, 1), (63, 5, 1), (130, 9, 1)]


def _values(kind, n, rng):
    x = rng.standard_normal(n).astype(np.float32)
    if kind.startswith("spread"):  # magnitudes in 2^0 .. 2^s, both ends present
        s = int(kind[6:])
        x = (np.sign(x) * rng.uniform(1, 2, n) * 2.0 ** rng.integers(0, s + 1, n)).astype(np.float32)
        x[rng.integers(0, n)] = np.float32(-1.0)
        x[rng.integers(0, n)] = np.float32(2.0 ** s)
    elif kind == "grow":           # each part of the row larger than what went before
        x *= (2.0 ** (np.arange(n) * 200.0 / n - 100)).astype(np.float32)
    elif kind == "wild":
        x *= (2.0 ** rng.integers(-120, 120, n)).astype(np.float32)
        x[rng.random(n) < 0.2] = 0.0
    elif kind == "subnormal":
        x = (rng.integers(-1000, 1000, n) * 2.0 ** -149).astype(np.float32)
        x[rng.random(n) < 0.1] = np.float32(2.0 ** -120)
    elif kind == "cancel":
        x[n // 2:] = -x[:n - n // 2][::-1]
    elif kind == "huge":
        x = np.where(x > 0, np.float32(3.0e38), np.float32(-2.9e38)).astype(np.float32)
    elif kind == "zeros":
        x = np.where(x > 0, np.float32(0.0), np.float32(-0.0))
    return x


KINDS = ["spread13", "spread24", "spread25", "spread26", "spread29", "grow", "wild", "subnormal", "cancel",
         "huge", "zeros"]


@pytest.mark.parametrize("kind", KINDS)
def test_sum_ranges_match_oracle(torch_gpu, kind):
    for A, B, C in SHAPES:
        x = _values(kind, A * B * C, np.random.default_rng(A + 7 * B + 13 * C))
        for mean in (False, True):
            note("sum", kind, (A, B, C), mean)
            got = rg.exact_sum(to_dev(torch_gpu, x), A, B, C, mean)
            want = O.exact_sum(x, A, B, C, mean)
            assert np.array_equal(bits(got), want.view(np.uint32)), (kind, A, B, C, mean)


@pytest.mark.parametrize("special", [np.nan, np.inf, -np.inf])
def test_sum_of_nonfinite_values_is_nan(torch_gpu, special):
    for A, B, C in SHAPES:
        for kind in ("spread13", "wild", "huge"):
            x = _values(kind, A * B * C, np.random.default_rng(3)).reshape(A, B, C)
            x[-1, B // 2, -1] = special
            note("sum nonfinite", kind, (A, B, C), special)
            got = bits(rg.exact_sum(to_dev(torch_gpu, x.ravel()), A, B, C))
            want = O.exact_sum(x.ravel(), A, B, C).view(np.uint32)
            assert np.array_equal(got, want) and np.isnan(want.view(np.float32)[B // 2])


@pytest.mark.parametrize("kind", ["softmax", "wild", "mixed"])
def test_long_sums_of_values_that_leave_binary64(torch_gpu, kind):
    """One chunk, so that a thread's share takes hundreds of batches: the superaccumulator resolves
    its carries many times, between batches that fit binary64 and batches that do not."""
    for A, B, C in ((60000, 3, 1), (1, 2, 90001), (4, 2, 20000)):
        rng = np.random.default_rng(A + C)
        x = _values("wild" if kind == "wild" else "spread13", A * B * C, rng)
        if kind == "softmax":
            x = np.exp(x / np.abs(x).max() * 40.0 - 40.0).astype(np.float32)
        elif kind == "mixed":  # runs of 4096 values of one magnitude, some of them with outliers
            x *= (2.0 ** (np.arange(x.size) // 4096 * 37 % 120 - 60)).astype(np.float32)
            x[::2999] = np.float32(3.0e38)
        for mean in (False, True):
            note("long sum", kind, (A, B, C), mean)
            cfg = rg.SumConfig(chunks=1, mean=mean)
            dx, out = to_dev(torch_gpu, x), torch_gpu.empty(B, device="cuda")
            ws = torch_gpu.empty(max(rg.make_sum_plan(A, B, C, cfg).workspace_bytes, 1), dtype=torch_gpu.uint8,
                                 device="cuda")
            assert rg.repro_sum_fp32_ws(dx.data_ptr(), out.data_ptr(), A, B, C, cfg, ws.data_ptr(), ws.numel(),
                                        torch_gpu.cuda.current_stream().cuda_stream) == 0
            want = O.exact_sum(x, A, B, C, mean)
            assert np.array_equal(bits(out), want.view(np.uint32)), (kind, A, B, C, mean)


def _fastest(torch, x, shape, mean=False):
    times = []
    for _ in range(8):
        ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        ev[0].record()
        for _ in range(20):
            rg.exact_sum(x, *shape, mean)
        ev[1].record()
        torch.cuda.synchronize()
        times.append(ev[0].elapsed_time(ev[1]))
    return min(times)


def test_wide_ranges_cost_little_more(torch_gpu):
    """Values that do not fit binary64 together cost at most 2.5 times as much as N(0, 1) ones (1.4-1.8
    measured; adding them one by one took 3.3-4.7 times as long)."""
    torch = torch_gpu
    torch.manual_seed(1)
    for shape in ((8192, 3072, 1), (256, 64, 3136)):
        x = torch.randn(*shape, device="cuda")
        wide = x * torch.exp2(torch.randint(-20, 21, shape, device="cuda").float())
        p = torch.softmax(4 * x.view(shape[0], -1), 1)
        p[:, 0] -= 1
        note("sum cost", shape)
        plain = _fastest(torch, x, shape)
        for y in (wide, p / shape[0]):
            assert _fastest(torch, y, shape) < 2.5 * plain, shape


def test_few_rows_cost_little_more(torch_gpu):
    """The mean of a few rows of such values takes at most 1.6 times as long as the sum of N(0, 1) ones
    (1.39 measured; with a batch of 16 for every few rows, and twelve 64-bit divisions, 1.86)."""
    torch = torch_gpu
    torch.manual_seed(1)
    shape = (11, 1000000, 1)
    x = torch.randn(*shape, device="cuda")
    wide = x * torch.exp2(torch.randint(-20, 21, shape, device="cuda").float())
    note("sum cost", shape)
    assert _fastest(torch, wide, shape, True) < 1.6 * _fastest(torch, x, shape)
