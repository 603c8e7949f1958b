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

# (A, B, C): one row per wave, rows in fours and not, single and several chunks, columns
SHAPES = [(1, 5, 3), (1, 3, 64), (1, 4, 260), (3, 5, 7), (7, 3, 1000), (2, 2, 20000), (1, 1, 300001),
          (70, 65, 1), (3000, 130, 1), (1, 1, 1)]


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
