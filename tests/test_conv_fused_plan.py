"""The fused convolution's plan on the host: which passes take it, and the conditions its patch
kernel relies on (a block's patch fits its LDS slot wherever the block starts; a channel group's
slot is free, and the next patch in it ready, before its first use)."""
import ctypes
import random
import time

import pytest

import bit_reproducible_training_amd as rg
from bit_reproducible_training_amd import _lib

FWD, DW, DX = 0, 1, 2
BLOCK = 128       # positions per block
PATCH = 384       # values per channel and slot


def fused(pass_, shape, S=3, num_cus=256, forced=False):
    info = (ctypes.c_int * 11)()
    g = rg.ConvShape(*shape).to_c()
    assert _lib.lib.rg_test_conv_plan(pass_, ctypes.byref(g), S, num_cus, int(forced), info) == 0, shape
    return dict(zip(("taken", "patch", "split", "classes", "strips", "width", "groups", "tf", "taps",
                     "stages", "channel_groups"), info))


def test_routes():
    resnet = (32, 64, 56, 56, 64, 3, 3, 1, 1, 1, 1)
    for pass_ in (FWD, DX):
        p = fused(pass_, resnet)
        assert p["taken"] and p["patch"] and p["split"] == 1, p
    assert fused(DW, resnet)["taken"]
    assert not fused(DW, (32, 512, 7, 7, 512, 3, 3, 1, 1, 1, 1))["taken"]    # many filters, few windows
    assert not fused(DW, (8, 64, 20, 20, 64, 3, 3, 3, 3, 1, 1))["taken"]     # column stride 3
    strided = (32, 64, 56, 56, 128, 3, 3, 2, 2, 1, 1)
    p = fused(DX, strided)
    assert p["taken"] and not p["patch"] and p["classes"] == 4
    assert fused(FWD, (32, 64, 56, 56, 256, 1, 1, 1, 1, 0, 0))["taken"]
    # Measured on both routes (us, fused against the pipeline):
    assert fused(FWD, strided)["taken"]                                       # 44, 56
    assert fused(FWD, (32, 512, 7, 7, 512, 3, 3, 1, 1, 1, 1))["split"] > 1    # 71, 81
    assert fused(FWD, (100, 6, 14, 14, 16, 5, 5, 1, 1, 0, 0))["taken"]        # 18.1, 18.9
    for shape in ((8, 256, 14, 14, 256, 3, 3, 1, 1, 1, 1),                    # 43, 37
                  (32, 128, 28, 28, 128, 3, 3, 2, 2, 1, 1),                   # 47, 36
                  (1, 64, 56, 56, 256, 3, 3, 1, 1, 1, 1),                     # 28, 24
                  (22, 828, 8, 8, 51, 7, 7, 2, 2, 0, 0),                      # 119, 42
                  (3, 750, 8, 7, 1714, 5, 5, 2, 2, 2, 2),                     # 238, 95
                  (1, 1149, 7, 9, 933, 5, 5, 1, 1, 2, 2)):                    # 220, 88
        assert not fused(FWD, shape)["taken"] and fused(FWD, shape, forced=True)["taken"], shape
    for shape in ((3, 1068, 14, 14, 53, 7, 7, 2, 2, 3, 3),                    # 92, 53
                  (2, 35, 10, 10, 124, 7, 7, 1, 1, 0, 0)):                    # 29, 22
        assert not fused(DW, shape)["taken"] and fused(DW, shape, forced=True)["taken"], shape
    assert not fused(FWD, (32, 3, 112, 112, 64, 7, 7, 2, 2, 3, 3))["taken"]   # 3 channels
    assert not fused(DX, (8, 8, 20, 20, 16, 5, 5, 3, 3, 2, 2))["taken"]       # nine classes
    bad = rg.ConvShape(1, 1, 3, 3, 1, 5, 5).to_c()      # kernel larger than the image
    info = (ctypes.c_int * 8)()
    assert _lib.lib.rg_test_conv_fused(FWD, ctypes.byref(bad), 3, 256, info) == 1
    assert _lib.lib.rg_test_conv_fused(7, ctypes.byref(bad), 3, 256, info) == 1


def test_plans_keep_to_the_launch_limit():
    """A launch takes fewer than 2^32 work items; a pass over the pixels takes four for each."""
    for S in (1, 2):
        for forced in (False, True):
            assert not fused(FWD, (2 ** 22, 1, 16, 17, 1, 2, 2, 2, 2, 0, 0), S, forced=forced)["taken"]
    assert fused(FWD, (2 ** 22, 1, 16, 15, 1, 2, 2, 2, 2, 0, 0), 1, forced=True)["taken"]
    assert not fused(DX, (2 ** 24, 4, 2, 2, 4, 2, 2, 2, 2, 0, 0), 1, forced=True)["taken"]  # a block per image
    assert fused(DX, (2 ** 24 - 9, 4, 2, 2, 4, 2, 2, 2, 2, 0, 0), 1, forced=True)["taken"]


def patch_shapes(count):
    rng = random.Random(11)
    while count:
        k = rng.choice([(2, 2), (3, 3), (3, 3), (5, 5), (7, 7), (2, 3), (1, 7), (5, 2)])
        n, c, f = rng.randint(1, 40), rng.choice([8, 13, 16, 33, 64, 130]), rng.choice([16, 33, 64])
        h, w = rng.randint(k[0], 90), rng.randint(k[1], 150)
        shape = (n, c, h, w, f, k[0], k[1], 1, 1, rng.randint(0, k[0] - 1), rng.randint(0, k[1] - 1))
        for pass_ in (FWD, DX):
            p = fused(pass_, shape, forced=True)
            if p["patch"]:
                count -= 1
                yield pass_, shape, p
                if not count:
                    return


def test_patch_fits_every_block():
    for pass_, shape, p in patch_shapes(60):
        N, C, H, W, F, KH, KW, _, _, PY, PX = shape
        OH, OW = H + 2 * PY - KH + 1, W + 2 * PX - KW + 1
        gh, gw = (OH, OW) if pass_ == FWD else (H, W)
        assert p["strips"] * p["width"] >= gw and p["groups"] * 64 <= PATCH, (shape, p)
        per = gh * p["width"]
        rows, width = N * p["strips"] * per, p["width"] + KW - 1

        def padded_row(r):
            img, g = divmod(r, per)
            return img * (gh + KH - 1) + g // p["width"]

        for r0 in range(0, rows, BLOCK):
            last = min(r0 + BLOCK, rows) - 1
            values = (padded_row(last) - padded_row(r0) + KH) * width
            assert values <= p["groups"] * 64, (shape, p, r0)


def schedule(pass_, T, s0, s1, groups):
    copied = (ctypes.c_int * groups)()
    assert _lib.lib.rg_test_conv_schedule(pass_, T, s0, s1, groups, copied) == 0
    return list(copied)


def test_patches_need_four_or_six_taps():
    """The slots' schedule serves four taps and six or more; plans hold no patches at others."""
    seen = set()
    for kh in range(1, 10):
        for kw in range(1, 10):
            for pass_ in (FWD, DX):
                p = fused(pass_, (4, 64, 20, 20, 64, kh, kw, 1, 1, 0, 0), forced=True)
                assert p["taken"] and bool(p["patch"]) <= (kh * kw == 4 or kh * kw >= 6), (kh, kw)
                if p["patch"]:
                    seen.add(p["taps"])
    assert 4 in seen and 6 in seen and 5 not in seen and max(seen) > 40
    for pass_, shape, p in patch_shapes(60):
        assert p["taps"] == 4 or p["taps"] >= 6, (pass_, shape)


@pytest.mark.parametrize("taps", [4] + list(range(6, 82)))
def test_patch_slots_are_free_and_ready(taps):
    """Stage s reads k groups 4 s .. 4 s + 3, group g channel group g // taps from slot
    (g // taps) % 2. Whatever stages a part has, a channel group is copied before the stage that first
    reads it, and after the last that reads the group before it in its slot."""
    for groups in (1, 2, 3, 9, 20):
        stages = -(-groups * taps // 4)
        starts = sorted({0, 1, 2, 3, taps // 4, stages // 3, stages // 2, stages - 2, stages - 1} - {-1, -2})
        for s0 in [s for s in starts if 0 <= s < stages]:
            for s1 in sorted({min(stages, s0 + n) for n in (1, 2, 3, 7, taps, 2 * taps, stages)}):
                copied = schedule(FWD, taps, s0, s1, groups)
                reads = {}  # channel group -> first and last stage (a group past the last reads any value)
                for s in range(s0, s1):
                    for g in range(4 * s, 4 * s + 4):
                        if g // taps < groups:
                            first, _ = reads.get(g // taps, (s, s))
                            reads[g // taps] = (first, s)
                for cg, (first, last) in reads.items():
                    at = copied[cg]
                    assert at == -1 or s0 <= at < first, (taps, groups, s0, s1, cg)
                    if cg - 2 in reads:
                        assert at != -1 and at > reads[cg - 2][1], (taps, groups, s0, s1, cg)


def test_weight_gradient_chunks_fit_every_block():
    """A chunk of RC output rows' source rows fits its patch slot wherever the chunk starts, and two
    to sixteen k steps of eight quads of four columns cover it."""
    rng = random.Random(12)
    found = 0
    while found < 60:
        k = rng.choice([(2, 2), (3, 3), (3, 3), (5, 5), (7, 7), (1, 7), (5, 2), (1, 1)])
        n, c, f = rng.randint(1, 40), rng.choice([1, 3, 13, 16, 64, 130]), rng.choice([6, 33, 64])
        h, w = rng.randint(k[0], 90), rng.randint(k[1], 300)
        sy, sx = rng.choice([1, 1, 2, 3]), rng.choice([1, 1, 2])
        shape = (n, c, h, w, f, k[0], k[1], sy, sx, rng.randint(0, k[0] - 1), rng.randint(0, k[1] - 1))
        p = fused(DW, shape, forced=True)
        if not p["taken"]:
            continue
        found += 1
        N, C, H, W, F, KH, KW, SY, SX, PY, PX = shape
        OH, OW = (H + 2 * PY - KH) // SY + 1, (W + 2 * PX - KW) // SX + 1
        rc, ns, sw = p["classes"], p["strips"], p["width"]
        assert sw % 4 == 0 and ns * sw >= OW > (ns - 1) * sw, (shape, p)
        channels = max((min(q + BLOCK, C * KH * KW) - 1) // (KH * KW) - q // (KH * KW) + 1
                       for q in range(0, C * KH * KW, BLOCK))
        assert channels * (64 * p["groups"] + 20) <= 6144 and p["groups"] <= 6, (shape, p)
        ph, pw = (OH - 1) * SY + KH, (sw - 1) * SX + KW
        assert 1 <= rc * sw // 4 <= 8 * 16, (shape, p)

        def padded(v):
            return v // OH * ph + v % OH * SY

        rows = N * ns * OH
        for v0 in range(0, rows, rc):
            last = min(v0 + rc, rows) - 1
            assert (padded(last) - padded(v0) + KH) * pw <= 64 * p["groups"], (shape, p, v0)


@pytest.mark.parametrize("steps", range(2, 17))
def test_weight_gradient_slots_are_free_and_ready(steps):
    """Stage s takes k steps 2 s and 2 s + 1, step j chunk j // steps from patch slot (chunk % 2) and
    table slot (chunk % 4). Tables 0 .. 3 are built before the first stage and table c + 2 where chunk c
    is copied; a chunk's quads are looked up when dY is loaded, two stages before their own."""
    for chunks in (1, 2, 3, 4, 5, 40):
        stages = -(-chunks * steps // 2)
        copied = schedule(DW, steps, 0, stages, chunks)
        for c in range(chunks):
            first, last = c * steps // 2, ((c + 1) * steps - 1) // 2
            if c < 2:
                assert copied[c] == -1
            else:
                assert 0 <= copied[c] < first, (steps, c)
                assert copied[c] > (((c - 1) * steps) - 1) // 2, (steps, c)   # chunk c - 2 is done
            if c >= 4:                                                          # table c
                assert copied[c - 2] >= 0 and copied[c - 2] + 1 <= first - 2, (steps, c)


def test_weight_gradient_chunks_take_two_steps_or_more():
    rng = random.Random(3)
    seen = set()
    for _ in range(3000):
        k = rng.randint(1, 7)
        shape = (rng.randint(1, 9), rng.randint(1, 64), rng.randint(k, 40), rng.randint(k, 60), rng.randint(1, 64),
                 k, k, rng.randint(1, 3), rng.randint(1, 2), 0, 0)
        p = fused(DW, shape, forced=True)
        if p["taken"]:
            seen.add(p["taps"])  # (k steps per chunk)
    assert min(seen) == 2 and max(seen) <= 16 and len(seen) > 5


def test_forced_algorithms_are_known():
    g = rg.ConvShape(2, 3, 9, 9, 4, 3, 3)
    for algo, known in ((3, True), (4, True), (5, False), (-1, False)):
        try:
            rg.repro_conv.conv2d_algo_workspace(FWD, g, 3, algo)
            code = 0
        except rg.ReproGemmError as e:
            code = e.code
        assert (code != 1) == known, algo  # (without a GPU a known one stops at the device query)


@pytest.mark.parametrize("pass_", [FWD, DW, DX])
@pytest.mark.parametrize("S", [1, 3])
def test_planning_wide_rows_takes_microseconds(pass_, S):
    """A call plans twice, so the search for strips and parts has to stay far below a launch (a search
    by every number of strips took 2 ms here, by every length of a part 5 us)."""
    for shape in ((1, 2, 31, 1000000, 4, 31, 31, 1, 1, 0, 0), (64, 64, 1, 16384, 64, 1, 3, 1, 1, 0, 1)):
        best = 1.0
        for _ in range(20):
            t = time.perf_counter()
            fused(pass_, shape, S)
            best = min(best, time.perf_counter() - t)
        assert best < 2e-4, (shape, best)
