"""The fused convolution's plan on the host: which passes take it, and the conditions its patch
kernel relies on (a block's patch fits its LDS slot wherever the block starts; a channel group's
slot is free, and the next patch in it ready, before its first use)."""
import ctypes
import random

import pytest

import bit_reproducible_training_amd as rg
from bit_reproducible_training_amd import _lib

FWD, DW, DX = 0, 1, 2
BLOCK = 128       # positions per block
PATCH = 384       # values per channel and slot


def fused(pass_, shape, S=3, num_cus=256):
    info = (ctypes.c_int * 8)()
    g = rg.ConvShape(*shape).to_c()
    assert _lib.lib.rg_test_conv_fused(pass_, ctypes.byref(g), S, num_cus, info) == 0, shape
    return dict(zip(("taken", "patch", "split", "classes", "strips", "width", "groups", "tf"), info))


def test_routes():
    resnet = (32, 64, 56, 56, 64, 3, 3, 1, 1, 1, 1)
    for pass_ in (FWD, DX):
        p = fused(pass_, resnet)
        assert p["taken"] and p["patch"] and p["split"] == 1, p
    assert not fused(DW, resnet)["taken"]
    strided = (32, 64, 56, 56, 128, 3, 3, 2, 2, 1, 1)
    assert not fused(FWD, strided)["taken"]             # overlapping windows, not at stride 1
    p = fused(DX, strided)
    assert p["taken"] and not p["patch"] and p["classes"] == 4
    assert fused(FWD, (32, 64, 56, 56, 256, 1, 1, 1, 1, 0, 0))["taken"]
    assert not fused(FWD, (8, 256, 14, 14, 256, 3, 3, 1, 1, 1, 1))["taken"]   # needs parts
    assert fused(FWD, (32, 512, 7, 7, 512, 3, 3, 1, 1, 1, 1))["split"] > 1    # past one-pass slicing
    assert not fused(FWD, (32, 3, 112, 112, 64, 7, 7, 2, 2, 3, 3))["taken"]   # 3 channels
    assert not fused(DX, (8, 8, 20, 20, 16, 5, 5, 3, 3, 2, 2))["taken"]       # nine classes
    bad = rg.ConvShape(1, 1, 3, 3, 1, 5, 5).to_c()      # kernel larger than the image
    info = (ctypes.c_int * 8)()
    assert _lib.lib.rg_test_conv_fused(FWD, ctypes.byref(bad), 3, 256, info) == 1
    assert _lib.lib.rg_test_conv_fused(7, ctypes.byref(bad), 3, 256, info) == 1


def patch_shapes(count):
    rng = random.Random(11)
    while count:
        k = rng.choice([(2, 2), (3, 3), (3, 3), (5, 5), (7, 7), (2, 3), (1, 7), (5, 2)])
        n, c, f = rng.randint(1, 40), rng.choice([8, 13, 16, 33, 64, 130]), rng.choice([16, 33, 64])
        h, w = rng.randint(k[0], 90), rng.randint(k[1], 150)
        shape = (n, c, h, w, f, k[0], k[1], 1, 1, rng.randint(0, k[0] - 1), rng.randint(0, k[1] - 1))
        for pass_ in (FWD, DX):
            p = fused(pass_, shape)
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


@pytest.mark.parametrize("taps", [4] + list(range(6, 82)))
def test_patch_slots_are_free_and_ready(taps):
    """Stage s reads k groups 4 s .. 4 s + 3, group g channel group g // taps from slot
    (g // taps) % 2. The kernel copies channel group cg >= 2 during the first stage that starts
    past the last group of cg - 2; that stage has to come before the first that reads cg."""
    for cg in range(2, 40):
        copied = -(-(cg - 1) * taps // 4)
        assert 4 * copied >= (cg - 1) * taps         # every read of cg - 2 is in an earlier stage
        assert copied < cg * taps // 4, (taps, cg)
        if cg > 2:                                   # one copy per stage at most
            assert copied > -(-(cg - 2) * taps // 4)
