"""GPU: images of flat ground and regular patterns (masks, halftones, textures on a ramp, one-row signals), where components
of the basin graph take each other in an order that follows the image and one round joins paths as long as the image.
Exact against the oracle, and bounded in time by uniform noise of the same size."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

dcf = pytest.importorskip("disccofan_amd")
torch = pytest.importorskip("torch")
from oracle.oracle import OracleTree  # noqa: E402

_BAYER = np.array([[0, 8, 2, 10], [12, 4, 14, 6], [3, 11, 1, 9], [15, 7, 13, 5]])


def pattern(kind, shape, seed=31):
    rng = np.random.default_rng(seed)
    y, x = np.indices(shape)
    ramp = (x * 7 + y) * (60000.0 / (7 * shape[1] + shape[0]))
    if kind == "checkerboard":
        return ((x + y) & 1).astype(np.uint8)
    if kind == "dots":
        return ((x % 4 == 0) & (y % 4 == 0)).astype(np.uint8)
    if kind == "salt":
        return (rng.random(shape) < 0.05).astype(np.uint8)
    if kind == "binary":
        return rng.integers(0, 2, shape).astype(np.uint8)
    if kind == "halftone":
        return (_BAYER[y % 4, x % 4] < ramp * (16 / 60000.0)).astype(np.uint8) * 255
    if kind == "ramp_checkerboard":  # every saddle of another grey
        return np.where((x + y) & 1, 65535, ramp.astype(np.int64)).astype(np.uint16)
    if kind == "ramp_dots":
        return np.where((x % 4 == 0) & (y % 4 == 0), 65535, ramp.astype(np.int64)).astype(np.uint16)
    if kind == "rising_peaks_float":  # a row of peaks whose saddles rise from left to right, all different
        return np.where(x & 1, 2.0, (x + y * shape[1]) / float(shape[0] * shape[1])).astype(np.float32)
    assert kind == "noise"
    return rng.integers(0, 256, shape).astype(np.uint8)


@pytest.fixture(scope="module")
def ctx():
    c = dcf.Context(0)
    yield c
    c.close()


def same_tree(ctx, img, conn, tree="max", attr=0):
    t = ctx.build(img, conn, tree, attr)
    o = OracleTree(img, conn, tree, attr)
    try:
        assert np.array_equal(t.parent(), o.parent().astype(np.int32))
        assert np.array_equal(t.check(attr), np.asarray(o.check(attr), dtype=np.float32).reshape(img.shape), equal_nan=True)
    finally:
        t.free()


def seconds(ctx, img, conn):
    """the fastest of five builds of an image that is on the GPU"""
    a = torch.from_numpy(img.view(np.int16) if img.dtype == np.uint16 else img).cuda()
    torch.cuda.synchronize()
    best = float("inf")
    for _ in range(6):
        ctx.synchronize()
        t0 = time.perf_counter()
        t = ctx.build_device(a.data_ptr(), img.dtype, img.shape, conn, "max", 0)
        ctx.synchronize()
        best = min(best, time.perf_counter() - t0)
        t.free()
    return best


PATTERNS = [("checkerboard", 4), ("dots", 8), ("salt", 8), ("halftone", 4), ("ramp_checkerboard", 4), ("ramp_dots", 8),
            ("rising_peaks_float", 4)]


@pytest.mark.parametrize("kind,conn", PATTERNS)
@pytest.mark.parametrize("shape", [(1, 25 * 2 + 1), (150, 200), (1, 40000)])
def test_pattern_trees(ctx, kind, conn, shape):
    """paths below, at and above the steps one thread walks, in memory and in one block's LDS; groups of both kinds"""
    img = pattern(kind, shape)
    same_tree(ctx, img, conn)
    same_tree(ctx, img, conn, "min", 0 if img.dtype == np.float32 else 9)


@pytest.mark.parametrize("kind,conn", [("checkerboard", 4), ("halftone", 4), ("ramp_checkerboard", 4)])
def test_large_pattern_trees(ctx, kind, conn):
    """above 2^22 pixels, where the forest is sized by its counts"""
    same_tree(ctx, pattern(kind, (2050, 2050)), conn)


def test_pattern_volume(ctx):
    z, y, x = np.indices((40, 50, 60))
    img = ((x + y + z) & 1).astype(np.uint8)
    same_tree(ctx, img, 6)
    same_tree(ctx, img, 26, "min")


@pytest.mark.parametrize("kind,conn,shape", [(k, c, (2048, 2048)) for k, c in PATTERNS] + [("binary", 4, (1, 1 << 20)),
                                                                                          ("checkerboard", 4, (1, 1 << 20))])
def test_pattern_time(ctx, kind, conn, shape):
    """no more than four times the noise's: with paths walked step by step these images take seconds"""
    assert seconds(ctx, pattern(kind, shape), conn) < 4 * seconds(ctx, pattern("noise", shape), conn)


def corridor(side):
    """a square spiral one pixel wide that rises to its middle, between walls of grey 0: ascents as long as the spiral"""
    a = np.zeros((side, side), np.uint16)
    y, x, dy, dx, k = 0, 0, 0, 1, 1
    a[0, 0] = 1

    def free(r, c):
        return 0 <= r < side and 0 <= c < side and a[r, c] == 0

    def steps(r, c):  # the next pixel is free and the one beyond it is no part of the spiral
        return free(r, c) and (not (0 <= r + dy < side and 0 <= c + dx < side) or a[r + dy, c + dx] == 0)
    while True:
        if not steps(y + dy, x + dx):
            dy, dx = dx, -dy
            if not steps(y + dy, x + dx):
                return a
        y, x, k = y + dy, x + dx, k + 1
        a[y, x] = k


@pytest.mark.parametrize("shape", [(1, 64 * 15), (1, 64 * 16 + 1), (1, 64 * 40), (64 * 300, 2), (2, 1, 16 * 300), (3, 16 * 150, 2),
                                   (1, (1 << 22) - 1), (1, (1 << 22) + 1), (2, 3, 800000)])
def test_long_plateaus(ctx, shape):
    """equal pixels in a row of 15, 16 and many more tiles, on both sides of 2^22 pixels, and with a step in the middle"""
    img = np.full(shape, 5, np.uint8)
    same_tree(ctx, img, 8)
    img.reshape(-1)[img.size // 2:] = 6
    img.reshape(-1)[0] = 4
    same_tree(ctx, img, 4, "min")


@pytest.mark.parametrize("side", [63, 250, 361])
def test_spiral(ctx, side):
    img = corridor(side)
    same_tree(ctx, img, 4)
    same_tree(ctx, img, 8, "min")


@pytest.mark.parametrize("shape", [(1, 1 << 22), (1, (1 << 23) + 1)])
def test_long_plateau_time(ctx, shape):
    """no more than the noise's"""
    img = np.full(shape, 5, np.uint8)
    assert seconds(ctx, img, 4) < seconds(ctx, pattern("noise", shape), 4)


def test_bin_in_parts(ctx):
    """more than 2^22 pixels of one grey and its double: 1089 tiles with one and two items each in one bin"""
    img = np.full((33 * 64, 33 * 64), 7, np.uint8)
    same_tree(ctx, img, 8)
    img[:, 1000:] = 8
    same_tree(ctx, img, 4)


def test_many_deep_hills(ctx):
    """400 hills of ten thousand greys each, over nearly all four million ranks: more pieces than one for 64 pixels, so wider ones"""
    y, x = np.indices((100, 100))
    order = np.argsort(np.argsort(-((x - 47.3) ** 2 + (y - 52.1) ** 2).ravel(), kind="stable")).reshape(100, 100)
    img = -np.random.default_rng(33).random((20 * 102, 20 * 102))
    for k in range(400):
        j, i = divmod(k, 20)
        img[102 * j:102 * j + 100, 102 * i:102 * i + 100] = order * 400 + k  # every grey once
    same_tree(ctx, img.astype(np.float32), 4)
