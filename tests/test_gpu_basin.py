"""GPU: the basin-graph build against the oracle at the sizes and contents where it can go wrong: tile edges (64x64,
16x16x16), plateaus (ascents across many tiles), isolated peaks, dense and sparse branches, every attribute group.
Trees and integer records are exact, so every comparison is an equality."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

dcf = pytest.importorskip("disccofan_amd")
from oracle.oracle import OracleTree  # noqa: E402


@pytest.fixture(scope="module")
def ctx():
    c = dcf.Context(0)
    yield c
    c.close()


def _contents(kind, shape, seed):
    rng = np.random.default_rng(seed)
    if kind == "constant":
        return np.full(shape, 9, np.uint8)
    if kind == "plateaus":  # large flat zones, ties everywhere
        return rng.integers(0, 3, shape).astype(np.uint8)
    if kind == "noise8":
        return rng.integers(0, 256, shape).astype(np.uint8)
    if kind == "noise16":  # sparse branches: a few pixels over thousands of greys
        return rng.integers(0, 65536, shape).astype(np.uint16)
    if kind == "ramp16":  # one dense branch
        return np.add.outer(np.arange(shape[0]) * 7, np.arange(shape[-1])).astype(np.uint16).reshape(shape)
    if kind == "peaks":  # isolated peaks of two heights on a grid
        g = np.indices(shape)
        return (np.all(g % 2 == 0, axis=0) * (1 + (g[0] // 2) % 2)).astype(np.uint8)
    if kind == "comb":  # ascents that run along every row and then down one column
        a = np.zeros(shape, np.uint16)
        a[::2] = np.arange(shape[-1])
        a[:, -1] = shape[-1] + np.arange(shape[0])
        return a
    if kind == "steps16":  # 70 thousand pixels over few and far greys, small noise on top: mid-sized sparse branches
        y, x = np.indices(shape)
        return ((np.sin(x / 40.0) + np.cos(y / 35.0) + 2) * 12000 + rng.integers(0, 3000, shape)).astype(np.uint16)
    assert kind == "float"
    return rng.normal(size=shape).astype(np.float32)


def _same_tree(ctx, img, conn, tree, attr):
    t = ctx.build(img, conn, tree, attr)
    o = OracleTree(img, conn, tree, attr)
    try:
        assert np.array_equal(t.parent(), o.parent().astype(np.int32))
        got, want = t.check(attr), np.asarray(o.check(attr), dtype=np.float32).reshape(img.shape)
        assert np.array_equal(got, want, equal_nan=True)
    finally:
        t.free()


@pytest.mark.parametrize("shape", [(1, 1), (1, 9), (9, 1), (64, 64), (65, 63), (63, 129), (130, 200)])
@pytest.mark.parametrize("kind", ["constant", "plateaus", "noise8", "noise16", "peaks", "float"])
def test_tile_edges_2d(ctx, kind, shape):
    img = _contents(kind, shape, 11)
    for conn in (4, 8):
        for tree in ("max", "min"):
            _same_tree(ctx, img, conn, tree, 0)


@pytest.mark.parametrize("shape", [(2, 1, 3), (16, 16, 16), (17, 15, 33), (3, 40, 18)])
@pytest.mark.parametrize("kind", ["constant", "plateaus", "noise8", "noise16", "peaks", "float"])
def test_tile_edges_3d(ctx, kind, shape):
    img = _contents(kind, shape, 12)
    for conn in (6, 26):
        for tree in ("max", "min"):
            _same_tree(ctx, img, conn, tree, 0)


@pytest.mark.parametrize("kind", ["ramp16", "comb", "steps16", "noise16"])
@pytest.mark.parametrize("attr", [0, 2, 7, 9, 13])
def test_attribute_groups_2d(ctx, kind, attr):
    _same_tree(ctx, _contents(kind, (270, 260), 13), 8, "max", attr)


@pytest.mark.parametrize("kind", ["plateaus", "noise8"])
@pytest.mark.parametrize("attr", [0, 1, 8, 11, 14])
def test_attribute_groups_3d(ctx, kind, attr):
    _same_tree(ctx, _contents(kind, (20, 35, 33), 14), 6, "min", attr)


def test_wide_plateau(ctx):
    """a constant image: every ascent crosses all the tiles of its row and then those of the last column"""
    _same_tree(ctx, np.full((700, 4200), 3, np.uint8), 8, "max", 0)


@pytest.mark.parametrize("shape,conn", [((400, 500), 8), ((30, 80, 90), 6)])
@pytest.mark.parametrize("scale", [0.02, 1.0])
def test_float_pieces(ctx, shape, conn, scale):
    """floats that are all different: a smooth hill with a little noise (a large dense branch) and with much (large
    branches of few pixels per key, cut into pieces)"""
    g = np.indices(shape).astype(np.float64)
    hill = sum(np.cos((a - s / 2) / s * 2) for a, s in zip(g, shape))
    img = (hill + scale * np.random.default_rng(15).normal(size=shape)).astype(np.float32)
    for tree in ("max", "min"):
        _same_tree(ctx, img, conn, tree, 0)


@pytest.mark.parametrize("kind", ["noise8", "plateaus", "noise16", "steps16", "float"])
def test_bins_2d(ctx, kind):
    """over 2^22 pixels, where slots are counted in bins: dense and sparse branches, tiles of more bins than descriptors"""
    img = _contents(kind, (2049, 2111), 16)
    _same_tree(ctx, img, 8, "max", 0)
    _same_tree(ctx, img, 4, "min", 7)


@pytest.mark.parametrize("kind", ["noise8", "noise16", "peaks"])
def test_bins_3d(ctx, kind):
    img = _contents(kind, (163, 161, 163), 17)
    _same_tree(ctx, img, 6, "max", 0)
    _same_tree(ctx, img, 26, "min", 0)


def test_bins_batch_of_small(ctx):
    """over 2^22 pixels in images of a few pixels each: one tile per image, most of them nearly empty"""
    rng = np.random.default_rng(18)
    imgs = [rng.integers(0, 65536, (7, int(w))).astype(np.uint16) for w in rng.integers(600, 640, 1000)]
    outs = ctx.batch_filter(imgs, [9.0] * len(imgs), 8, "max", 0)
    for i in range(0, len(imgs), 97):
        t = ctx.build(imgs[i], 8, "max", 0)
        try:
            assert np.array_equal(outs[i], t.filter(0, 9.0, out_dtype=np.uint16))
        finally:
            t.free()


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.float32])
@pytest.mark.parametrize("skip", [0, 1, 2, 3])
def test_filter_output_alignment(ctx, dtype, skip):
    """an output that starts at any element: four pixels a store where its address allows, one elsewhere"""
    torch = pytest.importorskip("torch")
    img = _contents("noise8", (37, 53), 19)
    t = ctx.build(img, 8, "max", 0)
    try:
        want = t.filter(0, 5.0, out_dtype=dtype)
        wide = torch.zeros((img.size + 8) * np.dtype(dtype).itemsize, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        t.filter_device(0, 5.0, 0, wide.data_ptr() + skip * np.dtype(dtype).itemsize, dtype)
        ctx.synchronize()
        got = wide.cpu().numpy().view(dtype)
        assert np.array_equal(got[skip:skip + img.size].reshape(img.shape), want)
        assert not got[:skip].any() and not got[skip + img.size:].any()
    finally:
        t.free()


@pytest.mark.parametrize("bins", [1, 2, 63, 64, 65, 1023, 1024, 1025, 2048, 2049])
def test_spectrum_copies(ctx, bins):
    """the copies of the LDS histogram at their limits (32 copies up to 64 bins, one above 1024), and no LDS above 2048"""
    img = _contents("noise16", (96, 131), 20)
    img[:40] //= 9000
    lv = np.linspace(0, 4000, bins, dtype=np.float32)
    t = ctx.build(img, 8, "max", 0)
    o = OracleTree(img, 8, "max", 0)
    try:
        assert np.array_equal(t.spectrum1d(0, lv), o.spectrum1d(0, lv))
    finally:
        t.free()


@pytest.mark.parametrize("pixels", [4094, 4095, 4096, 8191, 70000])
@pytest.mark.parametrize("attr", [7, 9, 13])
def test_prefixes_at_tile_edges(ctx, pixels, attr):
    """as many nodes as pixels (every grey once): prefixes of the sums at and around their tiles of 4096"""
    img = np.random.default_rng(21).permutation(pixels % 65536 if pixels < 65536 else 65536)
    img = np.resize(img, pixels).astype(np.uint16).reshape(1, pixels)
    _same_tree(ctx, img, 4, "max", attr)
