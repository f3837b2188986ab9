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
