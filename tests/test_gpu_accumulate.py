"""GPU: further attribute groups on a tree that is there, whose device image the caller may have changed meanwhile."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

dcf = pytest.importorskip("disccofan_amd")
torch = pytest.importorskip("torch")
from oracle.oracle import OracleTree  # noqa: E402


@pytest.fixture(scope="module")
def ctx():
    c = dcf.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("tree", ["max", "min"])
@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.float32])
@pytest.mark.parametrize("other", ["fewer nodes", "more nodes", "brighter"])
def test_image_changed_since_the_build(ctx, dtype, tree, other):
    """the attributes of other pixels are nobody's answer, but they stay in their arrays; with the pixels back they are right"""
    rng = np.random.default_rng(41)
    shape = (251, 333)
    noise, flat = rng.integers(0, 100, shape).astype(dtype), (np.indices(shape)[0] // 60).astype(dtype)
    img = flat if other == "more nodes" else noise
    now = {"fewer nodes": flat, "more nodes": noise, "brighter": (noise + 150).astype(dtype)}[other]
    as_int = (lambda a: a.view(np.int16)) if dtype is np.uint16 else (lambda a: a)
    d = torch.from_numpy(as_int(img).copy()).cuda()
    torch.cuda.synchronize()
    t = ctx.build_device(d.data_ptr(), img.dtype, shape, 8, tree, 0)
    try:
        nodes = t.num_nodes
        for attr in (1, 7, 13, 0):
            d.copy_(torch.from_numpy(as_int(now).copy()))
            torch.cuda.synchronize()
            t.accumulate(attr)
            ctx.synchronize()
            assert t.check(attr).shape == shape and t.num_nodes == nodes
        for attr in (1, 7, 13, 0):
            d.copy_(torch.from_numpy(as_int(img).copy()))
            torch.cuda.synchronize()
            t.accumulate(attr)
            o = OracleTree(img, 8, tree, attr)
            assert np.array_equal(t.check(attr), np.asarray(o.check(attr), dtype=np.float32).reshape(shape), equal_nan=True)
    finally:
        t.free()
