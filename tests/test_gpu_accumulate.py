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


def test_out_of_memory_half_way():
    """an accumulation that finds no memory leaves the tree with the group it had, or with none"""
    c = dcf.Context(0)
    img = np.random.default_rng(42).integers(0, 65536, (2100, 2100)).astype(np.uint16)
    t = c.build(img, 8, "max", 0)
    hold = []
    try:
        area = t.check(0)
        step = 64 << 20
        hold.append(torch.empty(torch.cuda.mem_get_info()[0] - 24 * step, dtype=torch.uint8, device="cuda"))
        while torch.cuda.mem_get_info()[0] > step:
            hold.append(torch.empty(step - (4 << 20), dtype=torch.uint8, device="cuda"))
        failed = 0
        while True:
            try:
                t.accumulate(13)
                break
            except dcf.DcfError as e:
                failed += 1
                assert e.code == -2, str(e)
            assert t.group in (0, -1)
            try:
                assert np.array_equal(t.check(0), area) and t.group == 0
            except dcf.DcfError as e:
                assert e.code == (-2 if t.group == 0 else -6)
            assert len(hold) > 1
            hold.pop()
            torch.cuda.empty_cache()
        assert failed > 1
        hold.clear()
        torch.cuda.empty_cache()
        want = OracleTree(img, 8, "max", 13).check(13)
        assert np.array_equal(t.check(13), np.asarray(want, dtype=np.float32).reshape(img.shape), equal_nan=True)
    finally:
        t.free()
        c.close()
        hold.clear()
        torch.cuda.empty_cache()
