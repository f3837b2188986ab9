"""The work a user of disccofan_amd has it do, as measurable cases.

A case is a dict of plain values.  `kind` names the call:

    image       build_device + filter_device (+ a 1D or 2D pattern spectrum) on an image resident in HBM
    batch       batch_filter_device over many images of uneven sizes, each with its own lambda
    pair        the max-tree and the min-tree of one image in one batch_filter_device call
    tiled       build_tiled_device over row slabs, then filter_device
    operations  run_operations on a host image: the reference's operation list, float results on the host
    rules       several filters and a spectrum on a tree that is already there

Images come from the seeded generators of disccofan_amd.synth, which are those of the benchmark and the
tests: blurred noise with disks, value noise with ellipses, blurred-noise volumes with spheres, and a
log-normal sky with Gaussian blobs (raw floats, or quantised to 16 bits).
"""
import math

import numpy as np
import torch

import disccofan_amd as dcf
from disccofan_amd import synth

_NP = {"u8": np.uint8, "u16": np.uint16, "f32": np.float32}
_BYTES = {"u8": 1, "u16": 2, "f32": 4}

# ranges: image sides 64..8192 in 2D, volume sides 24..512, batches of up to 256 images of 64..2048 a side
_MAX_PIXELS_2D = 8192 * 8192
_MAX_PIXELS_3D = 512 ** 3


def _image(name, kind="image", source="disks", dtype="u8", depth=1, height=256, width=256, conn=4, tree="max", attr=0,
           lam=100.0, decision=0, bins=0, bins2=0, count=1, slabs=1):
    return {"name": name, "kind": kind, "source": source, "dtype": dtype, "depth": depth, "height": height, "width": width,
            "conn": conn, "tree": tree, "attr": attr, "lam": float(lam), "decision": decision, "bins": bins, "bins2": bins2,
            "count": count, "slabs": slabs}


def listed():
    return [
        # one small image or crop, as an interactive tool or a per-object loop opens it: latency and launches
        _image("small_u8", height=256, width=320, lam=100),
        # an ordinary 8-bit photograph-sized image: area opening and its 32-bin area spectrum
        _image("disks1024_u8", height=1024, width=1024, lam=100, bins=32),
        # a 16-bit image of odd sides, its holes closed on the min-tree with 8-connectivity and the subtractive rule
        _image("odd_u16_min", source="vnoise", dtype="u16", height=769, width=1013, conn=8, tree="min", lam=60, decision=3),
        # shape analysis of a 16-bit sky: moments of inertia, filter by non-compactness, 2D non-compactness x area spectrum
        _image("blobs4096_shape", source="blobs", dtype="u16", height=4096, width=4096, conn=8, attr=17, lam=0.5, bins=32,
               bins2=32),
        # a raw float exposure of odd sides (every pixel its own grey), area opening
        _image("sky_f32", source="blobs", dtype="f32", height=1531, width=2048, conn=8, lam=25),
        # the large 16-bit mosaic: openings and closings of one image, max-tree and min-tree in one call
        _image("vnoise8192_pair", kind="pair", source="vnoise", dtype="u16", height=8192, width=8192, conn=8, lam=1000,
               decision=3),
        # the large 8-bit volume: volume opening with 6-connectivity and its 48-bin spectrum
        _image("spheres512", source="spheres", depth=512, height=512, width=512, conn=6, lam=500, bins=48),
        # an ordinary volume of odd sides, 26-connectivity, filtered by elongation (moments of inertia in 3D)
        _image("volume_elong_26", source="spheres", depth=151, height=187, width=203, conn=26, attr=14, lam=2.0),
        # a data set of 256 uneven 8- and 16-bit images, each with its own lambda, in one batched call
        _image("batch256", kind="batch", source="disks", height=2048, width=2048, lam=5000, count=256),
        # the reference's distributed build on one GPU: eight row slabs and the merge of their boundary trees
        _image("tiled_slabs", kind="tiled", source="vnoise", dtype="u16", height=4096, width=4096, conn=8, lam=300, slabs=8),
        # the drop-in driver: an operation list on a host image, across attribute groups, float results back on the host
        _image("operations_host", kind="operations", height=768, width=1024, lam=200),
        # one tree, many questions: a sweep of lambdas, a shape filter by each rule and a spectrum on a 2048^2 image
        _image("rules_sweep", kind="rules", height=2048, width=2048, conn=4, attr=17, lam=0.3, bins=32),
    ]


def draw(rng):
    """one more case of the same ranges"""

    def side(lo, hi):
        # log-uniform, odd as often as even
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(["image", "image", "image", "volume", "volume", "pair", "batch", "tiled", "operations", "rules"])
    lam = float(int(round(math.exp(rng.uniform(math.log(10), math.log(5000))))))
    tree = rng.choice(["max", "min"])
    if kind == "volume":
        d, h, w = side(24, 400), side(24, 512), side(24, 512)
        attr, lam = rng.choice([(0, lam), (0, lam), (14, 2.0), (3, 20.0)])
        c = _image("", source="spheres", depth=d, height=h, width=w, conn=rng.choice([6, 26]), tree=tree, attr=attr, lam=lam,
                   decision=rng.choice([0, 3]), bins=rng.choice([0, 48]))
    elif kind == "image":
        source, dtype = rng.choice([("disks", "u8"), ("disks", "u8"), ("disks", "u16"), ("vnoise", "u16"), ("blobs", "u16"),
                                    ("blobs", "f32")])
        top = 2048 if dtype == "f32" else 6000
        attr, lam = rng.choice([(0, lam), (0, lam), (0, lam), (17, 0.5), (2, 300.0)])
        c = _image("", source=source, dtype=dtype, height=side(64, top), width=side(64, top), conn=rng.choice([4, 8]), tree=tree,
                   attr=attr, lam=lam, decision=0 if dtype == "f32" else rng.choice([0, 0, 3]), bins=rng.choice([0, 32]))
    elif kind == "pair":
        c = _image("", kind="pair", source="vnoise", dtype="u16", height=side(512, 6000), width=side(512, 6000), conn=8, lam=lam,
                   decision=rng.choice([0, 3]))
    elif kind == "batch":
        c = _image("", kind="batch", source="disks", height=side(200, 2048), width=side(200, 2048), lam=5000,
                   count=rng.randint(3, 96), conn=rng.choice([4, 8]), tree=tree)
    elif kind == "tiled":
        c = _image("", kind="tiled", source="vnoise", dtype="u16", height=side(256, 4096), width=side(256, 4096), conn=8, tree=tree,
                   lam=lam, slabs=rng.randint(2, 8))
    elif kind == "operations":
        c = _image("", kind="operations", height=side(64, 1400), width=side(64, 1400), conn=rng.choice([4, 8]), tree=tree, lam=lam)
    else:
        c = _image("", kind="rules", height=side(256, 2048), width=side(256, 2048), conn=rng.choice([4, 8]), attr=17, lam=0.3,
                   tree=tree, bins=32)
    del c["name"]
    return c


# ---- inputs -----------------------------------------------------------------------------------------------------------
def _generate(case, seed):
    s = (synth.SEED[case["source"]] + 0x9E3779B97F4A7C15 * (seed + 1)) & 0xFFFFFFFFFFFFFFFF
    d, h, w = case["depth"], case["height"], case["width"]
    if case["source"] == "vnoise":
        return synth.vnoise(h, w, seed=s)
    if case["source"] == "spheres":
        return synth.spheres(d, h, w, seed=s)
    if case["source"] == "blobs":
        if case["dtype"] == "f32":
            return synth.blobs(h, w, seed=s, raw=True)[1]
        return synth.blobs(h, w, seed=s)
    return synth.disks(h, w, is16=case["dtype"] == "u16", seed=s)


def _shapes(case, seed):
    """(height, width, 16-bit, seed, lambda) of a batch's images; the sides are uniform up to the case's, as the
    benchmark's batch"""
    rng = np.random.default_rng(seed + 77)
    out = []
    for i in range(case["count"]):
        # sizes and lambdas belong to the case (its work is the same for every seed); the pixels to the seed
        fixed = np.random.default_rng(1000 + i)
        h, w = int(fixed.integers(64, case["height"] + 1)), int(fixed.integers(64, case["width"] + 1))
        out.append((h, w, i % 2 == 1, int(rng.integers(1, 2 ** 62)), float(int(fixed.uniform(10, case["lam"])))))
    return out


_SHARED = {}


def _context():
    """the process's context, on a stream of its own that torch's work is ordered with"""
    if not _SHARED:
        torch.cuda.init()
        _SHARED["stream"] = torch.cuda.Stream()
        _SHARED["ctx"] = dcf.Context(0)
        _SHARED["ctx"].set_stream(_SHARED["stream"].cuda_stream)
    return _SHARED["ctx"], _SHARED["stream"]


def _to_gpu(a):
    """16-bit greys as the int16 tensor of the same bits: torch has few operations on uint16"""
    return torch.from_numpy(a.view(np.int16) if a.dtype == np.uint16 else a).cuda()


def _lambdas(attr, bins):
    if attr == 0:
        return synth.log_lambdas(bins, 1, 2 ** 30)
    if attr == 17:
        return np.concatenate([[0], np.geomspace(0.1, 4, bins - 1)]).astype(np.float32)
    return synth.log_lambdas(bins, 1, 2 ** 12)


def prepare(case, seed):
    ctx, stream = _context()
    state = {"case": case, "ctx": ctx, "stream": stream}
    if case["kind"] == "batch":
        # the results of one type lie back to back in one buffer
        shapes = _shapes(case, seed)
        outs = [torch.empty(sum(h * w for h, w, is16, _, _ in shapes if is16 == wide), dtype=t, device="cuda")
                for wide, t in ((False, torch.uint8), (True, torch.int16))]
        items, keep, at = [], [], [0, 0]
        for h, w, is16, s, lam in shapes:
            a = synth.disks(h, w, is16=is16, seed=s)
            t = _to_gpu(a)
            o = outs[is16][at[is16]:]
            at[is16] += h * w
            items.append((t.data_ptr(), a.dtype, a.shape, lam, o.data_ptr()))
            keep.append(t)
        state.update(items=items, keep=keep, outs=outs)
        return state
    img = _generate(case, seed)
    if case["kind"] == "operations":
        state["img"] = img
        state["ops"] = [("filter", 0, case["lam"]), ("extract", 0, 4 * case["lam"]), ("check", 12), ("filter", 17, 0.3)]
        return state
    state["img"] = _to_gpu(img)
    state["dtype"], state["shape"] = img.dtype, img.shape
    n_out = {"pair": 2, "rules": 7}.get(case["kind"], 1)
    state["outs"] = [torch.empty_like(state["img"]) for _ in range(n_out)]
    if case["bins"]:
        state["l1"] = _lambdas(case["attr"], case["bins"])
    if case["bins2"]:
        state["l2"] = _lambdas(0, case["bins2"])
    if case["kind"] == "rules":
        stream.wait_stream(torch.cuda.current_stream())
        state["tree"] = ctx.build_device(state["img"].data_ptr(), state["dtype"], state["shape"], case["conn"], case["tree"],
                                         case["attr"])
    return state


# ---- one pass ---------------------------------------------------------------------------------------------------------
def run(state):
    case, ctx, stream = state["case"], state["ctx"], state["stream"]
    kind = case["kind"]
    if kind == "operations":
        return ctx.run_operations(state["img"], state["ops"], connectivity=case["conn"], tree_type=case["tree"])
    stream.wait_stream(torch.cuda.current_stream())
    result = _device_pass(case, ctx, state)
    torch.cuda.current_stream().wait_stream(stream)
    return result


def _device_pass(case, ctx, state):
    kind, attr, lam, rule = case["kind"], case["attr"], case["lam"], case["decision"]
    if kind == "batch":
        ctx.batch_filter_device(state["items"], connectivity=case["conn"], tree_type=case["tree"], attr_idx=attr, decision=rule)
        return state["outs"]
    ptr, dtype, shape, outs = state["img"].data_ptr(), state["dtype"], state["shape"], state["outs"]
    if kind == "pair":
        ctx.batch_filter_device([(ptr, dtype, shape, lam, outs[0].data_ptr(), "max"),
                                 (ptr, dtype, shape, lam, outs[1].data_ptr(), "min")],
                                connectivity=case["conn"], attr_idx=attr, decision=rule)
        return outs
    if kind == "rules":
        tree = state["tree"]
        for i in range(4):
            tree.filter_device(attr, lam * 2 ** i, 0, outs[i].data_ptr(), dtype)
        tree.filter_device(attr, lam, 1, outs[4].data_ptr(), dtype)
        tree.filter_device(attr, lam, 2, outs[5].data_ptr(), dtype)
        tree.filter_device(attr, lam, 3, outs[6].data_ptr(), dtype)
        return outs + [tree.spectrum1d(attr, state["l1"])]
    if kind == "tiled":
        tree = ctx.build_tiled_device(ptr, dtype, shape, (1, case["slabs"]), case["conn"], case["tree"], attr)
    else:
        tree = ctx.build_device(ptr, dtype, shape, case["conn"], case["tree"], attr)
    tree.filter_device(attr, lam, rule, outs[0].data_ptr(), dtype)
    result = list(outs)
    if case["bins2"]:
        result.append(tree.spectrum2d(attr, state["l1"], 0, state["l2"]))
    elif case["bins"]:
        result.append(tree.spectrum1d(attr, state["l1"]))
    tree.free()
    return result


# ---- what a pass cannot do without --------------------------------------------------------------------------------------
def work(case):
    """bytes: every input image read once and every output written once; flops: one comparison per pixel and neighbour
    of each tree that is built (a filter of a tree that is there: one per pixel)"""
    kind = case["kind"]
    if kind == "batch":
        px = [(h * w, 2 if is16 else 1) for h, w, is16, _, _ in _shapes(case, 0)]
        return {"bytes": float(sum(2 * n * b for n, b in px)), "flops": float(case["conn"] * sum(n for n, _ in px))}
    n, b = case["depth"] * case["height"] * case["width"], _BYTES[case["dtype"]]
    if kind == "pair":
        return {"bytes": float(3 * n * b), "flops": float(2 * case["conn"] * n)}
    if kind == "operations":
        return {"bytes": float(n * (b + 4 * 4)), "flops": float(case["conn"] * n)}
    if kind == "rules":
        # the tree is the input: each pixel's node, and the results
        return {"bytes": float(n * (4 + 7 * b) + 8 * case["bins"]), "flops": float(7 * n)}
    return {"bytes": float(2 * n * b + 8 * case["bins"] * max(1, case["bins2"])), "flops": float(case["conn"] * n)}


# ---- the same in plain Python, 64 bits ----------------------------------------------------------------------------------
_EXACT_PIXELS = 300000


def _plain_tree(g, shape, conn):
    """parent pixel of every pixel (equal greys chained, -1 at the root) and the pixels from the highest down"""
    h, w = shape
    order = np.argsort(g, kind="stable")[::-1].tolist()
    offs = [(-1, 0), (1, 0), (0, -1), (0, 1)]
    if conn == 8:
        offs += [(-1, -1), (-1, 1), (1, -1), (1, 1)]
    top, parent = [-1] * g.size, [-1] * g.size
    for p in order:
        top[p] = p
        y, x = divmod(p, w)
        for dy, dx in offs:
            yy, xx = y + dy, x + dx
            if not (0 <= yy < h and 0 <= xx < w):
                continue
            q = yy * w + xx
            if top[q] < 0:
                continue
            while top[q] != q:
                top[q] = top[top[q]]
                q = top[q]
            if q != p:
                top[q] = p
                parent[q] = p
    return parent, order


def _plain_area_filter(img, conn, tree, lam, bins):
    """area opening by the direct rule (the subtractive rule's result for the area) and the area spectrum"""
    v = img.astype(np.float64).ravel()
    top = v.max()
    g = top - v if tree == "min" else v
    parent, order = _plain_tree(g, img.shape, conn)
    size = np.ones(g.size, dtype=np.int64)
    for p in order:
        if parent[p] >= 0:
            size[parent[p]] += size[p]
    level = list(range(g.size))
    out = np.empty(g.size)
    spectrum = np.zeros(len(bins)) if bins is not None else None
    for p in reversed(order):
        q = parent[p]
        if q >= 0 and g[q] == g[p]:
            level[p] = level[q]
            out[p] = out[q]
            continue
        out[p] = g[p] if size[p] >= lam else (out[q] if q >= 0 else 0.0)
        if spectrum is not None:
            rise = g[p] - (g[q] if q >= 0 else 0.0)
            if rise:
                at = int(np.searchsorted(bins.astype(np.float64), size[p], side="right")) - 1
                spectrum[max(at, 0)] += rise * size[p]
    if tree == "min":
        out = top - out
    return out.reshape(img.shape), spectrum


def exact(case, seed):
    if case["kind"] != "image" or case["depth"] > 1 or case["attr"] != 0 or case["height"] * case["width"] > _EXACT_PIXELS:
        return None
    img = _generate(case, seed)
    bins = _lambdas(0, case["bins"]) if case["bins"] else None
    out, spectrum = _plain_area_filter(img, case["conn"], case["tree"], case["lam"], bins)
    if img.dtype == np.uint16:
        out = out.astype(np.uint16).view(np.int16)  # the results are tensors of the same bits
    return [out] if spectrum is None else [out, spectrum]
