"""Workloads of the stereo engine as its users run them, for timing and for comparing builds.

Every case goes through the package's public entry points (the ctypes binding over the C ABI) with
images resident in device memory, the way a program that keeps its frames on the GPU calls it:
the fused matchers over all five algorithms, small frames to 4K, odd and ragged sizes, both
output formats, the search around an initial map, many pairs in one call, the learned proposal, the
reference-format operators with their cross check and filters, and a training step of the proposal
network.  Sizes are those of the benchmark, the tests and the training script, and ragged
neighbours of them.

Images are torch tensors (rows padded to 256 bytes, as stereo_image_alloc lays them out) that the
engine reads and writes in place; scenes are textured planes at known disparities.
"""
import ctypes
import json
import math
import os
import random
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "module.clutec.cuda_amd")
sys.path.insert(0, _PKG)
import clutec_stereo as cs  # noqa: E402

_ALGO = {"sad": cs.ALGO_SAD, "census": cs.ALGO_CENSUS, "ncc": cs.ALGO_NCC, "aw1": cs.ALGO_AW1, "aw2": cs.ALGO_AW2}
# operations per pixel and disparity that the method asks for (cost, two running sums, two
# winner-take-alls)
_OPS = {"sad": 10, "census": 12, "ncc": 11, "aw1": 13, "aw2": 13}
_CTX = None


def listed():
    return [
        # the smallest frame in use (the smoke check's): launches and latency
        {"name": "census_320x120_d64", "op": "matcher", "algo": "census", "w": 320, "h": 120, "d": 64, "win": 9,
         "cw": 9, "ch": 7, "maps": False, "ids": False},
        # a live VGA camera: rectify both images, SAD, de-noise, colour
        {"name": "camera_sad_640x480_d64", "op": "camera", "w": 640, "h": 480, "d": 64, "win": 9},
        # the benchmark's headline frame
        {"name": "census_1920x1080_d256", "op": "matcher", "algo": "census", "w": 1920, "h": 1080, "d": 256, "win": 9,
         "cw": 9, "ch": 7, "maps": False, "ids": False},
        # a cropped 4K frame with all three maps, smaller windows: the largest, no size a tile multiple
        {"name": "census_3839x2161_d256_maps", "op": "matcher", "algo": "census", "w": 3839, "h": 2161, "d": 256,
         "win": 7, "cw": 7, "ch": 7, "maps": True, "ids": False},
        # normalised correlation at full HD
        {"name": "ncc_1920x1080_d256", "op": "matcher", "algo": "ncc", "w": 1920, "h": 1080, "d": 256, "win": 11,
         "cw": 0, "ch": 0, "maps": False, "ids": False},
        # normalised correlation around an initial map at a quarter of the size, odd frame
        {"name": "ncc_band_1023x769_d192", "op": "band", "algo": "ncc", "w": 1023, "h": 769, "d": 192, "win": 9,
         "cw": 0, "ch": 0, "scale": 4},
        # adaptive windows at 720p with the reference's pixel format
        {"name": "aw1_1280x720_d128_ids", "op": "matcher", "algo": "aw1", "w": 1280, "h": 720, "d": 128, "win": 5,
         "cw": 0, "ch": 0, "maps": False, "ids": True},
        # pairs of uneven size in one call
        {"name": "batch_sad7_20pairs", "op": "batch", "algo": "sad", "win": 7, "cw": 1, "ch": 1, "pairs": 20, "mix": 100},
        # the learned proposal at full HD
        {"name": "learned_1920x1080_d256", "op": "learned", "w": 1920, "h": 1080, "d": 256},
        # the reference's own sequence: NCC in both directions, cross check, de-noise, colour
        {"name": "reference_ncc_1280x720_d128", "op": "refncc", "w": 1280, "h": 720, "d": 128, "patch": 11},
        # the reference's BlockMatcher1 at full HD
        {"name": "bm1_1920x1080_d256", "op": "refblock", "kind": "bm1", "w": 1920, "h": 1080, "d": 256, "patch": 9},
        # one training step of the proposal network (the training script's batch and size): forward,
        # backward, update
        {"name": "train_16x240x135", "op": "train", "frames": 16, "w": 240, "h": 135},
    ]


def _size(rng, lo_w, hi_w):
    """A frame between lo_w and hi_w columns, odd widths among them, near the usual aspect ratios."""
    w = int(round(math.exp(rng.uniform(math.log(lo_w), math.log(hi_w)))))
    h = int(w * rng.uniform(0.45, 0.8)) + rng.randrange(3)
    return w, max(96, h)


def draw(rng):
    op = rng.choice(["matcher", "matcher", "matcher", "matcher", "camera", "band", "batch", "learned", "refncc",
                     "refblock", "train"])
    if op == "matcher":
        algo = rng.choice(["census", "census", "sad", "ncc", "aw1", "aw2"])
        w, h = _size(rng, 320, 3200 if algo in ("census", "sad") else 1920)
        d = 8 * rng.randint(4, 32 if w >= 640 else 8)
        win = rng.choice({"census": [5, 7, 9], "sad": [5, 7, 9], "ncc": [5, 7, 9, 11], "aw1": [3, 5], "aw2": [3, 5]}[algo])
        cw, ch = rng.choice([(9, 7), (7, 7), (5, 5)]) if algo == "census" else (0, 0)
        return {"op": op, "algo": algo, "w": w, "h": h, "d": d, "win": win, "cw": cw, "ch": ch,
                "maps": rng.random() < 0.4, "ids": rng.random() < 0.3}
    if op == "camera":
        w, h = _size(rng, 320, 1280)
        return {"op": op, "w": w, "h": h, "d": 8 * rng.randint(4, 16), "win": rng.choice([5, 7, 9])}
    if op == "band":
        algo = rng.choice(["census", "sad", "ncc", "aw1"])
        w, h = _size(rng, 480, 1920)
        return {"op": op, "algo": algo, "w": w, "h": h, "d": 8 * rng.randint(8, 32), "win": 5 if algo == "aw1" else 9,
                "cw": 9 if algo == "census" else 0, "ch": 7 if algo == "census" else 0, "scale": rng.choice([2, 4])}
    if op == "batch":
        algo = rng.choice(["sad", "census"])
        return {"op": op, "algo": algo, "win": 7 if algo == "sad" else 9, "cw": 1 if algo == "sad" else 9,
                "ch": 1 if algo == "sad" else 7, "pairs": rng.randint(8, 20), "mix": rng.randrange(1000)}
    if op == "learned":
        w, h = _size(rng, 800, 1920)
        return {"op": op, "w": w - w % 4, "h": h - h % 4, "d": 32 * rng.randint(3, 8)}
    if op == "refncc":
        w, h = _size(rng, 320, 1280)
        return {"op": op, "w": w, "h": h, "d": rng.randint(32, 128), "patch": rng.choice([5, 9, 11])}
    if op == "refblock":
        w, h = _size(rng, 320, 1280)
        kind = rng.choice(["bm1", "aw1"])
        return {"op": op, "kind": kind, "w": w, "h": h, "d": rng.randint(32, 128),
                "patch": rng.choice([5, 9, 11, 15] if kind == "bm1" else [9, 15])}
    return {"op": op, "frames": rng.randint(1, 16), "w": rng.randint(100, 240), "h": rng.randint(60, 135)}


# ---- inputs -------------------------------------------------------------------------

def _context():
    global _CTX
    if _CTX is None:
        _CTX = cs.Context(0)
    return _CTX


class _TensorImage:
    """A device image over a torch tensor of padded rows, for the binding's process calls."""

    # 16-bit ids are held as int16 patterns
    _TYPES = {cs.PIXEL_LUM_U8: (torch.uint8, 1), cs.PIXEL_LUM_U16: (torch.int16, 1), cs.PIXEL_LUM_I16: (torch.int16, 1),
              cs.PIXEL_RGBA_U16: (torch.int16, 4), cs.PIXEL_RGBA_U8: (torch.uint8, 4)}

    def __init__(self, w, h, pixel_type, data=None):
        dtype, ch = self._TYPES[pixel_type]
        size = torch.empty((), dtype=dtype).element_size()
        pitch = (w * ch * size + 255) // 256 * 256
        raw = torch.zeros((h, pitch // 2), dtype=torch.int16, device="cuda").view(dtype)
        self.view = raw[:, :w * ch] if ch == 1 else raw[:, :w * ch].unflatten(1, (w, ch))
        if data is not None:
            self.view.copy_(data)
        self.img = cs.Image(raw.data_ptr(), pitch, cs.ImageFormat(w, h, pixel_type))

    @property
    def ref(self):
        return ctypes.byref(self.img)


def _texture(gen, h, w):
    """Smooth shading with fine grain, its contrast fading in places (0 .. 255)."""
    rand = lambda a, b: torch.rand((1, 1, a, b), generator=gen, device="cuda")  # noqa: E731
    up = lambda t: torch.nn.functional.interpolate(t, size=(h, w), mode="bilinear", align_corners=False)  # noqa: E731
    coarse = up(rand(h // 24 + 2, w // 24 + 2))
    mid = up(rand(h // 5 + 2, w // 5 + 2)) - 0.5
    fine = rand(h, w) - 0.5
    contrast = (3.0 * up(rand(h // 90 + 2, w // 90 + 2)) - 0.4).clamp(0.02, 1.0)
    return (60 + 130 * coarse + contrast * (110 * mid + 60 * fine))[0, 0]


def _scene(seed, w, h, dmax):
    """A left / right pair (uint8) of rectangles on slanted or constant disparities, and the left
    image's disparity (int16, -1 where the right image does not show the point)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rng = random.Random(seed)
    xs = torch.arange(w, device="cuda", dtype=torch.float32)[None, :]
    ys = torch.arange(h, device="cuda", dtype=torch.float32)[:, None]
    top = float(dmax - 1)
    disp = (0.04 + 0.1 * rng.random()) * top + 0.06 * top * (ys / h) + 0 * xs
    for k in range(rng.randint(10, 20)):
        rw, rh = int(w * rng.uniform(0.08, 0.35)), int(h * rng.uniform(0.08, 0.4))
        x0, y0 = rng.randrange(max(1, w - rw)), rng.randrange(max(1, h - rh))
        d = top * rng.uniform(0.15, 0.97)
        slant = rng.choice([0.0, 0.0, 1.0]) * rng.uniform(-0.06, 0.06)
        box = (d + slant * (xs[:, x0:x0 + rw] - x0) + 0 * ys[y0:y0 + rh]).clamp(0, top)
        disp[y0:y0 + rh, x0:x0 + rw] = torch.maximum(disp[y0:y0 + rh, x0:x0 + rw], box)
    disp = disp.round().clamp(0, top).long()
    tex = _texture(gen, h, w + dmax)
    right = tex[:, dmax:]
    pos = torch.arange(w, device="cuda")[None, :] - disp
    left = torch.gather(tex, 1, pos + dmax)
    noise = lambda: torch.randint(-2, 3, (h, w), generator=gen, device="cuda")  # noqa: E731
    as_u8 = lambda t: (t.round().long() + noise()).clamp(0, 255).to(torch.uint8)  # noqa: E731
    return as_u8(left), as_u8(right), torch.where(pos >= 0, disp, -1).to(torch.int16)


def _pair(seed, w, h, dmax):
    left, right, disp = _scene(seed, w, h, dmax)
    return _TensorImage(w, h, cs.PIXEL_LUM_U8, left), _TensorImage(w, h, cs.PIXEL_LUM_U8, right), disp


def _batch_sizes(case):
    rng = random.Random(case["mix"])
    sizes = [(16 * rng.randint(20, 80), 16 * rng.randint(15, 60)) for _ in range(case["pairs"])]
    return sizes, [rng.choice([64, 128, 192, 256]) for _ in range(case["pairs"])]


def _camera(w, h):
    """A rectification of the tests' kind: OpenCV distortion and a small rotation."""
    f = 0.9 * w
    src = [f, 0.99 * f, 0.49 * w, 0.51 * h]
    dist = [-0.12, 0.04, 0.0005, -0.0004, -0.005]
    rect = [0.97 * f, 0.97 * f, 0.5 * w, 0.5 * h]
    a = 0.01
    return src + dist + rect + [math.cos(a), -math.sin(a), 0.0, math.sin(a), math.cos(a), 0.0, 0.0, 0.0, 1.0]


def _matcher(case, **more):
    return cs.Matcher(_context(), case["w"], case["h"], algorithm=_ALGO[case["algo"]], window=(case["win"], case["win"]),
                      census=(case["cw"] or 9, case["ch"] or 7), num_disp=case["d"], tol=1, **more)


def _train_data(case, seed):
    """A training batch: quarter-resolution pairs with a coarse map (holes in it), full-resolution labels and
    confidence targets, and initial parameters (layer by layer, He-normal)."""
    n, w, h = case["frames"], case["w"], case["h"]
    gen = torch.Generator(device="cuda").manual_seed(seed + 7)
    out = {"frames": []}
    for i in range(n):
        left, right, disp = _scene(1000 * seed + i, 4 * w, 4 * h, 128)
        quarter = lambda t: (t.float().view(h, 4, w, 4).mean(dim=(1, 3)) + 0.5).to(torch.uint8)  # noqa: E731
        hole = torch.rand((h // 6 + 1, w // 6 + 1), generator=gen, device="cuda") < 0.12
        hole = hole.repeat_interleave(6, 0)[:h].repeat_interleave(6, 1)[:, :w]
        seen = disp[2::4, 2::4]
        shift = torch.randint(-1, 2, (h, w), generator=gen, device="cuda")
        coarse = torch.where(hole | (seen < 0), -1, (seen.long() // 4 + shift).clamp(0, 31)).to(torch.int16)
        conf = torch.randint(0, 12, (h, w), generator=gen, device="cuda")
        conf = torch.where(conf == 0, 0, torch.where(conf == 1, 255, 1)).to(torch.uint8)
        out["frames"].append((quarter(left), quarter(right), coarse, disp, conf))
    rng = np.random.default_rng(seed)
    parts = []
    for cin, cout, _ in cs.CNN_LAYERS:
        parts.append((rng.standard_normal((cout, 3, 3, cin)) * math.sqrt(2.0 / (9 * cin))).astype(np.float32).ravel())
        parts.append((0.05 * rng.standard_normal(cout)).astype(np.float32))
    out["params"] = np.concatenate(parts)
    return out


def prepare(case, seed):
    op, ctx = case["op"], _context()
    s = {"case": case}
    if op == "train":
        data = _train_data(case, seed)
        w, h = case["w"], case["h"]
        net = cs.ProposalNet(ctx, w, h, max_frames=case["frames"])
        net.set_params(data["params"])
        keep = []
        for i, (l4, r4, coarse, disp, conf) in enumerate(data["frames"]):
            im = [_TensorImage(w, h, cs.PIXEL_LUM_U8, l4), _TensorImage(w, h, cs.PIXEL_LUM_U8, r4),
                  _TensorImage(w, h, cs.PIXEL_LUM_I16, coarse), _TensorImage(4 * w, 4 * h, cs.PIXEL_LUM_I16, disp),
                  _TensorImage(w, h, cs.PIXEL_LUM_U8, conf)]
            net.set_input(i, im[0], im[1], im[2])
            net.set_labels(i, im[3])
            net.set_conf_labels(i, im[4])
            keep.append(im)
        torch.cuda.synchronize()
        s.update(net=net)
        return s
    if op == "batch":
        sizes, ds = _batch_sizes(case)
        m = cs.BatchMatcher(ctx, sizes, ds, algorithm=_ALGO[case["algo"]], window=(case["win"], case["win"]),
                            census=(case["cw"], case["ch"]))
        pairs = [_pair(100 * seed + i, w, h, d)[:2] for i, ((w, h), d) in enumerate(zip(sizes, ds))]
        outs = [[_TensorImage(w, h, cs.PIXEL_LUM_I16) for (w, h) in sizes] for _ in range(3)]
        arr = lambda imgs: (cs.Image * len(sizes))(*[i.img for i in imgs])  # noqa: E731
        m.dev = tuple(arr(o) for o in outs) + (arr([p[0] for p in pairs]), arr([p[1] for p in pairs]))
        s.update(m=m, pairs=pairs, outs=outs)
        return s
    w, h, d = case["w"], case["h"], case["d"]
    left, right, disp = _pair(seed, w, h, d)
    s.update(left=left, right=right)
    i16 = lambda: _TensorImage(w, h, cs.PIXEL_LUM_I16)  # noqa: E731
    ids = lambda: _TensorImage(w, h, cs.PIXEL_RGBA_U16)  # noqa: E731
    if op == "matcher":
        s.update(m=_matcher(case), out=ids() if case["ids"] else i16(), lr=i16() if case["maps"] else None,
                 rl=i16() if case["maps"] else None)
    elif op == "band":
        k = case["scale"]
        init = disp[k // 2::k, k // 2::k]
        init = torch.where(init < 0, -1, init // k).to(torch.int16)
        init = init[:h // k, :w // k]
        s.update(m=_matcher(case, use_disp_input=True), out=i16(),
                 init=_TensorImage(init.shape[1], init.shape[0], cs.PIXEL_LUM_I16, init))
    elif op == "camera":
        s.update(rect=cs.Rectify(ctx, w, h, _camera(w, h)), rl=_TensorImage(w, h, cs.PIXEL_LUM_U8),
                 rr=_TensorImage(w, h, cs.PIXEL_LUM_U8),
                 m=cs.Matcher(ctx, w, h, algorithm=cs.ALGO_SAD, window=(case["win"], case["win"]), num_disp=d, tol=1),
                 disp=ids(), dn=cs.Denoise(ctx, w, h, patch=5, ref_format=True), clean=_TensorImage(w, h, cs.PIXEL_LUM_U16),
                 col=cs.ColorDisparity(ctx, w, h, pixel_type=cs.PIXEL_LUM_U16, disp_min=1, disp_max=d),
                 image=_TensorImage(w, h, cs.PIXEL_RGBA_U8))
    elif op == "learned":
        folder = os.path.join(_PKG, "weights")
        with open(os.path.join(folder, "proposal_cnn.bin.json")) as f:
            meta = json.load(f)
        params = np.fromfile(os.path.join(folder, "proposal_cnn.bin"), "<f4")
        s.update(m=cs.LearnedMatcher(ctx, w, h, params, num_disp=d, band=int(meta.get("band", 8)),
                                     chunk=int(meta.get("chunk", 32)), logit_thresh=float(meta["logit_thresh"])),
                 out=i16())
    elif op == "refncc":
        kw = dict(patch=case["patch"], disp_min=0, disp_max=d, min_delta_thresh=2, ncc_thresh=0.5, grad_thresh=2.0)
        s.update(ml=cs.BlockMatcherNCC(ctx, w, h, left_to_right=True, **kw),
                 mr=cs.BlockMatcherNCC(ctx, w, h, left_to_right=False, **kw), lr=ids(), rl=ids(),
                 check=cs.CrossCheck(ctx, w, h, thresh=1), kept=ids(),
                 dn=cs.Denoise(ctx, w, h, patch=5, ref_format=True), clean=_TensorImage(w, h, cs.PIXEL_LUM_U16),
                 col=cs.ColorDisparity(ctx, w, h, pixel_type=cs.PIXEL_LUM_U16, disp_min=1, disp_max=d),
                 image=_TensorImage(w, h, cs.PIXEL_RGBA_U8))
    else:
        if case["kind"] == "bm1":
            m = cs.BlockMatcher1(ctx, w, h, patch=case["patch"], disp_min=0, disp_max=d, min_delta_thresh=1.0,
                                 sim_thresh=60.0, grad_thresh=2.0)
        else:
            m = cs.BlockMatcherAW1(ctx, w, h, patch=case["patch"], disp_min=0, disp_max=d, min_delta_thresh=0.5,
                                   sim_thresh=60.0, grad_thresh=2.0)
        s.update(m=m, out=ids())
    return s


# ---- the calls ------------------------------------------------------------------------

def run(s):
    op = s["case"]["op"]
    if op == "matcher":
        s["m"].process(s["out"], s["lr"], s["rl"], s["left"], s["right"])
        return [s[k].view for k in ("out", "lr", "rl") if s[k] is not None]
    if op == "band":
        s["m"].process_init(s["out"], None, None, s["left"], s["right"], s["init"])
        return s["out"].view
    if op == "camera":
        s["rect"].process(s["rl"], s["left"])
        s["rect"].process(s["rr"], s["right"])
        s["m"].process(s["disp"], None, None, s["rl"], s["rr"])
        s["dn"].process(s["clean"], s["disp"])
        s["col"].process(s["image"], s["clean"], cs.COLOR_COLOR)
        return [s["disp"].view, s["clean"].view, s["image"].view]
    if op == "batch":
        s["m"].process()
        return [o.view for maps in s["outs"] for o in maps]
    if op == "learned":
        s["m"].process(s["out"], None, None, s["left"], s["right"])
        return s["out"].view
    if op == "refncc":
        s["ml"].process(s["lr"], s["left"], s["right"])
        s["mr"].process(s["rl"], s["right"], s["left"])
        s["check"].process(s["kept"], s["lr"], s["rl"])
        s["dn"].process(s["clean"], s["kept"])
        s["col"].process(s["image"], s["clean"], cs.COLOR_COLOR)
        return [s["lr"].view, s["rl"].view, s["kept"].view, s["clean"].view, s["image"].view]
    if op == "refblock":
        s["m"].process(s["out"], s["left"], s["right"])
        return s["out"].view
    loss = s["net"].train_step(s["case"]["frames"], 2e-3)
    return {"loss": loss, "grads": s["net"].grads()}


# ---- what a pass cannot do without ------------------------------------------------------

def work(case):
    op = case["op"]
    if op == "train":
        px = case["frames"] * case["w"] * case["h"]
        macs = sum(9 * cin * cout for cin, cout, _ in cs.CNN_LAYERS)
        first = 9 * cs.CNN_LAYERS[0][0] * cs.CNN_LAYERS[0][1]  # the input's gradient is not asked for
        # the input, the labels and targets; each hidden activation and gradient written and read
        return {"bytes": px * (4 + 12 + 4 * 2 * 32 * 2), "flops": 2.0 * px * (3 * macs - first)}
    if op == "batch":
        sizes, ds = _batch_sizes(case)
        px = sum(w * h for w, h in sizes)
        return {"bytes": px * (2 + 6), "flops": float(_OPS[case["algo"]]) * sum(w * h * d for (w, h), d in zip(sizes, ds))}
    px, d = case["w"] * case["h"], case["d"]
    if op == "matcher":
        return {"bytes": px * (2 + (8 if case["ids"] else 2) + (4 if case["maps"] else 0)),
                "flops": float(px) * d * _OPS[case["algo"]]}
    if op == "band":
        return {"bytes": px * (2 + 2 + 2.0 / case["scale"] ** 2), "flops": float(px) * d / 4 * _OPS[case["algo"]]}
    if op == "camera":
        return {"bytes": px * (2 + 2 + 2 + 8 + 8 + 2 + 2 + 4), "flops": float(px) * (d * _OPS["sad"] + 2 * 60)}
    if op == "learned":
        # the coarse match at a quarter of the size and range, the network, a quarter of the range
        macs = sum(9 * cin * cout for cin, cout, _ in cs.CNN_LAYERS)
        return {"bytes": px * 4, "flops": px * (d / 64.0 * 12 + 2.0 * macs / 16 + d / 4.0 * 12)}
    if op == "refncc":
        return {"bytes": px * (2 * (2 + 8) + 24 + 10 + 6), "flops": 2.0 * px * d * 12}
    return {"bytes": px * (2 + 8), "flops": float(px) * d * 12}


# ---- the training step in 64 bits -------------------------------------------------------

def _fill(coarse):
    """The coarse map with holes filled by the smaller of the nearest valid values within 64 columns."""
    h, w = coarse.shape
    x = torch.arange(w, device=coarse.device)[None, :].expand(h, w)
    ok = coarse >= 0
    near_l = torch.where(ok, x, -10 ** 6).cummax(dim=1).values
    near_r = torch.where(ok, x, 10 ** 6).flip(1).cummin(dim=1).values.flip(1)
    big = 10 ** 6
    val = coarse.long()
    a = torch.where(x - near_l <= 64, val.gather(1, near_l.clamp(0, w - 1)), big)
    b = torch.where(near_r - x <= 64, val.gather(1, near_r.clamp(0, w - 1)), big)
    m = torch.minimum(a, b)
    return torch.where(ok, val, torch.where(m == big, 0, m))


def _shifted(t, dy, dx):
    """t[n, y + dy, x + dx, c], zero outside."""
    n, h, w, c = t.shape
    out = torch.zeros_like(t)
    ys, xs = slice(max(0, -dy), min(h, h - dy)), slice(max(0, -dx), min(w, w - dx))
    yt, xt = slice(max(0, dy), min(h, h + dy)), slice(max(0, dx), min(w, w + dx))
    out[:, ys, xs] = t[:, yt, xt]
    return out


def exact(case, seed):
    if case["op"] != "train":
        return None  # whole numbers
    data = _train_data(case, seed)
    n, w, h = case["frames"], case["w"], case["h"]
    inputs, fills, labels, confs = [], [], [], []
    for l4, r4, coarse, disp, conf in data["frames"]:
        fill = _fill(coarse)
        x = torch.arange(w, device="cuda")[None, :]
        warped = r4.long().gather(1, (x - fill).clamp(0, w - 1))
        inputs.append(torch.stack([l4.double() / 255, warped.double() / 255], dim=-1))
        fills.append(fill.double())
        blocks = disp.long().view(h, 4, w, 4).permute(0, 2, 1, 3).reshape(h, w, 16)
        ok = blocks >= 0
        cnt, total = ok.sum(-1), torch.where(ok, blocks, 0).sum(-1)
        span = torch.where(ok, blocks, -1).amax(-1) - torch.where(ok, blocks, 10 ** 6).amin(-1)
        labels.append(torch.where((cnt >= 8) & (span <= 4), total.double() / (4 * cnt.clamp(min=1)), float("nan")))
        confs.append(torch.where(conf <= 1, conf.double(), float("nan")))
    x, fill, label, conf = (torch.stack(t) for t in (inputs, fills, labels, confs))
    weights, k = [], 0
    for cin, cout, dil in cs.CNN_LAYERS:
        wt = torch.from_numpy(data["params"][k:k + 9 * cin * cout].astype(np.float64)).cuda().view(cout, 9, cin)
        k += 9 * cin * cout
        b = torch.from_numpy(data["params"][k:k + cout].astype(np.float64)).cuda()
        k += cout
        weights.append((wt, b, dil))
    taps = [(t // 3 - 1, t % 3 - 1) for t in range(9)]
    acts = [x]
    for l, (wt, b, dil) in enumerate(weights):
        y = b + sum(_shifted(acts[-1], dy * dil, dx * dil).reshape(-1, wt.shape[2]).mm(wt[:, t].t()).view(n, h, w, -1)
                    for t, (dy, dx) in enumerate(taps))
        acts.append(y if l == len(weights) - 1 else y.clamp(min=0))
    o0, o1 = acts[-1][..., 0], acts[-1][..., 1]
    t = label - fill
    has = torch.isfinite(t)
    e = torch.where(has, o0 - t, 0.0)
    ae = e.abs()
    target = torch.where(has, (ae <= 2.0).double(), -1.0)
    target = torch.where(torch.isfinite(conf), conf, target)
    sure = target >= 0
    px = n * w * h
    huber = torch.where(has, torch.where(ae <= 1, 0.5 * e * e, ae - 0.5), 0.0).sum()
    bce = torch.where(sure, o1.clamp(min=0) - o1 * target + torch.log1p(torch.exp(-o1.abs())), 0.0).sum()
    count = (has | sure).sum().double()
    g = torch.zeros_like(acts[-1])
    g[..., 0] = torch.where(has, e.clamp(-1, 1), 0.0) / px
    g[..., 1] = torch.where(sure, 0.5 * (torch.sigmoid(o1) - target), 0.0) / px
    grads = [None] * len(weights)
    for l in range(len(weights) - 1, -1, -1):
        wt, b, dil = weights[l]
        flat = g.reshape(px, -1)
        dw = torch.stack([flat.t().mm(_shifted(acts[l], dy * dil, dx * dil).reshape(px, -1)) for dy, dx in taps], dim=1)
        grads[l] = torch.cat([dw.reshape(-1), flat.sum(0)])
        if l:
            g = sum(_shifted(g, -dy * dil, -dx * dil).reshape(px, -1).mm(wt[:, t]).view(n, h, w, -1)
                    for t, (dy, dx) in enumerate(taps))
            g = torch.where(acts[l] > 0, g, 0.0)
    loss = torch.stack([huber / count, bce / count, count, torch.where(sure, target, 0.0).sum() / count])
    return {"loss": loss, "grads": torch.cat(grads)}
