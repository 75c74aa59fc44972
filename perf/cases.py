"""The image work that a program built on this package has it do, as cases that can be timed and compared: through the
Python interface (`cvcuda_amd.pyapi`), on device memory that torch holds, as decoders and models hand it over.

`listed()` names one case per kind of program, from one camera frame to a batch of 4K float images; `draw()` gives
further cases of the same kinds over the ranges these stand for; `prepare()` makes what such a program has in hand
before the call and `run()` is one pass of it. `work()` counts the bytes that a pass cannot do without (each input
pixel that the result depends on read once, by whole spans of the rows that are touched; each output written once)
and its arithmetic.
"""
import math
import random

import numpy as np
import torch

from __graft_entry__ import load_package

load_package()
import cvcuda_amd.pyapi as cvcuda  # noqa: E402

INTERP = {"nearest": cvcuda.Interp.NEAREST, "linear": cvcuda.Interp.LINEAR, "cubic": cvcuda.Interp.CUBIC,
          "area": cvcuda.Interp.AREA}
BORDER = {"constant": cvcuda.Border.CONSTANT, "replicate": cvcuda.Border.REPLICATE}
TORCH = {"u8": torch.uint8, "f32": torch.float32}
SIZE = {"u8": 1, "f32": 4}
MEAN, STD = (0.485, 0.456, 0.406), (0.229, 0.224, 0.225)
MOST_BYTES = 500e6  # of a drawn case: about a third of the largest listed one's


def listed():
    return [
        # one camera frame scaled to a detector's square input: the smallest call, where latency and launches count
        {"name": "frame", "kind": "resize", "n": 1, "w": 1280, "h": 720, "c": 3, "dtype": "u8", "interp": "linear",
         "ow": 640, "oh": 640},
        # a classifier's batch of equal 1080p frames in one fused call (the benchmark's default workload)
        {"name": "classify_1080p", "kind": "fused", "n": 64, "w": 1920, "h": 1080, "short": 256, "crop": 224},
        # the same from a data loader: images of all sizes, made into an image batch for this one call
        {"name": "classify_loader", "kind": "fused_batch", "n": 61, "lo": 200, "hi": 1100, "short": 256, "crop": 224, "mix": 5},
        # the same preprocessing written as separate operators that allocate their outputs
        {"name": "classify_chain", "kind": "chain", "n": 16, "w": 1920, "h": 1080, "crop": 224},
        # previews of 1080p images by box filter, six times smaller
        {"name": "thumbnails", "kind": "resize", "n": 32, "w": 1920, "h": 1080, "c": 3, "dtype": "u8", "interp": "area",
         "ow": 320, "oh": 180},
        # a segmentation model's float maps enlarged to the odd-sized frames they belong to
        {"name": "mask_upsample", "kind": "resize", "n": 24, "w": 513, "h": 289, "c": 1, "dtype": "f32", "interp": "linear",
         "ow": 1917, "oh": 1079},
        # 4K float RGBA reduced bicubically (a benchmark configuration): the largest call
        {"name": "cubic_4k_f32", "kind": "resize", "n": 16, "w": 3840, "h": 2160, "c": 4, "dtype": "f32", "interp": "cubic",
         "ow": 640, "oh": 360},
        # decoded video frames to RGB (a benchmark configuration)
        {"name": "video_decode", "kind": "decode", "n": 32, "w": 1920, "h": 1080},
        # planar RGB from a model to the encoder's NV12, by way of interleaved RGB
        {"name": "video_encode", "kind": "encode", "n": 12, "w": 3840, "h": 2160},
        # augmentation of images of mixed sizes by rotation and scale (a benchmark configuration)
        {"name": "augment_rotate", "kind": "warp_batch", "n": 32, "wlo": 640, "whi": 1920, "hlo": 480, "hhi": 1080,
         "interp": "linear", "mix": 4},
        # page photographs straightened
        {"name": "straighten", "kind": "warp", "n": 16, "w": 1240, "h": 1754, "c": 3, "dtype": "u8", "interp": "cubic",
         "border": "replicate", "tilt": 0.15},
        # training crops, flipped at random and normalised
        {"name": "augment_crop", "kind": "augment", "n": 256, "wlo": 256, "whi": 512, "hlo": 256, "hhi": 384, "crop": 224, "mix": 7},
    ]


def _between(rng, lo, hi):
    """A whole number of lo .. hi, spread evenly over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def _fit(n, bytes_of_one):
    return max(1, min(n, int(MOST_BYTES / bytes_of_one)))


def draw(rng):
    kind = rng.choice(["resize"] * 5 + ["fused", "fused_batch", "chain", "decode", "encode", "warp", "warp", "warp_batch", "augment"])
    n = _between(rng, 1, 64)
    w, h = _between(rng, 200, 3840), _between(rng, 160, 2160)
    mix = rng.randrange(1000)
    if kind == "resize":
        c, dtype, interp = rng.choice([1, 3, 3, 3, 4]), rng.choice(["u8", "u8", "u8", "f32"]), rng.choice(sorted(INTERP))
        # enlarged up to 4 times or reduced up to 12 times, now and then not alike along both axes
        most = 1.0 if interp == "area" else 4.0
        factor = math.exp(rng.uniform(math.log(1 / 12), math.log(most)))
        other = factor if rng.random() < 0.7 else min(most, factor * math.exp(rng.uniform(-0.4, 0.4)))
        ow, oh = max(16, min(4096, round(w * factor))), max(16, min(4096, round(h * other)))
        if interp == "area":
            ow, oh = min(ow, w), min(oh, h)
        n = _fit(n, (w * h + ow * oh) * c * SIZE[dtype])
        return {"kind": kind, "n": n, "w": w, "h": h, "c": c, "dtype": dtype, "interp": interp, "ow": ow, "oh": oh}
    crop = rng.choice([224, 224, 160, 192, 299, 384])
    short = crop + crop // 7
    if kind == "fused":
        return {"kind": kind, "n": _fit(n, w * h * 3), "w": w, "h": h, "short": short, "crop": crop}
    if kind == "fused_batch":
        lo = _between(rng, 100, 700)
        return {"kind": kind, "n": n, "lo": lo, "hi": lo + _between(rng, 16, 900), "short": short, "crop": crop, "mix": mix}
    if kind == "chain":
        return {"kind": kind, "n": _fit(n, w * h * 3), "w": w, "h": h, "crop": crop}
    if kind in ("decode", "encode"):
        w, h = w & ~1, h & ~1
        return {"kind": kind, "n": _fit(n, w * h * (4.5 if kind == "decode" else 10.5)), "w": w, "h": h}
    if kind == "warp":
        c, dtype, interp = rng.choice([1, 3, 3, 4]), rng.choice(["u8", "u8", "u8", "f32"]), rng.choice(["nearest", "linear", "linear", "cubic"])
        w, h = min(w, 2048), min(h, 2048)
        return {"kind": kind, "n": _fit(n, w * h * c * SIZE[dtype] * (4 if interp == "cubic" else 2)), "w": w, "h": h, "c": c,
                "dtype": dtype, "interp": interp, "border": rng.choice(sorted(BORDER)), "tilt": round(rng.uniform(0.0, 0.3), 3)}
    if kind == "warp_batch":
        wlo, hlo = _between(rng, 64, 1200), _between(rng, 64, 900)
        return {"kind": kind, "n": min(n, 40), "wlo": wlo, "whi": wlo + _between(rng, 8, 800), "hlo": hlo,
                "hhi": hlo + _between(rng, 8, 600), "interp": rng.choice(["linear", "linear", "cubic"]), "mix": mix}
    lo = crop + rng.randrange(0, 64)
    return {"kind": kind, "n": 4 * n, "wlo": lo, "whi": lo + _between(rng, 8, 400), "hlo": lo, "hhi": lo + _between(rng, 8, 300),
            "crop": crop, "mix": mix}


# ---- inputs ----------------------------------------------------------------------------------------------------------
class _Photos:
    """Images as cameras give them: smooth shapes with noise on top, on the GPU, from the seed alone."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.host = random.Random(seed)

    def image(self, h, w, c, dtype="u8"):
        coarse = torch.rand((1, c, h // 48 + 2, w // 48 + 2), generator=self.gen, device="cuda")
        img = torch.nn.functional.interpolate(coarse, size=(h, w), mode="bilinear", align_corners=True)[0].permute(1, 2, 0)
        img = (img + 0.06 * (torch.rand((h, w, c), generator=self.gen, device="cuda") - 0.5)).clamp_(0, 1)
        return (img * 255).to(torch.uint8) if dtype == "u8" else img.contiguous()

    def batch(self, n, h, w, c, dtype="u8"):
        out = torch.empty((n, h, w, c), dtype=TORCH[dtype], device="cuda")
        for i in range(n):
            out[i] = self.image(h, w, c, dtype)
        return out


def _sizes(case):
    """(w, h) of every image of a batch of mixed sizes."""
    rng = random.Random(case["mix"])
    if case["kind"] == "fused_batch":
        return [(rng.randint(case["lo"], case["hi"]), rng.randint(case["lo"], case["hi"])) for _ in range(case["n"])]
    return [(rng.randint(case["wlo"], case["whi"]), rng.randint(case["hlo"], case["hhi"])) for _ in range(case["n"])]


def _scaled(w, h, short):
    """(w, h) with the shorter side at `short`."""
    return (short, max(short, round(h * short / w))) if w <= h else (max(short, round(w * short / h)), short)


def _rotation(w, h, rng):
    """2 x 3 forward matrix: a turn of up to 30 degrees and a scale of 0.8 to 1.2 about the centre."""
    t, s = math.radians(rng.uniform(-30, 30)), rng.uniform(0.8, 1.2)
    c, sn, cx, cy = s * math.cos(t), s * math.sin(t), (w - 1) / 2, (h - 1) / 2
    return [c, -sn, cx - c * cx + sn * cy, sn, c, cy - sn * cx - c * cy]


def _homography(w, h, tilt, rng):
    """3 x 3 forward matrix: a small turn about the centre and a perspective that shortens a side by up to `tilt`."""
    t, s = math.radians(rng.uniform(-8, 8)), rng.uniform(0.9, 1.1)
    c, sn, cx, cy = s * math.cos(t), s * math.sin(t), (w - 1) / 2, (h - 1) / 2
    m = [[c, -sn, cx - c * cx + sn * cy], [sn, c, cy - sn * cx - c * cy],
         [tilt * rng.uniform(-1, 1) / w, tilt * rng.uniform(-1, 1) / h, 1.0]]
    return np.asarray(m, np.float32)


def _dev(values, dtype=torch.float32):
    return torch.tensor(values, dtype=dtype, device="cuda")


def prepare(case, seed):
    kind, photos, s = case["kind"], _Photos(seed), {"kind": case["kind"], "case": case}
    n = case["n"]

    def wrapped(name, t, layout):
        s[name + "_torch"], s[name] = t, cvcuda.as_tensor(t, layout)

    def empty(*shape, dtype=torch.uint8):
        return torch.empty(shape, dtype=dtype, device="cuda")

    if kind == "resize":
        wrapped("src", photos.batch(n, case["h"], case["w"], case["c"], case["dtype"]), "NHWC")
        wrapped("dst", empty(n, case["oh"], case["ow"], case["c"], dtype=TORCH[case["dtype"]]), "NHWC")
    elif kind == "fused":
        wrapped("src", photos.batch(n, case["h"], case["w"], 3), "NHWC")
        wrapped("dst", empty(n, 3, case["crop"], case["crop"], dtype=torch.float32), "NCHW")
    elif kind == "fused_batch":
        s["surfaces"] = [photos.image(h, w, 3) for w, h in _sizes(case)]
    elif kind == "chain":
        wrapped("src", photos.batch(n, case["h"], case["w"], 3), "NHWC")
        wrapped("mean", _dev(MEAN).reshape(1, 1, 1, 3), "NHWC")
        wrapped("std", _dev(STD).reshape(1, 1, 1, 3), "NHWC")
    elif kind == "decode":
        # studio range: luma 16 .. 235, chroma about 128
        rgb = photos.batch(n, case["h"] * 3 // 2, case["w"], 1)
        wrapped("src", (rgb.to(torch.int16) * 219 // 255 + 16).to(torch.uint8), "NHWC")
        wrapped("dst", empty(n, case["h"], case["w"], 3), "NHWC")
    elif kind == "encode":
        wrapped("src", photos.batch(n, case["h"], case["w"], 3).permute(0, 3, 1, 2).contiguous(), "NCHW")
        wrapped("rgb", empty(n, case["h"], case["w"], 3), "NHWC")
        wrapped("dst", empty(n, case["h"] * 3 // 2, case["w"], 1), "NHWC")
    elif kind == "warp":
        wrapped("src", photos.batch(n, case["h"], case["w"], case["c"], case["dtype"]), "NHWC")
        wrapped("dst", empty(n, case["h"], case["w"], case["c"], dtype=TORCH[case["dtype"]]), "NHWC")
        s["xform"] = _homography(case["w"], case["h"], case["tilt"], photos.host)
    elif kind == "warp_batch":
        sizes = _sizes(case)
        s["src"] = cvcuda.as_images([photos.image(h, w, 3) for w, h in sizes])
        s["out"] = [empty(h, w, 3) for w, h in sizes]
        s["dst"] = cvcuda.as_images(s["out"])
        wrapped("xform", _dev([_rotation(w, h, photos.host) for w, h in sizes]), "NW")
    elif kind == "augment":
        sizes, crop = _sizes(case), case["crop"]
        s["src"] = cvcuda.as_images([photos.image(h, w, 3) for w, h in sizes])
        rects = [[[[photos.host.randint(0, w - crop), photos.host.randint(0, h - crop), crop, crop]]] for w, h in sizes]
        wrapped("rect", _dev(rects, torch.int32), "NHWC")
        wrapped("flip", _dev([[photos.host.choice([-1, 0, 1, 2])] for _ in sizes], torch.int32), "NC")
        wrapped("mean", 255 * _dev(MEAN).reshape(1, 1, 1, 3), "NHWC")
        wrapped("scale", 1 / (255 * _dev(STD)).reshape(1, 1, 1, 3), "NHWC")
        wrapped("dst", empty(n, 3, crop, crop, dtype=torch.float32), "NCHW")
    return s


def run(state):
    kind, case, s = state["kind"], state["case"], state
    if kind == "resize":
        cvcuda.resize_into(s["dst"], s["src"], INTERP[case["interp"]])
        return s["dst_torch"]
    if kind == "fused":
        dim, crop = _scaled(case["w"], case["h"], case["short"]), case["crop"]
        cvcuda.resize_crop_convert_reformat_into(s["dst"], s["src"], dim, cvcuda.Interp.LINEAR,
                                                 ((dim[0] - crop) // 2, (dim[1] - crop) // 2), scale=1 / (255 * 0.226),
                                                 offset=-0.449 / 0.226, srcCast=False)
        return s["dst_torch"]
    if kind == "fused_batch":
        short, crop = case["short"], case["crop"]
        batch = cvcuda.as_images(s["surfaces"], cvcuda.Format.RGB8)
        out = cvcuda.resize_crop_convert_reformat(batch, (short, short), cvcuda.Interp.LINEAR,
                                                  cvcuda.RectI((short - crop) // 2, (short - crop) // 2, crop, crop),
                                                  layout="NCHW", data_type=cvcuda.Type.F32, scale=1 / (255 * 0.226),
                                                  offset=-0.449 / 0.226, srcCast=False)
        return out.torch()
    if kind == "chain":
        crop = case["crop"]
        small = cvcuda.resize(s["src"], (case["n"], crop, crop, 3), cvcuda.Interp.LINEAR)
        unit = cvcuda.convertto(small, np.float32, scale=1 / 255)
        normal = cvcuda.normalize(unit, s["mean"], s["std"], cvcuda.NormalizeFlags.SCALE_IS_STDDEV)
        return cvcuda.reformat(normal, "NCHW").torch()
    if kind == "decode":
        cvcuda.cvtcolor_into(s["dst"], s["src"], cvcuda.ColorConversion.YUV2RGB_NV12)
        return s["dst_torch"]
    if kind == "encode":
        cvcuda.reformat_into(s["rgb"], s["src"])
        cvcuda.cvtcolor_into(s["dst"], s["rgb"], cvcuda.ColorConversion.RGB2YUV_NV12)
        return [s["dst_torch"], s["rgb_torch"]]
    if kind == "warp":
        cvcuda.warp_perspective_into(s["dst"], s["src"], s["xform"], INTERP[case["interp"]], border_mode=BORDER[case["border"]],
                                     border_value=[0, 0, 0, 0])
        return s["dst_torch"]
    if kind == "warp_batch":
        cvcuda.warp_affine_into(s["dst"], s["src"], s["xform"], INTERP[case["interp"]])
        return s["out"]
    cvcuda.crop_flip_normalize_reformat_into(s["dst"], s["src"], s["rect"], s["flip"], s["mean"], s["scale"])
    return s["dst_torch"]


# ---- what a pass cannot do without -----------------------------------------------------------------------------------
def _axis(src, new, first, count, interp):
    """(source indices referenced, length of the span they lie in) along one axis, for outputs first .. first + count."""
    scale = src / new
    d = np.arange(first, first + count) + 0.5
    if interp == "nearest":
        idx = np.minimum((d * scale).astype(np.int64), src - 1)
    elif interp == "area":
        return src, src
    else:
        lo, taps = np.floor(d * scale - 0.5).astype(np.int64), (0, 1) if interp == "linear" else (-1, 0, 1, 2)
        idx = np.clip(np.concatenate([lo + t for t in taps]), 0, src - 1)
    return len(np.unique(idx)), int(idx.max() - idx.min()) + 1


def _window(w, h, new, first, count, interp, pixel):
    """Source bytes of the outputs `first` .. `first` + `count` of a resize of (w, h) to `new`: touched rows by their span."""
    rows, _ = _axis(h, new[1], first[1], count[1], interp)
    _, span = _axis(w, new[0], first[0], count[0], interp)
    return rows * span * pixel


def _seen(w, h, matrix):
    """Share of a w x h source that the inverse image of a destination of the same size covers."""
    inv = np.linalg.inv(np.asarray(matrix, np.float64))
    g = 96
    x, y = np.meshgrid((np.arange(g) + 0.5) * w / g, (np.arange(g) + 0.5) * h / g)
    p = inv @ np.stack([x.ravel(), y.ravel(), np.ones(g * g)])
    u, v = p[0] / p[2] / w * 48, p[1] / p[2] / h * 48
    ok = (u >= 0) & (u < 48) & (v >= 0) & (v < 48)
    return len(set(zip(u[ok].astype(int), v[ok].astype(int)))) / 48.0 ** 2


TAP_FLOPS = {"nearest": 0, "linear": 8, "cubic": 40}  # per channel of an output pixel


def work(case):
    kind, n = case["kind"], case["n"]
    if kind == "resize":
        w, h, ow, oh, c, es = case["w"], case["h"], case["ow"], case["oh"], case["c"], SIZE[case["dtype"]]
        per = 2 * (w / ow) * (h / oh) if case["interp"] == "area" else TAP_FLOPS[case["interp"]]
        return {"bytes": n * (_window(w, h, (ow, oh), (0, 0), (ow, oh), case["interp"], c * es) + ow * oh * c * es),
                "flops": n * ow * oh * c * per}
    if kind in ("fused", "fused_batch"):
        crop, total = case["crop"], 0
        for w, h in [(case["w"], case["h"])] * n if kind == "fused" else _sizes(case):
            dim = _scaled(w, h, case["short"]) if kind == "fused" else (case["short"], case["short"])
            total += _window(w, h, dim, ((dim[0] - crop) // 2, (dim[1] - crop) // 2), (crop, crop), "linear", 3) + crop * crop * 12
        return {"bytes": total, "flops": n * crop * crop * 3 * 10}
    if kind == "chain":
        # the operators are separate calls: each one's input and output
        px = n * case["crop"] ** 2 * 3
        src = _window(case["w"], case["h"], (case["crop"],) * 2, (0, 0), (case["crop"],) * 2, "linear", 3) * n
        return {"bytes": src + px + 5 * px + 8 * px + 8 * px, "flops": px * 13}
    if kind == "decode":
        return {"bytes": n * case["w"] * case["h"] * 4.5, "flops": n * case["w"] * case["h"] * 9}
    if kind == "encode":
        return {"bytes": n * case["w"] * case["h"] * 10.5, "flops": n * case["w"] * case["h"] * 8}
    if kind == "warp":
        px = case["w"] * case["h"] * case["c"] * SIZE[case["dtype"]]
        m = _homography(case["w"], case["h"], case["tilt"], random.Random(1))
        return {"bytes": n * px * (1 + _seen(case["w"], case["h"], m)),
                "flops": n * case["w"] * case["h"] * (12 + case["c"] * TAP_FLOPS[case["interp"]])}
    if kind == "warp_batch":
        rng, total, px = random.Random(1), 0, 0
        for w, h in _sizes(case):
            m = _rotation(w, h, rng)
            total += w * h * 3 * (1 + _seen(w, h, [m[:3], m[3:], [0, 0, 1]]))
            px += w * h
        return {"bytes": total, "flops": px * (8 + 3 * TAP_FLOPS[case["interp"]])}
    px = n * case["crop"] ** 2 * 3
    return {"bytes": px * 5, "flops": px * 2}


def tolerance(case):
    """Bytes stay the same. Float results are float32 sums over taps whose places are float32 expressions: against the same
    formula with 64-bit places and sums, bilinear enlarging 513 x 289 to 1917 x 1079 differs by 3.0e-7 of the norm and
    3.2e-6 of the root mean square at most, bicubic reducing 4K to 640 x 360 by 0.8e-7 and 0.5e-6; the figures below are about
    four times the former. A perspective map divides by a third row that is itself rounded: its places are off by up to
    four times as much."""
    kind = case["kind"]
    if kind in ("decode", "encode", "warp_batch") or case.get("dtype") == "u8" or case.get("interp") == "nearest":
        return "exact"
    return {"rel": 5e-6, "max": 5e-5} if kind == "warp" else {"rel": 1.2e-6, "max": 1.3e-5}
