"""The work whose speed is watched: batches of decoded images through the augmentation ops and pipelines.

Every case is one batch of a program that trains on images or serves them: new parameters for the batch (crop windows, mirror
flags, colour factors, angles), then the op or the pipeline that applies them. The pixels are blurred noise with fine grain on
top, which is what decoded photographs look like to an interpolation."""
import math

import numpy as np
import torch

from rocal_amd import fn, ops, types
from rocal_amd import workloads as wl
from rocal_amd.pipeline import Pipeline

DTYPE = {"f32": ops.FP32, "f16": ops.FP16, "u8": ops.UINT8}
LAYOUT = {"nchw": ops.NCHW, "nhwc": ops.NHWC}
SIZE = {"f32": 4, "f16": 2, "u8": 1}
INTERP = {"linear": ops.LINEAR, "nearest": ops.NEAREST, "triangular": ops.TRIANGULAR}
MEAN = [float(v) for v in wl.MEAN]
STD = [float(v) for v in wl.STD]


def listed():
    return [
        # one image answered by a server, through the Python pipeline: latency and launches count
        {"name": "serve_1", "kind": "serve", "n": 1, "h": 299, "w": 299, "rs": 256, "oh": 224, "ow": 224, "dtype": "f16", "layout": "nchw"},
        # a detector's training step through the pipeline: crop, resize, colour, normalise, f32 planes of 300 x 300
        {"name": "chain_64", "kind": "chain", "n": 64, "h": 375, "w": 500, "oh": 300, "ow": 300, "dtype": "f32", "layout": "nchw"},
        # RandomResizedCrop of a classifier's training step on the padded batch of a loader (the benchmark's headline shapes)
        {"name": "rrc_256", "kind": "rrc", "n": 256, "h": 640, "w": 640, "lo": 240, "source": "padded", "interp": "linear", "oh": 224, "ow": 224,
         "dtype": "f16", "layout": "nchw"},
        # the same from images packed one behind the other without any padding, as a decoder writes them
        {"name": "rrc_packed_128", "kind": "rrc", "n": 128, "h": 640, "w": 640, "lo": 240, "source": "packed", "interp": "linear", "oh": 224, "ow": 224,
         "dtype": "f16", "layout": "nchw"},
        # the same windows with antialiasing
        {"name": "rrc_triangular_256", "kind": "rrc", "n": 256, "h": 640, "w": 640, "lo": 240, "source": "padded", "interp": "triangular", "oh": 224,
         "ow": 224, "dtype": "f16", "layout": "nchw"},
        # centre crop of resized images, mirrored at random, f32 planes
        {"name": "crop_128", "kind": "crop", "n": 128, "h": 256, "w": 256, "oh": 224, "ow": 224, "dtype": "f32", "layout": "nchw"},
        # colour augmentation in place of the image, rows of an odd number of bytes
        {"name": "twist_299", "kind": "colour", "op": "twist", "n": 128, "h": 299, "w": 299, "dtype": "u8", "layout": "nhwc"},
        # affine augmentation, the benchmark's shapes
        {"name": "warp_512", "kind": "warp", "n": 128, "h": 512, "w": 512, "interp": "linear", "dtype": "u8", "layout": "nhwc"},
        # rotation of images with rows of an odd number of bytes
        {"name": "rotate_299", "kind": "rotate", "n": 64, "h": 299, "w": 299, "interp": "linear", "dtype": "u8", "layout": "nhwc"},
        # full-HD frames brought down to a third with antialiasing, normalised
        {"name": "frames_1080", "kind": "fit", "n": 32, "h": 1080, "w": 1920, "interp": "triangular", "oh": 360, "ow": 640, "dtype": "f16", "layout": "nchw"},
        # label images: the nearest pixel, bytes in and out
        {"name": "labels_64", "kind": "labels", "n": 64, "h": 384, "w": 512, "oh": 256, "ow": 256, "dtype": "u8", "layout": "nhwc"},
        # normalisation by each image's own mean and deviation
        {"name": "normalize_64", "kind": "normalize", "n": 64, "h": 300, "w": 400, "dtype": "f32", "layout": "nchw"},
    ]


MOST_BYTES = 235e6  # a drawn case moves no more than the largest listed one


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _format(rng):
    """What a network is fed with: planes of half precision most of the time, f32 planes, and channels-last of either."""
    return rng.choice([("f16", "nchw"), ("f16", "nchw"), ("f32", "nchw"), ("f16", "nhwc"), ("f32", "nhwc")])


def draw(rng):
    kind = rng.choice(["serve", "chain", "rrc", "rrc", "rrc", "crop", "colour", "warp", "rotate", "fit", "labels", "normalize"])
    dtype, layout = _format(rng)
    c = {"kind": kind, "n": _log(rng, 8, 256)}
    if kind == "serve":
        c.update(n=_log(rng, 1, 32), h=_log(rng, 160, 720), w=_log(rng, 160, 960))
        c["oh"] = c["ow"] = rng.randint(96, 384)
        c.update(rs=int(c["oh"] * 256 / 224), dtype=dtype, layout=layout)
    elif kind == "chain":
        c.update(h=rng.randint(200, 640), w=rng.randint(200, 640), oh=rng.randint(96, 384), ow=rng.randint(96, 384), dtype=dtype, layout=layout)
    elif kind == "rrc":
        h, w, o = rng.randint(256, 720), rng.randint(256, 720), rng.choice([rng.randint(96, 384), rng.choice([128, 160, 192, 224, 256, 299])])
        c.update(h=h, w=w, lo=rng.randint(160, 256), source=rng.choice(["padded", "padded", "packed", "packed4"]),
                 interp=rng.choice(["linear", "linear", "triangular"]), oh=o, ow=o, dtype=dtype, layout=layout)
    elif kind == "crop":
        h, w = rng.randint(128, 400), rng.randint(128, 400)
        c.update(h=h, w=w, oh=rng.randint(h * 2 // 3, h), ow=rng.randint(w * 2 // 3, w), dtype=dtype, layout=layout)
    elif kind == "colour":
        c.update(op=rng.choice(["twist", "twist", "brightness", "contrast", "saturation"]), h=rng.randint(96, 512), w=rng.randint(96, 512), dtype="u8", layout="nhwc")
    elif kind in ("warp", "rotate"):
        c.update(h=rng.randint(96, 512), w=rng.randint(96, 512), interp=rng.choice(["linear", "linear", "nearest"]), dtype="u8", layout="nhwc")
    elif kind == "fit":
        c.update(n=_log(rng, 2, 32), h=rng.randint(480, 1080), w=rng.randint(640, 1920), interp=rng.choice(["linear", "triangular"]), dtype=dtype, layout=layout)
        shrink = rng.uniform(1.3, 3.5)
        c.update(oh=int(c["h"] / shrink), ow=int(c["w"] / shrink))
    elif kind == "labels":
        c.update(h=rng.randint(240, 640), w=rng.randint(240, 640), oh=rng.randint(128, 512), ow=rng.randint(128, 512), dtype="u8", layout="nhwc")
    else:
        c.update(h=rng.randint(96, 512), w=rng.randint(96, 512), dtype=dtype, layout=layout)
    while c["n"] > 1 and work(c)["bytes"] > MOST_BYTES:
        c["n"] -= 1 + c["n"] // 8
    return c


def _sizes(case, seed):
    """Widths and heights of the batch's images, and the crop windows of a RandomResizedCrop among them."""
    rng = np.random.default_rng(seed)
    n, h, w, lo = case["n"], case["h"], case["w"], case["lo"]
    H, W = rng.integers(lo, h + 1, n), rng.integers(lo, w + 1, n)
    return H, W, wl.random_crop_dec_windows(seed, H, W)


def work(case):
    n, px = case["n"], case["h"] * case["w"]
    out_px = case.get("oh", case["h"]) * case.get("ow", case["w"])
    kind = case["kind"]
    if kind == "rrc":  # the windows of such a batch, whatever its seed
        _, _, roi = _sizes(dict(case, n=512), 1)
        src_px = float((roi[:, 2].astype(np.float64) * roi[:, 3]).mean())
    elif kind == "chain":
        src_px = CHAIN_AREA * 0.77 * px  # (images of 75 to 100 % of either side)
    elif kind == "serve":
        src_px = px * (case["oh"] / case["rs"]) ** 2
    elif kind == "crop":
        src_px = out_px
    elif kind == "labels":
        src_px = min(px, out_px)
    else:
        src_px = px
    per_px = {"linear": 36, "nearest": 6}.get(case.get("interp", "linear"), 36)
    if case.get("interp") == "triangular":  # every source value into the columns that read it, every filtered row into its rows
        flops = src_px * 3 * 4 + out_px * 3 * 8
    else:
        flops = out_px * {"crop": 6, "labels": 6, "normalize": 15, "colour": 60, "chain": 96}.get(kind, per_px)
    return {"bytes": n * (3.0 * src_px + 3.0 * SIZE[case["dtype"]] * out_px), "flops": float(n * flops)}


def tolerance(case):
    # Bytes are the same bytes. Against 64 bits a half differs by the one rounding at its end (2.1e-4 of the result), an f32 multiply-add
    # by 7e-8, an f32 interpolation by 2e-6 (its coordinates), and a blend that is rounded to bytes before it is normalised by the
    # values that lie on a rounding boundary (1.6e-3).
    if case["dtype"] == "u8":
        return "exact"
    if case["kind"] in ("serve", "chain") or (case["kind"] == "rrc" and case["interp"] == "linear"):
        return {"rel": 3e-3}
    if case["dtype"] == "f16":
        return {"rel": 1e-3}
    return {"rel": 1e-5} if case["kind"] in ("rrc", "fit") else {"rel": 5e-7}


def _images(case, seed, n=None):
    """u8 [n, h, w, 3] on the GPU: blurred noise with grain."""
    n, h, w = n or case["n"], case["h"], case["w"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    out = torch.empty((n, h, w, 3), dtype=torch.uint8, device="cuda")
    for a in range(0, n, 64):
        m = min(64, n - a)
        coarse = torch.rand((m, 3, h // 12 + 2, w // 12 + 2), generator=gen, device="cuda") * 300 - 22
        img = torch.nn.functional.interpolate(coarse, size=(h, w), mode="bilinear", align_corners=False)
        img += torch.rand((m, 1, h, w), generator=gen, device="cuda") * 16 - 8
        out[a:a + m] = img.clamp_(0, 255).round_().to(torch.uint8).permute(0, 2, 3, 1)
    return out


CHAIN_AREA = 0.6


class _Piped:
    """A pipeline with its source fed from device memory and its output bound to a tensor of the program's own."""

    def __init__(self, case, seed):
        n = case["n"]
        rng = np.random.default_rng(seed)
        self.pipe = Pipeline(batch_size=n, device_id=0, seed=1)
        layout = types.NCHW if case["layout"] == "nchw" else types.NHWC
        dtype = {"f32": types.FLOAT, "f16": types.FLOAT16, "u8": types.UINT8}[case["dtype"]]
        low = 0.75 if case["kind"] == "chain" else 1.0
        self.widths = rng.integers(int(low * case["w"]), case["w"] + 1, n).astype(np.uint32)
        self.heights = rng.integers(int(low * case["h"]), case["h"] + 1, n).astype(np.uint32)
        self.images = _images(case, seed)
        with self.pipe:
            self.source = self.pipe.device_source(case["w"], case["h"])
            if case["kind"] == "serve":
                x = fn.resize(self.source, resize_width=case["rs"], resize_height=case["rs"])
                mirror = 0
            else:
                x = fn.resize_crop(self.source, resize_width=case["ow"], resize_height=case["oh"], crop_area_factor=CHAIN_AREA, crop_aspect_ratio=1.1,
                                   x_drift=0.4, y_drift=0.6)
                x = fn.color_twist(x, brightness=1.1, contrast=6.0, hue=12.0, saturation=1.2)
                mirror = 1
            self.out = fn.crop_mirror_normalize(x, crop=(case["oh"], case["ow"]), mean=MEAN, std=STD, mirror=mirror, output_layout=layout, output_dtype=dtype)
        self.pipe.set_outputs(self.out)
        self.pipe.build()
        self.dst = torch.zeros(_shape(case), dtype=ops.torch_dtype(DTYPE[case["dtype"]]), device="cuda")
        self.pipe.bind_output(self.out, self.dst)

    def run(self):
        self.pipe.feed(self.source, self.images, self.widths, self.heights)
        self.pipe.rocal_run()
        self.pipe.wait_on_stream()
        return self.dst

    def __del__(self):
        self.pipe.release()


def _shape(case):
    n, h, w = case["n"], case.get("oh", case["h"]), case.get("ow", case["w"])
    return (n, 3, h, w) if case["layout"] == "nchw" else (n, h, w, 3)


def _pack(images, H, W, dwords):
    """The images of a padded batch one behind the other: (buffer, offsets, row strides or None, bytes)."""
    stride = (W * 3 + 3) // 4 * 4 if dwords else W * 3
    ends = np.cumsum(stride * H)
    offsets = np.concatenate([[0], ends[:-1]]).astype(np.uint64)
    total = (int(ends[-1]) + 3) // 4 * 4
    buf = torch.zeros(total + 16, dtype=torch.uint8, device="cuda")
    for i in range(len(H)):
        h, w, o, st = int(H[i]), int(W[i]), int(offsets[i]), int(stride[i])
        buf[o:o + h * st].view(h, st)[:, :3 * w] = images[i, :h, :w].reshape(h, 3 * w)
    return buf, offsets, (stride.astype(np.uint32) if dwords else None), total


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("serve", "chain"):
        return _Piped(case, seed)
    rng = np.random.default_rng(seed)
    n, h, w = case["n"], case["h"], case["w"]
    oh, ow = case.get("oh", h), case.get("ow", w)
    ctx = ops.Context(0)
    sd = ops.desc(n, h, w, ops.NHWC, ops.UINT8)
    dd = ops.desc(n, oh, ow, LAYOUT[case["layout"]], DTYPE[case["dtype"]])
    whole = np.tile(np.array([0, 0, w, h], np.uint32), (n, 1))
    st = {"kind": kind, "ctx": ctx, "src": _images(case, seed)}
    scale = np.tile((1 / wl.STD).astype(np.float32), (n, 1))
    bias = np.tile((-wl.MEAN / wl.STD).astype(np.float32), (n, 1))
    mirror = (rng.random(n) < 0.5).astype(np.uint32)
    dw, dh = np.full(n, ow, np.uint32), np.full(n, oh, np.uint32)
    if kind == "rrc":
        H, W, roi = _sizes(case, seed)
        if case["source"] != "padded":
            st["src"], offsets, strides, total = _pack(st["src"], H, W, case["source"] == "packed4")
            st["packed"] = (offsets, W.astype(np.uint32), H.astype(np.uint32), total, strides)
        # (a bilinear node hands bytes on, the antialiasing one keeps its precision)
        op = ops.Resize(ctx, sd, dd, INTERP[case["interp"]], flags=ops.F_QUANTIZE_U8 if case["interp"] == "linear" else 0)
        st["args"] = (roi, dw, dh, scale, bias, mirror)
    elif kind == "fit":
        op = ops.Resize(ctx, sd, dd, INTERP[case["interp"]])
        st["args"] = (whole, dw, dh, scale, bias, mirror)
    elif kind == "labels":
        op = ops.Resize(ctx, sd, dd, ops.NEAREST)
        st["args"] = (whole, dw, dh, mirror)
    elif kind == "crop":
        op = ops.CropMirrorNormalize(ctx, sd, dd)
        st["args"] = (np.tile(np.array([(w - ow) // 2, (h - oh) // 2, ow, oh], np.uint32), (n, 1)), scale, bias, mirror)
    elif kind == "colour":
        u = lambda lo, hi: rng.uniform(lo, hi, n).astype(np.float32)  # noqa: E731
        op = {"twist": ops.ColorTwist, "brightness": ops.Brightness, "contrast": ops.Contrast, "saturation": ops.Saturation}[case["op"]](ctx, sd, dd)
        st["args"] = (whole,) + {"twist": lambda: (u(0.6, 1.4), u(-20, 20), u(-18, 18), u(0.6, 1.4)), "brightness": lambda: (u(0.6, 1.4), u(-20, 20)),
                                 "contrast": lambda: (u(0.6, 1.4), u(100, 150)), "saturation": lambda: (u(0.6, 1.4),)}[case["op"]]()
    elif kind == "warp":
        op = ops.WarpAffine(ctx, sd, dd, INTERP[case["interp"]])
        a = np.empty((n, 6), np.float32)
        for i in range(n):
            m = wl.inverse_affine(rng.uniform(-30, 30), rng.uniform(0.9, 1.1), rng.uniform(-16, 16), rng.uniform(-16, 16))
            a[i] = [m[0, 0], m[1, 0], m[0, 1], m[1, 1], m[0, 2], m[1, 2]]
        st["args"] = (whole, a, dw, dh)
    elif kind == "rotate":
        op = ops.Rotate(ctx, sd, dd, INTERP[case["interp"]])
        st["args"] = (whole, rng.uniform(-45, 45, n).astype(np.float32), dw, dh)
    else:
        op = ops.Normalize(ctx, sd, dd)
        st["args"] = (whole,)
    st["op"], st["dst"] = op, op.alloc_output()
    return st


def run(state):
    if isinstance(state, _Piped):
        return state.run()
    op = state["op"]
    if "packed" in state:
        op.set_ragged_source(*state["packed"])
    if state["kind"] in ("rrc", "fit"):
        op.update_cmn(*state["args"])
    else:
        op.update(*state["args"])
    op.launch(state["src"], state["dst"])
    return state["dst"]
