"""The performance cases of this framework: 2x luma passes of every model family in the
precisions and element types they are run in, a batched launch over uneven images, the
device-resident colour pipeline around a pass, and `Processor.process` on a host image.

A case is a dict of plain values; `prepare` makes what a program holds before the call
(device tensors or host arrays, the net, its workspace), `run` makes the one call.
"""
import math
import os
import random

import numpy as np
import torch
import torch.nn.functional as F

import anime4kcpp_amd
from anime4kcpp_amd import hip, processor

DEVICE = "cuda:0"
WEIGHTS = os.path.join(os.path.dirname(os.path.abspath(anime4kcpp_amd.__file__)), "weights")
DTYPES = {"u8": torch.uint8, "u16": torch.uint16, "f16": torch.float16, "f32": torch.float32}
BYTES = {"u8": 1, "u16": 2, "f16": 2, "f32": 4}


# ---- the cases ----

def listed():
    return [
        # a thumbnail or icon: launches and host time
        {"name": "thumb_fp32_u8", "op": "pass", "family": "legacy", "variant": "hdn0", "precision": "fp32", "dtype": "u8",
         "w": 128, "h": 96},
        # the 256 x 256 float image of the parity workload
        {"name": "luma256_fp32_f32", "op": "pass", "family": "legacy", "variant": "hdn0", "precision": "fp32",
         "dtype": "f32", "w": 256, "h": 256},
        # the default model at the frame size of the benchmark tool of the original project
        {"name": "sd_default_fp32", "op": "pass", "family": "acnet8", "variant": "b8_hdn", "precision": "fp32",
         "dtype": "u8", "w": 720, "h": 480},
        # a 1080p video frame to 4K, the headline workload, in both arithmetics
        {"name": "hd_fp32", "op": "pass", "family": "legacy", "variant": "hdn1", "precision": "fp32", "dtype": "u8",
         "w": 1920, "h": 1080},
        {"name": "hd_fp16", "op": "pass", "family": "legacy", "variant": "hdn2", "precision": "fp16", "dtype": "u8",
         "w": 1920, "h": 1080},
        # the same frame through the default model in FP16, as a serving loop runs it
        {"name": "hd_default_fp16", "op": "pass", "family": "acnet8", "variant": "b8_hdn", "precision": "fp16",
         "dtype": "u8", "w": 1920, "h": 1080},
        # the first pass of a 4K float image on its way to 16K
        {"name": "uhd_bf16_f32", "op": "pass", "family": "legacy", "variant": "gan", "precision": "bf16", "dtype": "f32",
         "w": 3840, "h": 2160},
        # the widest network on a 720p frame
        {"name": "artcnn32_720p", "op": "pass", "family": "artcnn", "variant": "f32", "precision": "fp32", "dtype": "u8",
         "w": 1280, "h": 720},
        # a ragged still in 16-bit samples (10-bit video words, PNG)
        {"name": "fsrcnnx8_ragged_u16", "op": "pass", "family": "fsrcnnx", "variant": "f8", "precision": "fp32",
         "dtype": "u16", "w": 1001, "h": 777},
        # a folder of stills of all sizes in one launch
        {"name": "batch24_fp16", "op": "batch", "precision": "fp16", "dtype": "u8", "n": 24, "lo": 128, "hi": 1024, "mix": 5},
        # an RGB frame that stays on the device: split, pass, chroma resize and merge
        {"name": "rgb_720p_fp16", "op": "rgb", "variant": "hdn3", "precision": "fp16", "dtype": "u8", "w": 1280, "h": 720},
        # the drop-in call on an RGB image in ordinary host memory
        {"name": "process_rgb_host", "op": "process", "model": "acnet-hdn", "type": "hip", "dtype": "u8", "w": 800, "h": 600},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng):
    """A width and a height, whole video formats now and then, else any, odd ones included."""
    if rng.random() < 0.25:
        return rng.choice([(256, 256), (640, 360), (640, 480), (720, 576), (1024, 768), (1280, 720), (1440, 1080),
                           (1920, 1080), (2560, 1440), (3840, 2160)])
    w = _log(rng, 64, 3840)
    return w, max(48, min(2160, int(round(w * rng.uniform(0.45, 1.4)))))


_FAMILIES = (
    # family, variants, precisions, weight in the draw
    ("legacy", hip.VARIANTS, ("fp32", "fp16", "bf16"), 5),
    ("acnet8", ("b4_hdn", "b8", "b8_hdn", "b18_box"), ("fp32", "fp16", "bf16"), 5),
    ("artcnn", hip.VARIANTS_ART, ("fp32",), 2),
    ("fsrcnnx", hip.VARIANTS_FSR, ("fp32",), 2),
)


def draw(rng):
    most = max(work(c)["flops"] for c in listed())
    while True:
        kind = rng.random()
        dtype = rng.choice(["u8"] * 6 + ["u16", "f16", "f32", "f32"])
        if kind < 0.72:
            family, variants, precisions, _ = rng.choices(_FAMILIES, [f[3] for f in _FAMILIES])[0]
            w, h = _size(rng)
            c = {"op": "pass", "family": family, "variant": rng.choice(variants), "precision": rng.choice(precisions),
                 "dtype": dtype, "w": w, "h": h}
        elif kind < 0.84:
            lo = _log(rng, 32, 256)
            c = {"op": "batch", "precision": rng.choice(["fp32", "fp16", "bf16"]), "dtype": dtype,
                 "n": _log(rng, 3, 48), "lo": lo, "hi": _log(rng, 2 * lo, 1600), "mix": rng.randrange(1 << 20)}
        elif kind < 0.93:
            w, h = _size(rng)
            c = {"op": "rgb", "variant": rng.choice(hip.VARIANTS), "precision": rng.choice(["fp32", "fp16", "bf16"]),
                 "dtype": "u8", "w": w, "h": h}
        else:
            w, h = _size(rng)
            c = {"op": "process", "model": rng.choice(["acnet-hdn", "acnet-legacy-hdn1", "fsrcnnx-f8"]),
                 "type": "hip", "dtype": "u8", "w": min(w, 1600), "h": min(h, 1200)}
        if work(c)["flops"] <= most:
            return c


# ---- inputs ----

def _to_type(x, dtype):
    if dtype == "f32":
        return x.contiguous()
    if dtype == "f16":
        return x.half().contiguous()
    top = 255.0 if dtype == "u8" else 65535.0
    v = (x * top).round()
    return v.to(torch.uint8) if dtype == "u8" else v.to(torch.int32).to(torch.uint16)


def _picture(w, h, seed, dtype, channels=1):
    """Drawn content: flat shaded areas with hard outlines, a soft gradient and a little grain, in [0, 1]."""
    g = torch.Generator(device=DEVICE).manual_seed(int(seed))

    def field(cells):
        a = torch.rand((1, 1, max(2, h // cells + 2), max(2, w // cells + 2)), generator=g, device=DEVICE)
        return F.interpolate(a, size=(h, w), mode="bilinear", align_corners=False)[0, 0]

    planes = []
    shade = torch.floor(field(48) * 7) / 7
    lines = (field(24) - 0.5).abs() < 0.02
    for _ in range(channels):
        x = 0.65 * shade + 0.25 * field(160) + 0.1 * torch.floor(field(12) * 3) / 3
        x = torch.where(lines, x * 0.15, x)
        x = x + (torch.rand((h, w), generator=g, device=DEVICE) - 0.5) * 0.02
        planes.append(x.clamp(0.0, 1.0))
    x = planes[0] if channels == 1 else torch.stack(planes, dim=-1)
    return _to_type(x, dtype)


def _batch_sizes(case):
    r = random.Random(case["mix"])
    return [(_log(r, case["lo"], case["hi"]), _log(r, case["lo"], case["hi"])) for _ in range(case["n"])]


def _net(case):
    family = case.get("family", "legacy")
    if family == "legacy":
        return hip.Net(case.get("variant", "hdn0"))
    if family == "acnet8":
        return hip.Net8(case["variant"])
    if family == "artcnn":
        return hip.NetArt(case["variant"])
    return hip.NetFsr(case["variant"])


def prepare(case, seed):
    op, t = case["op"], DTYPES[case["dtype"]]
    s = {"case": case}
    if op == "process":
        s["src"] = _picture(case["w"], case["h"], seed, "u8", 3).cpu().numpy()
        s["proc"] = processor.Processor(case["type"], 0, case["model"])
        if not s["proc"].ok():
            raise RuntimeError(s["proc"].error())
        return s
    s["net"] = _net(case)
    if op == "batch":
        sizes = _batch_sizes(case)
        s["src"] = [_picture(w, h, seed * 131 + i, case["dtype"]) for i, (w, h) in enumerate(sizes)]
        s["dst"] = [torch.empty((2 * h, 2 * w), dtype=t, device=DEVICE) for w, h in sizes]
        if case["precision"] == "fp32":
            s["ws"] = torch.empty(s["net"].batch_layers_bytes(s["src"]), dtype=torch.uint8, device=DEVICE)
        return s
    w, h = case["w"], case["h"]
    s["dst"] = torch.empty((2 * h, 2 * w), dtype=t, device=DEVICE)
    if op == "rgb":
        s["src"] = _picture(w, h, seed, "u8", 3)
        s["y"] = torch.empty((h, w), dtype=t, device=DEVICE)
        s["uv"] = torch.empty((h, w, 2), dtype=t, device=DEVICE)
        s["rgb"] = torch.empty((2 * h, 2 * w, 3), dtype=t, device=DEVICE)
    else:
        s["src"] = _picture(w, h, seed, case["dtype"])
    if case.get("family", "legacy") == "legacy":
        need = s["net"].workspace_bytes(w, h, precision=case["precision"], src_dtype=t)
        s["ws"] = torch.empty(max(need, 256), dtype=torch.uint8, device=DEVICE)
    return s


def run(s):
    c = s["case"]
    op = c["op"]
    if op == "process":
        rc, out = s["proc"].process(s["src"], 2.0)
        if rc != 0:
            raise RuntimeError(s["proc"].error())
        return out
    net = s["net"]
    if op == "batch":
        if c["precision"] == "fp32":
            return net.upscale_batch_layers(s["src"], s["dst"], workspace=s["ws"])
        return net.upscale_batch(s["src"], s["dst"], precision=c["precision"])
    if op == "rgb":
        hip.rgb2yuv(s["src"], s["y"], s["uv"])
        net.upscale(s["y"], s["dst"], precision=c["precision"], workspace=s["ws"])
        return hip.resize_yuv2rgb(s["dst"], s["uv"], mode=processor.RESIZE_CATMULL_ROM, out=s["rgb"])
    if c["family"] == "legacy":
        return net.upscale(s["src"], s["dst"], precision=c["precision"], workspace=s["ws"])
    if c["family"] == "acnet8":
        return net.upscale(s["src"], s["dst"], precision=c["precision"])
    return net.upscale(s["src"], s["dst"])


# ---- what a pass cannot do without ----

def _flops_per_pixel(case):
    family, v = case.get("family", "legacy"), case.get("variant", "")
    if case["op"] == "process":
        family = {"acnet-hdn": "acnet8", "acnet-legacy-hdn1": "legacy", "fsrcnnx-f8": "fsrcnnx"}[case["model"]]
        v = {"acnet8": "b8_hdn", "legacy": "hdn1", "fsrcnnx": "f8"}[family]
    if family == "legacy":
        macs = 9 * 8 + 72 * 8 * 8 + 8 * 4
    elif family == "acnet8":
        macs = 9 * 8 + 72 * 8 * int(v[1:].split("_")[0]) + 72 * 4
    else:
        f = int(v[1:].split("_")[0])
        macs = 9 * f + 9 * f * f * 5 + 36 * f if family == "artcnn" else 25 * f + 9 * f * f * 4 + f * f + 36 * f
    return 2 * macs


def work(case):
    op, e = case["op"], BYTES[case["dtype"]]
    if op == "batch":
        px = sum(w * h for w, h in _batch_sizes(case))
    else:
        px = case["w"] * case["h"]
    channels = 3 if op in ("rgb", "process") else 1
    # the luma network, and for colour images the split (about 15 operations a pixel) and the
    # chroma resize and merge (about 40 an output pixel)
    flops = px * _flops_per_pixel(case) + (px * (15 + 4 * 40) if channels == 3 else 0)
    return {"bytes": float(px * 5 * e * channels), "flops": float(flops)}


# ---- the networks in 64 bits ----

def _weights(case):
    family, v = case.get("family", "legacy"), case.get("variant", "hdn0")
    stem = {"legacy": "acnet_legacy", "acnet8": "acnet8", "artcnn": "artcnn", "fsrcnnx": "fsrcnnx"}[family] + "_" + v
    got = []
    for kind in ("kernels", "biases", "alphas"):
        p = os.path.join(WEIGHTS, "%s.%s.f32" % (stem, kind))
        got.append(torch.from_numpy(np.fromfile(p, dtype="<f4").astype(np.float64)).to(DEVICE) if os.path.exists(p) else None)
    return got


def _conv64(x, k, b, n, taps):
    """n x H x W from c x H x W: edge-replicated conv in 64 bits; k as [n][tap][c]."""
    c, h, w = x.shape
    r = {1: 0, 9: 1, 25: 2}[taps]
    side = 2 * r + 1
    k = k.reshape(n, taps, c)
    p = F.pad(x[None], (r, r, r, r), mode="replicate")[0]
    out = torch.empty((n, h, w), dtype=torch.float64, device=x.device)
    band = max(1, (1 << 21) // w)   # rows at a time: bounds the memory of the products
    for y in range(0, h, band):
        e = min(h, y + band)
        acc = b.reshape(n, 1).expand(n, (e - y) * w).clone()
        for t in range(taps):
            dy, dx = t // side, t % side
            acc += k[:, t].contiguous() @ p[:, y + dy:e + dy, dx:dx + w].reshape(c, -1)
        out[:, y:e] = acc.reshape(n, e - y, w)
    return out


def _net64(case, x):
    """2H x 2W from H x W in 64 bits: the case's network with its stored weights."""
    family, v = case.get("family", "legacy"), case.get("variant", "hdn0")
    k, b, a = _weights(case)
    pos = {"k": 0, "b": 0, "a": 0}

    def take(name, n):
        src = {"k": k, "b": b, "a": a}[name]
        pos[name] += n
        return src[pos[name] - n:pos[name]]

    def conv(t, n, taps=9):
        return _conv64(t, take("k", n * taps * t.shape[0]), take("b", n), n, taps)

    def prelu(t, n):
        s = take("a", n).reshape(n, 1, 1)
        return t.clamp(min=0) + s * t.clamp(max=0)

    def shuffle(t):
        return F.pixel_shuffle(t[None], 2)[0, 0]

    t = x[None]
    if family == "legacy":
        t = conv(t, 8).clamp(min=0)
        for _ in range(8):
            t = conv(t, 8).clamp(min=0)
        return shuffle((take("k", 32).reshape(4, 8) @ t.reshape(8, -1)).reshape(4, *x.shape))
    if family == "acnet8":
        t = prelu(conv(t, 8), 8)
        for _ in range(int(v[1:].split("_")[0])):
            t = prelu(conv(t, 8), 8)
        return shuffle(conv(t, 4)) + F.interpolate(x[None, None], scale_factor=2, mode="nearest")[0, 0]
    f = int(v[1:].split("_")[0])
    if family == "artcnn":
        feat = t = conv(t, f)
        for _ in range(4):
            t = conv(t, f).clamp(min=0)
        return shuffle(conv(conv(t, f) + feat, 4))
    feat = t = conv(t, f, 25)
    for _ in range(4):
        t = prelu(conv(t, f), f)
    t = prelu(conv(t, f, 1) + feat, f)
    return shuffle(conv(t, 4))


def exact(case, seed):
    """The floating outputs in 64 bits; whole-number outputs have no such value."""
    if case["dtype"] not in ("f32", "f16") or case["op"] not in ("pass", "batch"):
        return None
    if work(case)["flops"] > 1.0e11:
        return None
    if case["op"] == "pass":
        return _net64(case, _picture(case["w"], case["h"], seed, case["dtype"]).double()).clamp(0.0, 1.0)
    return [_net64(case, _picture(w, h, seed * 131 + i, case["dtype"]).double()).clamp(0.0, 1.0)
            for i, (w, h) in enumerate(_batch_sizes(case))]
