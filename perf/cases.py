"""The work that a user of fbcuda_amd has it do, as cases that can be timed and compared.

Five families, each through the package's public entry points:

  rows      fbfft1D then fbifft1D of a batch of rows
  planes    fbfft2D then fbifft2D of a batch of real windows inside N x N planes
  layer     the convolution layer's passes (conv_fprop / conv_bprop / conv_accgrad)
  tiled     FFTIteratedConvolution on tile descriptors, with or without a workspace
  composed  fbfft2D of images and filters, transposeMM, fbifft2D: the sequence that
            callers of the plane-major primitives run

Everything is fp32 on the current stream; operands, spectra and workspaces are allocated
once, as a program that runs the same layer again and again does.
"""
import math

import torch

import fbcuda_amd as F

PASSES = {"forward": (0,), "train": (0, 1, 2)}


def listed():
    return [
        # one mini-batch of short signals: four thousand rows of 32 points
        {"name": "rows_32", "family": "rows", "n": 32, "batch": 4096},
        # long rows in a batch far beyond the last-level cache (256 MiB of samples)
        {"name": "rows_256", "family": "rows", "n": 256, "batch": 262144},
        # every feature map of 128 images x 128 channels, planes that fill the transform
        {"name": "planes_32", "family": "planes", "n": 32, "batch": 16384, "h": 32, "w": 32,
         "pad": 0, "packed": False},
        # the largest transform, 256 MiB of samples
        {"name": "planes_128", "family": "planes", "n": 128, "batch": 4096, "h": 128, "w": 128,
         "pad": 0, "packed": False},
        # odd-sized feature maps (128 images x 64 channels of 27 x 27) inside a 32-point
        # transform: implicit zero padding on the way in, crop on the way out
        {"name": "planes_27", "family": "planes", "n": 32, "batch": 8192, "h": 27, "w": 27,
         "pad": 0, "packed": False},
        # one image through one layer, transform size left to the library: serving
        {"name": "layer_one_image", "family": "layer", "passes": "forward", "fft": 0, "batch": 1,
         "cin": 64, "cout": 192, "h": 27, "w": 27, "k": 5},
        # a training step of the same layer on a batch of 128
        {"name": "layer_train", "family": "layer", "passes": "train", "fft": 32, "batch": 128,
         "cin": 64, "cout": 192, "h": 27, "w": 27, "k": 5},
        # a training step of a late layer: small maps, many channels, library's transform size
        {"name": "layer_small_maps", "family": "layer", "passes": "train", "fft": 0, "batch": 128,
         "cin": 96, "cout": 256, "h": 13, "w": 13, "k": 3},
        # a training step on images much larger than the transform
        {"name": "layer_large_image", "family": "layer", "passes": "train", "fft": 32,
         "batch": 16, "cin": 32, "cout": 32, "h": 256, "w": 256, "k": 9},
        # a training step whose maps fit one 64-point transform
        {"name": "layer_64", "family": "layer", "passes": "train", "fft": 64, "batch": 32,
         "cin": 32, "cout": 64, "h": 60, "w": 60, "k": 5},
        # the tiled convolution on its own interface, no workspace, all three passes
        {"name": "tiled", "family": "tiled", "passes": "train", "fft": 32, "batch": 16, "cin": 32,
         "cout": 32, "h": 256, "w": 256, "k": 9, "workspace": False},
        # the forward convolution composed from the plane-major primitives
        {"name": "composed", "family": "composed", "fft": 32, "batch": 128, "cin": 64,
         "cout": 192, "h": 27, "w": 27, "k": 5, "packed": False},
    ]


# ---- sizes ----

def _windows(p, n, c):
    """Windows per image of pass p with n-point transforms."""
    h, w, k = c["h"], c["w"], c["k"]
    if h <= n and w <= n:
        return 1
    step = n - k + 1
    sy, sx = (h, w) if p == 1 else (h - k + 1, w - k + 1)
    return -(-sy // step) * -(-sx // step)


def _sizes(c):
    """Transform sizes that case c's convolution may run on."""
    if c["fft"]:
        return (c["fft"],)
    return tuple(n for n in (8, 16, 32) if n >= c["k"])


def _cost(c):
    """About how many seconds a pass takes: what draw() keeps below the largest listed case."""
    w = work(c)
    if c["family"] in ("rows", "planes", "composed"):
        return w["bytes"] / 4e12 + w["flops"] / 5e13
    t = 0.0
    for p in PASSES[c["passes"]]:
        n = max(_sizes(c))
        images = _windows(p, n, c) * c["batch"]
        pairs = images * c["cin"] * c["cout"]
        if c["family"] == "tiled" and not c["workspace"]:
            t += pairs * n * n * 5e-13
        else:
            planes = images * (c["cin"] + c["cout"]) + c["cin"] * c["cout"]
            t += planes * n * n * (8 / 4e12) * (2 if n > 32 else 1) + pairs * n * n * (3 / 1e14)
    return t


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_one(rng):
    family = rng.choice(["rows", "planes", "planes", "layer", "layer", "layer", "layer", "tiled", "composed"])
    if family == "rows":
        n = rng.choice([8, 16, 32, 64, 128, 256])
        return {"family": family, "n": n, "batch": _log(rng, 512, 2 ** 26 // n)}
    if family == "planes":
        n = rng.choice([8, 16, 32, 64, 128])
        c = {"family": family, "n": n, "batch": _log(rng, 16, 2 ** 26 // (n * n)), "h": n, "w": n,
             "pad": 0, "packed": n <= 32 and rng.random() < 0.25}
        if rng.random() < 0.5:
            c["h"], c["w"] = rng.randint(n // 2, n), rng.randint(n // 2, n)
            c["pad"] = rng.randint(0, min(2, n - c["h"], n - c["w"]))
        return c
    k = rng.randint(1, 11)
    c = {"family": family, "fft": 0, "batch": _log(rng, 1, 256), "cin": _log(rng, 3, 384),
         "cout": _log(rng, 8, 384), "h": 0, "w": 0, "k": k}
    if family == "layer":
        c["passes"] = rng.choice(["forward", "train"])
        c["fft"] = rng.choice([0, 0, 0, 32, 16, 64, 128])
        most = c["fft"] if c["fft"] > 32 else 256
    elif family == "tiled":
        c["passes"] = rng.choice(["forward", "train"])
        c["workspace"] = rng.random() < 0.5
        c["fft"] = rng.choice([16, 32])
        c["cin"], c["cout"] = _log(rng, 3, 96), _log(rng, 8, 96)
        most = 256
    else:
        c["fft"] = rng.choice([16, 32, 32])
        c["packed"] = rng.random() < 0.25
        most = c["fft"]
    least = max(7, k, 2 if c["fft"] <= 32 else c["fft"] // 2)
    c["h"] = _log(rng, least, most)
    c["w"] = min(most, max(least, c["h"] + rng.choice([0, 0, 0, -3, 1, 8])))
    return c


def draw(rng):
    limit = max(_cost(c) for c in listed())
    while True:
        c = _draw_one(rng)
        if 0 < c.get("fft", 0) < c.get("k", 0):
            continue
        if _cost(c) <= limit:
            return c


# ---- state ----

def _normal(gen, shape, std=1.0):
    t = torch.empty(shape, dtype=torch.float32, device="cuda")
    return t.normal_(0.0, std, generator=gen)


def _empty(*shape):
    return torch.zeros(shape, dtype=torch.float32, device="cuda")


def prepare(case, seed):
    c, gen = case, torch.Generator(device="cuda")
    gen.manual_seed(seed)
    if c["family"] == "rows":
        b, n = c["batch"], c["n"]
        return {"case": c, "x": _normal(gen, (b, n)), "spec": _empty(b, n // 2 + 1, 2),
                "back": _empty(b, n)}
    if c["family"] == "planes":
        b, n = c["batch"], c["n"]
        rows = n // 2 if c["packed"] else n // 2 + 1
        return {"case": c, "x": _normal(gen, (b, c["h"], c["w"])), "spec": _empty(b, rows, n, 2),
                "back": _empty(b, c["h"], c["w"])}
    b, cin, cout, h, w, k, n = (c[x] for x in ("batch", "cin", "cout", "h", "w", "k", "fft"))
    oh, ow = h - k + 1, w - k + 1
    # activations, filters at the usual initialisation scale, gradients that have shrunk
    s = {"case": c, "x": _normal(gen, (b, cin, h, w)),
         "weight": _normal(gen, (cout, cin, k, k), 1.0 / math.sqrt(cin * k * k)),
         "out": _empty(b, cout, oh, ow)}
    if c["family"] == "composed":
        rows = n // 2 if c["packed"] else n // 2 + 1
        s.update(xs=_empty(b, cin, rows, n, 2), ws=_empty(cout, cin, rows, n, 2),
                 os=_empty(b, cout, rows, n, 2))
        return s
    passes = PASSES[c["passes"]]
    if len(passes) > 1:
        s.update(grad=_normal(gen, (b, cout, oh, ow), 1e-2), gin=_empty(b, cin, h, w),
                 gw=_empty(cout, cin, k, k))
    size = 0
    if c["family"] == "layer":
        size = max(F.conv_workspace_image(p, b, cin, cout, h, w, k, k, n) for p in passes)
    else:
        s["tiles"] = [F.make_tile_grid(s["gin"] if p == 1 else s["x"],
                                       s["out"] if p == 0 else s["grad"], k, k, n, p)
                      for p in passes]
        if len(passes) > 1:
            # the weight-gradient pass writes through the weight operand
            s["filters"] = (s["weight"], s["weight"], s["gw"])
        else:
            s["filters"] = (s["weight"],)
        if c["workspace"]:
            size = max(F.iterated_conv_workspace(n, p, b, t[2], cin, cout)
                       for p, t in zip(passes, s["tiles"]))
    if size:
        s["space"] = torch.empty(size, dtype=torch.uint8, device="cuda")
    return s


# ---- one pass ----

def _done(code):
    if code != F.Success:
        raise RuntimeError(F.error_string(code))


def run(state):
    s, c = state, state["case"]
    family = c["family"]
    if family == "rows":
        _done(F.fbfft1D(s["x"], s["spec"]))
        _done(F.fbifft1D(s["back"], s["spec"]))
        return s["spec"], s["back"]
    if family == "planes":
        _done(F.fbfft2D(s["x"], s["spec"], c["pad"], c["pad"]))
        _done(F.fbifft2D(s["spec"], s["back"], c["pad"], c["pad"]))
        return s["spec"], s["back"]
    if family == "composed":
        b, cin, cout = c["batch"], c["cin"], c["cout"]
        x, w, o = s["x"], s["weight"], s["out"]
        _done(F.fbfft2D(x.flatten(0, 1), s["xs"].flatten(0, 1)))
        _done(F.fbfft2D(w.flatten(0, 1), s["ws"].flatten(0, 1)))
        _done(F.transposeMM(s["xs"], s["ws"], s["os"], 1.0 / c["fft"] ** 2,
                            conjugateTransposeB=True, packed=c["packed"]))
        _done(F.fbifft2D(s["os"].flatten(0, 1), o.flatten(0, 1)))
        return s["xs"], s["ws"], s["os"], o
    n = c["fft"]
    if family == "layer":
        _done(F.conv_fprop(s["x"], s["weight"], s["out"], n, s["space"]))
        if c["passes"] == "forward":
            return s["out"]
        _done(F.conv_bprop(s["grad"], s["weight"], s["gin"], n, s["space"]))
        _done(F.conv_accgrad(s["x"], s["grad"], s["gw"], n, s["space"]))
        return s["out"], s["gin"], s["gw"]
    for p, (ins, outs, count), weight in zip(PASSES[c["passes"]], s["tiles"], s["filters"]):
        if c["workspace"]:
            ok = F.FFTIteratedConvolutionWS(n, ins, outs, weight, p, 1.0, c["batch"], count, s["space"])
        else:
            ok = F.FFTIteratedConvolution(n, ins, outs, weight, p, 1.0, c["batch"], count)
        if not ok:
            raise RuntimeError("the tiled convolution was not launched")
    if c["passes"] == "forward":
        return s["out"]
    return s["out"], s["gin"], s["gw"]


# ---- what a pass cannot do without, and how far correct results may lie apart ----

def work(case):
    c = case
    if c["family"] == "rows":
        n, b = c["n"], c["batch"]
        return {"bytes": 2 * b * (4 * n + 8 * (n // 2 + 1)), "flops": 2 * b * 2.5 * n * math.log2(n)}
    if c["family"] == "planes":
        n, b = c["n"], c["batch"]
        rows = n // 2 if c["packed"] else n // 2 + 1
        return {"bytes": 2 * b * (4 * c["h"] * c["w"] + 8 * n * rows),
                "flops": 2 * b * 2.5 * n * n * 2 * math.log2(n)}
    b, cin, cout, h, w, k = (c[x] for x in ("batch", "cin", "cout", "h", "w", "k"))
    real = b * cin * h * w + cout * cin * k * k + b * cout * (h - k + 1) * (w - k + 1)

    def spectral(p, n):
        # 8 operations per complex multiply-add on n * n / 2 bins, and each plane's transform
        images = _windows(p, n, c) * b
        planes = images * (cin + cout) + cin * cout
        return 4 * n * n * images * cin * cout + planes * 2.5 * n * n * 2 * math.log2(n)

    if c["family"] == "composed":
        n = c["fft"]
        rows = n // 2 if c["packed"] else n // 2 + 1
        spectra = (b * cin + cout * cin + b * cout) * 8 * n * rows
        # every entry point reads its inputs once and writes its output once
        return {"bytes": 4 * real + 2 * spectra, "flops": spectral(0, n)}
    passes = PASSES[c["passes"]]
    return {"bytes": 4 * real * len(passes),
            "flops": sum(min(spectral(p, n) for n in _sizes(c)) for p in passes)}


def tolerance(case):
    # four times the largest distance seen between a result and the same path in 64 bits
    # over the listed and two dozen drawn cases: transforms 2.0e-7; convolutions 6.0e-7
    # (a weight gradient over 1936 windows, others 2e-7 to 4e-7), single values 2.4e-6
    if case["family"] in ("rows", "planes"):
        return {"rel": 8e-7}
    return {"rel": 2.4e-6, "max": 1e-5}
