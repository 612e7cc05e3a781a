"""The calls whose speed this repository watches: scoring frames and training
losses through the public functions of ``frame_analytics_amd``.

``listed()`` holds the fixed cases, ``draw(rng)`` gives further ones of the same
ranges, ``prepare`` makes what a program has in hand before the call, ``run``
makes one call (or one small group of calls that a program makes together on the
same frames), and ``exact`` gives the same outputs in float64 from plain torch.

A case is a dict: ``op`` says which calls, ``n, c, h, w`` the frames, ``dtype``
their element type, ``reduction`` what the scores are reduced to and ``crop`` the
border cropped before scoring (Y-channel scores only).
"""

from __future__ import annotations

import math

import torch

import frame_analytics_amd as fa

_DTYPES = {"uint8": torch.uint8, "float16": torch.float16, "bfloat16": torch.bfloat16,
           "float32": torch.float32}
_BYTES = {"uint8": 1, "float16": 2, "bfloat16": 2, "float32": 4}
_LOSSES = ("ssim_loss", "ms_ssim_loss", "gms_loss")


def _case(name, op, n, c, h, w, dtype="uint8", reduction="mean", crop=0):
    return {"name": name, "op": op, "n": n, "c": c, "h": h, "w": w, "dtype": dtype,
            "reduction": reduction, "crop": crop}


def listed():
    return [
        # one small grey frame: a thumbnail or a crop scored as it arrives, where
        # the call's own latency counts
        _case("psnr_gray_512", "psnr", 1, 1, 512, 512),
        # one decoded video frame against its source, as a per-frame filter does
        _case("ssim_frame_1080p", "ssim", 1, 3, 1080, 1920),
        # a batch of decoded frames: the repository's headline workload
        _case("ssim_batch_1080p", "ssim", 8, 3, 1080, 1920),
        # the largest frames in a batch, one value per frame batch
        _case("psnr_batch_4k", "psnr", 8, 3, 2160, 3840),
        # the two heavier scores over the same batch of decoded frames
        _case("ms_ssim_batch_1080p", "ms_ssim", 8, 3, 1080, 1920),
        _case("gmsd_batch_1080p", "gmsd", 8, 3, 1080, 1920),
        # super-resolution evaluation: Y-PSNR and Y-SSIM with a cropped border, one
        # image of an odd size at a time
        _case("y_scores_odd_image", "y_scores", 1, 3, 1021, 1357, crop=4),
        # a clip whose width is no multiple of 8, one value per frame
        _case("ragged_clip", "ssim_ms_ssim", 4, 3, 767, 1366, reduction="none"),
        # validation inside mixed-precision training: network output and target in
        # bfloat16, scored as they are
        _case("val_bf16", "psnr_ssim", 8, 3, 512, 768, dtype="bfloat16"),
        # training steps: the loss and its gradient, on patches and on whole frames
        _case("ssim_loss_patches", "ssim_loss", 16, 3, 256, 256, dtype="float32"),
        _case("ms_ssim_loss_1080p", "ms_ssim_loss", 8, 3, 1080, 1920, dtype="float32"),
        _case("gms_loss_540p", "gms_loss", 8, 3, 540, 960, dtype="float32"),
    ]


# op -> (draw weight, element types, smallest side, largest h, largest w, most
# images, fewest and most samples per tensor)
_RANGES = {
    "psnr": (2, ("uint8",), 48, 2160, 3840, 16, 1 << 18, 8 * 3 * 2160 * 3840),
    "ssim": (3, ("uint8", "uint8", "float32"), 48, 2160, 3840, 16, 1 << 18, 8 * 3 * 1080 * 1920),
    "ms_ssim": (2, ("uint8", "uint8", "float32"), 192, 2160, 3840, 16, 1 << 18,
                8 * 3 * 1080 * 1920),
    "gmsd": (2, ("uint8", "uint8", "float32"), 48, 2160, 3840, 16, 1 << 18, 8 * 3 * 1080 * 1920),
    "y_scores": (2, ("uint8",), 96, 2160, 3840, 4, 1 << 18, 4 * 3 * 1080 * 1920),
    "ssim_ms_ssim": (1, ("uint8",), 192, 1080, 1920, 8, 1 << 18, 8 * 3 * 720 * 1280),
    "psnr_ssim": (2, ("bfloat16", "float16", "float32"), 64, 1080, 1920, 16, 1 << 18,
                  8 * 3 * 720 * 1280),
    "ssim_loss": (2, ("float32",), 64, 720, 1280, 32, 1 << 18, 8 * 3 * 720 * 1280),
    "ms_ssim_loss": (2, ("float32",), 192, 1080, 1920, 16, 1 << 19, 8 * 3 * 1080 * 1920),
    "gms_loss": (2, ("float32",), 64, 1080, 1920, 32, 1 << 18, 8 * 3 * 720 * 1280),
}


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any op, sizes spread over the logarithm of its range, with
    odd sides as often as even ones."""
    ops = list(_RANGES)
    op = rng.choices(ops, [_RANGES[o][0] for o in ops])[0]
    _, dtypes, side, hmax, wmax, nmax, least, most = _RANGES[op]
    c = 3 if op == "y_scores" or rng.random() < 0.75 else 1
    while True:
        samples = _log_uniform(rng, least, most)
        aspect = rng.uniform(0.75, 2.0)
        n = _log_uniform(rng, 1, nmax)
        h = int(math.sqrt(samples / (n * c * aspect)))
        w = int(h * aspect)
        if h >= side and w >= side and h <= hmax and w <= wmax:
            break
    if rng.random() < 0.5:  # sizes that encoders and patch cutters make
        h, w = max(side, h // 8 * 8), max(side, w // 8 * 8)
    crop = rng.choice((0, 2, 3, 4)) if op == "y_scores" else 0
    reduction = "mean" if op in _LOSSES else rng.choice(("mean", "mean", "none"))
    case = _case("", op, n, c, h, w, rng.choice(dtypes), reduction, crop)
    del case["name"]
    return case


# --------------------------------------------------------------------------- #
# inputs
# --------------------------------------------------------------------------- #


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _frames(case, seed):
    """A pair of picture-like frames in [0, 1]: smooth shapes, texture and grain,
    and the same frames with a mild blur-free distortion, as coding noise is."""
    dev = _device()
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    n, c, h, w = case["n"], case["c"], case["h"], case["w"]

    def field(step):
        g = torch.rand(n, c, h // step + 2, w // step + 2, device=dev, generator=gen)
        return torch.nn.functional.interpolate(g, size=(h, w), mode="bilinear",
                                               align_corners=False)

    x = 0.55 * field(64) + 0.30 * field(12)
    x += 0.15 * torch.rand(n, c, h, w, device=dev, generator=gen)
    y = x + 0.03 * torch.randn(n, c, h, w, device=dev, generator=gen)
    return x.clamp_(0, 1), y.clamp_(0, 1)


def prepare(case, seed):
    x, y = _frames(case, seed)
    dt = _DTYPES[case["dtype"]]
    if dt == torch.uint8:
        x, y = ((255.0 * t).round_().to(torch.uint8) for t in (x, y))
    else:
        x, y = x.to(dt), y.to(dt)
    if case["op"] in _LOSSES:
        x.requires_grad_(True)
    return {"case": case, "x": x, "y": y}


# --------------------------------------------------------------------------- #
# one pass
# --------------------------------------------------------------------------- #


def _data_range(case):
    return 255.0 if case["dtype"] == "uint8" else 1.0


def run(state):
    case, x, y = state["case"], state["x"], state["y"]
    op, L, red = case["op"], _data_range(case), case["reduction"]
    if op == "psnr":
        return fa.psnr(x, y, data_range=L, reduction=red)
    if op == "ssim":
        return fa.ssim(x, y, data_range=L, reduction=red)
    if op == "ms_ssim":
        return fa.ms_ssim(x, y, data_range=L, reduction=red)
    if op == "gmsd":
        return fa.gmsd(x, y, data_range=L, reduction=red)
    if op == "y_scores":
        kw = dict(data_range=L, reduction=red, luma="matlab", crop_border=case["crop"])
        return fa.psnr(x, y, **kw), fa.ssim(x, y, **kw)
    if op == "ssim_ms_ssim":
        return (fa.ssim(x, y, data_range=L, reduction=red),
                fa.ms_ssim(x, y, data_range=L, reduction=red))
    if op == "psnr_ssim":
        return (fa.psnr(x, y, data_range=L, reduction=red),
                fa.ssim(x, y, data_range=L, reduction=red))
    # a training step's loss: its value and the gradient of the network's output
    x.grad = None
    if op == "ssim_loss":
        loss = 1.0 - fa.ssim(x, y, data_range=L)
    elif op == "ms_ssim_loss":
        loss = 1.0 - fa.ms_ssim(x, y, data_range=L)
    else:
        loss = 1.0 - fa.gms(x, y, data_range=L)
    loss.backward()
    return loss.detach(), x.grad


# --------------------------------------------------------------------------- #
# what a pass cannot do without
# --------------------------------------------------------------------------- #


def work(case):
    """Each input sample read once and each gradient written once; operations per
    output pixel of the textbook separable form: four moments under an 11-tap
    window both ways (176) and the formula (26) for SSIM, three more filtered maps
    (132) and their combination (16) for its gradient, all scales of a pyramid
    4/3 of its first; squares and a sum for PSNR; two 3 x 3 gradients per tensor
    and the similarity for GMSD, at a quarter of the samples."""
    op, c = case["op"], case["c"]
    samples = case["n"] * c * case["h"] * case["w"]
    nbytes = 2 * samples * _BYTES[case["dtype"]] + 8 * case["n"]
    if op in _LOSSES:
        nbytes += samples * 4
    per = {"psnr": 3, "ssim": 202, "ms_ssim": 202 * 4 / 3, "gmsd": 10, "y_scores": (202 + 13) / 3,
           "ssim_ms_ssim": 202 * 7 / 3, "psnr_ssim": 205, "ssim_loss": 350,
           "ms_ssim_loss": 350 * 4 / 3, "gms_loss": 25}[op]
    return {"bytes": int(nbytes), "flops": int(samples * per)}


def tolerance(case):
    """About four times the errors seen against :func:`exact`: exact integer sums
    and a float64 logarithm for PSNR of bytes; float32 moments with float64 sums for
    the SSIM scores (up to 7.5e-8); float32 terms with float64 sums for GMSD of bytes
    (2.5e-9); float32 gradients of float64 arithmetic (7.8e-8 through a pyramid,
    2.5e-8 where only the result is rounded)."""
    rel = {"psnr": 1e-12, "gmsd": 2e-8, "gms_loss": 1e-7}.get(case["op"], 3e-7)
    return {"rel": rel}


# --------------------------------------------------------------------------- #
# the same outputs in float64
# --------------------------------------------------------------------------- #

_WEIGHTS = (0.0448, 0.2856, 0.3001, 0.2363, 0.1333)


def _blur(t):
    d = torch.arange(11, dtype=torch.float64) - 5.0
    g = torch.exp(-d * d / (2.0 * 1.5 * 1.5))
    g = (g / g.sum()).tolist()
    h, w = t.shape[-2:]
    t = sum(g[i] * t[..., i:i + h - 10, :] for i in range(11))
    return sum(g[i] * t[..., i:i + w - 10] for i in range(11))


def _ssim_cs(x, y, L):
    """Per-plane means of SSIM and of its contrast-structure term."""
    C1, C2 = (0.01 * L) ** 2, (0.03 * L) ** 2
    mx, my = _blur(x), _blur(y)
    sxx = _blur(x * x) - mx * mx
    syy = _blur(y * y) - my * my
    sxy = _blur(x * y) - mx * my
    cs = (2 * sxy + C2) / (sxx + syy + C2)
    s = cs * (2 * mx * my + C1) / (mx * mx + my * my + C1)
    return s.mean(dim=(-2, -1)), cs.mean(dim=(-2, -1))


def _halve(t):
    h, w = t.shape[-2] // 2 * 2, t.shape[-1] // 2 * 2
    return 0.25 * (t[..., 0:h:2, 0:w:2] + t[..., 1:h:2, 0:w:2]
                   + t[..., 0:h:2, 1:w:2] + t[..., 1:h:2, 1:w:2])


def _ssim(x, y, L):
    return _ssim_cs(x, y, L)[0].mean()


def _ms_ssim(x, y, L):
    out = 1.0
    for i, e in enumerate(_WEIGHTS):
        if i:
            x, y = _halve(x), _halve(y)
        s, cs = _ssim_cs(x, y, L)
        out = out * (s if i == 4 else cs).clamp_min(0.0) ** e
    return out.mean()


def _gms_map(x, y, L):
    def grad2(t):
        t = _halve(t)
        rows = t[..., :-2, :] + t[..., 1:-1, :] + t[..., 2:, :]
        cols = t[..., :-2] + t[..., 1:-1] + t[..., 2:]
        gx = (rows[..., :-2] - rows[..., 2:]) / 3.0
        gy = (cols[..., :-2, :] - cols[..., 2:, :]) / 3.0
        return gx * gx + gy * gy + (1e-6 * L) ** 2

    a, b, T = grad2(x), grad2(y), 170.0 * (L / 255.0) ** 2
    return (2.0 * (a * b).sqrt() + T) / (a + b + T)


def _mse(x, y):
    d = x - y
    return (d * d).mean()


def _luma(t, L):
    k = (65.481 / 255.0, 128.553 / 255.0, 24.966 / 255.0)
    return k[0] * t[0:1] + k[1] * t[1:2] + k[2] * t[2:3] + 16.0 / 255.0 * L


def exact(case, seed):
    state = prepare(case, seed)
    op, L, n = case["op"], _data_range(case), case["n"]
    xs, ys = state["x"].detach(), state["y"]

    def pairs():  # image by image: float64 planes of whole batches are large
        for i in range(n):
            yield xs[i].double(), ys[i].double()

    def each(f):
        return torch.stack([f(x, y) for x, y in pairs()])

    def reduced(values):
        return values if case["reduction"] == "none" else values.mean()

    def db(mses):  # the batch's dB is that of its mean squared error
        return 10.0 * math.log10(L * L) - 10.0 * torch.log10(reduced(mses))

    if op == "psnr":
        return db(each(_mse))
    if op == "ssim":
        return reduced(each(lambda x, y: _ssim(x, y, L)))
    if op == "ms_ssim":
        return reduced(each(lambda x, y: _ms_ssim(x, y, L)))
    if op == "gmsd":
        return reduced(each(lambda x, y: _gms_map(x, y, L).std(correction=0)))
    if op == "y_scores":
        b = case["crop"]
        crop = lambda t: t[..., b:t.shape[-2] - b, b:t.shape[-1] - b]  # noqa: E731
        cut = lambda t: crop(_luma(t, L))  # noqa: E731
        return (db(each(lambda x, y: _mse(cut(x), cut(y)))),
                reduced(each(lambda x, y: _ssim(cut(x), cut(y), L))))
    if op == "ssim_ms_ssim":
        return (reduced(each(lambda x, y: _ssim(x, y, L))),
                reduced(each(lambda x, y: _ms_ssim(x, y, L))))
    if op == "psnr_ssim":
        return db(each(_mse)), reduced(each(lambda x, y: _ssim(x, y, L)))
    score = {"ssim_loss": _ssim, "ms_ssim_loss": _ms_ssim,
             "gms_loss": lambda x, y, L: _gms_map(x, y, L).mean()}[op]
    total, grads = 0.0, []
    for x, y in pairs():
        x.requires_grad_(True)
        v = score(x, y, L) / n
        grads.append(-torch.autograd.grad(v, x)[0])
        total = total + v.detach()
    return 1.0 - total, torch.stack(grads)
