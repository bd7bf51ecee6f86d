"""Performance cases of the detector: what a program that uses it has it do, call by call.

Every case goes through the public entry points (`FaceDetector.Detect`, `DetectDevice`,
`DetectBatch` and `skipnet.train`) over frames of the sizes that cameras, videos and photo
collections have, from the smallest call, where latency and launches count, to the deepest
pyramid. Frames are drawn on the GPU from a seed: smoothed noise at three octaves, a
Poisson number of face-like patches and a little noise per channel, as
`compactcnncascade_amd.synth` draws its frames on the CPU.

A case is a dict of plain values:

    call        "detect"  one host frame through Detect
                "device"  one frame in GPU memory through DetectDevice
                "batch"   `frames` host frames of each of `sizes` through DetectBatch
                "batch_device"  the same with the frames in GPU memory
                "train"   `epochs` epochs of the tile-skipping network on `frames` frames
    sizes       "WxH" or several, separated by commas
    channels    1 (gray), 3 (BGR) or 4 (BGRA)
    min_face, max_face, scale_factor, precision, facial   the detector's parameters
    skip        tile skipping with the shipped network at this operating point ("": off)

Detections have no 64-bit value of their own: which windows pass a threshold, and in which
order windows drop each other, is defined by the evaluation order in single precision.
The trained weights have one (`exact`).
"""
import math
import random

import numpy as np
import torch

from compactcnncascade_amd import api, skipnet

DEVICE = "cuda:0"
ROWS = 256          # detections a frame that are kept (DetectBatch's default capacity)


def _case(name, call, sizes, frames=1, channels=3, min_face=20, max_face=0, scale_factor=1.15, precision=0, facial=False,
          skip="", epochs=0):
    case = {"call": call, "sizes": sizes, "frames": frames, "channels": channels, "min_face": min_face,
            "max_face": max_face, "scale_factor": scale_factor, "precision": precision, "facial": facial, "skip": skip,
            "epochs": epochs}
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # a webcam: one small frame a call, where the launches and the host's part count
        _case("webcam", "detect", "640x480", min_face=40),
        # a camera's full-HD frames as the program gets them, one a call (host memory)
        _case("fhd_frame", "detect", "1920x1080", min_face=40, max_face=240),
        # the same from a hardware decoder, which leaves them in GPU memory
        _case("fhd_device", "device", "1920x1080", min_face=40, max_face=240),
        # a gray surveillance frame of odd size: scaled down in 8 bits before the pyramid
        _case("gray_odd", "detect", "1279x717", channels=1, min_face=61, scale_factor=1.2),
        # a portrait application: faces with their attributes (landmarks network)
        _case("attributes", "detect", "1280x720", min_face=40, facial=True),
        # a photograph searched down to the smallest faces in fine steps: the deepest pyramid
        _case("deep_photo", "detect", "4800x2400", min_face=15, scale_factor=1.05),
        # video analysis: many decoded full-HD frames at a time
        _case("fhd_batch", "batch_device", "1920x1080", frames=64, min_face=40, max_face=240),
        # many small camera streams at a time
        _case("vga_batch", "batch_device", "640x480", frames=64, min_face=40),
        # mixed sources, small faces; exact, and with the reduced-precision networks
        _case("mixed_batch", "batch_device", "640x480,1280x720,1920x1080,3840x2160", frames=4),
        _case("mixed_half", "batch_device", "640x480,1280x720,1920x1080,3840x2160", frames=4, precision=api.FP16_BF16),
        # a photo collection of ragged sizes from host memory, BGRA, with tile skipping
        _case("photos_skip", "batch", "3021x1999,1600x1104,1203x901,2047x1535", frames=2, channels=4, skip="recall"),
        # training the tile-skipping network: forward, backward and update
        _case("train", "train", "1280x720", frames=64, epochs=6),
    ]


def draw(rng):
    """One more case of the same ranges; no larger than the largest listed one."""
    most = max(work(c)["flops"] for c in listed() if c["call"] != "train")
    while True:
        call = rng.choice(["detect", "detect", "device", "batch", "batch_device", "batch_device", "train"])
        if call == "train":
            return _case("", call, "%dx%d" % (rng.randint(320, 1280), rng.randint(240, 720)), frames=rng.randint(8, 64),
                         epochs=rng.randint(2, 6))
        batch = call.startswith("batch")
        sizes = []
        for _ in range(rng.randint(1, 4) if batch else 1):
            w = round(math.exp(rng.uniform(math.log(240), math.log(3840 if batch else 4800))))
            sizes.append((w, max(180, round(w / rng.uniform(1.2, 2.0)))))
        low = min(100, max(16, min(h for _, h in sizes) // 10))     # several faces fit every frame
        skip = "recall" if batch and rng.random() < 0.2 else ""
        case = _case("", call, ",".join("%dx%d" % s for s in sizes),
                     frames=round(math.exp(rng.uniform(0.0, math.log(32)))) if batch else 1,
                     channels=rng.choice([1, 3, 3, 4]), min_face=20 if skip else rng.randint(15, low),
                     max_face=rng.choice([0, 0, 240]), scale_factor=1.15 if skip else round(rng.uniform(1.05, 1.3), 3),
                     precision=rng.choice([api.FP32, api.FP32, api.FP32, api.FP16_BF16, api.FP16_FP8, api.FP32_BF16]),
                     facial=not batch and rng.random() < 0.2, skip=skip)
        if work(case)["flops"] <= most:
            return case


def _sizes(case):
    return [tuple(int(v) for v in s.split("x")) for s in case["sizes"].split(",")]


def _levels(case, w, h):
    """Sizes of the pyramid levels of a w x h frame."""
    s = 27.0 / case["min_face"]
    if case["channels"] == 1 and s < 0.8:
        w, h, s = int(w * s), int(h * s), 1.0      # a gray frame is scaled down first
    low = 27.0 / case["max_face"] if case["max_face"] else 0.0
    out = []
    s = min(3.0, s)
    while s > low and int(w * s) >= 47 and int(h * s) >= 51:
        out.append((int(w * s), int(h * s)))
        s /= case["scale_factor"]
    return out


def work(case):
    """Bytes: every frame read once. Operations: stage 1 over every pyramid level (a
    multiply and an add per weight), and stage 2 on three of a thousand windows."""
    if case["call"] == "train":
        (w, h), n = _sizes(case)[0], case["frames"]
        cells = n * ((w + 7) // 8) * ((h + 7) // 8)
        macs = 9 * (8 + 64 + 8 * skipnet.SLOTS)
        return {"bytes": cells * (4 + skipnet.SLOTS), "flops": 6 * macs * cells * case["epochs"]}
    nbytes, macs = 0, 0
    for w, h in _sizes(case):
        nbytes += case["frames"] * w * h * case["channels"]
        for lw, lh in _levels(case, w, h):
            c1 = (lw - 3) * (lh - 3)
            c2 = ((lw - 3) // 2 - 2) * ((lh - 3) // 2 - 2)
            r = max(0, c2 // 4)
            macs += case["frames"] * (64 * c1 + 72 * c2 + 580 * r + 0.003 * 278496 * r)
    return {"bytes": nbytes, "flops": int(2 * macs)}


# -- frames ----------------------------------------------------------------------------
def _blur(a, sigma):
    r = int(3 * sigma)
    k = torch.exp(-0.5 * (torch.arange(-r, r + 1, dtype=torch.float32) / sigma) ** 2)
    k = (k / k.sum()).tolist()
    for dim in (0, 1):
        a = sum(kv * torch.roll(a, j - r, dim) for j, kv in enumerate(k))
    return a


def _face(rng, size, dev):
    """Gray values and opacity of one face-like patch."""
    half = int(size) // 2 + 2
    t = torch.arange(-half, half + 1, dtype=torch.float32, device=dev)
    ang = math.radians(rng.uniform(-15.0, 15.0))
    u = math.cos(ang) * t[None, :] + math.sin(ang) * t[:, None]
    v = -math.sin(ang) * t[None, :] + math.cos(ang) * t[:, None]
    alpha = ((1.0 - (u / (0.40 * size)) ** 2 - (v / (0.50 * size)) ** 2) * 6.0).clamp(0, 1)
    val = torch.full_like(u, 200.0)
    for ex in (-0.17 * size, 0.17 * size):
        val -= 140.0 * (1.5 - ((u - ex) ** 2 + (v + 0.12 * size) ** 2) / (0.085 * size) ** 2).clamp(0, 1)
    val -= 110.0 * (2.0 * (1.0 - u.abs() / (0.17 * size)).clamp(0, 1)
                    * (1.0 - (v - 0.24 * size).abs() / (0.04 * size + 0.5)).clamp(0, 1)).clamp(0, 1)
    val -= 40.0 * (1.0 - u.abs() / (0.05 * size + 0.5)).clamp(0, 1) * (1.0 - (v - 0.05 * size).abs() / (0.1 * size)).clamp(0, 1)
    return val, alpha


def _frame(seed, w, h, channels, min_face):
    """A uint8 frame [h, w, channels] (or [h, w]) on the GPU, with at least eight faces
    of sizes that the search looks for."""
    rng = random.Random(seed)
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    gray = torch.zeros(h, w, device=DEVICE)
    for factor, sigma, weight in ((2, 1.0, 0.35), (8, 1.5, 0.4), (32, 1.5, 0.25)):
        noise = torch.rand(h // factor + 2, w // factor + 2, generator=gen, device=DEVICE) * 255.0
        up = torch.nn.functional.interpolate(_blur(noise, sigma)[None, None], size=(h, w), mode="bilinear",
                                             align_corners=True)
        gray += weight * up[0, 0]
    gray = (118.0 + (gray - gray.mean()) * (24.0 / (gray.std() + 1e-9))).clamp(0, 255)
    n, p, limit = 8, rng.random(), math.exp(-4.0)        # 8 and a Poisson number more
    while p > limit:
        p *= rng.random()
        n += 1
    for _ in range(n):
        low, high = 1.2 * min_face, 0.6 * min(w, h, 500)
        size = math.exp(rng.uniform(math.log(min(low, high)), math.log(high)))
        val, alpha = _face(rng, size, DEVICE)
        ph, pw = val.shape
        x, y = rng.randint(0, max(0, w - pw)), rng.randint(0, max(0, h - ph))
        part = gray[y:y + ph, x:x + pw]
        val, alpha = val[:part.shape[0], :part.shape[1]], alpha[:part.shape[0], :part.shape[1]]
        part += alpha * ((185.0 + (val - 200.0) * rng.uniform(0.8, 1.4)).clamp(0, 255) - part)
    noise = torch.randn(h, w, channels, generator=gen, device=DEVICE) * 4.0
    shift = (torch.arange(channels, device=DEVICE) - 1.0) * 3.0 if channels > 1 else torch.zeros(1, device=DEVICE)
    frame = (gray[:, :, None] + noise + shift).round().clamp(0, 255).to(torch.uint8)
    return frame[:, :, 0].contiguous() if channels == 1 else frame


def _labels(seed, case):
    """Inputs of the tile-skipping network and its labels: a few face-sized spots a frame,
    each in the scale slot of its size."""
    (w, h), n = _sizes(case)[0], case["frames"]
    h8, w8 = (h + 7) // 8, (w + 7) // 8
    rng = np.random.default_rng(seed)
    xs = rng.normal(0.0, 0.08, (n, h8, w8)).astype(np.float32)
    ys = np.zeros((n, skipnet.SLOTS, h8, w8), np.uint8)
    for f in range(n):
        for _ in range(rng.poisson(10.0)):
            s, v, u = rng.integers(0, skipnet.SLOTS), rng.integers(0, h8), rng.integers(0, w8)
            r = 1 + int(s) // 6
            ys[f, s, max(0, v - 2):v + 3, max(0, u - 2):u + 3] = 1
            xs[f, max(0, v - r):v + r + 1, max(0, u - r):u + r + 1] += np.float32(rng.uniform(0.1, 0.3))
    return xs, ys


# -- what is measured ------------------------------------------------------------------
def prepare(case, seed):
    if case["call"] == "train":
        xs, ys = _labels(seed, case)
        return {"call": "train", "xs": xs, "ys": ys, "params": skipnet.init_params(seed), "epochs": case["epochs"]}
    sizes = _sizes(case)
    frames = [_frame(seed * 1009 + k, *sizes[k % len(sizes)], case["channels"], case["min_face"])
              for k in range(case["frames"] * len(sizes))]
    det = api.FaceDetector()
    param = api.Param(max_image_size=(max(w for w, _ in sizes), max(h for _, h in sizes)),
                      min_face_height=case["min_face"], max_face_height=case["max_face"],
                      scale_factor=case["scale_factor"], facial_analysis=case["facial"])
    if det.Init(param) != 0:
        raise RuntimeError("FaceDetector.Init failed")
    det.set_compute_precision(case["precision"])
    if case["skip"]:
        params, meta = skipnet.load()
        skipnet.apply_operating_point(det, skipnet.to_fp16(params), meta, case["skip"])
    state = {"call": case["call"], "det": det}
    if case["call"] in ("device", "batch_device"):
        torch.cuda.synchronize()
        state["tensors"] = frames
        state["frames"] = [(t.data_ptr(), t.shape[1], t.shape[0], case["channels"], t.shape[1] * case["channels"])
                           for t in frames]
    else:
        state["frames"] = [t.cpu().numpy() for t in frames]
    return state


def _table(found):
    """The detections as the rows of one table a frame, zeros after the last."""
    table = np.zeros((len(found), ROWS), api.FACE_DTYPE)
    for row, (_, faces) in zip(table, found):
        row[:len(faces)] = faces[:ROWS]
    ints = table.view(np.int32).reshape(len(found), ROWS, 8)
    return {"counts": np.array([n for n, _ in found]), "boxes": ints[:, :, :4], "attributes": ints[:, :, 5:],
            "scores": table["score"]}


def run(state):
    call = state["call"]
    if call == "train":
        params, losses = skipnet.train(api, state["xs"], state["ys"], epochs=state["epochs"], batch=len(state["xs"]),
                                       params=state["params"])
        return {"params": params, "losses": losses}
    det = state["det"]
    if call == "detect":
        return _table([det.Detect(state["frames"][0])])
    if call == "device":
        return _table([det.DetectDevice(*state["frames"][0])])
    if call == "batch":
        return _table(det.DetectBatch(images=state["frames"]))
    return _table(det.DetectBatch(device_frames=state["frames"]))


def _conv64(x, w, b):
    """3x3 convolution with zero padding, [n, ci, h, w] by [co, ci, 3, 3]."""
    h, wd = x.shape[2:]
    x = torch.nn.functional.pad(x, (1, 1, 1, 1))
    cols = torch.stack([x[:, :, ky:ky + h, kx:kx + wd] for ky in range(3) for kx in range(3)], 2)
    cols = cols.flatten(1, 2).flatten(2)                      # [n, ci * 9, h * w]
    out = torch.stack([w.flatten(1) @ c for c in cols])
    return out.unflatten(2, (h, wd)) + b[None, :, None, None]


def exact(case, seed):
    """The trained weights and the losses in 64 bits: weighted cross-entropy of the three
    convolutions, averaged over all outputs, and Adam over the whole set as one batch."""
    if case["call"] != "train":
        return None
    xs, ys = _labels(seed, case)
    x = torch.from_numpy(xs).to(DEVICE, torch.float64)[:, None]
    y = torch.from_numpy(ys).to(DEVICE, torch.float64)
    p = torch.from_numpy(skipnet.init_params(seed)).to(DEVICE, torch.float64)
    shapes = [(8, 1, 3, 3), (8,), (8, 8, 3, 3), (8,), (skipnet.SLOTS, 8, 3, 3), (skipnet.SLOTS,)]
    m, v, losses = torch.zeros_like(p), torch.zeros_like(p), []
    for t in range(1, case["epochs"] + 1):
        p = p.detach().requires_grad_(True)
        w1, b1, w2, b2, w3, b3 = (q.reshape(s) for q, s in zip(p.split([math.prod(s) for s in shapes]), shapes))
        total = 0.0
        g = torch.zeros_like(p)
        for k in range(0, len(x), 8):                         # a few frames at a time
            z = _conv64(_conv64(_conv64(x[k:k + 8], w1, b1).relu(), w2, b2).relu(), w3, b3)
            sp = z.clamp(min=0) + torch.log1p(torch.exp(-z.abs()))
            loss = torch.where(y[k:k + 8] > 0, 500.0 * (sp - z), sp).sum() / y.numel()
            g += torch.autograd.grad(loss, p, retain_graph=True)[0]
            total += float(loss.detach())
        with torch.no_grad():
            m = 0.9 * m + 0.1 * g
            v = 0.999 * v + 0.001 * g * g
            p = p - 3e-3 * (m / (1 - 0.9 ** t)) / ((v / (1 - 0.999 ** t)).sqrt() + 1e-8)
        losses.append(total)
    return {"params": p.detach().cpu().numpy(), "losses": np.array(losses)}
