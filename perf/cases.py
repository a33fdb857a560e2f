"""Performance cases: what a user of cujpegxl_amd has it do.

NV12 frames in device memory become `.jxl` files through a kept encoder, one
at a time (from the smallest frame the encoder takes to 8K, in the plain and
the learned + matrix-core form), from host memory, asynchronously with two
encoders, in batches; and the selection network's training pass.  Frames are
seeded noise, gratings and rectangles over chroma gradients, the same family
as cujpegxl_amd/synth.py, made on the GPU.
"""

from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import cujpegxl_amd as cj
from cujpegxl_amd import train_mlp

MODE_BOTH = cj.MODE_MFMA16 | cj.MODE_LEARNED
KINDS = ("frame", "frame", "frame", "host", "oneshot", "async", "noalloc", "batch", "batch", "train", "evaluate")
BATCH_SIZES = ((640, 360), (1280, 720), (1920, 1080), (2560, 1440), (3840, 2160))  # the bench's mixed batch
MAX_BATCH_PIXELS = 8 * 3840 * 2160
MAX_FRAME_PIXELS = 7680 * 4320
MAX_NOALLOC_PIXELS = 1920 * 1088
LR, LAMBDA, STEP = 2e-3, 0.1, 100


def listed():
    def frame(name, w, h, d, mode=0, pad=0):
        return {"name": name, "kind": "frame", "width": w, "height": h, "distance": d, "mode": mode, "pad": pad}

    mixed = "1920x1080:1.0 640x360:2.4 3840x2160:1.3 1280x720:0.9 2560x1440:1.8 1920x1080:2.9 640x360:1.1 1280x720:2.0 " \
            "3840x2160:2.2 640x360:0.8 1920x1080:1.5 2560x1440:1.0 1280x720:2.7 640x360:1.6 1920x1080:0.9 2560x1440:2.5"
    return [
        # A thumbnail: two AC groups, launches and latency only.
        frame("frame 320x240", 320, 240, 1.0),
        # A video-call or preview frame at a lower quality.
        frame("frame 1280x720 d2", 1280, 720, 2.0),
        # The common video frame.
        frame("frame 1920x1080", 1920, 1080, 1.0),
        # A cropped window in a larger surface: no dimension a multiple of 16 or of the
        # 32 and 64 pixel tiles, rows with a pitch.
        frame("frame 1368x776 pitched", 1368, 776, 1.5, MODE_BOTH, 168),
        # The headline workload, plain and in its fastest form.
        frame("frame 3840x2160", 3840, 2160, 1.0),
        frame("frame 3840x2160 learned", 3840, 2160, 1.0, MODE_BOTH),
        # The largest ordinary frame.
        frame("frame 7680x4320", 7680, 4320, 1.0),
        # A frame that a Python program holds in host memory, bytes back.
        {"name": "host 1920x1080", "kind": "host", "width": 1920, "height": 1080, "distance": 1.0, "mode": 0},
        # A capture loop that keeps two frames in flight.
        {"name": "async 2560x1440", "kind": "async", "width": 2560, "height": 1440, "distance": 0.8, "mode": 0},
        # Offline throughput: eight 4K frames, and a mixed batch of a server's requests.
        {"name": "batch 8x 3840x2160 learned", "kind": "batch", "frames": " ".join(["3840x2160:1.0"] * 8), "mode": MODE_BOTH},
        {"name": "batch 16 mixed", "kind": "batch", "frames": mixed, "mode": 0},
        # A training step of the selection network at the trainer's batch size.
        {"name": "train 4096", "kind": "train", "rows": 4096},
    ]


def _size(rng, pixels_max, side_max=7680):
    """A frame size, its pixels spread over their logarithm; sides multiples of 8."""
    while True:
        px = math.exp(rng.uniform(math.log(320 * 240), math.log(pixels_max)))
        aspect = rng.uniform(0.7, 2.2)
        w = 8 * round(math.sqrt(px * aspect) / 8)
        h = 8 * round(math.sqrt(px / aspect) / 8)
        if (w > 256 or h > 256) and 64 <= min(w, h) and max(w, h) <= side_max and w * h <= pixels_max:
            return w, h


def draw(rng):
    kind = rng.choice(KINDS)
    if kind in ("train", "evaluate"):
        return {"kind": kind, "rows": int(math.exp(rng.uniform(math.log(500), math.log(70000))))}
    distance = round(math.exp(rng.uniform(math.log(0.6), math.log(3.0))), 2)
    mode = rng.choice((0, 0, cj.MODE_MFMA16, cj.MODE_LEARNED, MODE_BOTH))
    if kind == "batch":
        frames, pixels = [], 0
        for _ in range(rng.randint(2, 16)):
            w, h = rng.choice(BATCH_SIZES) if rng.random() < 0.5 else _size(rng, 3840 * 2160, 4096)
            if pixels + w * h > MAX_BATCH_PIXELS:
                break
            pixels += w * h
            frames.append(f"{w}x{h}:{round(rng.uniform(0.8, 3.0), 2)}")
        return {"kind": kind, "frames": " ".join(frames), "mode": mode}
    if kind == "noalloc":
        w, h = _size(rng, MAX_NOALLOC_PIXELS, 4096)
        return {"kind": kind, "width": w, "height": h, "distance": distance, "mode": 0}
    if kind == "oneshot":
        w, h = _size(rng, 3840 * 2160)
        return {"kind": kind, "width": w, "height": h, "distance": distance, "mode": 0}
    w, h = _size(rng, MAX_FRAME_PIXELS if kind == "frame" else 3840 * 2160)
    case = {"kind": kind, "width": w, "height": h, "distance": distance, "mode": mode}
    if kind == "frame":
        case["pad"] = rng.choice((0, 0, 8 * rng.randint(1, 40)))
    return case


def _nv12(width, height, gen, pad=0):
    """Device NV12 as one (3/2 height, width + pad) byte tensor: luma rows, then
    interleaved chroma rows."""
    dev = "cuda"
    u = torch.rand(64, generator=gen, device=dev).tolist()
    yy = torch.arange(height, device=dev, dtype=torch.float32)[:, None]
    xx = torch.arange(width, device=dev, dtype=torch.float32)[None, :]
    y = torch.full((height, width), 128.0, device=dev)
    for k in range(3):
        theta, period = math.pi * u[4 * k], 16.0 + 112.0 * u[4 * k + 1]
        amp, phase = 12.0 + 16.0 * u[4 * k + 2], 2.0 * math.pi * u[4 * k + 3]
        y += amp * torch.sin((xx * math.cos(theta) + yy * math.sin(theta)) * (2.0 * math.pi / period) + phase)
    for k in range(8):
        a, b, c, d, level = u[12 + 5 * k : 17 + 5 * k]
        rw, rh = max(1, int(width * (0.03 + 0.22 * a))), max(1, int(height * (0.03 + 0.22 * b)))
        x0, y0 = int(c * (width - rw)), int(d * (height - rh))
        sub = y[y0 : y0 + rh, x0 : x0 + rw]
        sub.copy_(16.0 + 219.0 * level + 0.5 * (sub - 128.0))
    sigma = 2.0 + 4.0 * u[52]
    y += sigma * torch.randn(height, width, generator=gen, device=dev)
    out = torch.zeros(height * 3 // 2, width + pad, dtype=torch.uint8, device=dev)
    out[:height, :width] = y.round_().clamp_(16, 235).to(torch.uint8)
    ch, cw = height // 2, width // 2
    cy = torch.arange(ch, device=dev, dtype=torch.float32)[:, None] - ch / 2
    cx = torch.arange(cw, device=dev, dtype=torch.float32)[None, :] - cw / 2
    for k in range(2):
        a = 2.0 * math.pi * u[53 + k]
        p = 128.0 + (cx * math.cos(a) + cy * math.sin(a)) * (40.0 / (0.5 * math.hypot(cw, ch)))
        out[height:, k:width:2] = p.round().clamp_(88, 168).to(torch.uint8)
    return out


def _planes(nv12, height):
    """(luma, chroma, luma pitch, chroma pitch) of an _nv12 tensor."""
    pitch = nv12.stride(0)
    return nv12.data_ptr(), nv12.data_ptr() + pitch * height, pitch, pitch


class _File:
    """A batch's file buffer as an array that keeps the batch."""

    def __init__(self, owner, address, size):
        self.owner = owner
        self.__array_interface__ = {"version": 3, "shape": (size,), "typestr": "|u1", "data": (address, False)}


def _capacity(width, height):
    """Bytes of a file buffer of this frame size: twice the largest file of these frames."""
    return width * height * 3 // 4 + (1 << 16)


def _result(batch, i):
    """Where a batch keeps file i, and the file's size."""
    p, n = C.c_void_p(), C.c_uint64()
    if batch.lib.cjx_batch_result(batch.handle, i, C.byref(p), C.byref(n)) != cj.OK:
        raise RuntimeError("batch result failed")
    return p.value, n.value


def _parse(frames):
    out = []
    for f in frames.split():
        size, d = f.split(":")
        w, h = size.split("x")
        out.append((int(w), int(h), float(d)))
    return out


def _rows(case, gen):
    """Standardized features and labels of `rows` regions, parameters and Adam
    moments in the middle of a run."""
    n, dev = case["rows"], "cuda"
    x = torch.randn(n, train_mlp.IN, generator=gen, device=dev)
    lab = torch.zeros(n, train_mlp.LAB, device=dev)
    lab[:, :5] = (torch.rand(n, 5, generator=gen, device=dev) < 0.4).float()
    lab[:, 5] = 2.0 + 0.5 * torch.randn(n, generator=gen, device=dev)
    lab[:, 6:11] = (torch.rand(n, 5, generator=gen, device=dev) < 0.95).float()
    hid, inp, out = train_mlp.HID, train_mlp.IN, train_mlp.OUT
    p = torch.randn(train_mlp.PARAMS, generator=gen, device=dev)
    p[: hid * inp] *= math.sqrt(2.0 / inp)
    p[hid * inp : hid * inp + hid] *= 0.1
    p[hid * inp + hid :] *= math.sqrt(1.0 / hid)
    m = 1e-2 * torch.randn(train_mlp.PARAMS, generator=gen, device=dev)
    v = 1e-3 * (0.5 + torch.rand(train_mlp.PARAMS, generator=gen, device=dev))
    return x, lab, p, m, v


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind = case["kind"]
    if kind in ("train", "evaluate"):
        x, lab, p, m, v = _rows(case, gen)
        n = case["rows"]
        s = {"kind": kind, "n": n, "x": x, "lab": lab, "params": p, "m": m, "v": v}
        if kind == "train":
            s["grad"] = torch.zeros_like(p)
            s["loss"] = torch.zeros(1, device="cuda")
            s["partial"] = torch.empty(cj.stages_lib().cjx_mlp_partial_floats(n), device="cuda")
        else:
            s["z"] = torch.zeros(n, train_mlp.OUT, device="cuda")
        return s
    if kind == "batch":
        frames = _parse(case["frames"])
        nv12 = [_nv12(w, h, gen) for w, h, _ in frames]
        batch = cj.Batch([(w, h) for w, h, _ in frames], [d for _, _, d in frames], mode=case["mode"])
        batch.set_inputs([_planes(t, h) for t, (_, h, _) in zip(nv12, frames)])
        files = []
        for i, (fw, fh, _) in enumerate(frames):
            address = _result(batch, i)[0]
            C.memset(address, 0, _capacity(fw, fh))
            files.append(np.asarray(_File(batch, address, _capacity(fw, fh))))
        return {"kind": kind, "nv12": nv12, "batch": batch, "files": files}
    w, h, d = case["width"], case["height"], case["distance"]
    s = {"kind": kind, "width": w, "height": h, "distance": d}
    if kind == "noalloc":
        s["nv12"] = _nv12(w, h, gen)
        s["out"] = torch.zeros(_capacity(w, h), dtype=torch.uint8, device="cuda")
        s["size"] = torch.zeros(1, dtype=torch.int64, device="cuda")
        return s
    if kind in ("host", "oneshot"):
        s["nv12"] = _nv12(w, h, gen).reshape(-1).cpu().numpy()
    elif kind == "async":
        s["nv12"] = [_nv12(w, h, gen) for _ in range(2)]
    else:
        s["nv12"] = _nv12(w, h, gen, case["pad"])
    if kind != "oneshot":
        s["encoders"] = [cj.Encoder(w, h, d) for _ in range(2 if kind == "async" else 1)]
        for e in s["encoders"]:
            e.set_mode(case["mode"])
    # The caller's file buffers: page-locked for the synchronous encodes, ordinary memory elsewhere.
    if kind == "frame":
        s["out"] = torch.zeros(_capacity(w, h), dtype=torch.uint8, pin_memory=True)
    else:
        s["out"] = [np.zeros(_capacity(w, h), np.uint8) for _ in range(2 if kind == "async" else 1)]
    return s


def run(state):
    kind = state["kind"]
    if kind == "frame":
        out = state["out"]
        n = state["encoders"][0].encode_into(*_planes(state["nv12"], state["height"]), out.data_ptr(), out.numel())
        return out, n
    if kind == "host":
        e, base, w, out = state["encoders"][0], state["nv12"].ctypes.data, state["width"], state["out"][0]
        inp = cj.Nv12HostInput(base, base + w * state["height"], w, w)
        file = cj.Output(out.ctypes.data, 0, out.size)
        if e.lib.cujpegxl_encoder_encode_host(e.handle, C.byref(inp), C.byref(file)) != cj.OK:
            raise RuntimeError("encode_host failed")
        return out, file.size
    if kind == "oneshot":
        data = cj.encode(state["nv12"], state["width"], state["height"], state["distance"])
        state["out"][0][: len(data)] = np.frombuffer(data, np.uint8)
        return state["out"][0], len(data)
    if kind == "async":
        stream = torch.cuda.current_stream().cuda_stream
        for e, t in zip(state["encoders"], state["nv12"]):
            if e.encode_async(*_planes(t, state["height"]), stream) != cj.OK:
                raise RuntimeError("encode_async failed")
        sizes = []
        for e, out in zip(state["encoders"], state["out"]):
            file = cj.Output(out.ctypes.data, 0, out.size)
            if e.lib.cujpegxl_encoder_finish(e.handle, C.byref(file)) != cj.OK:
                raise RuntimeError("finish failed")
            sizes.append(file.size)
        return state["out"], sizes
    if kind == "batch":
        state["batch"].run(1)
        return state["files"], [_result(state["batch"], i)[1] for i in range(len(state["files"]))]
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "noalloc":
        w, h = state["width"], state["height"]
        cfg = cj.Config(w, h, state["distance"], 0)
        inp = cj.Nv12Input(*_planes(state["nv12"], h))
        out, size = state["out"], state["size"]
        if cj.public_lib().cujpegxl_encode_noalloc(C.byref(cfg), C.byref(inp), out.data_ptr(), out.numel(),
                                                   size.data_ptr(), stream) != cj.OK:
            raise RuntimeError("encode_noalloc failed")
        return out, size
    lib = cj.stages_lib()
    if kind == "train":
        t = state
        if lib.cjx_mlp_step(t["x"].data_ptr(), t["lab"].data_ptr(), t["n"], LAMBDA, t["partial"].data_ptr(),
                            t["grad"].data_ptr(), t["loss"].data_ptr(), t["params"].data_ptr(), t["m"].data_ptr(),
                            t["v"].data_ptr(), STEP, LR, stream) != cj.OK:
            raise RuntimeError("mlp step failed")
        return {k: t[k] for k in ("grad", "loss", "params", "m", "v")}
    if lib.cjx_mlp_forward(state["params"].data_ptr(), state["x"].data_ptr(), state["n"], state["z"].data_ptr(),
                           stream) != cj.OK:
        raise RuntimeError("mlp forward failed")
    return state["z"]


def work(case):
    """Bytes: the NV12 read once and the file written once (about 1.7 bits a
    pixel at distance 1, fewer above).  Operations: 4 N a pixel and channel of
    an N x N transform, the three sizes tried on Y and one taken on X and B."""
    hid, inp, out = train_mlp.HID, train_mlp.IN, train_mlp.OUT
    if case["kind"] in ("train", "evaluate"):
        n, p = case["rows"], train_mlp.PARAMS
        if case["kind"] == "train":
            return {"bytes": 4 * (n * (inp + train_mlp.LAB) + 8 * p), "flops": n * (2 * 2 * hid * inp + 3 * 2 * hid * out)}
        return {"bytes": 4 * (n * (inp + out) + p), "flops": n * 2 * (hid * inp + hid * out)}
    if case["kind"] == "batch":
        frames = _parse(case["frames"])
    else:
        frames = [(case["width"], case["height"], case["distance"])] * (2 if case["kind"] == "async" else 1)
    total = {"bytes": 0.0, "flops": 0.0}
    for w, h, d in frames:
        total["bytes"] += w * h * (1.5 + 0.21 / d)
        total["flops"] += w * h * 4 * (8 + 16 + 32 + 2 * 16)
    return total


def exact(case, seed):
    """The network's passes in 64 bits; files are bytes and have no such value."""
    if case["kind"] not in ("train", "evaluate"):
        return None
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    x, lab, p, m, v = (t.double() for t in _rows(case, gen))
    hid, inp, out, n = train_mlp.HID, train_mlp.IN, train_mlp.OUT, case["rows"]
    w1, b1 = p[: hid * inp].view(hid, inp), p[hid * inp : hid * inp + hid]
    w2, b2 = p[hid * inp + hid : -out].view(out, hid), p[-out:]
    h = (x @ w1.T + b1).clamp_min(0.0)
    z = h @ w2.T + b2
    if case["kind"] == "evaluate":
        return z
    lam = float(np.float32(LAMBDA))
    root = lab[:, 0] > 0.5
    lse = torch.logsumexp(z[:, :2], 1)
    loss = lab[:, 6] * (lse - torch.where(root, z[:, 1], z[:, 0]))
    loss = loss + (lab[:, 7:11] * (torch.nn.functional.softplus(z[:, 2:6], threshold=700.0) - lab[:, 1:5] * z[:, 2:6])).sum(1)
    loss = loss + lam * (z[:, 6] - lab[:, 5]) ** 2
    dz = torch.zeros_like(z)
    p1 = torch.exp(z[:, 1] - lse)
    dz[:, 0] = lab[:, 6] * ((1.0 - p1) - (~root).double())
    dz[:, 1] = lab[:, 6] * (p1 - root.double())
    dz[:, 2:6] = lab[:, 7:11] * (torch.sigmoid(z[:, 2:6]) - lab[:, 1:5])
    dz[:, 6] = 2.0 * lam * (z[:, 6] - lab[:, 5])
    dh = (dz @ w2) * (h > 0.0)
    grad = torch.cat([(dh.T @ x).reshape(-1), dh.sum(0), (dz.T @ h).reshape(-1), dz.sum(0)]) / n
    beta1, beta2, lr = (float(np.float32(t)) for t in (0.9, 0.999, LR))
    m1 = beta1 * m + (1.0 - beta1) * grad
    v1 = beta2 * v + (1.0 - beta2) * grad * grad
    step = lr * (m1 / (1.0 - beta1**STEP)) / ((v1 / (1.0 - beta2**STEP)).sqrt() + 1e-8)
    return {"grad": grad, "loss": loss.mean().reshape(1), "params": p - step, "m": m1, "v": v1}
