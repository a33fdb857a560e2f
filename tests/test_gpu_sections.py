"""GPU: the section layout at DC group edges.  A frame's DC groups are coded
in chunks of 1,024 items, each at its own bit positions, and joined by the
assembly: sizes whose last groups are one block wide or high (fewer chunks
than the largest group, items of one chunk straddling the header blobs), and
a batch that mixes them.  Files equal the oracle's byte for byte."""

from __future__ import annotations

import numpy as np
import pytest

import cujpegxl_amd as cj
from cujpegxl_amd.synth import synthetic_nv12

pytestmark = pytest.mark.gpu

# Plane addresses and pitches of every alignment (the chroma pairs and the
# luma bytes are read where they lie).
PLANES = [(1, 1, 0, 0), (0, 3, 1, 5), (2, 1, 7, 2), (5, 2, 64, 63)]

SIZES = [(2056, 264, 0.8), (264, 2056, 1.5), (2064, 2056, 1.0), (264, 8, 1.0), (4104, 64, 3.0)]


def device_frame(w, h, seed):
    luma, chroma = synthetic_nv12(w, h, seed)
    dev = cj.DeviceBuffer.from_array(np.concatenate([luma.ravel(), chroma.ravel()]))
    return luma, chroma, dev, (dev.ptr, dev.ptr + w * h, w, w)


@pytest.mark.parametrize("w,h,d", SIZES)
def test_dc_group_edges(jo, w, h, d):
    luma, chroma, dev, planes = device_frame(w, h, 7)
    enc = cj.Encoder(w, h, d)
    want = jo.encode_nv12(luma, chroma, w, h, d)
    for _ in range(2):
        assert enc.encode_device(*planes) == want
    enc.close()
    dev.close()


def test_batch_of_dc_group_edges(jo):
    frames = [device_frame(w, h, 11 + i) for i, (w, h, _) in enumerate(SIZES)]
    b = cj.Batch([(w, h) for w, h, _ in SIZES], [d for _, _, d in SIZES])
    b.set_inputs([f[3] for f in frames])
    want = [jo.encode_nv12(f[0], f[1], w, h, d) for f, (w, h, d) in zip(frames, SIZES)]
    for _ in range(2):
        b.run(1)
        assert b.files() == want
    b.close()
    for f in frames:
        f[2].close()


def test_more_sections_than_layout_threads(jo):
    # 4 x 256 AC groups and 32 DC groups: 1,058 sections, two rounds of the
    # layout's 1,024 threads.
    w, h, d = 776, 65536, 2.0
    luma, chroma = synthetic_nv12(w, 512, 21)
    luma, chroma = np.tile(luma, (128, 1)), np.tile(chroma, (128, 1))
    jo.set_threads(8)
    want = jo.encode_nv12(luma, chroma, w, h, d)
    jo.set_threads(1)
    dev = cj.DeviceBuffer.from_array(np.concatenate([luma.ravel(), chroma.ravel()]))
    enc = cj.Encoder(w, h, d)
    assert enc.encode_device(dev.ptr, dev.ptr + w * h, w, w) == want
    enc.close()
    dev.close()


@pytest.mark.parametrize("luma_at,chroma_at,luma_pad,chroma_pad", PLANES)
def test_unaligned_planes(jo, luma_at, chroma_at, luma_pad, chroma_pad):
    w, h, d = 296, 136, 1.0
    luma, chroma = synthetic_nv12(w, h, 5)
    lp, cp = w + luma_pad, w + chroma_pad
    base = (luma_at + h * lp + 255) & ~255
    buf = np.full(base + chroma_at + (h // 2) * cp, 255, np.uint8)
    for y in range(h):
        buf[luma_at + y * lp : luma_at + y * lp + w] = luma[y]
    for y in range(h // 2):
        buf[base + chroma_at + y * cp : base + chroma_at + y * cp + w] = chroma[y]
    dev = cj.DeviceBuffer.from_array(buf)
    enc = cj.Encoder(w, h, d)
    assert enc.encode_device(dev.ptr + luma_at, dev.ptr + base + chroma_at, lp, cp) == jo.encode_nv12(luma, chroma, w, h, d)
    enc.close()
    dev.close()
