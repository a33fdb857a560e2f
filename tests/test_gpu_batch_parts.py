"""GPU: batches large enough to be replayed as parallel branches (80,000
blocks a branch, at most three) give the files of the single-frame encoder:
two and three branches, a frame larger than a branch, a last branch of small
frames, one workgroup per region and a persistent region grid, one tokenizer
workgroup per frame, over several replays."""

from __future__ import annotations

import numpy as np
import pytest

import cujpegxl_amd as cj
from cujpegxl_amd.synth import synthetic_nv12

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [
    [(3840, 2160), (1920, 1080), (640, 360)],
    [(3840, 2160), (1920, 1080), (3840, 2160), (640, 360), (2560, 1440), (320, 240)],
    [(264, 520), (7680, 4320)],
])
@pytest.mark.parametrize("mode", [0, cj.MODE_LEARNED | cj.MODE_MFMA16])
def test_branches_match_single_frames(sizes, mode):
    print(f"[gpu] branches of a batch: {sizes}, mode {mode}", flush=True)
    devs, inputs, want = [], [], []
    dists = [0.9 + 0.4 * i for i in range(len(sizes))]
    for i, ((w, h), d) in enumerate(zip(sizes, dists)):
        luma, chroma = synthetic_nv12(w, h, 300 + i)
        devs.append(cj.DeviceBuffer.from_array(np.concatenate([luma.ravel(), chroma.ravel()])))
        inputs.append((devs[-1].ptr, devs[-1].ptr + w * h, w, w))
        enc = cj.Encoder(w, h, d, stages=True)
        enc.set_mode(mode)
        want.append(enc.encode_device(*inputs[-1]))
        enc.close()
    b = cj.Batch(sizes, dists, mode=mode)
    b.set_inputs(inputs)
    for _ in range(3):
        b.run(2)
        assert b.files() == want
    for shape in ((1, 64, 1536), (1024, 4, 8)):
        b.set_shape(*shape)
        b.run(2)
        assert b.files() == want, shape
    b.close()
    for d in devs:
        d.close()
