"""GPU: one encoder that moves between frames whose host copy one thread makes
and frames whose copy is shared with helper threads (from 1 MiB): the nearest
sizes on both sides of the line (1,048,512 and 1,048,608 bytes) and larger and
smaller ones in turn, pitched and not, give the file of the device-memory
encode each time."""

from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import cujpegxl_amd as cj
from cujpegxl_amd.synth import synthetic_nv12

pytestmark = pytest.mark.gpu
SIZES = [(688, 1016), (264, 2648), (688, 1016), (1920, 1080), (320, 240), (264, 2648)]


def test_host_frames_across_the_shared_copy_size():
    assert 688 * 1016 * 3 // 2 == 1048512 < 1 << 20 < 264 * 2648 * 3 // 2 == 1048608
    enc = cj.Encoder(*SIZES[0], 1.0)
    out = np.zeros(1 << 23, np.uint8)
    for k, (w, h) in enumerate(SIZES):
        pitch = w + 8 * (k % 3)
        print(f"[gpu] host frame {w}x{h}, pitch {pitch}", flush=True)
        assert enc.lib.cujpegxl_encoder_configure(enc.handle, C.byref(cj.Config(w, h, 1.0, 0))) == cj.OK
        for seed in (1, 2):
            luma, chroma = synthetic_nv12(w, h, 740 + 2 * k + seed)
            rows = np.full((h * 3 // 2, pitch), 99, np.uint8)
            rows[:h, :w], rows[h:, :w] = luma, chroma.reshape(h // 2, w)
            dev = cj.DeviceBuffer.from_array(rows)
            got = []
            for call, base, kind in ((enc.lib.cujpegxl_encoder_encode, dev.ptr, cj.Nv12Input),
                                     (enc.lib.cujpegxl_encoder_encode_host, rows.ctypes.data, cj.Nv12HostInput)):
                inp, res = kind(base, base + pitch * h, pitch, pitch), cj.Output(out.ctypes.data, 0, out.size)
                assert call(enc.handle, C.byref(inp), C.byref(res)) == cj.OK
                got.append(out[: res.size].tobytes())
            assert got[0] == got[1]
            dev.close()
    enc.close()
