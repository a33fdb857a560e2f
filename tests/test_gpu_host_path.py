"""GPU: frames from host memory and files to ordinary memory.  Planes of every
upload form (one short of and past the size that helper threads share, one and
several staging chunks, ragged last rows, pitched, page-locked) give the file
of the device-memory encode; files of one, two and more staging chunks, to
ordinary and page-locked memory, synchronous and asynchronous, are whole; two
threads with an encoder each do not meet."""

from __future__ import annotations

import ctypes as C
import threading

import numpy as np
import pytest

import cujpegxl_amd as cj
from cujpegxl_amd.synth import synthetic_nv12

pytestmark = pytest.mark.gpu


def host_encode(enc, base, w, h, pitch, out_ptr, capacity):
    inp = cj.Nv12HostInput(base, base + pitch * h, pitch, pitch)
    out = cj.Output(out_ptr, 0, capacity)
    assert enc.lib.cujpegxl_encoder_encode_host(enc.handle, C.byref(inp), C.byref(out)) == cj.OK
    return out.size


# 0.1 MB; 1,047,552 and 1,049,088 bytes around 1 MiB; 3.1 MB; 12.4 MB at a
# low and a high rate (files from one staging chunk to several).
CASES = [(320, 240, 1.0, 0), (1024, 682 // 8 * 8, 1.0, 0), (1032, 680, 1.0, 24), (1920, 1080, 1.0, 0),
         (1368, 776, 0.5, 168), (3840, 2160, 6.0, 0), (3840, 2160, 0.3, 64)]


@pytest.mark.parametrize("w,h,d,pad", CASES)
def test_host_frames_match_device_frames(w, h, d, pad):
    print(f"[gpu] host frame {w}x{h}, d {d}, pad {pad}", flush=True)
    enc = cj.Encoder(w, h, d)
    pitch = w + pad
    for seed in (1, 2):
        luma, chroma = synthetic_nv12(w, h, 700 + seed)
        rows = np.full((h * 3 // 2, pitch), 99, np.uint8)
        rows[:h, :w], rows[h:, :w] = luma, chroma.reshape(h // 2, w)
        dev = cj.DeviceBuffer.from_array(rows)
        want = enc.encode_device(dev.ptr, dev.ptr + pitch * h, pitch, pitch)
        pinned_in, pinned_out = cj.PinnedBuffer(rows.nbytes), cj.PinnedBuffer(enc.capacity + 8)
        C.memmove(pinned_in.ptr, rows.ctypes.data, rows.nbytes)
        ordinary = np.zeros(enc.capacity, np.uint8)
        for base in (rows.ctypes.data, pinned_in.ptr):
            ordinary[:] = 0
            n = host_encode(enc, base, w, h, pitch, ordinary.ctypes.data, ordinary.size)
            assert ordinary[:n].tobytes() == want
            # An unaligned page-locked output takes a copy.
            for at in (0, 1):
                n = host_encode(enc, base, w, h, pitch, pinned_out.ptr + at, enc.capacity)
                assert C.string_at(pinned_out.ptr + at, n) == want
        assert enc.encode_async(dev.ptr, dev.ptr + pitch * h, pitch, pitch) == cj.OK
        assert enc.finish() == want
        for b in (dev, pinned_in, pinned_out):
            b.close()
    enc.close()


def test_two_threads():
    print("[gpu] host frames from two threads", flush=True)
    jobs = []
    for seed, (w, h) in enumerate([(1920, 1080), (2560, 1440)]):
        luma, chroma = synthetic_nv12(w, h, 720 + seed)
        nv12 = np.concatenate([luma.ravel(), chroma.ravel()])
        enc = cj.Encoder(w, h, 1.0)
        jobs.append((enc, nv12, enc.encode_host(nv12), []))

    def work(enc, nv12, want, bad):
        for _ in range(20):
            if enc.encode_host(nv12) != want:
                bad.append(1)

    threads = [threading.Thread(target=work, args=j) for j in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for enc, _, _, bad in jobs:
        assert not bad
        enc.close()
