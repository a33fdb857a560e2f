"""GPU: every stream, event and memory block that an encoder creates may be
refused.  A configure that meets a refusal, whichever it is, leaves an encoder
that refuses to encode until a configure succeeds; a refused input frame (made
by the first encode from host memory) or feature buffer fails that one call."""

from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import cujpegxl_amd as cj
from cujpegxl_amd.synth import synthetic_nv12

pytestmark = pytest.mark.gpu
W, H = 520, 264


@pytest.fixture()
def refuse():
    L = cj.stages_lib()
    yield L.cjx_stage_fail_allocation_after
    L.cjx_stage_fail_allocation_after(0)


def frame(seed):
    luma, chroma = synthetic_nv12(W, H, seed)
    return np.concatenate([luma.ravel(), chroma.ravel()])


def test_every_refusal_of_a_configure(refuse):
    L = cj.stages_lib()
    dev = cj.DeviceBuffer.from_array(frame(11))
    enc = cj.Encoder(W, H, 1.0, stages=True)
    args = (dev.ptr, dev.ptr + W * H, W, W)
    want = enc.encode_device(*args)
    own, other = cj.Config(W, H, 1.0, 0), cj.Config(328, 264, 1.0, 0)
    refused = 0
    for n in range(1, 64):
        print(f"[gpu] configure with creation {n} refused", flush=True)
        assert L.cujpegxl_encoder_configure(enc.handle, C.byref(other)) == cj.OK
        refuse(n)
        status = L.cujpegxl_encoder_configure(enc.handle, C.byref(own))
        refuse(0)
        if status == cj.OK:
            break
        assert status == cj.INTERNAL_ERROR
        refused += 1
        assert enc.encode_status(*args, enc.capacity)[0] == cj.INTERNAL_ERROR
    # The last creation of a configure is the device memory: of what comes
    # before it, the five events of a frame's order at least.
    assert 6 <= refused < 62
    assert enc.encode_device(*args) == want
    enc.close()
    dev.close()


def test_refused_input_frame(refuse):
    print("[gpu] first host encode without memory for the input frame", flush=True)
    enc = cj.Encoder(W, H, 1.0, stages=True)
    nv12 = frame(12)
    inp = cj.Nv12HostInput(nv12.ctypes.data, nv12.ctypes.data + W * H, W, W)
    out = cj.Output(enc.out.ctypes.data, 0, enc.capacity)
    refuse(1)
    assert enc.lib.cujpegxl_encoder_encode_host(enc.handle, C.byref(inp), C.byref(out)) == cj.INTERNAL_ERROR
    dev = cj.DeviceBuffer.from_array(nv12)
    want = enc.encode_device(dev.ptr, dev.ptr + W * H, W, W)
    for _ in range(2):
        assert enc.encode_host(nv12) == want
    enc.close()
    dev.close()


def test_refused_feature_buffer(refuse):
    print("[gpu] feature export without memory", flush=True)
    enc = cj.Encoder(W, H, 1.0, stages=True)
    dev = cj.DeviceBuffer.from_array(frame(13))
    want = enc.encode_device(dev.ptr, dev.ptr + W * H, W, W)
    refuse(1)
    with pytest.raises(RuntimeError):
        enc.export_features(True)
    assert enc.encode_device(dev.ptr, dev.ptr + W * H, W, W) == want
    enc.export_features(True)
    assert enc.encode_device(dev.ptr, dev.ptr + W * H, W, W) == want
    enc.close()
    dev.close()
