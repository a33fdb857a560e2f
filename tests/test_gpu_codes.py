"""GPU: prefix codes of histograms at the edges of the one-wave builder
against the oracle: 2 to 256 symbols around the widths of a wave and of its
merge queues, equal counts, counts that need higher and higher floors to fit
15 bits, and ties between leaves and inner nodes at every size."""

from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import cujpegxl_amd as cj

pytestmark = pytest.mark.gpu


def oracle_code(jo, h):
    d = np.zeros(h.size, np.uint8)
    b = np.zeros(h.size, np.uint16)
    out = np.zeros(4096, np.uint8)
    nb = C.c_size_t(0)
    jo.lib().jo_huffman(jo.ptr(h), h.size, jo.ptr(d), jo.ptr(b), jo.ptr(out), out.size, C.byref(nb))
    return d, b, out, nb.value


def histograms(n):
    rng = np.random.default_rng(n)
    fib = [1, 1]
    while len(fib) < min(n, 30):
        fib.append(fib[-1] + fib[-2])
    yield np.ones(n, np.uint32)
    yield np.resize(np.array(fib, np.uint32), n)
    yield np.resize(np.array(fib, np.uint32), n)[::-1].copy()
    yield (2 ** rng.integers(0, 24, n)).astype(np.uint32)
    yield rng.integers(1, 4, n).astype(np.uint32)
    yield np.maximum(1, (1e6 * 0.8 ** np.arange(n))).astype(np.uint32)
    sparse = np.zeros(256, np.uint32)
    sparse[np.sort(rng.permutation(256)[:n])] = rng.integers(1, 1000, n)
    yield sparse


@pytest.mark.parametrize("n", [2, 3, 4, 5, 15, 16, 17, 31, 33, 60, 61, 62, 63, 64, 65, 127, 128, 129, 255, 256])
def test_codes_at_queue_widths(jo, n):
    print(f"[gpu] prefix codes of {n} symbols", flush=True)
    cases = list(histograms(n))
    padded = np.zeros((len(cases), 256), np.uint32)
    for i, h in enumerate(cases):
        padded[i, :h.size] = h
    got = cj.build_codes(padded)
    for g, h in zip(got, padded):
        size = int(np.flatnonzero(h)[-1]) + 1
        d, b, out, nb = oracle_code(jo, np.ascontiguousarray(h[:size]))
        assert np.array_equal(np.asarray(g["depth"])[:size], d)
        assert np.array_equal(np.asarray(g["bits"])[:size][d > 0], b[d > 0])
        assert g["header_bits"] == nb and g["header"] == out[:(nb + 7) // 8].tobytes()
