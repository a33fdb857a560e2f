"""GPU: the batch autotuner times each set of launches once.  A frame's share of
the tokenizer's 4,096 workgroups and the runs of its file bound the grids of
the candidate shapes, so several shapes stand for the same launches; between
those a choice would be by noise, so they carry one time and the first of them
stands for all.  (The files do not depend on the choice.)"""

from __future__ import annotations

import re

import numpy as np
import pytest

import cujpegxl_amd as cj
from cujpegxl_amd.synth import synthetic_nv12

pytestmark = pytest.mark.gpu


def up(a, b):
    return -(-a // b)


def launches(sizes, token_cap, assemble_words):
    """Grids of the two stages that a shape changes, frame by frame."""
    blocks = [w * h // 64 for w, h in sizes]
    out = []
    for (w, h), nb in zip(sizes, blocks):
        bw, bh = w // 8, h // 8
        ac, dc = up(bw, 32) * up(bh, 32), up(bw, 256) * up(bh, 256)
        gw, gh = min(bw, 256), min(bh, 256)  # the largest DC group
        chunks = up(2 + 6 * gw * gh + 2 * up(gw, 8) * up(gh, 8), 1024)
        words = (3 * nb * 384 + 48 * nb + (ac + dc) * 2048 + 16384 + 3) // 4
        runs = 4 + dc * chunks + ac * 96
        out.append((min(up(3 * nb, 8), token_cap, up(4096 * nb, sum(blocks))),
                    min(up(words, 256 * assemble_words), up(runs, 4))))
    return tuple(out)


@pytest.mark.parametrize("sizes", [[(1280, 720)] * 8, [(640, 360), (1920, 1080), (264, 520)], [(328, 264)] * 40])
def test_each_set_of_launches_is_timed_once(sizes):
    print(f"[gpu] tune of {len(sizes)} frames, {sizes[0]} ..", flush=True)
    b = cj.Batch(sizes, [1.0] * len(sizes))
    devs, inputs = [], []
    for i, (w, h) in enumerate(sizes):
        luma, chroma = synthetic_nv12(w, h, 500 + i)
        devs.append(cj.DeviceBuffer.from_array(np.concatenate([luma.ravel(), chroma.ravel()])))
        inputs.append((devs[-1].ptr, devs[-1].ptr + w * h, w, w))
    b.set_inputs(inputs)
    b.run(1)
    want = b.files()
    *lines, chosen = b.tune(2).strip().splitlines()
    b.run(1)
    assert b.files() == want
    shapes, ms = [], []
    for line in lines + [chosen]:
        *shape, t = re.findall(r"=([\d.]+)", line)
        shapes.append(tuple(map(int, shape)))
        ms.append(t)
    assert shapes[:12] == [(t, a, 0) for t in (256, 512, 1024, 2048) for a in (4, 16, 64)]
    first = {}  # launches -> their first candidate
    for i, (t, a, _) in enumerate(shapes[:12]):
        k = first.setdefault(launches(sizes, t, a), i)
        assert ms[i] == ms[k], (lines[i], lines[k])
    assert len(first) < 12  # the candidates of every one of these batches repeat themselves
    best = min(range(len(lines)), key=lambda i: float(ms[i]))  # the first of the fastest
    assert float(ms[-1]) == float(ms[best])
    at = shapes.index(shapes[-1])
    assert at >= 12 or at in first.values()
    b.close()
    for d in devs:
        d.close()
