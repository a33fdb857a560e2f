"""GPU: AC tokens of items at the edges of the tokenizer's steps of 64 scan
positions, against the oracle's codestream: items of every transform size
whose last non-zero coefficient is the first or last of a chunk of 32 or a
step of 64, one before or after it, or the item's own first or last; items
without non-zeros and with all of them; alone in their wave's pair or beside
an item of another size."""

from __future__ import annotations

import numpy as np
import pytest

import cujpegxl_amd as cj

pytestmark = pytest.mark.gpu

ORDER_AT = {8: 0, 16: 64, 32: 320}


def scan_orders():
    L = cj.stages_lib()
    orders = np.zeros(64 + 256 + 1024, np.uint16)
    assert L.cjx_host_table(2, orders.ctypes.data, orders.nbytes) == orders.nbytes
    return {n: orders[at:at + n * n].astype(np.int64) for n, at in ORDER_AT.items()}


def ends(n):
    """Last non-zero positions worth a visit, in scan order."""
    first = (n // 8) ** 2
    near = [first + s + d for s in range(0, n * n, 32) for d in (-1, 0, 1)]
    return [-1] + sorted({p for p in near + [n * n - 2, n * n - 1] if first <= p < n * n})


@pytest.mark.parametrize("w,h,density", [(264, 296, 0.0), (264, 296, 0.3), (1032, 520, 1.0), (512, 512, 0.05)])
def test_last_coefficients_around_steps(jo, w, h, density):
    print(f"[gpu] tokens around step edges, {w}x{h}, density {density}", flush=True)
    orders = scan_orders()
    rng = np.random.default_rng(w + int(100 * density))
    bw, bh = w // 8, h // 8
    acs = np.full((bh, bw), 8, np.int8)
    ac = np.zeros((3, bh, bw, 64), np.int16)
    turn = {8: 0, 16: 0, 32: 0}
    for y in range(0, bh, 4):
        for x in range(0, bw, 4):
            n = int(rng.choice([8, 16, 32])) if x + 4 <= bw and y + 4 <= bh else 8
            m = n // 8
            for by in range(y, min(y + 4, bh), m):
                for bx in range(x, min(x + 4, bw), m):
                    acs[by:by + m, bx:bx + m] = 0
                    acs[by, bx] = n
                    for c in range(3):
                        choice = ends(n)
                        last = choice[turn[n] % len(choice)]
                        turn[n] += 1
                        if last < 0:
                            continue
                        raw = np.zeros(n * n, np.int16)
                        at = orders[n][m * m:last + 1]
                        keep = rng.random(at.size) < density
                        keep[-1] = True
                        size = rng.choice([1, 1, 1, 2, 15, 16, 300, 20000], at.size)
                        raw[at[keep]] = (size * rng.choice([-1, 1], at.size))[keep]
                        ac[c, by:by + m, bx:bx + m] = raw.reshape(m, m, 64)
    nblk = bw * bh
    dc = rng.integers(-50, 50, size=3 * nblk).astype(np.int32)
    qf = rng.integers(1, 64, size=nblk).astype(np.int32)
    enc = cj.Encoder(w, h, 1.0, any_size=True)
    data = enc.encode_coefficients(ac.ravel(), dc, acs.ravel(), qf, None, None, 2048, 300)
    enc.close()
    cs = jo.write_codestream(jo.make_frame(w, h, 2048, 300, dc, ac.ravel(), acs.ravel(), qf, None, None))
    assert data[40:] == cs or data[48:] == cs
