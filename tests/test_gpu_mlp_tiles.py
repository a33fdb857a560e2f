"""GPU: the selection network's training and evaluation kernels at the edges
of their tiles: one row, one short of and past a tile of 32, more tiles than
the 512 workgroups of a launch, and inputs at addresses of any float.

Inputs and parameters are small multiples of 1/8, so the hidden units and the
outputs are exact in FP32 in any order of summation: the outputs must equal
the float64 ones.  The gradient's error has two sources: the loss gradient at
an output (a few roundings of values up to 1: below 2^-20 of the mask, or of
the residual for the seventh), and sums of at most 33 + 512 FP32 terms; both
stay below 2^-14 of the sum of the terms' largest magnitudes.
"""

from __future__ import annotations

import numpy as np
import pytest

import cujpegxl_amd as cj

pytestmark = pytest.mark.gpu

IN, HID, OUT, LAB = 96, 64, 7, 12
LAMBDA = 0.25
B1, W2, B2, PARAMS = 6144, 6208, 6656, 6663


def batch(n):
    rng = np.random.default_rng(n)
    eighths = lambda lo, hi, *shape: (rng.integers(lo, hi + 1, shape) / 8.0).astype(np.float32)
    p = np.concatenate([eighths(-2, 2, B1), eighths(-8, 8, HID), eighths(-1, 1, OUT * HID), eighths(-8, 8, OUT)])
    x = eighths(-4, 4, n, IN)
    lab = np.zeros((n, LAB), np.float32)
    lab[:, 0:5] = rng.integers(0, 2, (n, 5))
    lab[:, 5] = eighths(-16, 16, n)
    lab[:, 6:11] = rng.integers(0, 2, (n, 5))
    return p, x, lab


def forward(p, x):
    p, x = p.astype(np.float64), x.astype(np.float64)
    h = np.maximum(x @ p[:B1].reshape(HID, IN).T + p[B1:W2], 0.0)
    return h, h @ p[W2:B2].reshape(OUT, HID).T + p[B2:]


def loss_grad(p, x, lab):
    """Mean loss, gradient, and the gradient of the terms' magnitudes."""
    h, z = forward(p, x)
    lab = lab.astype(np.float64)
    n = x.shape[0]
    root = lab[:, 6]
    e = np.exp(z[:, :2] - z[:, :2].max(axis=1, keepdims=True))
    soft = e / e.sum(axis=1, keepdims=True)
    hot = np.stack([1.0 - lab[:, 0], lab[:, 0]], axis=1)
    loss = -root * np.log((soft * hot).sum(axis=1))
    mask, y, v = lab[:, 7:11], lab[:, 1:5], z[:, 2:6]
    loss = loss + (mask * (np.logaddexp(0.0, v) - y * v)).sum(axis=1) + LAMBDA * (z[:, 6] - lab[:, 5]) ** 2
    dz = np.concatenate([root[:, None] * (soft - hot), mask * (1.0 / (1.0 + np.exp(-v)) - y),
                         2.0 * LAMBDA * (z[:, 6:] - lab[:, 5:6])], axis=1)
    most = np.concatenate([np.repeat(root[:, None], 2, axis=1), mask, np.abs(dz[:, 6:])], axis=1)
    w2 = p[W2:B2].reshape(OUT, HID).astype(np.float64)

    def grads(dz, w2, h, x):
        dh = (dz @ w2) * (h > 0)
        return np.concatenate([(dh.T @ x).ravel(), dh.sum(axis=0), (dz.T @ h).ravel(), dz.sum(axis=0)]) / n

    return loss.mean(), grads(dz, w2, h, x.astype(np.float64)), grads(most, np.abs(w2), h, np.abs(x.astype(np.float64)))


def shifted(a, floats):
    """A device copy of `a` that starts `floats` floats into its buffer."""
    b = cj.DeviceBuffer.from_array(np.concatenate([np.zeros(floats, np.float32), a.ravel()]))
    return b, b.ptr + 4 * floats


@pytest.mark.parametrize("n,offset", [(1, 0), (31, 1), (32, 2), (33, 3), (1000, 1), (512 * 32 + 33, 1)])
def test_training_pass_at_tile_edges(n, offset):
    p, x, lab = batch(n)
    L = cj.stages_lib()
    print(f"[gpu] network kernels, {n} rows, {offset} floats in", flush=True)
    (bp, dp), (bx, dx), (bl, dl) = shifted(p, offset), shifted(x, offset), shifted(lab, offset)
    zeros = np.zeros(PARAMS, np.float32)
    g, m, v = (cj.DeviceBuffer.from_array(zeros) for _ in range(3))
    loss, part = cj.DeviceBuffer(4), cj.DeviceBuffer(4 * L.cjx_mlp_partial_floats(n))
    guard = np.full(n * OUT + 64, 7.5, np.float32)
    dz = cj.DeviceBuffer.from_array(guard)
    try:
        assert L.cjx_mlp_forward(dp, dx, n, dz.ptr, 0) == cj.OK
        assert L.cjx_mlp_step(dx, dl, n, LAMBDA, part.ptr, g.ptr, loss.ptr, dp, m.ptr, v.ptr, 1, 0.0, 0) == cj.OK
        L.cjx_device_synchronize()
        z, grad = dz.to_host(np.float32), g.to_host(np.float32).astype(np.float64)
        got = float(loss.to_host(np.float32)[0])
    finally:
        for b in (bp, bx, bl, g, m, v, loss, part, dz):
            b.close()
    assert np.array_equal(z[:n * OUT].reshape(n, OUT), forward(p, x)[1])
    assert np.array_equal(z[n * OUT:], guard[n * OUT:])
    want_loss, want, most = loss_grad(p, x, lab)
    assert abs(got - want_loss) <= 2.0 ** -14 * max(want_loss, 1.0)
    assert (np.abs(grad - want) <= 2.0 ** -14 * most + 2.0 ** -40).all()
