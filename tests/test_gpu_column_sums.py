"""Column sums at the edges of their kernels' plans: launch_bias_grad (one
launch up to 512 rows, chunks of rows above; columns in blocks of 64) and the
weight normalisation (16 columns a workgroup and 24 rows a lane in registers, or
4 and 64: 1536 and 4096 rows, and past them), against double."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import TOL, assert_bits_equal, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1), (15, 64), (512, 65), (513, 3), (1000, 130), (65537, 64), (4097, 1000),
                                   (2049, 40000)], ids=lambda s: "x".join(map(str, s)))
def test_bias_grad_plans(L, rng, shape):
    rows, N = shape
    print(f"[case] bias grad {shape}", flush=True)
    g = rng.standard_normal(shape).astype(np.float32)
    gd, out = L.to_device(g), L.alloc(N)
    L.launch_bias_grad(out.p, gd.p, rows, N, None)
    L.sync()
    d = g.astype(np.float64)
    assert rel_err(out.download(), d.sum(0), floor=np.sqrt((d * d).sum(0))) <= TOL


@pytest.mark.parametrize("shape", [(1, 1), (27, 3), (255, 5), (256, 4), (257, 66), (4032, 12), (4096, 9), (4097, 6),
                                   (9000, 10)], ids=lambda s: "x".join(map(str, s)))
def test_weight_norm_plans(L, rng, shape):
    n, m = shape
    print(f"[case] weight norm {shape}", flush=True)
    W = rng.standard_normal(shape).astype(np.float32)
    M = rng.standard_normal(shape).astype(np.float32)
    wd, gd = L.to_device(W), L.to_device(M)
    L.launch_weight_normalize(wd.p, n, m, 1e-4, None)
    gain, gg = L.to_device(np.array([1.3], np.float32)), L.to_device(np.array([0.5], np.float32))
    ws = L.to_device(np.zeros(L.nnhip_weight_normalize_backward_workspace(m), np.float32))
    L.launch_weight_normalize_backward_ws(gd.p, wd.p, gain.p, gg.p, n, m, ws.p, None)
    L.sync()
    w64, m64 = W.astype(np.float64), M.astype(np.float64)
    wn = w64 / np.sqrt((w64 * w64).sum(0) + 1e-4)
    dot = (wn * m64).sum(0)
    assert rel_err(wd.download(shape=shape), wn) <= TOL
    ref = 1.3 * (m64 - dot * wn)
    # near (1, m) the two terms cancel: relative to what is subtracted
    assert rel_err(gd.download(shape=shape), ref, floor=np.sqrt(np.mean(m64 * m64))) <= TOL
    assert abs(gg.download()[0] - (0.5 + dot.sum())) <= TOL * np.sqrt((wn * wn * m64 * m64).sum() + 1)
    assert ws.download(1).view(np.uint32)[0] == 0  # the counter is armed again


def _tree(a, axis):
    """Neighbours added pairwise until one is left (fp32)."""
    a = np.moveaxis(a, axis, 0)
    while len(a) > 1:
        a = a[0::2] + a[1::2]
    return a[0]


def _one_by_one(a):
    t = np.zeros_like(a[0])
    for v in a:
        t = t + v
    return t


def _weight_norm_dots(wn, m):
    """The kernel's column sums and their sum in its order, in fp32: rows r, r + 64, ... of a lane one by one, trees
    of 4 lanes, 16 of those one by one; trees of 16 columns, each 64th of which a wave lane adds, a tree of the 16
    lanes of a row, 4 rows one by one."""
    n, cols = wn.shape
    terms = np.zeros((-(-n // 64) * 64, cols), np.float32)
    terms[:n] = wn * m
    lanes = _one_by_one(terms.reshape(-1, 64, cols))
    dots = _one_by_one(_tree(lanes.reshape(16, 4, cols), 1))
    padded = np.zeros(-(-cols // 1024) * 1024, np.float32)
    padded[:cols] = dots
    lane = _one_by_one(_tree(padded.reshape(-1, 64, 16), 2))
    return dots, _one_by_one(_tree(lane.reshape(4, 16), 1))


@pytest.mark.parametrize("shape", [(1, 1), (27, 3), (513, 17), (1152, 128), (1600, 512), (4096, 66), (4500, 20),
                                   (70, 1100)],
                         ids=lambda s: "x".join(map(str, s)))
def test_weight_norm_backward_order(L, rng, shape):
    """The gain gradient is a sum of terms of either sign and may be a small part of what it adds, so its order is
    part of the result: bit for bit what that order gives in fp32 on the CPU, with and without a workspace."""
    n, m = shape
    print(f"[case] weight norm order {shape}", flush=True)
    W = (rng.standard_normal(shape) / np.sqrt(n)).astype(np.float32)
    M = rng.standard_normal(shape).astype(np.float32)
    dots, total = _weight_norm_dots(W, M)
    gain = np.float32(1.3)
    for ws in (True, False):
        wd, gd, gn, gg = L.to_device(W), L.to_device(M), L.to_device(np.array([gain])), L.to_device(np.zeros(1, np.float32))
        if ws:
            w = L.to_device(np.zeros(L.nnhip_weight_normalize_backward_workspace(m), np.float32))
            L.launch_weight_normalize_backward_ws(gd.p, wd.p, gn.p, gg.p, n, m, w.p, None)
        else:
            L.launch_weight_normalize_backward(gd.p, wd.p, gn.p, gg.p, n, m, None)
        L.sync()
        assert_bits_equal(gg.download(), np.array([total]), "gain gradient")
        assert_bits_equal(gd.download(shape=shape), gain * (M - dots * W), "weight gradient")
