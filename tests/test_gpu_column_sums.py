"""Column sums at the edges of their kernels' plans: launch_bias_grad (one
launch up to 512 rows, chunks of rows above; columns in blocks of 64) and the
weight normalisation (4 columns a workgroup, 16 rows a lane in registers, 4096
rows, and past them), against double."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import TOL, rel_err

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
