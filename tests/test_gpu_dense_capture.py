"""Weight gradients captured in a HIP graph where the eager call takes the tiled
kernel: every replay gives what the eager call gave, bit for bit, when the
sequence ran once on the stream before (its scratch is then cached) and wherever
the tiled kernel needs no scratch; a stream without the scratch takes the small
tiles, within the reduction bar."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from helpers import TOL, assert_bits_equal, rel_err
from module_abi import Module

pytestmark = pytest.mark.gpu

P, I = C.c_void_p, C.c_int
CONV_SCRATCH_FREE = (4, 16, 16, 1024, 1024, 3, 1, 1)  # 576 tiles: one split


def _stream(L):
    s = L.dll.nnhip_stream_create()
    assert s
    return s


def _captured(L, s, issue):
    assert L.dll.nnhip_graph_capture_begin(s) == 0
    issue()
    g = L.dll.nnhip_graph_capture_end(s)
    assert g
    return g


def _tiled(L, *geom):
    f = L.dll.nnk_conv_weight_grad_tiled
    f.argtypes = [I] * 8
    return f(*geom)


@pytest.mark.parametrize("warm", [True, False], ids=["warm", "cold"])
def test_linear_backward_replays(L, rng, warm):
    B, ni, no = 4096, 512, 512
    print(f"[case] linear backward captured, {'scratch cached' if warm else 'no scratch'}", flush=True)
    assert _tiled(L, B, 1, 1, ni, no, 1, 1, 0)
    s = _stream(L)
    m = Module(L, "linear_create", ni, no, stream=s)
    sets = [(rng.standard_normal((B, ni), dtype=np.float32), rng.standard_normal((B, no), dtype=np.float32)) for _ in range(2)]
    xd, gd, y, gx = L.alloc(B * ni), L.alloc(B * no), L.alloc(B * no), L.alloc(B * ni)

    def issue():
        m.forward(xd.p, y.p, B)
        m.backward(xd.p, y.p, gd.p, gx.p, B)

    def load(k):
        L.dll.nnhip_stream_synchronize(s)
        xd.upload(sets[k][0])
        gd.upload(sets[k][1])

    def results():
        L.dll.nnhip_stream_synchronize(s)
        L.sync()
        return [y.download(), gx.download(), m.get(0, True), m.get(1, True)]

    def eager():
        refs = []
        for k in range(2):
            load(k)
            issue()
            refs.append(results())
        return refs

    refs = eager() if warm else None
    graph = _captured(L, s, issue)
    L.check("capture")
    got = []
    for k in (0, 1, 0, 1, 1):
        load(k)
        assert L.dll.nnhip_graph_launch(graph, s) == 0
        got.append((k, results()))
        if warm:  # eager work on the same stream and scratch between the replays
            issue()
            results()
    refs = refs or eager()
    for k, outs in got:
        for a, b, what in zip(outs, refs[k], ("y", "gx", "gw", "gb")):
            if warm or what in ("y", "gx"):
                assert_bits_equal(a, b, f"{what}, inputs {k}")
        x64, g64 = (v.astype(np.float64) for v in sets[k])
        assert rel_err(outs[2].reshape(ni, no), x64.T @ g64, floor=np.sqrt((x64 * x64).T @ (g64 * g64))) <= TOL
        assert rel_err(outs[3], g64.sum(0), floor=np.sqrt((g64 * g64).sum(0))) <= TOL
    L.dll.nnhip_graph_destroy(graph)
    m.free()
    L.dll.nnhip_stream_destroy(s)


def test_one_split_needs_no_scratch(L, rng):
    B, H, W, Ci, Co, K, st, p = CONV_SCRATCH_FREE
    print(f"[case] captured weight gradient of one split {CONV_SCRATCH_FREE}", flush=True)
    assert _tiled(L, *CONV_SCRATCH_FREE)
    d = L.dll
    d.nnk_conv_weight_grad.argtypes, d.nnk_conv_weight_grad.restype = [P] * 4 + [I] * 10 + [P, P], None
    xd, gd = (L.to_device(rng.standard_normal(B * H * W * c, dtype=np.float32)) for c in (Ci, Co))
    gw, gb = L.alloc(K * K * Ci * Co), L.alloc(Co)
    s = _stream(L)

    def issue():
        d.nnk_conv_weight_grad(gw.p, gb.p, xd.p, gd.p, B, H, W, Ci, Co, K, st, p, H, W, None, s)

    graph = _captured(L, s, issue)
    outs = []
    for replay in (True, False, True):
        gw.fill_bytes(0xFF)
        L.sync()
        if replay:
            assert d.nnhip_graph_launch(graph, s) == 0
        else:
            issue()
        d.nnhip_stream_synchronize(s)
        outs.append((gw.download(), gb.download()))
    L.check("captured weight gradient")
    for a, b in outs[1:]:
        assert_bits_equal(outs[0][0], a, "gw")
        assert_bits_equal(outs[0][1], b, "gb")
    d.nnhip_graph_destroy(graph)
    d.nnhip_stream_destroy(s)
