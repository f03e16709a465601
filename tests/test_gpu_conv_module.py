"""The products of the conv2d and linear modules (host/conv_api.h) at
any channel counts and alignment, at the edges of the small tiles (32 x 32
outputs and 16 k a step, or 16 x 16 and 32 k, 4 / 8 / 16 waves) and of the tiled kernels' ragged forms,
against double; bar as in test_gpu_conv_implicit.py.  Geometries past each rule
of the choice between them: few tiles (small), many (128, 64 or 32 columns)."""
from __future__ import annotations

import ctypes as C
from pathlib import Path

import numpy as np
import pytest

from helpers import TOL, assert_bits_equal
from module_abi import Module
from test_gpu_conv_split import _conv64

pytestmark = pytest.mark.gpu

P, I = C.c_void_p, C.c_int

GEOMS = [
    # B, H, W, C_in, C_out, K, stride, pad, offset of every tensor in floats
    (1, 1, 1, 1, 1, 1, 1, 0, 0),        # one product
    (33, 1, 1, 17, 31, 1, 1, 0, 0),     # dense, ragged, two row tiles
    (128, 1, 1, 512, 512, 1, 1, 0, 0),  # dense
    (5, 1, 1, 64, 96, 1, 1, 0, 1),      # dense, misaligned
    (8, 7, 7, 128, 128, 3, 1, 1, 0),    # small tiles, 72 steps
    (2, 6, 5, 40, 33, 3, 1, 1, 0),      # C_in no multiple of 16
    (1, 17, 1, 72, 17, 1, 1, 0, 0),     # tiles of 16 with one row and column more, 4 waves
    (1, 5, 3, 248, 16, 1, 1, 0, 1),     # fewer rows than one, misaligned, 8 waves
    (2, 5, 8, 4, 320, 5, 1, 2, 0),      # a long k range, few outputs: 250 steps on 16 waves
    (4, 16, 16, 256, 96, 3, 1, 1, 0),   # tiles of 32 forward and back, many of them
    (64, 32, 32, 3, 64, 3, 1, 1, 0),    # an image in: ragged rows, tiled
    (64, 32, 32, 64, 3, 3, 1, 1, 0),    # an image out
    (3, 65, 64, 20, 70, 3, 1, 1, 0),    # ragged, 128 columns of which 70 are
    (40, 32, 32, 24, 48, 3, 1, 1, 0),   # halo rows with a partial slice, 64 columns
    (40, 32, 32, 48, 96, 3, 1, 1, 1),   # misaligned: 4-byte loads
    (16, 33, 31, 10, 130, 5, 2, 2, 0),  # strided, even channels in pairs
    (90, 16, 16, 5, 7, 3, 2, 1, 0),
    (700, 7, 7, 6, 34, 1, 1, 0, 0),     # weight gradient of many splits and few elements
]


def _api(L):
    d = L.dll
    d.nnk_conv_forward.argtypes = [P] * 5 + [I] * 10 + [P, P]
    d.nnk_conv_input_grad.argtypes = [P] * 4 + [I] * 7 + [P, P]
    d.nnk_conv_weight_grad.argtypes = [P] * 4 + [I] * 10 + [P, P]
    d.nnk_conv_weight_grad_workspace.argtypes = [I] * 6
    d.nnk_conv_weight_grad_workspace.restype = C.c_size_t
    for f in (d.nnk_conv_forward, d.nnk_conv_input_grad, d.nnk_conv_weight_grad):
        f.restype = None
    return d


def _within(got, ref, floor):
    err = np.abs(got.astype(np.float64) - ref) / np.maximum(np.maximum(np.abs(ref), floor), 1e-30)
    assert float(err.max()) <= TOL


@pytest.mark.parametrize("geom", GEOMS, ids=lambda g: "x".join(map(str, g)))
def test_conv_products(L, rng, geom):
    B, H, W, Ci, Co, K, s, p, off = geom
    print(f"[case] conv products {geom}", flush=True)
    d = _api(L)
    Ho, Wo = (H + 2 * p - K) // s + 1, (W + 2 * p - K) // s + 1
    x = rng.standard_normal((B, H, W, Ci)).astype(np.float32)
    w = (rng.standard_normal((K * K * Ci, Co)) / np.sqrt(K * K * Ci)).astype(np.float32)
    g = rng.standard_normal((B, Ho, Wo, Co)).astype(np.float32)
    bias = rng.standard_normal(Co).astype(np.float32)

    def dev(a):
        t = L.alloc(a.size + off)
        t.upload(np.concatenate([np.zeros(off, np.float32), a.ravel()]))
        return t

    def get(t, shape):
        return t.download()[off:].reshape(shape)

    xd, wd, gd, bd, gain = dev(x), dev(w), dev(g), L.to_device(bias), L.to_device(np.array([0.7], np.float32))
    y, gx, gw, gb = L.alloc(g.size + off), L.alloc(x.size + off), L.alloc(w.size + off), L.alloc(Co)
    o = off
    geo = (B, H, W, Ci, Co, K, s, p, Ho, Wo)
    d.nnk_conv_forward(y.offset(o), xd.offset(o), wd.offset(o), bd.p, None, *geo, None, None)
    ws = L.alloc(max(1, d.nnk_conv_weight_grad_workspace(B, Ci, Co, K, Ho, Wo)))
    d.nnk_conv_weight_grad(gw.offset(o), gb.p, xd.offset(o), gd.offset(o), *geo, ws.p, None)
    if s == 1:
        d.nnk_conv_input_grad(gx.offset(o), gd.offset(o), wd.offset(o), gain.p, B, H, W, Ci, Co, K, p, None, None)
    L.sync()
    L.check("conv products")
    ref, floor = _conv64(x, w, K, s, p)
    _within(get(y, ref.shape), ref + bias, floor)
    # the gradients tap by tap
    xp = np.pad(x.astype(np.float64), ((0, 0), (p, p), (p, p), (0, 0)))
    g64 = g.astype(np.float64).reshape(-1, Co)
    gxp, gxq = np.zeros_like(xp), np.zeros_like(xp)
    rw, fw = [], []
    for t in range(K * K):
        i, j = divmod(t, K)
        at = np.s_[:, i:i + s * (Ho - 1) + 1:s, j:j + s * (Wo - 1) + 1:s]
        a = xp[at].reshape(-1, Ci)
        rw.append(a.T @ g64)
        fw.append(np.sqrt((a * a).T @ (g64 * g64)))
        wt = w[t * Ci:(t + 1) * Ci].astype(np.float64)
        gxp[at] += (g64 @ wt.T).reshape(B, Ho, Wo, Ci)
        gxq[at] += ((g64 * g64) @ (wt * wt).T).reshape(B, Ho, Wo, Ci)
    _within(get(gw, w.shape), np.concatenate(rw), np.concatenate(fw))
    _within(gb.download(), g64.sum(0), np.sqrt((g64 * g64).sum(0)))
    if s == 1:
        cut = np.s_[:, p:p + H, p:p + W]
        _within(get(gx, x.shape), 0.7 * gxp[cut], 0.7 * np.sqrt(gxq[cut]))


@pytest.mark.parametrize("geom", [(2, 5, 6, 24, 40, 3, 1, 1), (1, 4, 4, 64, 64, 3, 1, 1)],
                         ids=lambda g: "x".join(map(str, g)))
def test_small_tiles_fused_epilogues(L, nn, rng, geom):
    """The epilogues on the small tiles against the separate launches, bit for bit."""
    B, H, W, Ci, Co, K, s, p = geom
    print(f"[case] small tile epilogues {geom}", flush=True)
    d = _api(L)
    n = B * H * W * Co
    xd = L.to_device(rng.standard_normal((B, H, W, Ci)).astype(np.float32))
    wd = L.to_device((rng.standard_normal((K * K * Ci, Co)) / np.sqrt(K * K * Ci)).astype(np.float32))
    gain = L.to_device(np.array([0.91], np.float32))
    cond = L.to_device((0.5 * rng.standard_normal((B, Co))).astype(np.float32))
    res = L.to_device(rng.standard_normal(n).astype(np.float32))
    y, want, got, y2 = L.alloc(n), L.alloc(n), L.alloc(n), L.alloc(n)
    geo = (B, H, W, Ci, Co, K, s, p, H, W)
    d.nnk_conv_forward(y.p, xd.p, wd.p, None, gain.p, *geo, None, None)
    f = nn.NnConvFusion(cond=cond.p, y2=y2.p, act=nn.ACT_MP_SILU)
    d.nnk_conv_forward(got.p, xd.p, wd.p, None, gain.p, *geo, C.addressof(f), None)
    L.launch_spatial_modulate_act_forward(want.p, y.p, cond.p, B, H * W, 1, Co, nn.ACT_MP_SILU, None)
    L.sync()
    assert_bits_equal(got.download(), y.download(), "y")
    assert_bits_equal(y2.download(), want.download(), "y2")
    f = nn.NnConvFusion(res=res.p, res_w=0.83, out_w=0.55)
    d.nnk_conv_forward(got.p, xd.p, wd.p, None, gain.p, *geo, C.addressof(f), None)
    L.launch_weighted_sum(want.p, res.p, y.p, 0.83, 0.55, n, None)
    L.sync()
    assert_bits_equal(got.download(), want.download(), "residual")


COLUMNS = [
    # B, H, W, C_in, C_out, K, stride, pad, mp: input gradients by columns
    (64, 32, 32, 3, 64, 3, 1, 1, 0),   # an image in
    (20, 11, 11, 8, 448, 5, 1, 2, 1),  # a long k range, with a gain: the library's products
    (20, 11, 11, 8, 448, 5, 1, 2, 0),  # ... and without
    (3, 9, 8, 40, 24, 3, 2, 1, 1),     # strided: the library product
    (3, 9, 8, 40, 24, 3, 2, 1, 0),
    (2, 10, 7, 5, 33, 5, 3, 0, 0),     # stride past the padding: pixels that no column reaches
]


@pytest.mark.parametrize("geom", COLUMNS, ids=lambda g: "x".join(map(str, g)))
def test_input_gradient_by_columns(L, geom):
    """The conv2d module against its im2col + GEMM + col2im sequence: different
    summation orders of the same fp32 products, so 4 sqrt(terms) 2^-24 relative
    to max(|v|, rms(v)); the longest sum has 25 * 448 terms (2.5e-5)."""
    lib = C.CDLL(str(Path(__file__).resolve().parent / "_build" / "libgradcheck.so"))
    lib.nn_convcheck.argtypes = [C.c_int] * 10 + [C.POINTER(C.c_float)]
    lib.nn_convcheck.restype = C.c_double
    print(f"[case] input gradient by columns {geom}", flush=True)
    B, H, W, Ci, Co, K, s, p, mp = geom
    by = L.dll.nnk_conv_input_grad_by_columns
    by.argtypes, by.restype = [I] * 7, I
    assert s > 1 or by(B, H, W, Ci, Co, K, p)
    worst = lib.nn_convcheck(*geom, 1, (C.c_float * 4)())
    terms = max(K * K * Ci, K * K * Co, B * ((H + 2 * p - K) // s + 1) * ((W + 2 * p - K) // s + 1))
    assert worst <= 4 * terms ** 0.5 * 2.0 ** -24


def test_rule_for_columns(L):
    by = L.dll.nnk_conv_input_grad_by_columns
    by.argtypes, by.restype = [I] * 7, I
    assert not by(8, 7, 7, 128, 128, 3, 1)
    assert not by(128, 32, 32, 128, 128, 3, 1)
    assert not by(64, 32, 32, 3, 64, 1, 0)       # one tap: nothing to sum
    assert not by(1 << 20, 64, 64, 3, 64, 3, 1)  # rows past 32 bits


def test_module_holds_no_im2col_matrix(L):
    """A convolution whose products all go by the kernels: weights, gradients and partial sums, without the 75 MB of
    an im2col matrix that nothing reads."""
    print("[case] conv module memory", flush=True)
    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()

    def now():
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    small = Module(L, "conv2d_create", 8, 8, 1, 1, 0, 2, 2, 1, 0, 1.0)  # the context and what the library keeps for it
    L.sync()
    before = now()
    m = L.dll.conv2d_create(C.byref(small.ctx), 128, 128, 3, 1, 1, 32, 32, 16, 0, C.c_float(1.0))
    assert not L.dll.nnk_conv_input_grad_by_columns(16, 32, 32, 128, 128, 3, 1)
    own = 2 * 4 * (9 * 128 * 128 + 128)
    ws = L.dll.nnk_conv_weight_grad_workspace
    ws.argtypes, ws.restype = [I] * 6, C.c_size_t
    assert before - now() <= own + 4 * ws(16, 128, 128, 3, 32, 32) + (8 << 20)  # allocation granularity
    m.contents.free(m)
    small.free()
