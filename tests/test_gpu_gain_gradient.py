"""The weight-normalised modules (mp_linear, conv2d in mp mode).  Their gain
gradient is sum_j <Wn_j, gW_j>, a sum of terms of either sign that may leave a
hundredth of what it adds: its value depends on the order of every sum before
it.  So the products keep their order (the fp32 matrix cores for convolutions,
rocBLAS for dense layers and the convolutions' library path) and the results are
held to the bit; and they are held against double, relative to the root of the
summed squares of the terms."""
from __future__ import annotations

import ctypes as C
import hashlib

import numpy as np
import pytest

from helpers import TOL, assert_bits_equal, rel_err
from module_abi import Module

pytestmark = pytest.mark.gpu

CONVS = [
    # B, H, W, C_in, C_out, K, stride, pad, NNHIP_CONV_PATH; gain gradient, and what all results hash to
    # (None: the library's products, whose bits are its own)
    ((4, 8, 8, 64, 128, 3, 1, 1), "implicit", "-0x1.09e7acp+7", "20313578f5b1a5cc"),
    ((3, 9, 7, 128, 64, 3, 1, 1), "implicit", "0x1.b4a14p+6", "b8aec5eaedbfb692"),  # 64 columns, a ragged last tile, rows split in 2
    ((2, 11, 10, 32, 192, 3, 2, 1), "implicit", "-0x1.639598p+7", None),  # strided; the input gradient is the library's
    ((5, 6, 6, 64, 64, 5, 1, 2), "implicit", "0x1.65b47ep+6", "c380b5dcbc39fb20"),
    ((2, 8, 8, 64, 64, 3, 1, 1), None, None, None),  # few pixels: the library's products
    ((3, 6, 5, 12, 10, 3, 1, 1), None, None, None),
]


def conv_results(L, monkeypatch, geom, path):
    B, H, W, Ci, Co, K, s, p = geom
    rng = np.random.default_rng(7)
    Ho, Wo = (H + 2 * p - K) // s + 1, (W + 2 * p - K) // s + 1
    x = rng.standard_normal((B, H, W, Ci), dtype=np.float32)
    w = rng.standard_normal((K * K * Ci, Co), dtype=np.float32)
    g = rng.standard_normal((B, Ho, Wo, Co), dtype=np.float32)
    if path:
        monkeypatch.setenv("NNHIP_CONV_PATH", path)
    else:
        monkeypatch.delenv("NNHIP_CONV_PATH", raising=False)
    m = Module(L, "conv2d_create", Ci, Co, K, s, p, H, W, B, 1, 1.0)
    m.set(0, w)
    m.set(1, [0.8])
    xd, gd, y, gx = L.to_device(x), L.to_device(g), L.alloc(g.size), L.alloc(x.size)
    m.forward(xd.p, y.p, B)
    m.backward(xd.p, y.p, gd.p, gx.p, B)
    L.sync()
    L.check("conv2d mp")
    got = {"y": y.download(shape=(-1, Co)), "gx": gx.download(shape=x.shape), "wn": m.get(0).reshape(-1, Co),
           "gw": m.get(0, True).reshape(-1, Co), "gain": m.get(1, True)}
    m.free()
    return (x, w, g), got


def digest(got):
    return hashlib.sha1(b"".join(np.ascontiguousarray(got[k]).tobytes() for k in ("y", "gx", "wn", "gw", "gain"))).hexdigest()[:16]


@pytest.mark.parametrize("geom,path,gain,sha", CONVS, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else "")
def test_conv_module_with_gain(L, monkeypatch, geom, path, gain, sha):
    B, H, W, Ci, Co, K, s, p = geom
    print(f"[case] conv2d with gain {geom} {path}", flush=True)
    (x, w, g), got = conv_results(L, monkeypatch, geom, path)
    if gain:
        assert got["gain"][0] == np.float32(float.fromhex(gain))
    if sha:
        assert digest(got) == sha
    w64 = w.astype(np.float64)
    wn = w64 / np.sqrt((w64 * w64).sum(0) + 1e-4)
    assert rel_err(got["wn"], wn) <= TOL
    Ho, Wo = (H + 2 * p - K) // s + 1, (W + 2 * p - K) // s + 1
    xp = np.pad(x.astype(np.float64), ((0, 0), (p, p), (p, p), (0, 0)))
    g64 = g.astype(np.float64).reshape(-1, Co)
    y = sq = 0.0
    gw, gs = [], []
    gxp, gxq = np.zeros_like(xp), np.zeros_like(xp)
    for t in range(K * K):
        i, j = divmod(t, K)
        at = np.s_[:, i:i + s * (Ho - 1) + 1:s, j:j + s * (Wo - 1) + 1:s]
        a, b = xp[at].reshape(-1, Ci), wn[t * Ci:(t + 1) * Ci]
        y, sq = y + a @ b, sq + (a * a) @ (b * b)
        gw.append(a.T @ g64)
        gs.append((a * a).T @ (g64 * g64))
        gxp[at] += (g64 @ b.T).reshape(B, Ho, Wo, Ci)
        gxq[at] += ((g64 * g64) @ (b * b).T).reshape(B, Ho, Wo, Ci)
    cut = np.s_[:, p:p + H, p:p + W]
    assert rel_err(got["y"], 0.8 * y, floor=0.8 * np.sqrt(sq)) <= TOL
    # a strided convolution leaves pixels that no output reads: zero, on a floor of the others
    assert rel_err(got["gx"], 0.8 * gxp[cut], floor=np.maximum(0.8 * np.sqrt(gxq[cut]), 1e-3)) <= TOL
    gw, gs = np.concatenate(gw), np.concatenate(gs)
    dots = (wn * gw).sum(0)
    assert rel_err(got["gw"], 0.8 * (gw - dots * wn), floor=np.sqrt(gs)) <= TOL
    assert abs(got["gain"][0] - dots.sum()) <= TOL * np.sqrt((wn * wn * gs).sum())


@pytest.mark.parametrize("shape", [(128, 256, 512), (7, 30, 18), (1, 64, 64)], ids=lambda s: "x".join(map(str, s)))
def test_mp_linear_is_the_library_product(L, shape):
    """Bit for bit the launches and rocBLAS products that the module stands for."""
    B, ni, no = shape
    print(f"[case] mp_linear {shape}", flush=True)
    rng = np.random.default_rng(8)
    x, w, g = (rng.standard_normal(s, dtype=np.float32) for s in ((B, ni), (ni, no), (B, no)))
    m = Module(L, "mp_linear_create", ni, no, 1.0)
    m.set(0, w)
    m.set(1, [0.8])
    xd, gd, y, gx = L.to_device(x), L.to_device(g), L.alloc(g.size), L.alloc(x.size)
    m.forward(xd.p, y.p, B)
    m.backward(xd.p, y.p, gd.p, gx.p, B)
    L.sync()
    wd, gw, y2, gx2, gain = L.to_device(w), L.alloc(w.size), L.alloc(g.size), L.alloc(x.size), L.to_device(np.array([0.8], np.float32))
    gg, ws = L.to_device(np.zeros(1, np.float32)), L.to_device(np.zeros(L.nnhip_weight_normalize_backward_workspace(no), np.float32))
    one, zero = C.c_float(1.0), C.c_float(0.0)
    sgemm = C.CDLL("librocblas.so").rocblas_sgemm
    none, tr = 111, 112

    def gemm(ta, tb, mm, nn, kk, a, lda, b, ldb, c, ldc):
        assert sgemm(C.c_void_p(m.ctx.blas), ta, tb, mm, nn, kk, C.byref(one), C.c_void_p(a.p), lda, C.c_void_p(b.p), ldb,
                     C.byref(zero), C.c_void_p(c.p), ldc) == 0

    L.launch_weight_normalize(wd.p, ni, no, 1e-4, None)
    gemm(none, none, no, B, ni, wd, no, xd, ni, y2, no)
    L.launch_scale_by_scalar(y2.p, gain.p, B * no, None)
    gemm(none, tr, no, ni, B, gd, no, xd, ni, gw, no)
    L.launch_weight_normalize_backward_ws(gw.p, wd.p, gain.p, gg.p, ni, no, ws.p, None)
    gemm(tr, none, ni, B, no, wd, no, gd, no, gx2, ni)
    L.launch_scale_by_scalar(gx2.p, gain.p, B * ni, None)
    L.sync()
    for got, want, what in ((y.download(), y2.download(), "y"), (gx.download(), gx2.download(), "gx"),
                            (m.get(0), wd.download(), "weight"), (m.get(0, True), gw.download(), "gw"),
                            (m.get(1, True), gg.download(), "gain gradient")):
        assert_bits_equal(got, want, what)
    w64 = w.astype(np.float64)
    wn = w64 / np.sqrt((w64 * w64).sum(0) + 1e-4)
    x64, g64 = x.astype(np.float64), g.astype(np.float64)
    assert rel_err(y.download(shape=g.shape), 0.8 * x64 @ wn, floor=0.8 * np.sqrt((x64 * x64) @ (wn * wn))) <= TOL
    terms = (wn * wn * ((x64 * x64).T @ (g64 * g64))).sum()
    assert abs(m.get(1, True)[0] - (wn * (x64.T @ g64)).sum()) <= TOL * np.sqrt(terms)
    m.free()


@pytest.mark.parametrize("geom", [(3, 5, 7, 32, 128, 3, 1), (2, 9, 9, 64, 64, 3, 1), (2, 8, 8, 64, 192, 1, 0), (1, 9, 9, 128, 64, 5, 2)],
                         ids=lambda g: "x".join(map(str, g)))
def test_fused_epilogues_of_the_fp32_kernels(L, nn, rng, geom):
    """Tiles that end within the tensor and both tile widths: the neighbours in the epilogue against the separate
    launches, bit for bit."""
    B, H, W, Ci, Co, K, p = geom
    print(f"[case] fp32 kernels' epilogues {geom}", flush=True)
    d, P, I = L.dll, C.c_void_p, C.c_int
    d.nnk_conv_f32_forward.argtypes, d.nnk_conv_f32_forward.restype = [P] * 4 + [I] * 10 + [P, P], None
    d.nnk_conv_f32_input_grad.argtypes, d.nnk_conv_f32_input_grad.restype = [P] * 4 + [I] * 7 + [P, P], None
    n, ni = B * H * W * Co, B * H * W * Ci

    def dev(*shape, scale=1.0):
        return L.to_device((scale * rng.standard_normal(shape)).astype(np.float32))

    xd, wd, cond, res = dev(ni), dev(K * K * Ci, Co, scale=0.1), dev(B, Co, scale=0.5), dev(n)
    gain = L.to_device(np.array([0.91], np.float32))
    y, want, got, y2 = L.alloc(n), L.alloc(n), L.alloc(n), L.alloc(n)
    geo = (B, H, W, Ci, Co, K, 1, p, H, W)
    d.nnk_conv_f32_forward(y.p, xd.p, wd.p, gain.p, *geo, None, None)
    f = nn.NnConvFusion(cond=cond.p, y2=y2.p, act=nn.ACT_MP_SILU)
    d.nnk_conv_f32_forward(got.p, xd.p, wd.p, gain.p, *geo, C.addressof(f), None)
    L.launch_spatial_modulate_act_forward(want.p, y.p, cond.p, B, H * W, 1, Co, nn.ACT_MP_SILU, None)
    L.sync()
    L.check("modulate")
    assert_bits_equal(got.download(), y.download(), "y")
    assert_bits_equal(y2.download(), want.download(), "y2")
    f = nn.NnConvFusion(res=res.p, res_w=0.83, out_w=0.55)
    d.nnk_conv_f32_forward(got.p, xd.p, wd.p, gain.p, *geo, C.addressof(f), None)
    L.launch_weighted_sum(want.p, res.p, y.p, 0.83, 0.55, n, None)
    L.sync()
    assert_bits_equal(got.download(), want.download(), "residual")
    if Ci % 64 or Co % 32:
        return
    gd, act, resi, dx, t = dev(n), dev(ni), dev(ni), L.alloc(ni), L.alloc(ni)
    d.nnk_conv_f32_input_grad(dx.p, gd.p, wd.p, gain.p, B, H, W, Ci, Co, K, p, None, None)
    f = nn.NnConvFusion(act_in=act.p, act=nn.ACT_MP_SILU, res=resi.p, res_w=0.83, out_w=1.0)
    d.nnk_conv_f32_input_grad(t.p, gd.p, wd.p, gain.p, B, H, W, Ci, Co, K, p, C.addressof(f), None)
    L.sync()
    L.check("activation gradient")
    fused = t.download()
    L.launch_activation_backward(t.p, dx.p, act.p, ni, nn.ACT_MP_SILU, None)
    L.launch_weighted_sum(t.p, resi.p, t.p, 0.83, 1.0, ni, None)
    L.sync()
    assert_bits_equal(fused, t.download(), "input gradient")
