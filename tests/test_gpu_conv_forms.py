"""Every form of the convolution kernels by name (host/conv_api.h, nnk_conv_*_as):
the small tiles, the tiled kernel with 32, 64 and 128 columns and each way of
staging its activations (halo rows, rows gathered per tap, ragged loads), plain and
flipped; the weight gradient's small tiles and its tiled kernel with each way of
loading.  The rules give small shapes to the small tiles, so a shape alone does not
reach the edges of the others.  Against double; bar as in test_gpu_conv_implicit.py:
1e-5 relative to max(|ref|, sqrt(sum of the squared products))."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from helpers import TOL, assert_bits_equal
from test_gpu_conv_split import _check, _conv64

pytestmark = pytest.mark.gpu

P, I = C.c_void_p, C.c_int
HALO, GATHER, RAGGED = 0, 1, 2
FORMS = [(0, -1)] + [(n, m) for n in (32, 64, 128) for m in (HALO, GATHER, RAGGED)]  # columns, staging
LOADS = [(0, -1), (1, 0), (1, 1), (1, 2)]  # tiled, loads

GEOMS = [
    # B, H, W, C_in, C_out, K, stride, pad
    (3, 5, 3, 32, 64, 3, 1, 1),    # images smaller than a tile
    (1, 43, 3, 64, 64, 3, 1, 1),   # 129 rows: the second tile has one
    (2, 4, 63, 32, 64, 5, 1, 2),   # the widest 5 x 5 halo
    (1, 4, 70, 32, 64, 5, 1, 2),   # ... and past it: rows gathered per tap
    (1, 3, 140, 32, 64, 3, 1, 1),
    (2, 9, 7, 32, 64, 3, 1, 0),    # output smaller than the input
    (2, 9, 7, 32, 64, 7, 1, 3),    # more taps than bits
    (2, 6, 6, 160, 64, 1, 2, 0),   # strided 1 x 1
    (1, 5, 6, 40, 72, 1, 1, 0),    # 1 x 1, a slice and columns in part
    (2, 13, 9, 24, 70, 3, 1, 1),   # less than a slice, 70 columns
    (4, 8, 12, 130, 200, 3, 1, 1), # two k tiles and two column tiles of the weight gradient, rows in fours
    (3, 9, 9, 8, 7, 3, 2, 1),
    (2, 7, 8, 5, 33, 3, 1, 1),     # odd channels: ragged only
    (1, 1, 1, 1, 1, 1, 1, 0),
    (70, 1, 1, 17, 31, 1, 1, 0),   # dense
]


class Api:
    def __init__(self, L):
        self.L, d = L, L.dll
        d.nnk_conv_forward_as.argtypes = [I, I] + [P] * 5 + [I] * 10 + [P, P]
        d.nnk_conv_input_grad_as.argtypes = [I, I] + [P] * 4 + [I] * 7 + [P, P]
        d.nnk_conv_weight_grad_as.argtypes = [I, I] + [P] * 4 + [I] * 10 + [P, P]
        d.nnk_conv_weight_grad_workspace.argtypes, d.nnk_conv_weight_grad_workspace.restype = [I] * 6, C.c_size_t
        d.nnk_conv_tile.argtypes, d.nnk_conv_weight_grad_tiled.argtypes = [I] * 9, [I] * 8
        for f in (d.nnk_conv_forward_as, d.nnk_conv_input_grad_as, d.nnk_conv_weight_grad_as):
            f.restype = None
        self.d = d

    def forward(self, form, x, w, K, s, p, bias=None):
        B, H, W, Ci = x.shape
        Co = w.shape[1]
        Ho, Wo = (H + 2 * p - K) // s + 1, (W + 2 * p - K) // s + 1
        xd, wd, y = self.L.to_device(x), self.L.to_device(w), self.L.alloc(B * Ho * Wo * Co)
        y.fill_bytes(0x7F)
        bd = self.L.to_device(bias) if bias is not None else None
        self.d.nnk_conv_forward_as(*form, y.p, xd.p, wd.p, bd and bd.p, None, B, H, W, Ci, Co, K, s, p, Ho, Wo, None, None)
        self.done(f"forward as {form}")
        return y.download(shape=(B * Ho * Wo, Co)).astype(np.float64)

    def input_grad(self, form, dy, w, shape, K, p):
        B, H, W, Ci = shape
        Co = dy.shape[-1]
        dd, wd, dx = self.L.to_device(dy), self.L.to_device(w), self.L.alloc(B * H * W * Ci)
        dx.fill_bytes(0x7F)
        self.d.nnk_conv_input_grad_as(*form, dx.p, dd.p, wd.p, None, B, H, W, Ci, Co, K, p, None, None)
        self.done(f"input gradient as {form}")
        return dx.download(shape=shape).astype(np.float64)

    def weight_grad(self, form, x, dy, K, s, p):
        B, H, W, Ci = x.shape
        Ho, Wo, Co = dy.shape[1:]
        xd, dd = self.L.to_device(x), self.L.to_device(dy)
        gw, gb = self.L.alloc(K * K * Ci * Co), self.L.alloc(Co)
        gw.fill_bytes(0x7F)
        ws = self.L.alloc(max(1, self.d.nnk_conv_weight_grad_workspace(B, Ci, Co, K, Ho, Wo)))
        self.d.nnk_conv_weight_grad_as(*form, gw.p, gb.p, xd.p, dd.p, B, H, W, Ci, Co, K, s, p, Ho, Wo, ws.p, None)
        self.done(f"weight gradient as {form}")
        return gw.download(shape=(K * K * Ci, Co)).astype(np.float64), gb.download().astype(np.float64)

    def done(self, what):
        self.L.sync()
        self.L.check(what)


@pytest.fixture(scope="module")
def api(L):
    return Api(L)


def _dgrad64(dy, w, shape, K, p):
    """Input gradient of a stride-1 convolution and the root sum of its squared products, in double."""
    B, H, W, Ci = shape
    Ho, Wo, Co = dy.shape[1:]
    g, w = dy.astype(np.float64).reshape(-1, Co), w.astype(np.float64)
    y, sq = np.zeros((B, H + 2 * p, W + 2 * p, Ci)), np.zeros((B, H + 2 * p, W + 2 * p, Ci))
    for t in range(K * K):
        i, j = divmod(t, K)
        b = w[t * Ci:(t + 1) * Ci]
        y[:, i:i + Ho, j:j + Wo] += (g @ b.T).reshape(B, Ho, Wo, Ci)
        sq[:, i:i + Ho, j:j + Wo] += ((g * g) @ (b * b).T).reshape(B, Ho, Wo, Ci)
    cut = np.s_[:, p:p + H, p:p + W]
    return y[cut], np.sqrt(sq[cut])


def _wgrad64(x, dy, K, s, p):
    Ho, Wo, Co = dy.shape[1:]
    xp = np.pad(x.astype(np.float64), ((0, 0), (p, p), (p, p), (0, 0)))
    g = dy.astype(np.float64).reshape(-1, Co)
    col = np.concatenate([xp[:, i:i + s * (Ho - 1) + 1:s, j:j + s * (Wo - 1) + 1:s].reshape(-1, x.shape[-1])
                          for i in range(K) for j in range(K)], 1)
    return col.T @ g, np.sqrt((col * col).T @ (g * g))


@pytest.mark.parametrize("geom", GEOMS, ids=lambda g: "x".join(map(str, g)))
def test_edges_of_every_form(api, rng, geom):
    B, H, W, Ci, Co, K, s, p = geom
    print(f"[case] conv forms {geom}", flush=True)
    Ho, Wo = (H + 2 * p - K) // s + 1, (W + 2 * p - K) // s + 1
    x = rng.standard_normal((B, H, W, Ci)).astype(np.float32)
    w = (rng.standard_normal((K * K * Ci, Co)) / np.sqrt(K * K * Ci)).astype(np.float32)
    g = rng.standard_normal((B, Ho, Wo, Co)).astype(np.float32)
    bias = rng.standard_normal(Co).astype(np.float32)
    ref, floor = _conv64(x, w, K, s, p)
    for form in FORMS:
        _check(api.forward(form, x, w, K, s, p, bias), ref + bias, floor)
    if s == 1 and p <= K - 1:
        ref, floor = _dgrad64(g, w, x.shape, K, p)
        for form in FORMS:
            _check(api.input_grad(form, g, w, x.shape, K, p), ref, floor)
    ref, floor = _wgrad64(x, g, K, s, p)
    g64 = g.astype(np.float64).reshape(-1, Co)
    for form in LOADS:
        gw, gb = api.weight_grad(form, x, g, K, s, p)
        _check(gw, ref, floor)
        _check(gb, g64.sum(0), np.sqrt((g64 * g64).sum(0)))


@pytest.mark.parametrize("form", FORMS, ids=lambda f: f"{f[0]}-{f[1]}")
@pytest.mark.parametrize("stride", [1, 2])
def test_values_outside_the_split(api, rng, form, stride):
    """Infinities and NaN give what fp32 gives; 3e38 rounds to infinity in bf16 and stays finite in the product."""
    print(f"[case] conv form {form} with inf, nan and huge operands, stride {stride}", flush=True)
    K, p = 3, 1
    x = rng.standard_normal((4, 16, 16, 32)).astype(np.float32)
    w = (np.abs(rng.standard_normal((9 * 32, 64))) + 0.1).astype(np.float32) * np.float32(1e-3)
    x[0, 3, 4, 5], x[1, 0, 0, 0], x[1, 15, 15, 1], x[2, 8, 8, 2] = np.inf, -np.inf, np.nan, 3.4e38
    x[3, 2, 2, 0], x[3, 2, 3, 0] = np.inf, -np.inf  # inf - inf where both are seen
    with np.errstate(invalid="ignore"):
        ref, floor = _conv64(x, w, K, stride, p)
        _check(api.forward(form, x, w, K, stride, p), ref, np.where(np.isfinite(floor), floor, 0.0))


@pytest.mark.parametrize("form", LOADS, ids=lambda f: f"{f[0]}-{f[1]}")
def test_weight_gradient_outside_the_split(api, rng, form):
    print(f"[case] weight gradient form {form} with inf and huge operands", flush=True)
    x = rng.standard_normal((4, 16, 16, 32)).astype(np.float32)
    x[2, 8, 8, 2] = 3.4e38
    dy = (1e-3 * rng.standard_normal((4, 16, 16, 64))).astype(np.float32)  # 3.4e38 dy stays finite
    dy[0, 0, 7, 3] = np.inf
    with np.errstate(invalid="ignore"):
        ref, floor = _wgrad64(x, dy, 3, 1, 1)
        _check(api.weight_grad(form, x, dy, 3, 1, 1)[0], ref, np.where(np.isfinite(floor), floor, 0.0))


# Factors on the activations per image, on the weight per column and per row: operands whose last plane would lie below the
# smallest normal number (2^-103 and below), all of them, beside ordinary ones, and against large ones.
SCALES = [(1e-36, 1.0, 1.0), (1e-33, 1.0, 1.0), (1e-30, 1.0, 1.0), (1e30, 1.0, 1.0),
          ((1.0, 1e-36), 1.0, 1.0), ((1e-34, 1.0), 1.0, 1.0), (1.0, (1.0, 1e-36), 1.0), (1e-36, 1e15, 1.0),
          ((1.0, 1e-35), 1e12, 1.0), (1e15, 1e-36, 1.0), ((1e9, 1e-36), (1e-36, 1e9), 1.0)]


def _scaled(x, w, scales):
    sx, sw, _ = scales
    x = x.copy()
    for b in range(len(x)):
        x[b] *= np.float32(sx[b * len(sx) // len(x)] if isinstance(sx, tuple) else sx)
    w = w.copy()
    for n in range(w.shape[1]):
        w[:, n] *= np.float32(sw[n % len(sw)] if isinstance(sw, tuple) else sw)
    return x, w


@pytest.mark.parametrize("scales", SCALES, ids=str)
def test_scales_outside_the_split(api, rng, scales):
    print(f"[case] conv forms at scales {scales}", flush=True)
    x = rng.standard_normal((2, 7, 8, 40)).astype(np.float32)
    w = (rng.standard_normal((9 * 40, 48)) / 19).astype(np.float32)
    x, w = _scaled(x, w, scales)
    ref, floor = _conv64(x, w, 3, 1, 1)
    for form in FORMS:
        _check(api.forward(form, x, w, 3, 1, 1), ref, floor)
    # the same operands as an input gradient's: dy = x, and a weight whose rows are the columns above
    wt = np.ascontiguousarray(w.reshape(9, 40, 48).transpose(0, 2, 1)).reshape(9 * 48, 40)
    ref, floor = _dgrad64(x, wt, (2, 7, 8, 48), 3, 1)
    for form in FORMS:
        _check(api.input_grad(form, x, wt, (2, 7, 8, 48), 3, 1), ref, floor)
    # and as a weight gradient's: channels of x and of dy
    a = rng.standard_normal((3, 9, 8, 40)).astype(np.float32)
    d = rng.standard_normal((3, 9, 8, 48)).astype(np.float32)
    for t, f in ((a, scales[0]), (d, scales[1])):
        for c in range(t.shape[-1]):
            t[..., c] *= np.float32(f[c % len(f)] if isinstance(f, tuple) else f)
    ref, floor = _wgrad64(a, d, 3, 1, 1)
    for form in LOADS:
        _check(api.weight_grad(form, a, d, 3, 1, 1)[0], ref, floor)


@pytest.mark.parametrize("form", [(32, HALO), (64, GATHER), (128, HALO), (128, RAGGED)], ids=lambda f: f"{f[0]}-{f[1]}")
def test_outputs_are_not_shifted(api, rng, form):
    """As in test_gpu_conv_split.py, for the tiled kernel: the mean error within 4 standard errors plus 3e-9, the rms
    below a plain fp32 sum's."""
    print(f"[case] conv mean error, form {form}", flush=True)
    x = rng.standard_normal((4, 32, 32, 128)).astype(np.float32)
    w = (rng.standard_normal((9 * 128, 128)) / 34).astype(np.float32)
    ref, _ = _conv64(x, w, 3, 1, 1)
    err = (api.forward(form, x, w, 3, 1, 1) - ref) / np.sqrt(np.mean(ref * ref))
    print(f"mean {err.mean():.2e} rms {np.sqrt(np.mean(err * err)):.2e}", flush=True)
    assert abs(err.mean()) <= 4.4e-9
    assert np.sqrt(np.mean(err * err)) <= 6.1e-7


@pytest.mark.parametrize("form", [(n, m) for n in (32, 64, 128) for m in (HALO, GATHER)], ids=lambda f: f"{f[0]}-{f[1]}")
def test_fused_epilogues_of_the_tiled_forms(api, L, nn, rng, form):
    """Against the separate launches, bit for bit, with rows and columns that end within a tile."""
    print(f"[case] fused epilogues, form {form}", flush=True)
    B, H, W, Ci, Co, K, p = 3, 9, 7, 24, 72, 3, 1
    n, ni = B * H * W * Co, B * H * W * Ci
    d = api.d

    def dev(*shape, scale=1.0):
        return L.to_device((scale * rng.standard_normal(shape)).astype(np.float32))

    xd, wd, gd, cond, res, resi, act = dev(ni), dev(K * K * Ci, Co, scale=0.1), dev(n), dev(B, Co, scale=0.5), dev(n), dev(ni), dev(ni)
    gain = L.to_device(np.array([0.91], np.float32))
    y, want, got, y2, dx, t = L.alloc(n), L.alloc(n), L.alloc(n), L.alloc(n), L.alloc(ni), L.alloc(ni)
    geo = (B, H, W, Ci, Co, K, 1, p, H, W)
    d.nnk_conv_forward_as(*form, y.p, xd.p, wd.p, None, gain.p, *geo, None, None)
    for a in (nn.ACT_SILU, nn.ACT_MP_SILU):
        f = nn.NnConvFusion(cond=cond.p, y2=y2.p, act=a)
        d.nnk_conv_forward_as(*form, got.p, xd.p, wd.p, None, gain.p, *geo, C.addressof(f), None)
        L.launch_spatial_modulate_act_forward(want.p, y.p, cond.p, B, H * W, 1, Co, a, None)
        api.done("modulate")
        assert_bits_equal(got.download(), y.download(), "y")
        assert_bits_equal(y2.download(), want.download(), "y2")
    f = nn.NnConvFusion(res=res.p, res_w=0.83, out_w=0.55)
    d.nnk_conv_forward_as(*form, got.p, xd.p, wd.p, None, gain.p, *geo, C.addressof(f), None)
    L.launch_weighted_sum(want.p, res.p, y.p, 0.83, 0.55, n, None)
    api.done("residual")
    assert_bits_equal(got.download(), want.download(), "residual")
    d.nnk_conv_input_grad_as(*form, dx.p, gd.p, wd.p, gain.p, B, H, W, Ci, Co, K, p, None, None)
    for a in (nn.ACT_SILU, nn.ACT_MP_SILU):
        f = nn.NnConvFusion(act_in=act.p, act=a, res=resi.p, res_w=0.83, out_w=1.0)
        d.nnk_conv_input_grad_as(*form, t.p, gd.p, wd.p, gain.p, B, H, W, Ci, Co, K, p, C.addressof(f), None)
        api.done("activation gradient")
        fused = t.download()
        L.launch_activation_backward(t.p, dx.p, act.p, ni, a, None)
        L.launch_weighted_sum(t.p, resi.p, t.p, 0.83, 1.0, ni, None)
        api.done("separate")
        assert_bits_equal(fused, t.download(), "input gradient")


def test_which_form_the_calls_take(api):
    """The shapes whose kernels the tests above stand for."""
    tile, tiled = api.d.nnk_conv_tile, api.d.nnk_conv_weight_grad_tiled
    assert tile(16, 64, 64, 256, 256, 3, 1, 1, 0) == 128       # a full level: halo rows
    assert tile(32, 64, 64, 64, 128, 3, 2, 1, 0) == 64          # between levels: gathered rows
    assert tile(64, 32, 32, 3, 64, 3, 1, 1, 0) in (32, 64)      # three channels: ragged
    assert tile(8, 7, 7, 128, 128, 3, 1, 1, 0) == 0
    assert tile(8, 7, 7, 128, 128, 3, 1, 1, 1) == 0
    assert tiled(16, 64, 64, 256, 256, 3, 1, 1) and tiled(64, 32, 32, 3, 64, 3, 1, 1)
    assert not tiled(8, 7, 7, 128, 128, 3, 1, 1) and not tiled(128, 1, 1, 512, 512, 1, 1, 0)
