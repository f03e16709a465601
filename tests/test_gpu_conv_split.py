"""Where the split of fp32 operands into bf16 planes can go wrong, in the
convolutions' matrix-core kernels: operands that are infinite, NaN or so large
that they round to infinity in bf16, operands too small for the split, a mean
error that sums would show, and the edges of the staging (halo rows at image
borders and between samples, tiles past the end, widths that leave the halo
form), by the launchers and so in the form that the rules choose: for shapes as
small as these the small tiles.  test_gpu_conv_forms.py runs them in every form.
Reference: the same sums in double.  Bar for finite values as in
test_gpu_conv_implicit.py: 1e-5 relative to max(|ref|, sqrt(sum of the squared
products))."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import TOL

pytestmark = pytest.mark.gpu


def _conv64(x, w, K, s, p):
    """[B, H, W, Ci] * [K*K*Ci, Co] -> (y, root sum of the squared products) in double"""
    x, w = x.astype(np.float64), w.astype(np.float64)
    B, H, W, Ci = x.shape
    Ho, Wo = (H + 2 * p - K) // s + 1, (W + 2 * p - K) // s + 1
    xp = np.pad(x, ((0, 0), (p, p), (p, p), (0, 0)))
    y = sq = 0.0
    for t in range(K * K):
        i, j = divmod(t, K)
        a = xp[:, i:i + s * (Ho - 1) + 1:s, j:j + s * (Wo - 1) + 1:s].reshape(-1, Ci)
        b = w[t * Ci:(t + 1) * Ci]
        y, sq = y + a @ b, sq + (a * a) @ (b * b)
    return y, np.sqrt(sq)


def _forward(L, x, w, K, s, p):
    B, H, W, Ci = x.shape
    Co = w.shape[1]
    Ho, Wo = (H + 2 * p - K) // s + 1, (W + 2 * p - K) // s + 1
    xd, wd, yd = L.to_device(x), L.to_device(w), L.alloc(B * Ho * Wo * Co)
    L.launch_conv2d_forward_implicit(yd.p, xd.p, wd.p, None, None, B, H, W, Ci, Co, K, s, p, Ho, Wo, None)
    L.sync()
    return yd.download(shape=(B * Ho * Wo, Co)).astype(np.float64)


def _wgrad(L, x, dy, K, p):
    B, H, W, Ci = x.shape
    Co = dy.shape[-1]
    xd, dd, gw = L.to_device(x), L.to_device(dy), L.alloc(K * K * Ci * Co)
    L.launch_conv2d_weight_grad_implicit(gw.p, xd.p, dd.p, B, H, W, Ci, Co, K, 1, p, H, W, None, None)
    L.sync()
    return gw.download(shape=(K * K * Ci, Co)).astype(np.float64)


def _check(got, ref, floor):
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    inf = np.isinf(ref)
    assert np.array_equal(got[inf], ref[inf])
    fine = np.isfinite(ref)
    err = np.abs(got - ref)[fine] / np.maximum(np.maximum(np.abs(ref), floor)[fine], 1e-44)
    assert float(err.max()) <= TOL


STAGING = [
    # B, H, W, C_in, C_out, K, stride, pad: halo rows across samples and image borders
    (3, 5, 3, 32, 64, 3, 1, 1),     # images smaller than a tile
    (1, 43, 3, 64, 64, 3, 1, 1),    # 129 rows: the second tile has one
    (2, 4, 63, 32, 64, 5, 1, 2),    # the widest 5 x 5 halo
    (1, 4, 70, 32, 64, 5, 1, 2),    # ... and past it: rows gathered per tap
    (1, 3, 140, 32, 64, 3, 1, 1),
    (2, 9, 7, 32, 64, 3, 1, 0),     # output smaller than the input
    (2, 9, 7, 32, 64, 7, 1, 3),     # more taps than bits
    (2, 6, 6, 40 * 4, 64, 1, 2, 0),
]


@pytest.mark.parametrize("geom", STAGING, ids=lambda g: "x".join(map(str, g)))
def test_staging_edges(L, rng, geom):
    B, H, W, Ci, Co, K, s, p = geom
    print(f"[case] conv staging {geom}", flush=True)
    x = rng.standard_normal((B, H, W, Ci)).astype(np.float32)
    w = (rng.standard_normal((K * K * Ci, Co)) / np.sqrt(K * K * Ci)).astype(np.float32)
    _check(_forward(L, x, w, K, s, p), *_conv64(x, w, K, s, p))


@pytest.mark.parametrize("stride", [1, 2])
def test_values_outside_the_split(L, rng, stride):
    """Infinities and NaN give what fp32 gives; 3e38 rounds to infinity in bf16
    and stays finite in the product."""
    print(f"[case] conv with inf, nan and huge operands, stride {stride}", flush=True)
    B, H, W, Ci, Co, K, p = 4, 16, 16, 32, 64, 3, 1
    x = rng.standard_normal((B, H, W, Ci)).astype(np.float32)
    w = (np.abs(rng.standard_normal((K * K * Ci, Co))) + 0.1).astype(np.float32) * np.float32(1e-3)
    x[0, 3, 4, 5] = np.inf
    x[1, 0, 0, 0] = -np.inf
    x[1, 15, 15, 1] = np.nan
    x[2, 8, 8, 2] = 3.4e38
    x[3, 2, 2, 0], x[3, 2, 3, 0] = np.inf, -np.inf  # inf - inf where both are seen
    with np.errstate(invalid="ignore"):
        ref, floor = _conv64(x, w, K, stride, p)
        _check(_forward(L, x, w, K, stride, p), ref, np.where(np.isfinite(floor), floor, 0.0))
        if stride == 1:
            dy = (1e-3 * rng.standard_normal((B * H * W, Co))).astype(np.float32)  # 3.4e38 dy stays finite
            dy[7, 3] = np.inf
            # each infinite or NaN operand meets finite ones only in the columns it belongs to
            xt = x.copy()
            xt[~np.isfinite(xt)] = 1.0
            col = np.stack([np.pad(xt, ((0, 0), (1, 1), (1, 1), (0, 0)))[:, i:i + H, j:j + W].reshape(-1, Ci)
                            for i in range(3) for j in range(3)], 1).reshape(-1, 9 * Ci).astype(np.float64)
            d = dy.astype(np.float64)
            ref, floor = col.T @ d, np.sqrt((col * col).T @ (d * d))
            _check(_wgrad(L, xt, dy, K, p), ref, np.where(np.isfinite(floor), floor, 0.0))


@pytest.mark.parametrize("scale", [1e-36, 1e-33, 1e-30, 1e30])
def test_scales_outside_the_split(L, rng, scale):
    """Operands whose last plane would lie below the smallest bf16 (1e-36 and
    1e-33), and ranges well inside."""
    print(f"[case] conv at scale {scale}", flush=True)
    x = (rng.standard_normal((2, 8, 8, 64)) * scale).astype(np.float32)
    w = (rng.standard_normal((9 * 64, 128)) / 24).astype(np.float32)
    _check(_forward(L, x, w, 3, 1, 1), *_conv64(x, w, 3, 1, 1))


@pytest.mark.parametrize("images,weight", [((1.0, 1e-36), 1.0), ((1e-35, 1.0), 1.0), ((1e-36, 1e-36), 1e15), ((1.0, 1e-35), 1e12)],
                         ids=str)
def test_small_operands_beside_others(L, rng, images, weight):
    """Operands below the split's range where not all results are small: an image of
    them beside an ordinary one in the same tile, and against large weights."""
    print(f"[case] conv of images scaled by {images}, weight by {weight}", flush=True)
    x = rng.standard_normal((2, 5, 5, 64)).astype(np.float32)
    for b, f in enumerate(images):
        x[b] *= np.float32(f)
    w = (rng.standard_normal((9 * 64, 128)) / 24 * weight).astype(np.float32)
    _check(_forward(L, x, w, 3, 1, 1), *_conv64(x, w, 3, 1, 1))


def test_outputs_are_not_shifted(L, rng):
    """The matrix core cuts addends off towards minus infinity; with the small
    products in the large one's accumulator the mean of the outputs' errors is
    -6e-8 of their root mean square (the kernel's comment), with an accumulator
    of their own 2e-10.  Bar: 4 standard errors of the mean (rms error 2.5e-7
    over 524288 outputs: 1.4e-9) plus 3e-9."""
    print("[case] conv mean error", flush=True)
    x = rng.standard_normal((4, 32, 32, 128)).astype(np.float32)
    w = (rng.standard_normal((9 * 128, 128)) / 34).astype(np.float32)
    ref, _ = _conv64(x, w, 3, 1, 1)
    err = (_forward(L, x, w, 3, 1, 1) - ref) / np.sqrt(np.mean(ref * ref))
    print(f"mean {err.mean():.2e} rms {np.sqrt(np.mean(err * err)):.2e}", flush=True)
    assert abs(err.mean()) <= 4.4e-9
    # no further off than a plain fp32 sum of 1152 products (6.1e-7 with the fp32 MFMA)
    assert np.sqrt(np.mean(err * err)) <= 6.1e-7
