"""GroupNorm of channel counts and alignments the float4 kernels do not take
(csrc/k_gn_slab.hip), against the CPU oracle at the bars of
test_gpu_groupnorm.py, at the edges of its plan: slabs of one and many groups,
a last slab with fewer groups, more pixels than the registers hold, channels
per group up to the limit and past it, misaligned tensors."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import TOL, gn_param_floor, rel_err
from test_gpu_groupnorm import make_inputs

pytestmark = pytest.mark.gpu

SHAPES = [
    # B, H, W, C, G, offset in floats
    (24, 28, 28, 96, 32, 0),    # 3 channels per group, 784 pixels
    (3, 5, 7, 15, 5, 0),        # a few values per thread
    (2, 33, 31, 66, 22, 0),     # slabs that do not divide the groups
    (40, 9, 9, 64, 32, 0),      # 2 channels per group, wide slabs
    (1, 1, 1, 6, 3, 0),         # one pixel
    (2, 64, 64, 80, 8, 0),      # 10 channels per group: past the registers
    (1, 70, 70, 24, 2, 0),      # 12, a slab of one group past the registers
    (2, 3, 3, 1000, 1, 0),      # a thread per channel
    (2, 3, 3, 1024, 1, 0),
    (2, 3, 3, 1025, 1, 0),      # past the limit: the generic kernels
    (3, 8, 8, 128, 32, 1),      # 4 per group, not 16-byte aligned
]


@pytest.mark.parametrize("act", [0, 3, 2], ids=["identity", "silu", "gelu"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_groupnorm_slab(L, orc, rng, shape, act):
    B, H, W, C, G, off = shape
    print(f"[case] groupnorm slab {shape} act={act}", flush=True)
    x, gamma, beta, dy = make_inputs(rng, B, H, W, C)

    def dev(a):
        d = L.alloc(a.size + off)
        d.upload(np.concatenate([np.zeros(off, np.float32), a.ravel()]))
        return d

    xd, dyd, yd, dxd = dev(x), dev(dy), L.alloc(x.size + off), L.alloc(x.size + off)
    gd, bd, ggd, gbd = L.to_device(gamma), L.to_device(beta), L.alloc(C), L.alloc(C)
    mud, rsd = L.alloc(B * G), L.alloc(B * G)
    L.launch_groupnorm_act_forward(yd.offset(off), mud.p, rsd.p, xd.offset(off), gd.p, bd.p, B, H * W, C, G, 1e-5, act,
                                   None)
    L.launch_groupnorm_act_backward(dxd.offset(off), ggd.p, gbd.p, dyd.offset(off), xd.offset(off), gd.p, bd.p, mud.p,
                                    rsd.p, B, H * W, C, G, act, None)
    L.sync()
    y_ref, mu_ref, rs_ref = orc.groupnorm_forward(x, gamma, beta, G, 1e-5, act)
    dx_ref, gg_ref, gb_ref = orc.groupnorm_backward(dy, x, gamma, beta, mu_ref, rs_ref, G, act)
    if H * W * (C // G) > 2:  # two values have a variance of rounding
        assert rel_err(yd.download()[off:].reshape(x.shape), y_ref) <= TOL
        assert rel_err(dxd.download()[off:].reshape(x.shape), dx_ref, floor=np.sqrt(np.mean(dy * dy))) <= TOL
    assert rel_err(mud.download(), mu_ref.ravel(), floor=1.0 / np.sqrt(H * W * (C // G))) <= TOL
    v = x.reshape(B, H * W, G, C // G).astype(np.float64)
    xhat = ((v - v.mean((1, 3), keepdims=True)) / np.sqrt(v.var((1, 3), keepdims=True) + 1e-5)).reshape(x.shape)
    fg, fb = gn_param_floor(dy, xhat, C)
    assert rel_err(ggd.download(), gg_ref, floor=fg) <= TOL
    assert rel_err(gbd.download(), gb_ref, floor=fb) <= TOL
