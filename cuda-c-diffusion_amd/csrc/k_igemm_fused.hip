// k_igemm_fused.hip -- the implicit-GEMM convolutions with a neighbouring pass
// of the diffusion blocks folded in, so that the tensor between the two is
// never written to HBM or read back:
//   forward + residual        y = wa res + wb conv           (src/cond_conv_residual.c:34-35,
//                                                              src/conv_residual.c:38-39)
//   forward + modulate + act  y = conv, y2 = act(y (c + 1))  (src/cond_conv_residual.c:29, 31-33)
//   input gradient + act' + residual
//                             dx = wa res + 1 (conv^T(dy) act'(x))
//                                                            (src/cond_conv_residual.c:53-54, 61)
// The kernels are those of k_igemm.hip (igemm.h) with the pass in the
// epilogue; each computes with the replaced pass's operation order, so the
// outputs equal the separate launches' bit for bit.  Only these combinations
// are built.
#include "igemm.h"

namespace {

bool act_fusable(int act) { return act == ACT_SILU || act == ACT_MP_SILU; }

}  // namespace

void nnk_conv_forward_fused(float* Y, const float* X, const float* Wt, const ConvShape& sh, ConvEpi ep,
    const NnConvFusion& f, hipStream_t s, ConvPick pick) {
    ep.res = f.res;
    ep.wa = f.res_w;
    ep.wb = f.out_w;
    ep.cond = f.cond;
    ep.y2 = f.y2;
    ep.hw = FastDiv((uint32_t)(sh.Ho * sh.Wo));
    ep.mp = f.act == ACT_MP_SILU;
    if (f.res) conv_launch<false, kXeRes>(Y, X, Wt, sh, ep, s, pick);
    else conv_launch<false, kXeMod>(Y, X, Wt, sh, ep, s, pick);
}

void nnk_conv_input_grad_fused(float* dX, const float* dY, const float* Wt, const ConvShape& sh, ConvEpi ep,
    const NnConvFusion& f, hipStream_t s, ConvPick pick) {
    ep.res = f.res;
    ep.xa = f.act_in;
    ep.wa = f.res_w;
    ep.wb = f.out_w;
    ep.mp = f.act == ACT_MP_SILU;
    conv_launch<true, kXeActG | kXeRes>(dX, dY, Wt, sh, ep, s, pick);
}

extern "C" {

void launch_conv2d_forward_implicit_fused(float* Y, const float* X, const float* Wt, const float* bias,
    const float* gain, int batch, int H, int W, int C_in, int C_out, int K, int stride, int pad, int H_out,
    int W_out, const NnConvFusion* f, hipStream_t s) {
    const char* what = "launch_conv2d_forward_implicit_fused";
    NNK_REQUIRE(f, what, "%s: null fusion", what);
    NNK_REQUIRE(!f->act_in, what, "%s: act_in belongs to the input gradient", what);
    NNK_REQUIRE((f->res != nullptr) != (f->cond != nullptr), what,
        "%s: exactly one of res (residual) and cond (modulate + activation) is fused", what);
    if (f->cond) {
        NNK_REQUIRE(act_fusable(f->act), what, "%s: the modulate epilogue takes ACT_SILU or ACT_MP_SILU, not %d",
            what, (int)f->act);
    }
    ConvShape sh;
    if (fwd_setup(what, Y, X, Wt, bias, gain, batch, H, W, C_in, C_out, K, stride, pad, H_out, W_out, sh) <= 0)
        return;
    NNK_REQUIRE(!f->cond || f->y2, what, "%s: null y2", what);
    ConvEpi ep{};
    ep.bias = bias;
    ep.gain = gain;
    nnk_conv_forward_fused(Y, X, Wt, sh, ep, *f, s);
    nnk_after_launch(what, s);
}

void launch_conv2d_input_grad_implicit_fused(float* dX, const float* dY, const float* Wt, const float* gain,
    int batch, int H, int W, int C_in, int C_out, int K, int pad, const NnConvFusion* f, hipStream_t s) {
    const char* what = "launch_conv2d_input_grad_implicit_fused";
    NNK_REQUIRE(f, what, "%s: null fusion", what);
    NNK_REQUIRE(!f->cond && !f->y2, what, "%s: cond and y2 belong to the forward", what);
    NNK_REQUIRE(f->act_in && f->res, what, "%s: builds act_in with res", what);
    NNK_REQUIRE(act_fusable(f->act), what,
        "%s: the activation-gradient epilogue takes ACT_SILU or ACT_MP_SILU, not %d", what, (int)f->act);
    ConvShape sh;
    if (dgrad_setup(what, dX, dY, Wt, batch, H, W, C_in, C_out, K, pad, sh) <= 0) return;
    ConvEpi ep{};
    ep.gain = gain;
    nnk_conv_input_grad_fused(dX, dY, Wt, sh, ep, *f, s);
    nnk_after_launch(what, s);
}

}  // extern "C"
