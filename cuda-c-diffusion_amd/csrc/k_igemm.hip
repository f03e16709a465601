// k_igemm.hip -- NHWC convolution forward as an implicit GEMM on the matrix
// cores, replacing im2col + GEMM + bias/gain pass of the reference's conv2d
// forward (src/conv2d.c:17-34: launch_im2col, gemm_forward, launch_add_bias or
// launch_scale_by_scalar), the stride-1 input gradient as the same kernel over
// dy with the kernel flipped (replacing gemm_dX + col2im, src/conv2d.c:48-65),
// and the weight gradient (src/conv2d.c:44-47).
//
//   Y[m, n] = sum_k A[m, k] Wt[k, n]  (+ bias[n] | * gain[0])
//   m = (b, oh, ow), k = (kh, kw, ci), A[m, k] = X[b, oh s + kh - p, ow s + kw - p, ci]
//   (0 outside the image), Wt = the reference's [K*K*C_in, C_out] weight.
//
// The im2col matrix is never written and the weight is read in the reference's
// layout, with no transposed, flipped or converted copy in memory.
//
// fp32 products on the bf16 matrix cores.  v_mfma_f32_32x32x2f32 holds 134
// TFLOP/s here, v_mfma_f32_32x32x16_bf16 1780 (register-only loops, 512
// workgroups): 13 times.  Each fp32 operand is split exactly into three bf16
// planes and six of the nine plane products are formed (conv_common.h), 297
// TFLOP/s of fp32 products at most.  With data from memory a large bf16 product of
// the vendor library holds 1250 TFLOP/s, because the clock falls to 1.7 GHz under
// that load, so 208 is what to expect.  Measured, each kernel by itself: 3x3, 128 ->
// 128 at [128, 32, 32] forward 320 -> 184 us (210 TFLOP/s), 256 -> 256 at [16, 64,
// 64] 627 -> 355 us (218), their input gradients 317 -> 188 and 620 -> 358 us, their
// weight gradients (with the sum of the splits) 337 -> 227 and 657 -> 442 us, 5 %
// more on boxes that clock lower; the forward's matrix cores are busy 0.69 of the
// time at 1.67 GHz, the weight gradient's 0.46 (it splits each operand
// again in all nine k tiles, and decodes pixels).  On the way: the fp32 kernel's
// staging (both operands through LDS per tap, a split of each) 230-260 us;
// activations staged once per 32 channels for all taps, weights split in
// registers by the one wave that needs them 205-214; the next step's loads and
// splits between the MFMAs 184-191.  Error against 64 bits: below the fp32 MFMA's
// at every size measured (conv_common.h).  Convolutions with a trained gain stay on
// the fp32 MFMA all the same (k_igemm_f32.hip).
//
// Lane layout of v_mfma_f32_32x32x16_bf16 (checked on the device): lane l
// supplies A[l % 32][8 (l / 32) .. + 7] and B[8 (l / 32) .. + 7][l % 32];
// accumulator register r of lane l holds D[8 (r / 4) + 4 (l / 32) + r % 4][l %
// 32].
//
// Summation order: each output is a fixed-order sum, the same on every run: in the
// tiled kernels (igemm.h) slices of 32 channels, taps, halves of 16, in every staging
// form; in the small tiles (k_conv_small.hip) a wave's taps and channels, then the
// waves.  Which of them a shape takes is fixed too (conv_tile, small_us).  Orders
// differ from each other and from a library GEMM's by rounding only.
#include "igemm.h"

#include "conv_api.h"

extern "C" {

int nnhip_conv2d_implicit_supported(int C_in, int C_out) {
    return C_in > 0 && C_out > 0 && C_in % kBK == 0 && C_out % kBNmin == 0;
}

void launch_conv2d_forward_implicit(float* Y, const float* X, const float* Wt, const float* bias,
    const float* gain, int batch, int H, int W, int C_in, int C_out, int K, int stride, int pad, int H_out,
    int W_out, hipStream_t s) {
    const char* what = "launch_conv2d_forward_implicit";
    ConvShape sh;
    if (fwd_setup(what, Y, X, Wt, bias, gain, batch, H, W, C_in, C_out, K, stride, pad, H_out, W_out, sh) <= 0)
        return;
    ConvEpi ep{};
    ep.bias = bias;
    ep.gain = gain;
    conv_launch<false, kXeNone>(Y, X, Wt, sh, ep, s);
    nnk_after_launch(what, s);
}

int nnhip_conv2d_input_grad_implicit_supported(int C_in, int C_out, int K, int stride, int pad) {
    return stride == 1 && K > 0 && pad >= 0 && pad <= K - 1 && nnhip_conv2d_implicit_supported(C_out, C_in);
}

void launch_conv2d_input_grad_implicit(float* dX, const float* dY, const float* Wt, const float* gain, int batch,
    int H, int W, int C_in, int C_out, int K, int pad, hipStream_t s) {
    const char* what = "launch_conv2d_input_grad_implicit";
    ConvShape sh;
    if (dgrad_setup(what, dX, dY, Wt, batch, H, W, C_in, C_out, K, pad, sh) <= 0) return;
    ConvEpi ep{};
    ep.gain = gain;
    conv_launch<true, kXeNone>(dX, dY, Wt, sh, ep, s);
    nnk_after_launch(what, s);
}

int nnhip_conv2d_wgrad_implicit_supported(int C_in, int C_out) {
    return C_in > 0 && C_out > 0 && C_in % 4 == 0 && C_out % kBNmin == 0;
}

size_t nnhip_conv2d_wgrad_workspace(int batch, int C_in, int C_out, int K, int H_out, int W_out) {
    if (batch <= 0 || !nnhip_conv2d_wgrad_implicit_supported(C_in, C_out)) return 0;
    const long long M = (long long)batch * H_out * W_out;
    if (M <= 0 || M >= (1LL << 31)) return 0;
    const int S = wgrad_most_splits((int)M, K * K * C_in, C_out);
    return S > 1 ? (size_t)S * K * K * C_in * C_out : 0;
}

void launch_conv2d_weight_grad_implicit(float* gW, const float* X, const float* dY, int batch, int H, int W,
    int C_in, int C_out, int K, int stride, int pad, int H_out, int W_out, float* workspace, hipStream_t s) {
    wgrad_launch("launch_conv2d_weight_grad_implicit", gW, X, dY, batch, H, W, C_in, C_out, K, stride, pad, H_out,
        W_out, workspace, s);
}

// ---- the host modules' products (conv_api.h) ----

int nnk_conv_fits(int batch, int H, int W, int C_in, int C_out, int K, int H_out, int W_out) {
    const long long most = 1LL << 31, kk = (long long)K * K * C_in;
    return C_in < kMostChannels && C_out < kMostChannels && kk < kMostIndex && kk * C_out < most &&
           (long long)batch * H * W < kMostIndex && (long long)batch * H * W * C_in < most &&
           (long long)batch * H_out * W_out < kMostIndex && (long long)batch * H_out * W_out * C_out < most;
}

void nnk_conv_forward_as(int columns, int staging, float* y, const float* x, const float* w, const float* bias,
    const float* gain, int batch, int H, int W, int C_in, int C_out, int K, int stride, int pad, int H_out, int W_out,
    const NnConvFusion* f, hipStream_t s) {
    const char* what = "conv2d forward";
    NNK_REQUIRE(nnk_conv_fits(batch, H, W, C_in, C_out, K, H_out, W_out), what, "%s: tensor exceeds the 32-bit index range", what);
    if (batch <= 0) return;
    const ConvShape sh{batch, H, W, C_in, C_out, K, stride, pad, H_out, W_out, batch * H_out * W_out, K * K * C_in,
        FastDiv((uint32_t)W_out), FastDiv((uint32_t)H_out)};
    ConvEpi ep{};
    ep.bias = bias;
    ep.gain = gain;
    const ConvPick pick{columns, staging};
    if (f) nnk_conv_forward_fused(y, x, w, sh, ep, *f, s, pick);
    else conv_launch<false, kXeNone>(y, x, w, sh, ep, s, pick);
    nnk_after_launch(what, s);
}

void nnk_conv_forward(float* y, const float* x, const float* w, const float* bias, const float* gain, int batch,
    int H, int W, int C_in, int C_out, int K, int stride, int pad, int H_out, int W_out, const NnConvFusion* f,
    hipStream_t s) {
    nnk_conv_forward_as(-1, -1, y, x, w, bias, gain, batch, H, W, C_in, C_out, K, stride, pad, H_out, W_out, f, s);
}

int nnk_conv_tile(int batch, int H, int W, int C_in, int C_out, int K, int stride, int pad, int flip) {
    const int Ho = (H + 2 * pad - K) / stride + 1, Wo = (W + 2 * pad - K) / stride + 1;
    return conv_tile(ConvShape{batch, H, W, C_in, C_out, K, stride, pad, Ho, Wo, batch * Ho * Wo, K * K * C_in,
        FastDiv((uint32_t)Wo), FastDiv((uint32_t)Ho)}, flip != 0);
}

int nnk_conv_weight_grad_tiled(int batch, int H, int W, int C_in, int C_out, int K, int stride, int pad) {
    const int Ho = (H + 2 * pad - K) / stride + 1, Wo = (W + 2 * pad - K) / stride + 1;
    return !wgrad_small_wins(ConvShape{batch, H, W, C_in, C_out, K, stride, pad, Ho, Wo, batch * Ho * Wo, K * K * C_in,
        FastDiv((uint32_t)Wo), FastDiv((uint32_t)Ho)});
}

static ConvShape dgrad_shape(int batch, int H, int W, int C_in, int C_out, int K, int pad) {
    return ConvShape{batch, H + 2 * pad - K + 1, W + 2 * pad - K + 1, C_out, C_in, K, 1, K - 1 - pad, H, W,
        batch * H * W, K * K * C_out, FastDiv((uint32_t)W), FastDiv((uint32_t)H)};
}

// With few input channels the direct kernel's columns are mostly padding (its
// tiles have 32 or 16), K * K times over; the product dY W^T has K * K * C_in of
// them.  Times in us: conv_tile's of both products, and for the pass that sums
// the columns a launch and its bytes at 4.5 TB/s; a quarter and 2 us of margin,
// for the fit and the buffer.  Direct / by columns measured: 3x3 3 -> 64 [64, 32,
// 32] 22.5 / 18.7, 16 -> 64 22 / 38; 8 -> 64 [28, 56, 57] 27 / 43; 128 -> 128 [8, 7,
// 7] 6.6 / 15.5; 5x5 8 -> 448 [53, 11, 11] 68 / 43, 16 -> 256 [43, 14, 14] 67 / 40.
int nnk_conv_input_grad_by_columns(int batch, int H, int W, int C_in, int C_out, int K, int pad) {
    const int Ho = H + 2 * pad - K + 1, Wo = W + 2 * pad - K + 1;
    const long long rows = (long long)batch * Ho * Wo, kg = (long long)K * K * C_in;
    if (K == 1 || rows <= 0 || rows >= (1LL << 31) || !nnk_conv_fits((int)rows, 1, 1, (int)kg, C_out, 1, 1, 1)) return 0;
    double direct, product;
    conv_tile(dgrad_shape(batch, H, W, C_in, C_out, K, pad), true, &direct);
    conv_tile(dgrad_shape((int)rows, 1, 1, (int)kg, C_out, 1, 0), true, &product);
    const double pass = 3.0 + 4.0 * ((double)rows * kg + (double)batch * H * W * C_in) / 4.5e6;
    return 1.25 * (product + pass) + 2.0 < direct;
}

void nnk_conv_input_grad_as(int columns, int staging, float* dx, const float* dy, const float* w, const float* gain,
    int batch, int H, int W, int C_in, int C_out, int K, int pad, const NnConvFusion* f, hipStream_t s) {
    const char* what = "conv2d input gradient";
    NNK_REQUIRE(nnk_conv_fits(batch, H, W, C_in, C_out, K, H + 2 * pad - K + 1, W + 2 * pad - K + 1), what, "%s: tensor exceeds the 32-bit index range", what);
    if (batch <= 0) return;
    const ConvShape sh = dgrad_shape(batch, H, W, C_in, C_out, K, pad);
    ConvEpi ep{};
    ep.gain = gain;
    const ConvPick pick{columns, staging};
    if (f) nnk_conv_input_grad_fused(dx, dy, w, sh, ep, *f, s, pick);
    else conv_launch<true, kXeNone>(dx, dy, w, sh, ep, s, pick);
    nnk_after_launch(what, s);
}

void nnk_conv_input_grad(float* dx, const float* dy, const float* w, const float* gain, int batch, int H, int W,
    int C_in, int C_out, int K, int pad, const NnConvFusion* f, hipStream_t s) {
    nnk_conv_input_grad_as(-1, -1, dx, dy, w, gain, batch, H, W, C_in, C_out, K, pad, f, s);
}

size_t nnk_conv_weight_grad_workspace(int batch, int C_in, int C_out, int K, int H_out, int W_out) {
    const long long M = (long long)batch * H_out * W_out;
    if (M <= 0 || M >= (1LL << 31)) return 0;
    const int S = wgrad_most_splits((int)M, K * K * C_in, C_out);
    return S > 1 ? (size_t)S * (K * K * C_in + 1) * C_out : 0;
}

void nnk_conv_weight_grad_as(int tiled, int loads, float* gw, float* gb, const float* x, const float* dy, int batch,
    int H, int W, int C_in, int C_out, int K, int stride, int pad, int H_out, int W_out, float* workspace,
    hipStream_t s) {
    const char* what = "conv2d weight gradient";
    NNK_REQUIRE(nnk_conv_fits(batch, H, W, C_in, C_out, K, H_out, W_out), what, "%s: tensor exceeds the 32-bit index range", what);
    const int KKC = K * K * C_in;
    if (batch <= 0) {
        nnhip_fill_f32(gw, 0.0f, (size_t)KKC * C_out, s);
        if (gb) nnhip_fill_f32(gb, 0.0f, (size_t)C_out, s);
        return;
    }
    const ConvShape sh{batch, H, W, C_in, C_out, K, stride, pad, H_out, W_out, batch * H_out * W_out, KKC,
        FastDiv((uint32_t)W_out), FastDiv((uint32_t)H_out)};
    if (tiled < 0 ? wgrad_small_wins(sh) : !tiled) {
        nnk_wgrad_small(gw, gb, x, dy, sh, s);
    } else if (const size_t n = workspace || !nnk_capturing(s) ? 0 : wgrad_scratch(sh, gb != nullptr)) {
        // A capture cannot allocate: the block that the same call left on the stream
        // when it ran eagerly, so that a replay gives what it gave, bit for bit; a
        // stream that has none takes the small tiles, which need none.
        float* part = nnk_scratch_cached(n, s);
        if (part) wgrad_run(what, gw, gb, x, dy, sh, part, s, ConvPick{-1, loads});
        else nnk_wgrad_small(gw, gb, x, dy, sh, s);
        nnk_scratch_release(part, s);
    } else {
        wgrad_run(what, gw, gb, x, dy, sh, workspace, s, ConvPick{-1, loads});
    }
    nnk_after_launch(what, s);
}

void nnk_conv_weight_grad(float* gw, float* gb, const float* x, const float* dy, int batch, int H, int W, int C_in,
    int C_out, int K, int stride, int pad, int H_out, int W_out, float* workspace, hipStream_t s) {
    nnk_conv_weight_grad_as(-1, -1, gw, gb, x, dy, batch, H, W, C_in, C_out, K, stride, pad, H_out, W_out, workspace, s);
}

}  // extern "C"
