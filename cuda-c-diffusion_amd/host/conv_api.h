/* conv_api.h -- the products inside the conv2d and linear modules, on the
 * matrix-core kernels (csrc/igemm.h, csrc/k_conv_small.hip).  Unlike the
 * launchers of nn_hip.h they take any channel counts and 4-byte alignment, and
 * pick the tiled or the small-tile kernels by the work's size.  A dense layer
 * is a convolution with H = W = K = 1.  Tensors below 2^31 elements, fewer than
 * 2^24 channels (nnk_conv_fits); errors go to the launch layer's record.
 */
#ifndef NN_CONV_API_H
#define NN_CONV_API_H

#include "nn_hip.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Whether every tensor of the convolution is within the kernels' index range. */
int nnk_conv_fits(int batch, int H, int W, int C_in, int C_out, int K, int H_out, int W_out);

/* y = conv(x) + bias | * gain[0], then the neighbour in f (may be NULL) as in
   launch_conv2d_forward_implicit_fused. */
void nnk_conv_forward(float* y, const float* x, const float* w, const float* bias, const float* gain, int batch,
    int H, int W, int C_in, int C_out, int K, int stride, int pad, int H_out, int W_out, const NnConvFusion* f,
    hipStream_t s);
/* dx of a stride-1 convolution with pad <= K - 1, * gain[0]; f (may be NULL) as
   in launch_conv2d_input_grad_implicit_fused. */
void nnk_conv_input_grad(float* dx, const float* dy, const float* w, const float* gain, int batch, int H, int W,
    int C_in, int C_out, int K, int pad, const NnConvFusion* f, hipStream_t s);
/* Whether that is faster as the product dy w^T (a dense layer's input gradient
   with C_in * K * K inputs, into batch * H_out * W_out rows of memory of the
   caller's) and launch_col2im_set. */
int nnk_conv_input_grad_by_columns(int batch, int H, int W, int C_in, int C_out, int K, int pad);
/* gw, and with gb non-NULL the column sums of dy.  workspace:
   nnk_conv_weight_grad_workspace floats, enough for every smaller batch. */
void nnk_conv_weight_grad(float* gw, float* gb, const float* x, const float* dy, int batch, int H, int W, int C_in,
    int C_out, int K, int stride, int pad, int H_out, int W_out, float* workspace, hipStream_t s);
size_t nnk_conv_weight_grad_workspace(int batch, int C_in, int C_out, int K, int H_out, int W_out);
/* Which kernel a forward takes (flip: an input gradient, given as the convolution
   of dy with the flipped kernel): 128, 64 or 32 columns a workgroup, 0 the small
   tiles; whether a weight gradient takes the tiled kernel. */
int nnk_conv_tile(int batch, int H, int W, int C_in, int C_out, int K, int stride, int pad, int flip);
int nnk_conv_weight_grad_tiled(int batch, int H, int W, int C_in, int C_out, int K, int stride, int pad);
/* The three products in a named form, for tests: columns as nnk_conv_tile gives
   them, tiled as nnk_conv_weight_grad_tiled, staging 0 halo rows, 1 gathered, 2
   ragged, loads 0 fours, 1 pairs, 2 singles of pixels (a more special one than the
   shape allows is not taken); negative: as the call without a name. */
void nnk_conv_forward_as(int columns, int staging, float* y, const float* x, const float* w, const float* bias,
    const float* gain, int batch, int H, int W, int C_in, int C_out, int K, int stride, int pad, int H_out, int W_out,
    const NnConvFusion* f, hipStream_t s);
void nnk_conv_input_grad_as(int columns, int staging, float* dx, const float* dy, const float* w, const float* gain,
    int batch, int H, int W, int C_in, int C_out, int K, int pad, const NnConvFusion* f, hipStream_t s);
void nnk_conv_weight_grad_as(int tiled, int loads, float* gw, float* gb, const float* x, const float* dy, int batch,
    int H, int W, int C_in, int C_out, int K, int stride, int pad, int H_out, int W_out, float* workspace,
    hipStream_t s);
/* The same sums on the fp32 matrix cores, for conv2d modules with a gain
   (csrc/k_igemm_f32.hip says why): channel counts, alignment and index range as
   the launchers of nn_hip.h, outputs times gain[0].  f (may be NULL): res, or cond
   and y2 with MP-SiLU; for the input gradient act_in with MP-SiLU, and res.
   workspace as above. */
void nnk_conv_f32_forward(float* y, const float* x, const float* w, const float* gain, int batch, int H, int W,
    int C_in, int C_out, int K, int stride, int pad, int H_out, int W_out, const NnConvFusion* f, hipStream_t s);
void nnk_conv_f32_input_grad(float* dx, const float* dy, const float* w, const float* gain, int batch, int H, int W,
    int C_in, int C_out, int K, int pad, const NnConvFusion* f, hipStream_t s);
void nnk_conv_f32_weight_grad(float* gw, const float* x, const float* dy, int batch, int H, int W, int C_in,
    int C_out, int K, int stride, int pad, int H_out, int W_out, float* workspace, hipStream_t s);
size_t nnk_conv_f32_weight_grad_workspace(int batch, int C_in, int C_out, int K, int H_out, int W_out);
/* launch_weight_normalize_backward_ws with *g_gain overwritten. */
void nnk_weight_normalize_backward_set(float* gW, const float* Wn, const float* gain, float* g_gain, int in,
    int out, float* workspace, hipStream_t s);

#ifdef __cplusplus
}
#endif

#endif /* NN_CONV_API_H */
