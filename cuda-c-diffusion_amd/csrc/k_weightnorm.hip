// k_weightnorm.hip -- forced unit-norm weight normalisation (forward, in place)
// and its backward with the gain gradient.
// Reference maths: src/kernels.cu:255-297 with launchers 330-344.
//
// W is [in, out] row-major and every output column j is normalised over its
// `in` rows.  A workgroup owns 16 whole columns with 64 lanes each (or 4, wn_cols):
// lane (r, c) walks rows r, r + 64, ... of its column and keeps up to 24 (64) of them
// in registers, all loaded at once; more are read again from cache, in batches.
// The work is one round trip of loads and one of stores, so what counts is that
// no round follows another.  Against 8 rows at a time, read twice: forward 19.9 ->
// 11.4 us and backward 35.9 -> 18.2 at [4032, 448], 6.6 -> 4.6 and 9.7 -> 6.7 at
// [1152, 128], 4.5 -> 4.6 and 8.3 -> 5.2 at [512, 512].  Neighbouring blocks share
// 128-byte lines, so they run on one XCD.
//
// The order of a column's sum is fixed and part of the results: the lane's rows
// one by one, then the lanes 4 q .. 4 q + 3 as a tree, then q = 0 .. 15 one by one;
// of the sum over the columns: 16 columns as a tree, of which wave lane l adds
// the blocks l, l + 64, ..., and a tree over the lanes.  A gain gradient is
// such a sum of terms of either sign, in which what is left can be a hundredth of
// what was added: another order is as right and a different number.
//   forward : column sum of squares, then W *= rsqrt(sum + eps)    (one launch;
//             the second read of W comes from cache)
//   backward: dot_j = <Wn_j, gW_j>, then gW = gain * (gW - dot_j Wn) (one
//             launch), and *g_gain += sum_j dot_j in a fixed order: with a
//             lent workspace the last workgroup to finish adds the
//             per-workgroup sums; otherwise a one-wave launch does (the
//             reference adds each column with atomicAdd).
#include "conv_api.h"
#include "nnk_common.h"

namespace {

using namespace nnk;

constexpr int kRows = 64;              // lanes of a column
constexpr int kMore = 8;               // rows in flight beyond those in registers
constexpr int kTree = 16;              // columns of a tree of the sum over columns

// Rows i0 + u kRows of this lane's column, 0 past the end.
template <int N>
__device__ __forceinline__ void column_rows(float (&v)[N], const float* __restrict__ A, int i0, int in, int out,
    int j) {
#pragma unroll
    for (int u = 0; u < N; ++u) {
        const int i = i0 + u * kRows;
        v[u] = i < in ? A[(size_t)i * out + j] : 0.0f;
    }
}

// Total of the lanes' s over the column (identical on all its lanes, in every
// wave).
template <int COLS>
__device__ __forceinline__ float column_total(float s, float (*l)[COLS]) {
    const int r = threadIdx.x / COLS, c = threadIdx.x % COLS;
    s += __shfl_xor(s, COLS, kWave);
    s += __shfl_xor(s, 2 * COLS, kWave);
    if (r % 4 == 0) l[r / 4][c] = s;
    __syncthreads();
    float t = l[0][c];
#pragma unroll
    for (int q = 1; q < kRows / 4; ++q) t += l[q][c];
    return t;
}

template <int COLS, int KEEP>
__global__ __launch_bounds__(kRows * COLS) void wn_forward(float* __restrict__ W, int in, int out, float eps) {
    __shared__ float l[kRows / 4][COLS];
    const int bid = xcd_swizzle(blockIdx.x, gridDim.x);
    const int i0 = threadIdx.x / COLS;
    const int j = bid * COLS + threadIdx.x % COLS, jc = min(j, out - 1);
    float v[KEEP], s = 0.0f;
    column_rows(v, W, i0, in, out, jc);
#pragma unroll
    for (int u = 0; u < KEEP; ++u) s += v[u] * v[u];
    for (int i = i0 + KEEP * kRows; i < in; i += kMore * kRows) {
        float x[kMore];
        column_rows(x, W, i, in, out, jc);
#pragma unroll
        for (int u = 0; u < kMore; ++u) s += x[u] * x[u];
    }
    const float inv = rsqrtf(column_total(s, l) + eps);
    if (j >= out) return;
#pragma unroll
    for (int u = 0; u < KEEP; ++u) {
        const int i = i0 + u * kRows;
        if (i < in) W[(size_t)i * out + j] = v[u] * inv;
    }
    for (int i = i0 + KEEP * kRows; i < in; i += kRows) W[(size_t)i * out + j] *= inv;
}

// The sum over the columns from the n workgroups' sums of 4 or 16 columns each (a
// wave; the order of the file's head).
__device__ __forceinline__ float blocks_total(const float* part, int n, int cols) {
    float t = 0.0f;
    for (int k = threadIdx.x & (kWave - 1); k * kTree < n * cols; k += kWave) {
        if (cols == kTree) {
            t += part[k];
        } else {
            float q[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) q[u] = 4 * k + u < n ? part[4 * k + u] : 0.0f;
            t += (q[0] + q[1]) + (q[2] + q[3]);
        }
    }
    return wave_sum(t);
}

// gW = gain * (gW - dot_j * Wn); part[b] = sum of block b's dot_j.
// kAddGain, kSetGain: the last workgroup to arrive (counter) adds part[0..gridDim.x)
// in index order to *g_gain, or to zero, and re-arms the counter.  A module's
// gain gradient is new in every backward pass: to set it saves the launch that
// cleared it (embedding MLP of two layers, 256 -> 512 -> 512 at batch 128:
// 59 -> 56 us a pass; convolution block [128, 32, 32, 128] 1400 -> 1375).
enum { kPartsOnly, kAddGain, kSetGain };
template <int COLS, int KEEP, int GAIN>
__global__ __launch_bounds__(kRows * COLS) void wn_backward(float* __restrict__ gW, const float* __restrict__ Wn,
    const float* __restrict__ gain, float* __restrict__ part, unsigned* __restrict__ counter,
    float* __restrict__ g_gain, int in, int out) {
    __shared__ float l[kRows / 4][COLS];
    __shared__ int last;
    const int bid = xcd_swizzle(blockIdx.x, gridDim.x);
    const int i0 = threadIdx.x / COLS;
    const int j = bid * COLS + threadIdx.x % COLS, jc = min(j, out - 1);
    float a[KEEP], b[KEEP], s = 0.0f;
    column_rows(a, gW, i0, in, out, jc);
    column_rows(b, Wn, i0, in, out, jc);
    const float g = gain[0];
#pragma unroll
    for (int u = 0; u < KEEP; ++u) s += b[u] * a[u];
    for (int i = i0 + KEEP * kRows; i < in; i += kMore * kRows) {
        float x[kMore], y[kMore];
        column_rows(x, gW, i, in, out, jc);
        column_rows(y, Wn, i, in, out, jc);
#pragma unroll
        for (int u = 0; u < kMore; ++u) s += y[u] * x[u];
    }
    const float dot = column_total(s, l);  // its barrier orders every read of gW before the writes below
    if (threadIdx.x < kWave) {
        // lanes 0..COLS-1 hold the block's column totals
        const float t = wave_sum(threadIdx.x < COLS && j < out ? dot : 0.0f);
        if (threadIdx.x == 0) part[bid] = t;
    }
    if constexpr (GAIN != kPartsOnly) {
        __syncthreads();
        if (threadIdx.x == 0) {
            __threadfence();  // this block's part is visible before it is counted
            last = atomicAdd(counter, 1u) == gridDim.x - 1;
        }
        __syncthreads();
        if (last && threadIdx.x < kWave) {
            __threadfence();  // every counted block's part is visible here
            const float t = blocks_total(part, (int)gridDim.x, COLS);
            if (threadIdx.x == 0) {
                g_gain[0] = (GAIN == kSetGain ? 0.0f : g_gain[0]) + t;
                *counter = 0u;
            }
        }
    }
    if (j < out) {
#pragma unroll
        for (int u = 0; u < KEEP; ++u) {
            const int i = i0 + u * kRows;
            if (i < in) gW[(size_t)i * out + j] = g * (a[u] - dot * b[u]);
        }
        for (int i = i0 + KEEP * kRows; i < in; i += kRows) {
            const size_t o = (size_t)i * out + j;
            gW[o] = g * (gW[o] - dot * Wn[o]);
        }
    }
}

// *g_gain += the sum over the columns (one wave).
__global__ __launch_bounds__(kWave) void wn_gain_sum(float* __restrict__ g_gain, const float* __restrict__ part,
    int n, int cols) {
    const float t = blocks_total(part, n, cols);
    if (threadIdx.x == 0) g_gain[0] = g_gain[0] + t;
}

// Columns per workgroup.  16 hold up to 24 rows a lane in registers (1024 threads);
// above, 4 hold 64 and spread a weight over four times the CUs, which wins until
// the workgroups' arrivals at one counter take longer (20 ns each).  Forward +
// backward in us with 16 / 4 columns: [512, 1024] 10.1 / 15.9, [256, 4096] 14.5 /
// 37.5, [2304, 512] 17.3 / 19.4, [4032, 1024] 33 / 38; [4032, 448] 36 / 30, [4096, 66]
// 45 / 24, [2304, 256] 16.7 / 16.6.
int wn_cols(int in, int out) { return in > 24 * kRows && out < 512 ? 4 : kTree; }
int wn_blocks(int out, int cols) { return (out + cols - 1) / cols; }

bool wn_backward_args(const char* what, float* gW, const float* Wn, const float* gain, float* g_gain, int in,
    int out) {
    NNK_REQUIRE_RET(in >= 0 && out >= 0, false, what, "%s: bad shape in=%d out=%d", what, in, out);
    if (out == 0) return false;
    NNK_REQUIRE_RET(gW && Wn && gain && g_gain, false, what, "%s: null pointer", what);
    return true;
}

// KERNEL<COLS, KEEP, ...> for the shape.  A lane keeps the rows of 512, 1536 or
// 4096 input rows in registers (fewer registers and loads to skip where the column
// is short; 1024 threads have room for 24).
#define NNK_WN(KERNEL, COLS_, KEEP_, ARGS, ...)                                                               \
    KERNEL<COLS_, KEEP_ __VA_ARGS__><<<dim3((unsigned)wn_blocks(out, COLS_)), kRows * COLS_, 0, s>>> ARGS
#define NNK_WN_LAUNCH(KERNEL, ARGS, ...)                                                 \
    do {                                                                                 \
        if (wn_cols(in, out) == 16) {                                                    \
            if (in <= 8 * kRows) NNK_WN(KERNEL, 16, 8, ARGS, __VA_ARGS__);               \
            else NNK_WN(KERNEL, 16, 24, ARGS, __VA_ARGS__);                              \
        } else if (in <= 8 * kRows) NNK_WN(KERNEL, 4, 8, ARGS, __VA_ARGS__);             \
        else if (in <= 24 * kRows) NNK_WN(KERNEL, 4, 24, ARGS, __VA_ARGS__);             \
        else NNK_WN(KERNEL, 4, 64, ARGS, __VA_ARGS__);                                   \
    } while (0)

}  // namespace

extern "C" {

void launch_weight_normalize(float* W, int in, int out, float eps, hipStream_t s) {
    const char* what = "launch_weight_normalize";
    NNK_REQUIRE(in >= 0 && out >= 0, what, "%s: bad shape in=%d out=%d", what, in, out);
    if (in == 0 || out == 0) return;
    NNK_REQUIRE(W, what, "%s: null pointer", what);
    NNK_WN_LAUNCH(wn_forward, (W, in, out, eps));
    nnk_after_launch(what, s);
}

void launch_weight_normalize_backward(float* gW, const float* Wn, const float* gain,
    float* g_gain, int in, int out, hipStream_t s) {
    const char* what = "launch_weight_normalize_backward";
    if (!wn_backward_args(what, gW, Wn, gain, g_gain, in, out)) return;
    const int blocks = wn_blocks(out, wn_cols(in, out));
    float* part = nnk_scratch_acquire((size_t)blocks, s, what);
    if (!part) return;
    NNK_WN_LAUNCH(wn_backward, (gW, Wn, gain, part, nullptr, g_gain, in, out), , kPartsOnly);
    wn_gain_sum<<<dim3(1), kWave, 0, s>>>(g_gain, part, blocks, wn_cols(in, out));
    nnk_scratch_release(part, s);
    nnk_after_launch(what, s);
}

size_t nnhip_weight_normalize_backward_workspace(int out) {
    return out > 0 ? (size_t)64 + (size_t)wn_blocks(out, 4) : 0;
}

void launch_weight_normalize_backward_ws(float* gW, const float* Wn, const float* gain, float* g_gain,
    int in, int out, float* workspace, hipStream_t s) {
    const char* what = "launch_weight_normalize_backward_ws";
    if (!wn_backward_args(what, gW, Wn, gain, g_gain, in, out)) return;
    NNK_REQUIRE(workspace, what, "%s: null workspace", what);
    unsigned* counter = reinterpret_cast<unsigned*>(workspace);
    NNK_WN_LAUNCH(wn_backward, (gW, Wn, gain, workspace + 64, counter, g_gain, in, out), , kAddGain);
    nnk_after_launch(what, s);
}

// As launch_weight_normalize_backward_ws on a *g_gain of 0 (host/conv_api.h).
void nnk_weight_normalize_backward_set(float* gW, const float* Wn, const float* gain, float* g_gain, int in,
    int out, float* workspace, hipStream_t s) {
    const char* what = "weight normalisation backward";
    if (!wn_backward_args(what, gW, Wn, gain, g_gain, in, out)) return;
    NNK_REQUIRE(workspace, what, "%s: null workspace", what);
    NNK_WN_LAUNCH(wn_backward, (gW, Wn, gain, workspace + 64, reinterpret_cast<unsigned*>(workspace), g_gain, in, out), ,
        kSetGain);
    nnk_after_launch(what, s);
}

}  // extern "C"
