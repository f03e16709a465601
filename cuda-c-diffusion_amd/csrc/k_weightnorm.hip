// k_weightnorm.hip -- forced unit-norm weight normalisation (forward, in place)
// and its backward with the gain gradient.
// Reference maths: src/kernels.cu:255-297 with launchers 330-344.
//
// W is [in, out] row-major and every output column j is normalised over its
// `in` rows.  One 1024-thread workgroup owns COLS whole columns: a wave
// instruction covers 64 / COLS rows, lane (r, c) walks rows of column COLS b + c
// and keeps up to kKeep of them in registers, all loaded at once; its partial,
// the row lanes of the wave and then the 16 waves are added in a fixed order.
// Each column total therefore has a fixed order and needs no scratch or second
// pass.  The work is one round trip of loads and one of stores, so what counts
// is how many CUs share it and that no round follows another: COLS = 4 puts
// [1152, 128] on 32 CUs with 5 rows a lane and [4032, 448] on 112 with 16 (rows
// longer than kKeep steps are read again from cache, in batches).  Neighbouring
// blocks share 128-byte lines, so they run on one XCD.  Against 16 columns a
// workgroup and 8 rows at a time: forward 20.1 -> 12.2 us and backward 37.0 ->
// 19.6 at [4032, 448], 6.7 -> 5.2 and 11.3 -> 8.4 at [1152, 128].
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

constexpr int kTpb = 1024;
constexpr int kNw = kTpb / kWave;
constexpr int kCols = 4;               // columns per workgroup
constexpr int kRowsPerWave = kWave / kCols;
constexpr int kRowStep = kNw * kRowsPerWave;
constexpr int kKeep = 16;              // rows a lane keeps in registers
constexpr int kMore = 8;               // rows in flight beyond those

// Rows i0 + u kRowStep of this lane's column, 0 past the end.
template <int N>
__device__ __forceinline__ void column_rows(float (&v)[N], const float* __restrict__ A, int i0, int in, int out,
    int j) {
#pragma unroll
    for (int u = 0; u < N; ++u) {
        const int i = i0 + u * kRowStep;
        v[u] = i < in ? A[(size_t)i * out + j] : 0.0f;
    }
}

// Total of the lanes' s over the column (identical on all its lanes, in every
// wave).  `l` is [kNw][kCols].
__device__ __forceinline__ float column_total(float s, float (*l)[kCols]) {
    const int lane = threadIdx.x & (kWave - 1);
    const int c = lane % kCols;
#pragma unroll
    for (int o = kCols; o < kWave; o <<= 1) s += __shfl_xor(s, o, kWave);
    if (lane < kCols) l[threadIdx.x / kWave][c] = s;
    __syncthreads();
    float t = l[0][c];
#pragma unroll
    for (int w = 1; w < kNw; ++w) t += l[w][c];
    return t;
}

__global__ __launch_bounds__(kTpb) void wn_forward(float* __restrict__ W, int in, int out, float eps) {
    __shared__ float l[kNw][kCols];
    const int bid = xcd_swizzle(blockIdx.x, gridDim.x);
    const int lane = threadIdx.x & (kWave - 1);
    const int i0 = threadIdx.x / kWave * kRowsPerWave + lane / kCols;
    const int j = bid * kCols + lane % kCols, jc = min(j, out - 1);
    float v[kKeep], s = 0.0f;
    column_rows(v, W, i0, in, out, jc);
#pragma unroll
    for (int u = 0; u < kKeep; ++u) s += v[u] * v[u];
    for (int i = i0 + kKeep * kRowStep; i < in; i += kMore * kRowStep) {
        float x[kMore];
        column_rows(x, W, i, in, out, jc);
#pragma unroll
        for (int u = 0; u < kMore; ++u) s += x[u] * x[u];
    }
    const float inv = rsqrtf(column_total(s, l) + eps);
    if (j >= out) return;
#pragma unroll
    for (int u = 0; u < kKeep; ++u) {
        const int i = i0 + u * kRowStep;
        if (i < in) W[(size_t)i * out + j] = v[u] * inv;
    }
    for (int i = i0 + kKeep * kRowStep; i < in; i += kRowStep) W[(size_t)i * out + j] *= inv;
}

// gW = gain * (gW - dot_j * Wn); part[b] = sum of block b's dot_j.
// kAddGain, kSetGain: the last workgroup to arrive (counter) adds part[0..gridDim.x)
// in index order to *g_gain, or to zero, and re-arms the counter.  A module's
// gain gradient is new in every backward pass: to set it saves the launch that
// cleared it (embedding MLP of two layers, 256 -> 512 -> 512 at batch 128:
// 59 -> 56 us a pass; convolution block [128, 32, 32, 128] 1400 -> 1375).
enum { kPartsOnly, kAddGain, kSetGain };
template <int GAIN>
__global__ __launch_bounds__(kTpb) void wn_backward(float* __restrict__ gW, const float* __restrict__ Wn,
    const float* __restrict__ gain, float* __restrict__ part, unsigned* __restrict__ counter,
    float* __restrict__ g_gain, int in, int out) {
    __shared__ float l[kNw][kCols];
    __shared__ int last;
    const int bid = xcd_swizzle(blockIdx.x, gridDim.x);
    const int lane = threadIdx.x & (kWave - 1);
    const int wid = threadIdx.x / kWave;
    const int i0 = wid * kRowsPerWave + lane / kCols;
    const int j = bid * kCols + lane % kCols, jc = min(j, out - 1);
    float a[kKeep], b[kKeep], s = 0.0f;
    column_rows(a, gW, i0, in, out, jc);
    column_rows(b, Wn, i0, in, out, jc);
    const float g = gain[0];
#pragma unroll
    for (int u = 0; u < kKeep; ++u) s += b[u] * a[u];
    for (int i = i0 + kKeep * kRowStep; i < in; i += kMore * kRowStep) {
        float x[kMore], y[kMore];
        column_rows(x, gW, i, in, out, jc);
        column_rows(y, Wn, i, in, out, jc);
#pragma unroll
        for (int u = 0; u < kMore; ++u) s += y[u] * x[u];
    }
    const float dot = column_total(s, l);  // its barrier orders every read of gW before the writes below
    if (wid == 0) {
        // lanes 0..kCols-1 hold the block's column totals
        const float t = wave_sum(lane < kCols && j < out ? dot : 0.0f);
        if (lane == 0) part[bid] = t;
    }
    if constexpr (GAIN != kPartsOnly) {
        __syncthreads();
        if (threadIdx.x == 0) {
            __threadfence();  // this block's part is visible before it is counted
            last = atomicAdd(counter, 1u) == gridDim.x - 1;
        }
        __syncthreads();
        if (last && wid == 0) {
            __threadfence();  // every counted block's part is visible here
            float t = 0.0f;
            for (int k = lane; k < (int)gridDim.x; k += kWave) t += part[k];
            t = wave_sum(t);
            if (lane == 0) {
                g_gain[0] = (GAIN == kSetGain ? 0.0f : g_gain[0]) + t;
                *counter = 0u;
            }
        }
    }
    if (j < out) {
#pragma unroll
        for (int u = 0; u < kKeep; ++u) {
            const int i = i0 + u * kRowStep;
            if (i < in) gW[(size_t)i * out + j] = g * (a[u] - dot * b[u]);
        }
        for (int i = i0 + kKeep * kRowStep; i < in; i += kRowStep) {
            const size_t o = (size_t)i * out + j;
            gW[o] = g * (gW[o] - dot * Wn[o]);
        }
    }
}

// *g_gain += part[0] + part[1] + ... (one wave, fixed order).
__global__ __launch_bounds__(kWave) void wn_gain_sum(float* __restrict__ g_gain, const float* __restrict__ part,
    int n) {
    float t = 0.0f;
    for (int k = threadIdx.x; k < n; k += kWave) t += part[k];
    t = wave_sum(t);
    if (threadIdx.x == 0) g_gain[0] = g_gain[0] + t;
}

int wn_blocks(int out) { return (out + kCols - 1) / kCols; }

bool wn_backward_args(const char* what, float* gW, const float* Wn, const float* gain, float* g_gain, int in,
    int out) {
    NNK_REQUIRE_RET(in >= 0 && out >= 0, false, what, "%s: bad shape in=%d out=%d", what, in, out);
    if (out == 0) return false;
    NNK_REQUIRE_RET(gW && Wn && gain && g_gain, false, what, "%s: null pointer", what);
    return true;
}

}  // namespace

extern "C" {

void launch_weight_normalize(float* W, int in, int out, float eps, hipStream_t s) {
    const char* what = "launch_weight_normalize";
    NNK_REQUIRE(in >= 0 && out >= 0, what, "%s: bad shape in=%d out=%d", what, in, out);
    if (in == 0 || out == 0) return;
    NNK_REQUIRE(W, what, "%s: null pointer", what);
    wn_forward<<<dim3((unsigned)wn_blocks(out)), kTpb, 0, s>>>(W, in, out, eps);
    nnk_after_launch(what, s);
}

void launch_weight_normalize_backward(float* gW, const float* Wn, const float* gain,
    float* g_gain, int in, int out, hipStream_t s) {
    const char* what = "launch_weight_normalize_backward";
    if (!wn_backward_args(what, gW, Wn, gain, g_gain, in, out)) return;
    const int blocks = wn_blocks(out);
    float* part = nnk_scratch_acquire((size_t)blocks, s, what);
    if (!part) return;
    wn_backward<kPartsOnly><<<dim3((unsigned)blocks), kTpb, 0, s>>>(gW, Wn, gain, part, nullptr, g_gain, in, out);
    wn_gain_sum<<<dim3(1), kWave, 0, s>>>(g_gain, part, blocks);
    nnk_scratch_release(part, s);
    nnk_after_launch(what, s);
}

size_t nnhip_weight_normalize_backward_workspace(int out) {
    return out > 0 ? (size_t)64 + (size_t)wn_blocks(out) : 0;
}

void launch_weight_normalize_backward_ws(float* gW, const float* Wn, const float* gain, float* g_gain,
    int in, int out, float* workspace, hipStream_t s) {
    const char* what = "launch_weight_normalize_backward_ws";
    if (!wn_backward_args(what, gW, Wn, gain, g_gain, in, out)) return;
    NNK_REQUIRE(workspace, what, "%s: null workspace", what);
    unsigned* counter = reinterpret_cast<unsigned*>(workspace);
    wn_backward<kAddGain><<<dim3((unsigned)wn_blocks(out)), kTpb, 0, s>>>(gW, Wn, gain, workspace + 64, counter,
        g_gain, in, out);
    nnk_after_launch(what, s);
}

// As launch_weight_normalize_backward_ws on a *g_gain of 0 (host/conv_api.h).
void nnk_weight_normalize_backward_set(float* gW, const float* Wn, const float* gain, float* g_gain, int in,
    int out, float* workspace, hipStream_t s) {
    const char* what = "weight normalisation backward";
    if (!wn_backward_args(what, gW, Wn, gain, g_gain, in, out)) return;
    NNK_REQUIRE(workspace, what, "%s: null workspace", what);
    wn_backward<kSetGain><<<dim3((unsigned)wn_blocks(out)), kTpb, 0, s>>>(gW, Wn, gain, workspace + 64,
        reinterpret_cast<unsigned*>(workspace), g_gain, in, out);
    nnk_after_launch(what, s);
}

}  // extern "C"
