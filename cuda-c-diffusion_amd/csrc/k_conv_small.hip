// k_conv_small.hip -- convolutions and dense layers (a convolution of one pixel)
// with few output tiles: 32 x 32 or 16 x 16 outputs a workgroup, whose waves share
// the k range, so that a few hundred rows still spread over the device.  The
// tiled kernels (igemm.h) put the reference DDPM's 7 x 7 x 128 level (392 rows) on
// four workgroups.
//
// A wave loads the fragments of its steps of 16 or 32 k straight from memory
// (eight k of a row or column a lane), a step ahead, splits both operands in
// registers and adds up its part of the tile; the parts are added in wave order
// through LDS and go through the epilogue, so one launch does all and nothing is
// kept in memory between.  Both operands are split per tile, four times as often
// as in the tiled kernels (eight with tiles of 16): ~90 vector instructions beside
// 6 MFMAs a step bound it, at about half the tiled kernels' full rate, but from
// the first workgroup on; with few tiles, the round trips of loads.  The rules
// between them are small_us (conv_common.h), conv_tile and wgrad_small_wins
// (igemm.h).
// Against im2col, rocBLAS and the bias pass at [8, 7 x 7, 128 -> 128]: forward 17 ->
// 6.2 us, input gradient 12 -> 6.9, weight gradient with the bias gradient 30 ->
// 8.2; dense [128, 512 -> 512] with bias 8 -> 4.9, its weight and bias gradients 11
// -> 4.9.
#include "conv_common.h"

#include <type_traits>

namespace {

using namespace nnk;
using namespace nnk::conv;

constexpr int kT = 32;     // tile edge
// Steps whose operands are on their way.  Two measured 5-20 % slower: the vector
// work of the four waves on a SIMD, not the loads, bounds a step.
constexpr int kAhead = 1;

// Parts in LDS, [wave][row][column]; accumulator register r of lane l holds row
// 8 (r / 4) + 4 (l / 32) + r % 4 of column l % 32 (tiles of 16: row 4 (l / 16) + r
// of column l % 16).
template <int T, class V>
__device__ __forceinline__ void put_part(float* lds, int w, int fr, int fh, const V& v) {
#pragma unroll
    for (int r = 0; r < T * T / 64; ++r) lds[w * T * T + (8 * (r >> 2) + 4 * fh + (r & 3)) * T + fr] = v[r];
}

// the sum of the waves' parts of element i, in wave order
template <int T, int WAVES>
__device__ __forceinline__ float sum_parts(const float* lds, int i) {
    float v = lds[i];
#pragma unroll
    for (int q = 1; q < WAVES; ++q) v += lds[q * T * T + i];
    return v;
}

// fp32 products of 2 k (tiles of 32) or 4 k (tiles of 16), one a lane
__device__ __forceinline__ void mfma_f32(float a, float b, f32x16& d) {
    d = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, d, 0, 0, 0);
}
__device__ __forceinline__ void mfma_f32(float a, float b, f32x4& d) {
    d = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, d, 0, 0, 0);
}

// VEC: channel counts are multiples of 8 and the pointers 16-byte aligned, so
// that 8 k of a pixel (and of a flipped weight's row) are two 16-byte loads.
template <int T, int WAVES, bool FLIP, bool VEC>
__global__ __launch_bounds__(64 * WAVES) void conv_small(float* __restrict__ Y, const float* __restrict__ X,
    const float* __restrict__ Wt, ConvShape sh, ConvEpi ep, int xe) {
    using Acc = std::conditional_t<T == 32, f32x16, f32x4>;
    constexpr int SK = 512 / T;  // k a step, 8 a lane
    __shared__ float lds[WAVES * T * T];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane % T, fh = lane / T;
    const int nt = (sh.Cout + T - 1) / T;
    const int tl = xcd_order((int)blockIdx.x, (int)gridDim.x);
    const int m0 = tl / nt * T, n0 = tl % nt * T;
    const int nc = min(n0 + fr, sh.Cout - 1);
    const int KK = sh.K * sh.K, nk = (sh.Cin + SK - 1) / SK, steps = KK * nk;
    const int per = (steps + WAVES - 1) / WAVES, s0 = w * per, s1 = min(steps, s0 + per);
    uint32_t q, ow, b, oh;
    sh.wo.divmod((uint32_t)min(m0 + fr, sh.M - 1), q, ow);  // a row past the end computes the last, stores nothing
    sh.ho.divmod(q, b, oh);
    const int ih0 = (int)oh * sh.stride - sh.pad, iw0 = (int)ow * sh.stride - sh.pad;
    const float* xb = X + (size_t)b * sh.H * sh.W * sh.Cin;

    // the operands of the next kAhead steps; channels past C_in are zeroed in
    // the activations (both read valid ones)
    struct Ops {
        float va[8], vw[8];
        bool ok;
        int c;
    };
    Ops o[kAhead];
    int tap = s0 / nk, cs = s0 - tap * nk;
    auto load = [&](Ops& r) {
        const int kh = tap / sh.K, kw = tap - kh * sh.K, ih = ih0 + kh, iw = iw0 + kw;
        r.ok = ((unsigned)ih < (unsigned)sh.H) & ((unsigned)iw < (unsigned)sh.W);
        const float* x = xb + (size_t)(r.ok ? ih * sh.W + iw : 0) * sh.Cin;
        r.c = SK * cs + 8 * fh;
        const size_t wt = FLIP ? ((size_t)(KK - 1 - tap) * sh.Cout + nc) * sh.Cin : (size_t)tap * sh.Cin * sh.Cout + nc;
        if constexpr (VEC) {
            const int cc = min(r.c, sh.Cin - 8);
            const float4 u = ld4(x + cc), z = ld4(x + cc + 4);
            r.va[0] = u.x, r.va[1] = u.y, r.va[2] = u.z, r.va[3] = u.w;
            r.va[4] = z.x, r.va[5] = z.y, r.va[6] = z.z, r.va[7] = z.w;
            if constexpr (FLIP) {
                const float4 g = ld4(Wt + wt + cc), h = ld4(Wt + wt + cc + 4);
                r.vw[0] = g.x, r.vw[1] = g.y, r.vw[2] = g.z, r.vw[3] = g.w;
                r.vw[4] = h.x, r.vw[5] = h.y, r.vw[6] = h.z, r.vw[7] = h.w;
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) r.vw[i] = Wt[wt + (size_t)(cc + i) * sh.Cout];
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int cc = min(r.c + i, sh.Cin - 1);
                r.va[i] = x[cc];
                r.vw[i] = Wt[FLIP ? wt + cc : wt + (size_t)cc * sh.Cout];
            }
        }
        if (++cs == nk) cs = 0, tap = min(tap + 1, KK - 1);  // past the last step: a harmless reload
    };
    Acc acc[1][1], cor[1][1];
    acc[0][0] = cor[0][0] = (Acc){};
    if (s0 < s1) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) load(o[u]);
    }
    for (int s = s0; s < s1; s += kAhead) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            uint4 pa[kPlanes], pw[kPlanes], a[kPlanes][1], bb[kPlanes][1];
            const bool in = o[u].ok && s + u < s1;  // a step past the wave's last adds zeros
#pragma unroll
            for (int i = 0; i < 8; ++i) o[u].va[i] = keep(o[u].va[i], in && (VEC ? o[u].c : o[u].c + i) < sh.Cin);
            split8(o[u].va, pa);
            split8(o[u].vw, pw);
            load(o[u]);
#pragma unroll
            for (int p = 0; p < kPlanes; ++p) a[p][0] = pa[p], bb[p][0] = pw[p];
            products<1, 1>(a, bb, acc, cor);
        }
    }
    acc[0][0] += cor[0][0];
    if (split_failed<1, 1>(acc)) {
        // straight from memory in fp32, one k a lane; rare, so simple
        acc[0][0] = (Acc){};
        for (int s = s0; s < s1; ++s) {
            const int t = s / nk, kh = t / sh.K, kw = t - kh * sh.K, ih = ih0 + kh, iw = iw0 + kw;
            const bool in = ((unsigned)ih < (unsigned)sh.H) & ((unsigned)iw < (unsigned)sh.W);
            for (int i = 0; i < SK; i += 64 / T) {
                const int ci = SK * (s - t * nk) + i + fh, cc = min(ci, sh.Cin - 1);
                const float x = xb[(size_t)(in ? ih * sh.W + iw : 0) * sh.Cin + cc];
                const float y = FLIP ? Wt[((size_t)(KK - 1 - t) * sh.Cout + nc) * sh.Cin + cc]
                                     : Wt[((size_t)t * sh.Cin + cc) * sh.Cout + nc];
                mfma_f32(in && ci < sh.Cin ? x : 0.0f, ci < sh.Cin ? y : 0.0f, acc[0][0]);
            }
        }
    }
    put_part<T>(lds, w, fr, fh, acc[0][0]);
    __syncthreads();
    const float gain = ep.gain ? ep.gain[0] : 1.0f;
    for (int i = tid; i < T * T; i += 64 * WAVES) {
        const int m = m0 + i / T, n = n0 + i % T;
        if (m >= sh.M || n >= sh.Cout) continue;
        uint32_t co = 0;
        if (xe & kXeMod) {
            uint32_t bb, r;
            ep.hw.divmod((uint32_t)m, bb, r);
            co = bb * (uint32_t)sh.Cout + (uint32_t)n;
        }
        epilogue_store(Y, sum_parts<T, WAVES>(lds, i), xe, (uint32_t)m * (uint32_t)sh.Cout + (uint32_t)n, co, ep,
            ep.bias ? ep.bias[n] : 0.0f, gain);
    }
}

// gW[k, n] = sum_m A[m, k] dY[m, n], A gathered from X; gb[n] = sum_m dY[m, n]
// from the workgroups of the first k tile.  A step is 16 rows m; all loads are
// 4 bytes a lane along k and n, so any channel counts and alignments do.
// DENSE: 1 x 1, stride 1, no padding: the input pixel is the output pixel.
template <int WAVES, bool DENSE>
__global__ __launch_bounds__(64 * WAVES) void wgrad_small(float* __restrict__ gW, float* __restrict__ gb,
    const float* __restrict__ X, const float* __restrict__ dY, ConvShape sh) {
    __shared__ float lds[WAVES * kT * kT];
    __shared__ float bl[WAVES][64];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 31, fh = lane >> 5;
    const int nt = (sh.Cout + kT - 1) / kT;
    const int tl = xcd_order((int)blockIdx.x, (int)gridDim.x);
    const int k0 = tl / nt * kT, n0 = tl % nt * kT;
    const bool sums = gb != nullptr && k0 == 0;
    const int nc = min(n0 + fr, sh.Cout - 1), k = min(k0 + fr, sh.KKC - 1);
    const int tap = k / sh.Cin, ci = k - tap * sh.Cin, kh = tap / sh.K - sh.pad, kw = tap % sh.K - sh.pad;
    const int steps = (sh.M + 15) / 16, per = (steps + WAVES - 1) / WAVES;
    const int s0 = w * per, s1 = min(steps, s0 + per);

    struct Ops {
        float va[8], vd[8];
        bool in[8];
    };
    Ops o[kAhead];
    auto load = [&](Ops& r, int s) {
        int m = 16 * s + 8 * fh;
        if constexpr (DENSE) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t mm = (uint32_t)min(m + i, sh.M - 1);
                r.in[i] = m + i < sh.M;
                r.va[i] = X[mm * (uint32_t)sh.Cin + (uint32_t)ci];
                r.vd[i] = dY[mm * (uint32_t)sh.Cout + (uint32_t)nc];
            }
            return;
        }
        uint32_t q, ow, b, oh;
        sh.wo.divmod((uint32_t)min(m, sh.M - 1), q, ow);
        sh.ho.divmod(q, b, oh);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int ih = (int)oh * sh.stride + kh, iw = (int)ow * sh.stride + kw;
            r.in[i] = (m + i < sh.M) & ((unsigned)ih < (unsigned)sh.H) & ((unsigned)iw < (unsigned)sh.W);
            r.va[i] = X[(uint32_t)((r.in[i] ? ((int)b * sh.H + ih) * sh.W + iw : 0) * sh.Cin + ci)];
            r.vd[i] = dY[(uint32_t)(min(m + i, sh.M - 1) * sh.Cout + nc)];
            if (++ow == (uint32_t)sh.Wo) {
                ow = 0;
                if (++oh == (uint32_t)sh.Ho) oh = 0, ++b;
            }
        }
    };
    f32x16 acc[1][1], cor[1][1];
    acc[0][0] = cor[0][0] = (f32x16){};
    float bs = 0.0f;
    if (s0 < s1) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) load(o[u], min(s0 + u, s1 - 1));
    }
    for (int s = s0; s < s1; s += kAhead) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            uint4 pa[kPlanes], pd[kPlanes], a[kPlanes][1], d[kPlanes][1];
            const bool mine = s + u < s1;  // a step past the wave's last adds zeros
            if (sums) {
#pragma unroll
                for (int i = 0; i < 8; ++i) bs += mine && 16 * (s + u) + 8 * fh + i < sh.M ? o[u].vd[i] : 0.0f;
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) o[u].va[i] = keep(o[u].va[i], mine && o[u].in[i]);
            split8(o[u].va, pa);
            split8(o[u].vd, pd);
            load(o[u], min(s + u + kAhead, s1 - 1));  // the last one again: harmless, and no branch
#pragma unroll
            for (int p = 0; p < kPlanes; ++p) a[p][0] = pa[p], d[p][0] = pd[p];
            products<1, 1>(a, d, acc, cor);
        }
    }
    acc[0][0] += cor[0][0];
    if (split_failed<1, 1>(acc)) {
        // straight from memory in fp32, 2 rows per MFMA; rare, so simple
        acc[0][0] = (f32x16){};
        for (int m2 = 16 * s0; m2 < min(16 * s1, sh.M); m2 += 2) {
            const int m = m2 + fh;
            uint32_t q, ow, b, oh;
            sh.wo.divmod((uint32_t)min(m, sh.M - 1), q, ow);
            sh.ho.divmod(q, b, oh);
            const int ih = (int)oh * sh.stride + kh, iw = (int)ow * sh.stride + kw;
            const bool inside = (m < sh.M) & ((unsigned)ih < (unsigned)sh.H) & ((unsigned)iw < (unsigned)sh.W);
            const float x = X[(size_t)(inside ? ((int)b * sh.H + ih) * sh.W + iw : 0) * sh.Cin + ci];
            const float y = dY[(size_t)min(m, sh.M - 1) * sh.Cout + nc];
            mfma_f32(inside ? x : 0.0f, m < sh.M ? y : 0.0f, acc[0][0]);
        }
    }
    put_part<kT>(lds, w, fr, fh, acc[0][0]);
    if (sums) bl[w][lane] = bs;
    __syncthreads();
    for (int i = tid; i < kT * kT; i += 64 * WAVES) {
        const int kk = k0 + i / kT, n = n0 + i % kT;
        if (kk < sh.KKC && n < sh.Cout) gW[(size_t)kk * sh.Cout + n] = sum_parts<kT, WAVES>(lds, i);
    }
    if (sums && tid < kT && n0 + tid < sh.Cout) {
        float t = 0.0f;
#pragma unroll
        for (int q = 0; q < WAVES; ++q) t += bl[q][tid] + bl[q][tid + 32];
        gb[n0 + tid] = t;
    }
}

}  // namespace

void nnk_conv_small(bool flip, int xe, float* Y, const float* X, const float* Wt, const ConvShape& sh,
    const ConvEpi& ep, hipStream_t s) {
    const int t = small_us(sh, flip, 16) < small_us(sh, flip, 32) ? 16 : 32;
    const unsigned grid = (unsigned)((sh.M + t - 1) / t) * (unsigned)((sh.Cout + t - 1) / t);
    const int waves = waves_for(sh.K * sh.K * ((sh.Cin + 512 / t - 1) / (512 / t)));
    const bool vec = sh.Cin % 8 == 0 && aligned16(X) && (!flip || aligned16(Wt));
#define NNK_SMALL(T_, W_, F_, V_) conv_small<T_, W_, F_, V_><<<grid, 64 * W_, 0, s>>>(Y, X, Wt, sh, ep, xe)
#define NNK_SMALL_W(T_, F_, V_)                        \
    do {                                               \
        if (waves == 4) NNK_SMALL(T_, 4, F_, V_);      \
        else if (waves == 8) NNK_SMALL(T_, 8, F_, V_); \
        else NNK_SMALL(T_, 16, F_, V_);                \
    } while (0)
#define NNK_SMALL_T(F_, V_)                  \
    do {                                     \
        if (t == 16) NNK_SMALL_W(16, F_, V_); \
        else NNK_SMALL_W(32, F_, V_);        \
    } while (0)
    if (flip) {
        if (vec) NNK_SMALL_T(true, true);
        else NNK_SMALL_T(true, false);
    } else {
        if (vec) NNK_SMALL_T(false, true);
        else NNK_SMALL_T(false, false);
    }
#undef NNK_SMALL_T
#undef NNK_SMALL_W
#undef NNK_SMALL
}

void nnk_wgrad_small(float* gW, float* gb, const float* X, const float* dY, const ConvShape& sh, hipStream_t s) {
    const unsigned grid = (unsigned)((sh.KKC + kT - 1) / kT) * (unsigned)((sh.Cout + kT - 1) / kT);
    const int waves = waves_for((sh.M + 15) / 16);
    const bool dense = sh.K == 1 && sh.stride == 1 && sh.pad == 0;
#define NNK_WSMALL(W_)                                                                             \
    do {                                                                                           \
        if (dense) wgrad_small<W_, true><<<grid, 64 * W_, 0, s>>>(gW, gb, X, dY, sh);              \
        else wgrad_small<W_, false><<<grid, 64 * W_, 0, s>>>(gW, gb, X, dY, sh);                   \
    } while (0)
    if (waves == 4) NNK_WSMALL(4);
    else if (waves == 8) NNK_WSMALL(8);
    else NNK_WSMALL(16);
#undef NNK_WSMALL
}
