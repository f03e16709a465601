// k_gn_slab.hip -- GroupNorm (+ activation) of any channels per group and any
// alignment, for the shapes the float4 kernels (gn_kernels.h, gn_stream.h) do
// not take.  Reference maths: src/kernels.cu:622-717 with the activation of
// :21-68, as gn_kernels.h.
//
// A workgroup owns a slab of GB neighbouring groups of one sample: CW = GB cpg
// channels, contiguous in every pixel, so that a wave's 4-byte accesses cover
// whole runs of CW floats instead of cpg (12 bytes at 3 channels per group).
// Thread t always meets channel t % CW, of the pixels t / CW + k PSTEP, and
// keeps the first NV of them in registers: x (and dy) cross HBM once; a group
// too large for that reads the rest again.  Sums are taken per channel (threads
// of a channel over LDS, in a fixed order), then over the group's channels, so
// the backward's dgamma / dbeta partials of the sample come out of the same
// pass.  Bound by the round trips of loads and of the sums' barriers at small
// sizes, by HBM above.
// [24, 28 x 28, 96], 3 channels per group, forward + backward: 157 -> 25 us,
// against one 256-thread workgroup per group, three passes over x and a kernel
// of its own for the partials; with slabs of 96 bytes on 96 workgroups 30.
#include "gn_kernels.h"

namespace {

using namespace nnk;

struct Slab {
    int G, HW, C, cpg;
    int gb, cw, pstep, seg;  // groups and channels of a slab, pixels per step, partial sums per channel
    FastDiv dcw, dcpg;
};

// Total of a and b over the workgroup, on every thread: a slab of one group (ONE)
// needs no sums by channel for it.  One thread adding a group's channels one by
// one took longer than all else from about 100 channels on: forward + backward
// [1, 1, 1, 1024] in one group 48 -> 17 us, [64, 8, 8, 1000] 111 -> 69.  l is [2][TPB /
// 64]; the barriers order it after earlier uses of l.
template <int TPB>
__device__ __forceinline__ void slab_sum2(float& a, float& b, float* l) {
    a = wave_sum(a);
    b = wave_sum(b);
    const int w = threadIdx.x / kWave;
    __syncthreads();
    if (threadIdx.x % kWave == 0) {
        l[w] = a;
        l[TPB / kWave + w] = b;
    }
    __syncthreads();
    a = l[0];
    b = l[TPB / kWave];
#pragma unroll
    for (int i = 1; i < TPB / kWave; ++i) {
        a += l[i];
        b += l[TPB / kWave + i];
    }
}

// red[0..TPB) holds the threads' values (0 past pstep * cw); leaves in out[s *
// cw + c], s < seg, the sums of channel c over the pixels s, s + seg, ...
__device__ __forceinline__ void channel_segments(float* out, const float* red, const Slab& sl) {
    const int t = threadIdx.x;
    if (t < sl.seg * sl.cw) {
        uint32_t s, c;
        sl.dcw.divmod((uint32_t)t, s, c);
        float a = 0.0f;
        for (int p = (int)s; p < sl.pstep; p += sl.seg) a += red[p * sl.cw + (int)c];
        out[t] = a;
    }
}

template <int TPB, int NV, bool ONE, int ACT>
__global__ __launch_bounds__(TPB) void gn_fwd_slab(float* __restrict__ y, float* __restrict__ mu_out,
    float* __restrict__ rstd_out, const float* __restrict__ x, const float* __restrict__ gamma,
    const float* __restrict__ beta, Slab sl, float eps) {
    __shared__ float red[TPB], part[TPB], stat[TPB];
    const int slabs = (sl.G + sl.gb - 1) / sl.gb;
    const int work = xcd_swizzle(blockIdx.x, gridDim.x);
    const int b = work / slabs, g0 = (work - b * slabs) * sl.gb, ng = min(sl.gb, sl.G - g0);
    uint32_t p0, ch;
    sl.dcw.divmod(threadIdx.x, p0, ch);
    const bool on = (int)p0 < sl.pstep && (int)ch < ng * sl.cpg;
    const int c = g0 * sl.cpg + (on ? (int)ch : 0), gl = on ? (int)sl.dcpg.div(ch) : 0;
    const int last = on ? sl.HW : 0;  // a thread that is not on has no pixel
    const size_t base = (size_t)b * sl.HW * sl.C + c;
    float v[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int p = (int)p0 + k * sl.pstep;
        v[k] = p < last ? x[base + (size_t)p * sl.C] : 0.0f;
    }
    const float gm = gamma[c], bt = beta[c];
    const int more = (int)p0 + NV * sl.pstep;
    const float n = (float)(sl.HW * sl.cpg);
    // the group's total of s, per thread's own group
    auto group_total = [&](float s) {
        if constexpr (ONE) {
            float z = 0.0f;
            slab_sum2<TPB>(s, z, red);
            return s;
        }
        __syncthreads();
        red[threadIdx.x] = s;
        __syncthreads();
        channel_segments(part, red, sl);
        __syncthreads();
        if ((int)threadIdx.x < ng) {
            float a = 0.0f;
            for (int q = 0; q < sl.seg; ++q)
                for (int i = 0; i < sl.cpg; ++i) a += part[q * sl.cw + (int)threadIdx.x * sl.cpg + i];
            stat[threadIdx.x] = a;
        }
        __syncthreads();
        return stat[gl];
    };
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; ++k) s += v[k];
    for (int p = more; p < last; p += sl.pstep) s += x[base + (size_t)p * sl.C];
    const float mean = group_total(s) / n;
    float q = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const float d = (int)p0 + k * sl.pstep < last ? v[k] - mean : 0.0f;
        q += d * d;
    }
    for (int p = more; p < last; p += sl.pstep) {
        const float d = x[base + (size_t)p * sl.C] - mean;
        q += d * d;
    }
    const float rs = rsqrtf(group_total(q) / n + eps);
    if (on && p0 == 0 && (int)ch == gl * sl.cpg) {
        mu_out[b * sl.G + g0 + gl] = mean;
        rstd_out[b * sl.G + g0 + gl] = rs;
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int p = (int)p0 + k * sl.pstep;
        if (p < last) y[base + (size_t)p * sl.C] = act_fwd<ACT>(gm * ((v[k] - mean) * rs) + bt);
    }
    for (int p = more; p < last; p += sl.pstep) {
        const size_t o = base + (size_t)p * sl.C;
        y[o] = act_fwd<ACT>(gm * ((x[o] - mean) * rs) + bt);
    }
}

template <int TPB, int NV, bool ONE, int ACT>
__global__ __launch_bounds__(TPB) void gn_bwd_slab(float* __restrict__ dx, float* __restrict__ part_g,
    float* __restrict__ part_b, const float* __restrict__ dy, const float* __restrict__ x,
    const float* __restrict__ gamma, const float* __restrict__ beta, const float* __restrict__ mu,
    const float* __restrict__ rstd, Slab sl) {
    __shared__ float red[2][TPB], part[2][TPB], stat[2][TPB];
    const int slabs = (sl.G + sl.gb - 1) / sl.gb;
    const int work = xcd_swizzle(blockIdx.x, gridDim.x);
    const int b = work / slabs, g0 = (work - b * slabs) * sl.gb, ng = min(sl.gb, sl.G - g0);
    uint32_t p0, ch;
    sl.dcw.divmod(threadIdx.x, p0, ch);
    const bool on = (int)p0 < sl.pstep && (int)ch < ng * sl.cpg;
    const int c = g0 * sl.cpg + (on ? (int)ch : 0), gl = on ? (int)sl.dcpg.div(ch) : 0;
    const int last = on ? sl.HW : 0;
    const size_t base = (size_t)b * sl.HW * sl.C + c;
    float xv[NV], gv[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int p = (int)p0 + k * sl.pstep;
        const bool in = p < last;
        xv[k] = in ? x[base + (size_t)p * sl.C] : 0.0f;
        gv[k] = in ? dy[base + (size_t)p * sl.C] : 0.0f;
    }
    const float mean = mu[b * sl.G + g0 + gl], rs = rstd[b * sl.G + g0 + gl], gm = gamma[c];
    float bt = 0.0f;
    if constexpr (ACT != ACT_IDENTITY) bt = beta[c];
    auto d_of = [&](float g, float xh) {
        if constexpr (ACT != ACT_IDENTITY) return g * act_grad<ACT>(gm * xh + bt);
        else return g;
    };
    const int more = (int)p0 + NV * sl.pstep;
    float sg = 0.0f, sb = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const bool in = (int)p0 + k * sl.pstep < last;
        const float xh = (xv[k] - mean) * rs, d = d_of(gv[k], xh);
        sg += in ? d * xh : 0.0f;
        sb += in ? d : 0.0f;
        xv[k] = xh;
        gv[k] = d * gm;
    }
    for (int p = more; p < last; p += sl.pstep) {
        const size_t o = base + (size_t)p * sl.C;
        const float xh = (x[o] - mean) * rs, d = d_of(dy[o], xh);
        sg += d * xh;
        sb += d;
    }
    red[0][threadIdx.x] = sg;
    red[1][threadIdx.x] = sb;
    __syncthreads();
    channel_segments(part[0], red[0], sl);
    channel_segments(part[1], red[1], sl);
    __syncthreads();
    // channel totals (into red), then the group's sums of d gamma and of d gamma xhat
    float a = 0.0f, e = 0.0f;
    if ((int)threadIdx.x < ng * sl.cpg) {
        for (int q = 0; q < sl.seg; ++q) {
            a += part[0][q * sl.cw + (int)threadIdx.x];
            e += part[1][q * sl.cw + (int)threadIdx.x];
        }
        const int cc = g0 * sl.cpg + (int)threadIdx.x;
        part_g[(size_t)b * sl.C + cc] = a;
        part_b[(size_t)b * sl.C + cc] = e;
        a *= gamma[cc];
        e *= gamma[cc];
        red[0][threadIdx.x] = a;
        red[1][threadIdx.x] = e;
    }
    if constexpr (ONE) {
        slab_sum2<TPB>(a, e, stat[0]);
    } else {
        __syncthreads();
        if ((int)threadIdx.x < ng) {
            a = e = 0.0f;
            for (int i = 0; i < sl.cpg; ++i) {
                a += red[0][(int)threadIdx.x * sl.cpg + i];
                e += red[1][(int)threadIdx.x * sl.cpg + i];
            }
            stat[0][threadIdx.x] = a;
            stat[1][threadIdx.x] = e;
        }
        __syncthreads();
        a = stat[0][gl];
        e = stat[1][gl];
    }
    const float inv_n = 1.0f / (float)(sl.HW * sl.cpg);
    const float pgx = a, m1 = e * inv_n;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int p = (int)p0 + k * sl.pstep;
        if (p < last) dx[base + (size_t)p * sl.C] = rs * ((gv[k] - m1) - xv[k] * pgx * inv_n);
    }
    for (int p = more; p < last; p += sl.pstep) {
        const size_t o = base + (size_t)p * sl.C;
        const float xh = (x[o] - mean) * rs, gg = d_of(dy[o], xh) * gm;
        dx[o] = rs * ((gg - m1) - xh * pgx * inv_n);
    }
}

// A slab starts as one group and doubles while it is narrower than kSlabMin
// bytes, the least that a memory transaction moves, and half of the CUs
// still get a workgroup (a small tensor is bound by latency, not by its
// transactions); then up to kSlabMax while that leaves two workgroups per CU
// and the registers hold it.
constexpr int kSlabMin = 64, kSlabMax = 256, kFew = 128, kEnough = 512, kHeld = 1024 * 16;

// Threads by the slab's size: a thread keeps 4 or 16 values (its loads are all
// in flight at once), 32 only where 1024 threads do not hold the slab with 16.
struct SlabPlan {
    int cfg;  // 0: 256 x 4, 1: 256 x 16, 2: 1024 x 16, 3: 1024 x 32
    unsigned grid;
    Slab sl;
};
SlabPlan plan(int B, int G, int HW, int C) {
    const int cpg = C / G;
    int gb = 1;
    while (2 * gb <= G && 2 * gb * cpg <= 256 &&
           ((4 * gb * cpg < kSlabMin && (long long)B * G >= 2LL * gb * kFew) ||
               (8 * gb * cpg <= kSlabMax && (long long)B * G >= 2LL * gb * kEnough &&
                   (long long)HW * 2 * gb * cpg <= kHeld)))
        gb *= 2;
    SlabPlan p;
    p.sl.G = G, p.sl.HW = HW, p.sl.C = C, p.sl.cpg = cpg;
    p.sl.gb = gb;
    p.sl.cw = gb * cpg;
    const long long n = (long long)HW * p.sl.cw;
    p.cfg = n <= 256 * 4 ? 0 : n <= 256 * 16 ? 1 : n <= 1024 * 16 ? 2 : 3;
    if (p.sl.cw > 256 && p.cfg < 2) p.cfg = 2;
    const int tpb = p.cfg < 2 ? 256 : 1024;
    p.sl.pstep = tpb / p.sl.cw;
    p.sl.seg = p.sl.pstep < 8 ? p.sl.pstep : 8;
    p.sl.dcw = FastDiv((uint32_t)p.sl.cw);
    p.sl.dcpg = FastDiv((uint32_t)cpg);
    p.grid = (unsigned)B * (unsigned)((G + gb - 1) / gb);
    return p;
}

}  // namespace

bool nnk_gn_slab_takes(int HW, int C, int G) { return C / G <= 1024 && HW <= 1 << 30; }

// (a slab of one group has kernels of its own: the others lose 4 % to the branch)
#define NNK_SLAB_ONE(KERNEL, TPB_, NV_, ...)                                              \
    do {                                                                                 \
        if (p.sl.gb == 1) KERNEL<TPB_, NV_, true, A><<<p.grid, TPB_, 0, s>>>(__VA_ARGS__); \
        else KERNEL<TPB_, NV_, false, A><<<p.grid, TPB_, 0, s>>>(__VA_ARGS__);             \
    } while (0)
#define NNK_SLAB(KERNEL, ...)                                             \
    NNK_ACT_DISPATCH(act, A, {                                            \
        if (p.cfg == 0) NNK_SLAB_ONE(KERNEL, 256, 4, __VA_ARGS__);        \
        else if (p.cfg == 1) NNK_SLAB_ONE(KERNEL, 256, 16, __VA_ARGS__);  \
        else if (p.cfg == 2) NNK_SLAB_ONE(KERNEL, 1024, 16, __VA_ARGS__); \
        else NNK_SLAB_ONE(KERNEL, 1024, 32, __VA_ARGS__);                 \
    })

void nnk_gn_fwd_slab(int act, float* y, float* mu, float* rstd, const float* x, const float* gamma, const float* beta,
    int B, int G, int HW, int C, float eps, hipStream_t s) {
    const SlabPlan p = plan(B, G, HW, C);
    NNK_SLAB(gn_fwd_slab, y, mu, rstd, x, gamma, beta, p.sl, eps);
}

void nnk_gn_bwd_slab(int act, float* dx, float* part_g, float* part_b, const float* dy, const float* x,
    const float* gamma, const float* beta, const float* mu, const float* rstd, int B, int G, int HW, int C,
    hipStream_t s) {
    const SlabPlan p = plan(B, G, HW, C);
    NNK_SLAB(gn_bwd_slab, dx, part_g, part_b, dy, x, gamma, beta, mu, rstd, p.sl);
}
