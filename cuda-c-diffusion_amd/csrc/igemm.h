// igemm.h -- the tiled implicit-GEMM convolution kernels on the matrix cores,
// shared by k_igemm.hip (the plain launchers) and k_igemm_fused.hip (the
// launchers with a neighbouring pass folded into a kernel's operand loads or
// epilogue).  Design notes: k_igemm.hip.
#pragma once
#include <math.h>

#include <atomic>

#include "conv_common.h"

namespace {

using namespace nnk;
using namespace nnk::conv;

constexpr int kTpb = 256;

// LDS tiles hold rows of 32 k, 64 bytes (four 16-byte chunks) a plane, and
// every access is 16 bytes a lane.  The order of a row's chunks depends on the
// row (swz), so that the fragment reads, 16 consecutive rows at one chunk,
// fall on 16 distinct 16-byte groups of the 64 banks (5.3 cycles a wave read
// against 8 with chunks ordered by (row / 2) % 4), and so do the writes of
// lanes along a row, 4 rows x 4 chunks.
//   rowslot: the three planes of a row beside each other (the convolution's
//     activations, read at any row offset);
//   stage_slot: a plane of its own with 16 k a row (the weight gradient's tiles):
//     32 bytes a row, the two chunks swapped on alternate groups of 8 rows.
__device__ __forceinline__ int swz(int row, int c) { return c ^ ((row >> 2) & 3); }
constexpr int kRowSlots = 4 * kPlanes;  // uint4 per row of all planes
__device__ __forceinline__ int rowslot(int row, int c) { return row * kRowSlots + swz(row, c); }
constexpr int kStage4 = 2;  // uint4 per row of one plane
__device__ __forceinline__ int stage_slot(int row, int c) { return row * kStage4 + (c ^ ((row >> 3) & 1)); }
// ... written stride uint4 apart
__device__ __forceinline__ void put8(uint4* t, int stride, const float (&v)[8]) {
    uint4 p[kPlanes];
    split8(v, p);
#pragma unroll
    for (int i = 0; i < kPlanes; ++i) t[i * stride] = p[i];
}

// a buffer resource at a uniform address: loads then take a scalar base and a
// 32-bit lane offset instead of a 64-bit address in vector registers
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const float* p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, -1, 0x00020000);
}

// The order of a step's instructions: after each MFMA up to VALU
// vector instructions, and an access of LDS or a load from memory where one is left.
template <int MFMAS, int VALU = 6>
__device__ __forceinline__ void sched() {
#pragma unroll
    for (int i = 0; i < MFMAS; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, VALU, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
        __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // LDS write
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // memory read
    }
}

// How the activations reach LDS:
//   kHalo: the rows of all taps once per 32 channels (stride 1, output as large
//     as the input: the input pixel of output pixel m and tap (kh, kw) is m +
//     (kh - pad) W + kw - pad, so the pixels of 128 consecutive outputs lie in
//     128 + 2 pad (W + 1) consecutive rows; taps outside the image read a row of
//     zeros instead);
//   kGather: 128 rows per tap and 32 channels, any geometry;
//   kRagged: as kGather for channel counts that are no multiple of 8 or
//     pointers that are not 16-byte aligned, loads of 4 bytes.
enum { kHalo = 0, kGather = 1, kRagged = 2 };

// Y[m, n] = sum_k A[m, k] B[k, n] with the fused epilogue; FLIP: B is the input
// gradient's flipped weight (sh is then the gradient's convolution: C_in = the
// layer's C_out, C_out = the layer's C_in, so Wt is [K*K*sh.Cout][sh.Cin]).
//
// A workgroup computes 128 x BN outputs with four waves of 32 columns and 32 T
// rows.  k runs over slices of 32 channels and, within one, over the taps.
// Only the activations go through LDS, where the waves share them: they are
// split into planes as they are stored.  A wave needs its weight columns
// alone, so it loads them straight into the fragment's registers, a slice
// ahead, and splits them there; no element of either is split twice per
// workgroup and slice, and with kHalo none of the activations is per tap.
// Two workgroups share a CU: one computes while the other stages.
template <int BN, int MODE, bool FLIP, int XE>
__global__ __launch_bounds__(kTpb, 2) void conv_x3(float* __restrict__ Y, const float* __restrict__ X,
    const float* __restrict__ Wt, ConvShape sh, ConvEpi ep) {
    constexpr int WN = BN / 32, T = WN;  // waves along n; row tiles per wave (4 / (4 / WN))
    extern __shared__ uint4 As[];        // rowslot(): kHalo halo rows and a row of zeros, else 128 rows
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 31, fh = lane >> 5;
    const int nb = (sh.Cout + BN - 1) / BN;
    const int tl = xcd_order((int)blockIdx.x, (int)gridDim.x);
    const int m0 = tl / nb * kBM, n0 = tl % nb * BN;
    const int wrow = w / WN * 32 * T;  // the wave's first row of the tile
    const int n = n0 + 32 * (w % WN) + fr, nc = min(n, sh.Cout - 1);
    const int nu = min(n0 + 32 * (w % WN), sh.Cout - 1);  // the wave's first column
    const int KK = sh.K * sh.K, ncs = (sh.Cin + kBK - 1) / kBK;

    // fragment rows: the lane's row of each row tile, as its LDS offset or
    // (kHalo) its place among the halo rows of tap 0, with the taps that lie
    // inside the image as bits
    const char* as_bytes = reinterpret_cast<const char*>(As);
    int arow[T];
    uint32_t inside[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int r = wrow + 32 * t + fr;
        arow[t] = MODE == kHalo ? r : 16 * rowslot(r, fh);
        if constexpr (MODE == kHalo) {
            const int m = m0 + r;
            uint32_t q, ow, b, oh, cols = 0;
            sh.wo.divmod((uint32_t)min(m, sh.M - 1), q, ow);
            sh.ho.divmod(q, b, oh);
            for (int kw = 0; kw < sh.K; ++kw) cols |= (uint32_t)((unsigned)((int)ow + kw - sh.pad) < (unsigned)sh.W) << kw;
            inside[t] = 0;
            for (int kh = 0; kh < sh.K; ++kh)
                if ((unsigned)((int)oh + kh - sh.pad) < (unsigned)sh.H) inside[t] |= cols << (kh * sh.K);
            if (m >= sh.M) inside[t] = 0;
        }
    }

    // activation loader: chunk ch (8 channels) of rows r0, r0 + 64, ...
    const int ch = tid & 3, r0 = tid >> 2;
    float v0[8], v1[8];  // kGather: the rows r0, r0 + 64 of the next tap
    bool ok0 = false, ok1 = false;
    int pix[2], ihb[2], iwb[2];
    const int halo = kBM + 2 * sh.pad * (sh.W + 1);
    if constexpr (MODE == kHalo) {
        if (tid < kRowSlots) As[halo * kRowSlots + tid] = make_uint4(0, 0, 0, 0);
    } else {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int m = m0 + r0 + 64 * q;
            uint32_t t, ow, b, oh;
            sh.wo.divmod((uint32_t)(m < sh.M ? m : 0), t, ow);  // a row past the end computes row 0, stores nothing
            sh.ho.divmod(t, b, oh);
            pix[q] = (int)b * sh.H * sh.W;
            ihb[q] = (int)oh * sh.stride - sh.pad;
            iwb[q] = (int)ow * sh.stride - sh.pad;
        }
    }
    // 8 channels from c on of pixel p; channels past the end are left to the
    // caller to zero (they read valid ones)
    auto pixel8 = [&](float (&v)[8], int p, int c) {
        const float* x = X + (size_t)p * sh.Cin;
        if constexpr (MODE == kRagged) {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = x[min(c + i, sh.Cin - 1)];
        } else {
            const float4 u = ld4(x + min(c, sh.Cin - 8)), z = ld4(x + min(c, sh.Cin - 8) + 4);
            v[0] = u.x, v[1] = u.y, v[2] = u.z, v[3] = u.w, v[4] = z.x, v[5] = z.y, v[6] = z.z, v[7] = z.w;
        }
    };
    // zeroed by masking the bits (a select of values would become a select of
    // their addresses); channels past C_in too
    auto put_row = [&](int row, float (&v)[8], bool ok, int c) {
        if constexpr (MODE == kRagged) {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = keep(v[i], ok && c + i < sh.Cin);
        } else if constexpr (MODE == kGather) {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = keep(v[i], ok && c < sh.Cin);
        } else if (!ok) {  // kHalo: ok is uniform but in the last slice
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = 0.0f;
        }
        put8(As + rowslot(row, ch), 4, v);
    };
    auto gather = [&](int cs, int kh, int kw) {
        const int c = cs * kBK + 8 * ch;
        ok0 = ((unsigned)(ihb[0] + kh) < (unsigned)sh.H) & ((unsigned)(iwb[0] + kw) < (unsigned)sh.W);
        ok1 = ((unsigned)(ihb[1] + kh) < (unsigned)sh.H) & ((unsigned)(iwb[1] + kw) < (unsigned)sh.W);
        pixel8(v0, ok0 ? pix[0] + (ihb[0] + kh) * sh.W + iwb[0] + kw : 0, c);
        pixel8(v1, ok1 ? pix[1] + (ihb[1] + kh) * sh.W + iwb[1] + kw : 0, c);
    };
    auto stage_halo = [&](int cs) {
        const int c = cs * kBK + 8 * ch, base = m0 - sh.pad * (sh.W + 1);
        constexpr int NB = 2;  // rows in flight
        for (int r = r0; r < halo; r += 64 * NB) {
            float v[NB][8];
#pragma unroll
            for (int q = 0; q < NB; ++q) pixel8(v[q], min(max(base + r + 64 * q, 0), sh.M - 1), c);
#pragma unroll
            for (int q = 0; q < NB; ++q)
                if (r + 64 * q < halo) put_row(r + 64 * q, v[q], c < sh.Cin, c);
        }
    };

    // weight loader: the lane's 8 k (8 fh .. + 7) of 16 at column nc, for the
    // 16 channels c0 .. of a tap.  Channels past the end read valid ones: the
    // activations are zero there.
    float wv[2][8];
    auto weights = [&](float (&v)[8], int tap, int c0) {
        if constexpr (MODE == kRagged) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int c = min(c0 + 8 * fh + i, sh.Cin - 1);
                v[i] = FLIP ? Wt[((size_t)(KK - 1 - tap) * sh.Cout + nc) * sh.Cin + c]
                            : Wt[(size_t)(tap * sh.Cin + c) * sh.Cout + nc];
            }
        } else {
            const int cu = min(c0, sh.Cin - 8);  // c0 may lie past the end
            const int lh = cu + 16 > sh.Cin ? 0 : fh;
            // a uniform base in scalar registers and a 32-bit lane offset (at
            // most 31 rows of C_in, or 16 of C_out)
            if constexpr (FLIP) {
                const auto q = buffer(Wt + ((size_t)(KK - 1 - tap) * sh.Cout + nu) * sh.Cin + cu);
                const int lo = 4 * ((nc - nu) * sh.Cin + 8 * lh);
                const f32x4 u = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(q, lo, 0, 0));
                const f32x4 z = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(q, lo, 16, 0));
                v[0] = u.x, v[1] = u.y, v[2] = u.z, v[3] = u.w, v[4] = z.x, v[5] = z.y, v[6] = z.z, v[7] = z.w;
            } else {
                const auto q = buffer(Wt + (size_t)(tap * sh.Cin + cu) * sh.Cout + nu);
                const int lo = 4 * (8 * lh * sh.Cout + nc - nu);
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    v[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(q, lo, 4 * i * sh.Cout, 0));
            }
        }
    };

    f32x16 acc[T][1], cor[T][1];
#pragma unroll
    for (int t = 0; t < T; ++t) acc[t][0] = cor[t][0] = (f32x16){};

    // Steps of 16 k: (slice, tap, half).  A step's MFMAs read fragments that are
    // in registers when it begins; between them it reads the next step's
    // activation fragments into the registers of planes that are done with,
    // splits the next step's weights and loads those of the step after.  The
    // pattern (sched) keeps the compiler from drawing those to one side of the
    // MFMAs: a wave by itself then leaves the matrix core few gaps, where two
    // waves that take their vector work and their MFMAs in turns fall into step
    // and leave it idle together.
    uint4 a[kPlanes][T], b[2][kPlanes][1];
    auto split_w = [&](int h) {
        uint4 q[kPlanes];
        split8(wv[h], q);
#pragma unroll
        for (int p = 0; p < kPlanes; ++p) b[h][p][0] = q[p];
    };
    auto rows_of = [&](int tap, int shift, int (&as)[T]) {  // byte offsets of the lane's fragment rows
#pragma unroll
        for (int t = 0; t < T; ++t) {
            as[t] = arow[t];
            if constexpr (MODE == kHalo) {
                // the row's slot where the tap is inside, else the zeros: a bit
                // select, which stays free of branches
                const int row = arow[t] + shift, in = -(int)((inside[t] >> tap) & 1);
                as[t] = ((__mul24(row, 16 * kRowSlots) + 16 * swz(row, fh)) & in) | (halo * kRowSlots * 16 & ~in);
            }
        }
    };
    auto frag = [&](int p, const int (&as)[T], int ks) {
#pragma unroll
        for (int t = 0; t < T; ++t)
            a[p][t] = *reinterpret_cast<const uint4*>(as_bytes + (as[t] ^ 32 * ks) + 64 * p);
    };
    auto mul = [&](int i, int j, int h, f32x16 (&d)[T][1]) {
#pragma unroll
        for (int t = 0; t < T; ++t)
            d[t][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[i][t]),
                __builtin_bit_cast(bf16x8, b[h][j][0]), d[t][0], 0, 0, 0);
    };
    // One step: half h of a tap, whose rows are `as`; (nas, h ^ 1) the next
    // step's rows and half; (ntap, nc0) the tap and channels of the weights two
    // steps on.  Planes 1 and 2 of the activations are in registers when the
    // step begins, plane 0 is read during the first three products.
    auto step = [&](int h, const int (&as)[T], const int (&nas)[T], int ntap, int nc0) {
        frag(0, as, h);
        mul(2, 0, h, cor);
        split_w(h ^ 1);
        mul(1, 1, h, cor);
        mul(1, 0, h, cor);
        sched<3 * T>();
        __builtin_amdgcn_sched_barrier(0);
        frag(2, nas, h ^ 1);
        frag(1, nas, h ^ 1);
        weights(wv[h ^ 1], ntap, nc0);  // into the registers just split
        mul(0, 2, h, cor);
        mul(0, 1, h, cor);
        mul(0, 0, h, acc);
        sched<3 * T>();
        __builtin_amdgcn_sched_barrier(0);
    };
    weights(wv[0], 0, 0);
    weights(wv[1], 0, 16);
    if constexpr (MODE != kHalo) gather(0, 0, 0);
    split_w(0);
    weights(wv[0], KK > 1 ? 1 : 0, KK > 1 ? 0 : min(kBK, sh.Cin - 1));
    int as[T];
    for (int cs = 0; cs < ncs; ++cs) {
        if constexpr (MODE == kHalo) {
            if (cs) __syncthreads();  // the slice before has been read
            stage_halo(cs);
            __syncthreads();
            // vmcnt(0): the slice's first weights came with the rows, and the waits in the
            // loop over taps are for its own loads (to the compiler, else, for all of them)
            __builtin_amdgcn_s_waitcnt(0x0f70);
            rows_of(0, 0, as);
            frag(2, as, 0);
            frag(1, as, 0);
        }
        int kh = 0, kw = 0;  // of the tap after this one
        for (int tap = 0; tap < KK; ++tap) {
            const bool last = tap + 1 == KK;
            const int t1 = last ? 0 : tap + 1, s1 = last ? cs + 1 : cs;        // the next tap
            const int t2 = t1 + 1 == KK ? 0 : t1 + 1, s2 = t1 + 1 == KK ? s1 + 1 : s1;  // and the one after
            if (++kw == sh.K) kw = 0, ++kh;
            if (last) kh = 0;
            if constexpr (MODE != kHalo) {
                if (cs | tap) __syncthreads();  // the tap before has been read
                const int c = cs * kBK + 8 * ch;
                put_row(r0, v0, ok0, c);
                put_row(r0 + 64, v1, ok1, c);
                gather(min(s1, ncs - 1), kh, kw);  // the last one: a harmless reload, and no branch
                __syncthreads();
                rows_of(0, 0, as);
                frag(2, as, 0);
                frag(1, as, 0);
            }
            step(0, as, as, t1, s1 * kBK + 16);
            int nas[T];
            rows_of(t1, kh * sh.W + kw, nas);  // after the last tap: tap 0, read again once staged
            step(1, as, nas, t2, s2 * kBK);
#pragma unroll
            for (int t = 0; t < T; ++t) as[t] = nas[t];
        }
    }
#pragma unroll
    for (int t = 0; t < T; ++t) acc[t][0] += cor[t][0];
    if (split_failed<T, 1>(acc)) {
        // straight from memory in fp32, 2 k per MFMA; rare, so simple
#pragma unroll
        for (int t = 0; t < T; ++t) acc[t][0] = (f32x16){};
        for (int tap = 0; tap < KK; ++tap) {
            const int kh = tap / sh.K, kw = tap - kh * sh.K;
            const float* xp[T];
            bool ok[T];
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const int m = m0 + wrow + 32 * t + fr;
                uint32_t q, ow, b, oh;
                sh.wo.divmod((uint32_t)min(m, sh.M - 1), q, ow);
                sh.ho.divmod(q, b, oh);
                const int ih = (int)oh * sh.stride - sh.pad + kh, iw = (int)ow * sh.stride - sh.pad + kw;
                ok[t] = (m < sh.M) & ((unsigned)ih < (unsigned)sh.H) & ((unsigned)iw < (unsigned)sh.W);
                xp[t] = X + (size_t)(ok[t] ? ((int)b * sh.H + ih) * sh.W + iw : 0) * sh.Cin;
            }
            for (int c0 = 0; c0 < sh.Cin; c0 += 2) {
                const int c = min(c0 + fh, sh.Cin - 1);
                const bool in = c0 + fh < sh.Cin;
                const float wgt = FLIP ? Wt[((size_t)(KK - 1 - tap) * sh.Cout + nc) * sh.Cin + c]
                                       : Wt[(size_t)(tap * sh.Cin + c) * sh.Cout + nc];
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    const float x = xp[t][c];
                    acc[t][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(in && ok[t] ? x : 0.0f, in ? wgt : 0.0f, acc[t][0], 0, 0, 0);
                }
            }
        }
    }
    // Epilogue: lanes 0-31 and 32-63 each write 32 consecutive outputs of a row
    // 8 (r / 4) + 4 fh + r % 4.  The fused operands of a row tile are loaded
    // together; a row past M reads row M - 1 (harmless) and stores nothing.  Offsets are 32-bit
    // (the launcher bounds the tensors below 2^31 elements).
    const int mrow = m0 + wrow + 4 * fh;
    const bool mp = ep.mp != 0;
    const float bn = ep.bias ? ep.bias[nc] : 0.0f, g = ep.gain ? ep.gain[0] : 1.0f;
    auto off = [&](int t, int r) {
        return (uint32_t)(min(mrow + 32 * t + 8 * (r >> 2) + (r & 3), sh.M - 1) * sh.Cout + nc);
    };
    const bool full = m0 + kBM <= sh.M && n0 + BN <= sh.Cout;  // stores with no test per row
#pragma unroll
    for (int t = 0; t < T; ++t) {
        float e1[16], e2[16];
        if constexpr (XE != kXeNone) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                if constexpr ((XE & kXeRes) != 0) e1[r] = ep.res[off(t, r)];
                if constexpr ((XE & kXeActG) != 0) e2[r] = ep.xa[off(t, r)];
                if constexpr ((XE & kXeMod) != 0) {
                    uint32_t bb, q;
                    ep.hw.divmod((uint32_t)min(mrow + 32 * t + 8 * (r >> 2) + (r & 3), sh.M - 1), bb, q);
                    e2[r] = ep.cond[bb * (uint32_t)sh.Cout + (uint32_t)nc];
                }
            }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            if (!full && (mrow + 32 * t + 8 * (r >> 2) + (r & 3) >= sh.M || n >= sh.Cout)) continue;
            float v = acc[t][0][r];
            if (ep.bias) v = v + bn;
            else if (ep.gain) v = v * g;
            if constexpr ((XE & kXeActG) != 0) {
                const float d = act_grad<ACT_SILU, false>(e2[r]);
                v = v * (mp ? d * kMpSiluScale : d);
            }
            if constexpr ((XE & kXeRes) != 0) v = ep.wa * e1[r] + ep.wb * v;
            Y[off(t, r)] = v;
            if constexpr ((XE & kXeMod) != 0) {
                const float z = act_fwd<ACT_SILU, false>(v * (e2[r] + 1.0f));
                ep.y2[off(t, r)] = mp ? z * kMpSiluScale : z;
            }
        }
    }
}

// Host side: how the activations are staged, the tile, and the launch.

// Halo rows that leave room for two workgroups on a CU (160 KB of LDS), with
// the taps' bits in 32.
inline int conv_mode(const ConvShape& sh, const float* X, const float* Wt, bool flip) {
    const bool vec = sh.Cin % 8 == 0 && aligned16(X) && (!flip || aligned16(Wt));
    if (!vec) return kRagged;
    const int halo = kBM + 2 * sh.pad * (sh.W + 1);
    return sh.stride == 1 && sh.Ho == sh.H && sh.Wo == sh.W && sh.K <= 5 && (halo + 1) * kRowSlots * 16 <= 80000 ? kHalo
                                                                                                             : kGather;
}

// Columns per workgroup of the tiled kernels, or 0 for the small tiles: the
// least of the times, in us, that fit a sweep of 23 shapes (1x1 to 5x5, 3 to
// 1024 channels, 3 to 131072 rows).  A tiled workgroup by itself takes 0.75 us to
// stage a slice of 32 channels and `lone` us for each of its taps; the filled
// device 0.0014 us for a slice, `full` for a tap and 0.005 for the rest of each
// tile.  The small tiles (small_us) are bound by a wave's round trips of loads or by
// their vector work (which a flipped weight's scattered rows lengthen).  Forward
// at [8, 7 x 7, 128 -> 128]: small 6.2, 32 / 64 / 128 columns 25 / 33 / 46; [64, 8
// x 8, 448 -> 448]: 169, 111 / 103 / 138; [20, 40 x 40, 80 -> 200]: 177, 88 / 81 /
// 74; [4, 16 x 16, 256 -> 256]: 15, 45 / 59 / 80; [16, 16 x 16, 256 -> 256]: 56,
// 46 / 59 / 80.
inline int conv_tile(const ConvShape& sh, bool flip, double* best_us = nullptr) {
    struct Tile {
        int bn;
        double lone, full;
    };
    const Tile kTiles[] = {{128, 1.07, 0.00485}, {64, 0.74, 0.00255}, {32, 0.54, flip ? 0.00195 : 0.00175}};
    const double KK = (double)sh.K * sh.K;
    const double slices = (sh.Cin + 31) / 32;
    const double s16 = small_us(sh, flip, 16), s32 = small_us(sh, flip, 32);
    double best = s16 < s32 ? s16 : s32;
    if (best_us) *best_us = best;
    if (sh.Cin >= kMostChannels || sh.Cout >= kMostChannels) return 0;
    int bn = 0;
    for (const Tile& t : kTiles) {
        const double tiles = (double)((sh.M + kBM - 1) / kBM) * ((sh.Cout + t.bn - 1) / t.bn);
        // 128 columns reach the full rate with two workgroups on each CU only
        const double lone = slices * (0.75 + KK * t.lone);
        const double full = tiles * (slices * (0.0014 + KK * t.full) + 0.005) * (t.bn == 128 && tiles < 512 ? 1.16 : 1.0);
        const double us = 5.0 + (lone > full ? lone : full);
        if (us < best) best = us, bn = t.bn;
    }
    if (best_us) *best_us = best;
    return bn;
}

// Raises kernel fn's LDS limit to 80 KB (two workgroups a CU) on the current device,
// once a device: `done` has a bit for each that it was raised on.  False after
// recording an error.
inline bool lds_raised(const void* fn, std::atomic<unsigned long long>& done, const char* what) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess && dev >= 64) e = hipErrorInvalidDevice;
    if (e == hipSuccess && !(done.load(std::memory_order_relaxed) >> dev & 1)) {
        e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 81920);
        if (e == hipSuccess) done.fetch_or(1ull << dev, std::memory_order_relaxed);
    }
    if (e == hipSuccess) return true;
    (void)hipGetLastError();
    nnk_set_error((int)e, "%s: LDS of 80 KB on device %d: %s", what, dev, hipGetErrorString(e));
    return false;
}

template <bool FLIP, int XE>
void conv_launch(float* Y, const float* X, const float* Wt, const ConvShape& sh, const ConvEpi& ep, hipStream_t s,
    ConvPick pick = {}) {
    const int BN = pick.columns >= 0 ? pick.columns : conv_tile(sh, FLIP);
    const int own = conv_mode(sh, X, Wt, FLIP), mode = own > pick.staging ? own : pick.staging;
    if (BN == 0) {
        nnk_conv_small(FLIP, XE, Y, X, Wt, sh, ep, s);
        return;
    }
    const unsigned grid = (unsigned)((sh.M + kBM - 1) / kBM) * (unsigned)((sh.Cout + BN - 1) / BN);
    const int rows = mode == kHalo ? kBM + 2 * sh.pad * (sh.W + 1) + 1 : kBM;
    const size_t lds = (size_t)rows * kRowSlots * sizeof(uint4);
#define NNK_CONV(BN_, MODE_)                                                                                      \
    do {                                                                                                          \
        if (MODE_ == kHalo) {                                                                                     \
            static std::atomic<unsigned long long> done;                                                          \
            if (!lds_raised((const void*)conv_x3<BN_, MODE_, FLIP, XE>, done, "convolution")) return;             \
        }                                                                                                         \
        conv_x3<BN_, MODE_, FLIP, XE><<<grid, kTpb, lds, s>>>(Y, X, Wt, sh, ep);                                  \
    } while (0)
#define NNK_CONV_MODE(MODE_)                 \
    do {                                     \
        if (BN == 128) NNK_CONV(128, MODE_); \
        else if (BN == 64) NNK_CONV(64, MODE_); \
        else NNK_CONV(32, MODE_);            \
    } while (0)
    if (mode == kHalo) NNK_CONV_MODE(kHalo);
    else if (mode == kGather) NNK_CONV_MODE(kGather);
    else if constexpr (XE == kXeNone) NNK_CONV_MODE(kRagged);
    else nnk_conv_small(FLIP, XE, Y, X, Wt, sh, ep, s);  // the ragged form has no fused epilogues
#undef NNK_CONV_MODE
#undef NNK_CONV
}

// ---------------------------------------------------------------------------
// Weight gradient: gW[k, n] = sum_m A[m, k] dY[m, n] (the reference's
// gemm_dW over the im2col matrix, src/conv2d.c:44-47), with A gathered from X
// as in the forward.  The m reduction (B * Ho * Wo rows) is split over S
// workgroups per 128 x 128 output tile; split z writes its fixed-order partial
// tile to part[z], and a second launch adds the S partials in split order.
//
// Per stage a workgroup stages 16 pixel rows m of A (its 128 k columns) and of
// dY (its BN n columns) in LDS transposed and split: per plane and column, 16
// consecutive m, so that a lane's MFMA operands run along the pixel reduction.
// A loader thread's registers hold consecutive rows of a column, which is the
// transpose.
//
// What bounds it is the vector work beside the MFMAs: each wave splits its share
// of both operands and writes it to LDS in every stage (165 vector instructions
// to 48 MFMAs).  So the stages are pipelined: three LDS buffers and one barrier a
// stage, the next stage's fragment reads and splits and the one after's loads
// spread between the MFMAs.  3x3 128 -> 128 at [128, 32, 32]: 264 us with two
// barriers a stage, 247 so on one box (337 on the fp32 MFMA), 227 on a faster one;
// 256 -> 256 at [16, 64, 64]: 484, 457, 442.  The column sums of dY (a convolution's bias gradient) come from
// the rows that the workgroups of the first k tile hold anyway, instead of a
// pass over dY of two launches (5 us and more).
// ---------------------------------------------------------------------------
constexpr int kStage = 16;  // rows per stage

// How the activation columns are loaded: kSingles one by one, for any channel
// counts and alignments; kPairs two at a time (C_in even, x 8-byte aligned);
// kQuads also with W_out a multiple of 4, so that the four consecutive pixels of
// a loader thread lie in one output row and are decoded once (the decoding is
// scalar work, which a wave issues in turn with the rest: 148 scalar
// instructions beside 165 vector ones a stage without it).
enum { kQuads = 0, kPairs = 1, kSingles = 2 };

template <int BN, int LOADS>
__global__ __launch_bounds__(kTpb, 2) void igemm_wgrad(float* __restrict__ part, float* __restrict__ sums,
    size_t stride, const float* __restrict__ X, const float* __restrict__ dY, ConvShape sh, int rows_per_split) {
    constexpr int UT = BN / 64;                                // 32-column accumulator tiles per wave
    constexpr int PA = 128 * kStage4, PD = BN * kStage4;       // uint4 per plane
    constexpr int kBuf = kPlanes * (PA + PD);                  // and per stage buffer
    extern __shared__ uint4 lds[];                             // three stage buffers: A planes, dY planes
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 31, fh = lane >> 5;
    const int wk = w >> 1, wn = w & 1;
    // tile (k tile, n tile, split z), k tile fastest, in XCD-aware order
    const int KT = (sh.KKC + 127) / 128, NT = (sh.Cout + BN - 1) / BN;
    const int tl = xcd_order((int)blockIdx.x, (int)gridDim.x);
    const int k0 = (tl % KT) * 128, n0 = ((tl / KT) % NT) * BN, z = tl / (KT * NT);
    const int mbeg = z * rows_per_split;
    const int mend = min(sh.M, mbeg + rows_per_split);
    // loader roles.  A: columns k0 + 2 lane, + 1 of the stage's rows 4 w .. + 3
    // (the pixels of a wave are the same in all lanes, so they are decoded in
    // scalar registers); column 2 l + j goes to tile row l + 64 j, so that a
    // wave's 8-byte writes go to consecutive rows.  dY: column n0 + nd of rows
    // 8 md .. + 7 (with BN = 64 the upper two waves store none).
    constexpr int NC = LOADS == kSingles ? 2 : 1;  // column addresses of a pair
    int kh[NC], kw[NC];
    uint32_t xo[NC];  // the column's offset from the output pixel's input pixel (wraps below it)
#pragma unroll
    for (int j = 0; j < NC; ++j) {
        // columns past the end compute the last ones, stored nowhere
        const int kcol = min(k0 + 2 * lane + j, sh.KKC - (NC == 2 ? 1 : 2)), tap = kcol / sh.Cin;
        kh[j] = tap / sh.K - sh.pad;
        kw[j] = tap % sh.K - sh.pad;
        xo[j] = (uint32_t)((kh[j] * sh.W + kw[j]) * sh.Cin + kcol - tap * sh.Cin);
    }
    const int nd = tid % BN, md = (w / (BN / 64)) & 1;
    const bool dput = tid < 2 * BN;
    const int dlo = 4 * (min(n0 + nd, sh.Cout - 1) - n0);

    // Every lane loads (rows past the end, padding and columns past the end read
    // a valid address): a branch around a load would make the compiler's later
    // waits drain the whole vector-memory counter.  A's rows past the end and
    // padding are zeroed as they are split.
    float2 va[4];
    float vd[8];
    uint32_t aok[NC][4];  // all ones where the pixel counts: a mask, as a select would become a branch
    auto load = [&](int ms) {
        // decode the first of the 4 rows, then step along the output row
        const int mf = ms + 4 * w;
        uint32_t t, ow, b, oh;
        sh.wo.divmod((uint32_t)(mf < sh.M ? mf : 0), t, ow);
        sh.ho.divmod(t, b, oh);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int ih = (int)oh * sh.stride, iw = (int)(LOADS == kQuads ? ow + q : ow) * sh.stride;
            // 32-bit element offsets (the host bounds x below 2^31 elements)
            const uint32_t px = (((uint32_t)b * sh.H + ih) * sh.W + iw) * sh.Cin;
            float v[NC + 1];
#pragma unroll
            for (int j = 0; j < NC; ++j) {
                aok[j][q] = -(uint32_t)((mf + q < mend) & ((unsigned)(ih + kh[j]) < (unsigned)sh.H) &
                                        ((unsigned)(iw + kw[j]) < (unsigned)sh.W));
                const uint32_t o = (px + xo[j]) & aok[j][q];
                if constexpr (NC == 2) v[j] = X[o];
                else va[q] = *reinterpret_cast<const float2*>(X + o);
            }
            if constexpr (NC == 2) va[q] = make_float2(v[0], v[1]);
            if constexpr (LOADS != kQuads) {
                if (++ow == (uint32_t)sh.Wo) {
                    ow = 0;
                    if (++oh == (uint32_t)sh.Ho) {
                        oh = 0;
                        ++b;
                    }
                }
            }
        }
        const int dm = min(ms + 8 * md, mend - 1);
        const auto db = buffer(dY + (size_t)dm * sh.Cout + n0);
        const int dlim = 4 * min(7, mend - 1 - dm) * sh.Cout;  // rows past the end read the last
#pragma unroll
        for (int q = 0; q < 8; ++q)
            vd[q] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(db, dlo,
                min(4 * q * sh.Cout, dlim), 0));
    };
    const int wa = stage_slot(lane, w >> 1) * 2 + (w & 1), wb = stage_slot(lane + 64, w >> 1) * 2 + (w & 1);
    const int wd = stage_slot(nd, md);
    auto store = [&](uint4* buf) {
        uint2* a2 = reinterpret_cast<uint2*>(buf);
        uint32_t lo[kPlanes], hi[kPlanes];
        split2(__uint_as_float(__float_as_uint(va[0].x) & aok[0][0]), __uint_as_float(__float_as_uint(va[1].x) & aok[0][1]), lo);
        split2(__uint_as_float(__float_as_uint(va[2].x) & aok[0][2]), __uint_as_float(__float_as_uint(va[3].x) & aok[0][3]), hi);
#pragma unroll
        for (int p = 0; p < kPlanes; ++p) a2[p * PA * 2 + wa] = make_uint2(lo[p], hi[p]);
        split2(__uint_as_float(__float_as_uint(va[0].y) & aok[NC - 1][0]), __uint_as_float(__float_as_uint(va[1].y) & aok[NC - 1][1]), lo);
        split2(__uint_as_float(__float_as_uint(va[2].y) & aok[NC - 1][2]), __uint_as_float(__float_as_uint(va[3].y) & aok[NC - 1][3]), hi);
#pragma unroll
        for (int p = 0; p < kPlanes; ++p) a2[p * PA * 2 + wb] = make_uint2(lo[p], hi[p]);
        uint4 d[kPlanes];
        split8(vd, d);
        if (BN == 128 || dput) {
#pragma unroll
            for (int p = 0; p < kPlanes; ++p) buf[kPlanes * PA + p * PD + wd] = d[p];
        }
    };
    // Column sums of dY, from the workgroups of the first k tile: the rows that
    // are about to be split, once a stage (a uniform branch of its own, outside
    // the scheduled parts).
    const bool summing = sums != nullptr && k0 == 0;
    float bs = 0.0f;
    auto add_rows = [&](int ms) {
        if (!summing) return;
        float v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = ms + 8 * md + q < mend ? vd[q] : 0.0f;
        bs += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    };
    f32x16 acc[2][UT], cor[2][UT];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int u = 0; u < UT; ++u) acc[t][u] = cor[t][u] = (f32x16){};

    // Stages of 16 rows in three buffers: while stage s is computed, stage s + 2
    // is split and written to the buffer that stage s - 1 left, the fragments of
    // stage s + 1 are read and the rows of stage s + 3 loaded, all between the
    // MFMAs (sched), with one barrier a stage.  Planes 1 and 2 of A and 0 and 1
    // of dY are in registers when the stage begins (dY's in two sets, as both
    // halves of a stage use them); the others are read during the first half.
    const int sa = stage_slot(wk * 64 + fr, fh), sd = stage_slot(wn * (BN / 2) + fr, fh);
    uint4 a[kPlanes][2], d2[UT], ds[2][2][UT];
    auto frag_a = [&](const uint4* buf, int p) {
#pragma unroll
        for (int t = 0; t < 2; ++t) a[p][t] = buf[p * PA + 32 * t * kStage4 + sa];
    };
    auto frag_d = [&](const uint4* buf, int p, uint4 (&d)[UT]) {
#pragma unroll
        for (int u = 0; u < UT; ++u) d[u] = buf[kPlanes * PA + p * PD + 32 * u * kStage4 + sd];
    };
    auto mul = [&](int i, const uint4 (&d)[UT], f32x16 (&o)[2][UT]) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int u = 0; u < UT; ++u)
                o[t][u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[i][t]),
                    __builtin_bit_cast(bf16x8, d[u]), o[t][u], 0, 0, 0);
    };
    const int nst = (mend - mbeg + kStage - 1) / kStage;
    auto row = [&](int s) { return mbeg + min(s, nst - 1) * kStage; };  // past the last: a harmless reload
    uint4 *b0 = lds, *b1 = lds + kBuf, *b2 = lds + 2 * kBuf;
    auto stage = [&](int s, const uint4 (&d)[2][UT], uint4 (&dn)[2][UT]) {
        add_rows(mbeg + (s + 2) * kStage);  // past the last stage: no rows
        frag_a(b0, 0);
        frag_d(b0, 2, d2);
        mul(2, d[0], cor);
        mul(1, d[1], cor);
        mul(1, d[0], cor);
        store(b2);
        sched<6 * UT, 8>();
        __builtin_amdgcn_sched_barrier(0);
        frag_a(b1, 2);
        frag_a(b1, 1);
        frag_d(b1, 0, dn[0]);
        frag_d(b1, 1, dn[1]);
        load(row(s + 3));  // into the registers just split
        mul(0, d2, cor);
        mul(0, d[1], cor);
        mul(0, d[0], acc);
        sched<6 * UT>();
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        uint4* t = b0;
        b0 = b1;
        b1 = b2;
        b2 = t;
    };
    if (nst > 0) {
        load(row(0));
        add_rows(mbeg);
        store(b0);
        load(row(1));
        add_rows(mbeg + kStage);
        store(b1);
        load(row(2));
        __syncthreads();
        frag_a(b0, 2);
        frag_a(b0, 1);
        frag_d(b0, 0, ds[0][0]);
        frag_d(b0, 1, ds[0][1]);
        for (int s = 0;;) {
            stage(s, ds[0], ds[1]);
            if (++s == nst) break;
            stage(s, ds[1], ds[0]);
            if (++s == nst) break;
        }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int u = 0; u < UT; ++u) acc[t][u] += cor[t][u];
    if (split_failed<2, UT>(acc)) {
        // straight from memory in fp32, 2 pixels per MFMA; rare, so simple
        int tp[2], cc[2];
        bool ck[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int k = k0 + 2 * (32 * t + fr) + wk;  // the column of tile row wk 64 + 32 t + fr
            ck[t] = k < sh.KKC;
            tp[t] = ck[t] ? k / sh.Cin : 0;
            cc[t] = ck[t] ? k - tp[t] * sh.Cin : 0;
#pragma unroll
            for (int u = 0; u < UT; ++u) acc[t][u] = (f32x16){};
        }
        for (int ms = mbeg; ms < mend; ms += 2) {
            const int m = ms + fh;
            const bool in = m < mend;
            uint32_t q, ow, b, oh;
            sh.wo.divmod((uint32_t)(in ? m : mbeg), q, ow);
            sh.ho.divmod(q, b, oh);
            float av[2], dv[UT];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int th = tp[t] / sh.K, tw = tp[t] - th * sh.K;
                const int ih = (int)oh * sh.stride - sh.pad + th, iw = (int)ow * sh.stride - sh.pad + tw;
                const bool ok = in & ck[t] & ((unsigned)ih < (unsigned)sh.H) & ((unsigned)iw < (unsigned)sh.W);
                const float v = X[(size_t)(ok ? ((int)b * sh.H + ih) * sh.W + iw : 0) * sh.Cin + cc[t]];
                av[t] = ok ? v : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < UT; ++u) {
                const float v = dY[(size_t)(in ? m : mbeg) * sh.Cout + min(n0 + wn * (BN / 2) + 32 * u + fr, sh.Cout - 1)];
                dv[u] = in ? v : 0.0f;
            }
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int u = 0; u < UT; ++u)
                    acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[t], dv[u], acc[t][u], 0, 0, 0);
        }
    }
    // partial tile: D[row][n], rows 32 t + 8 (r / 4) + 4 fh + r % 4 of the wave's
    // 64, which hold the even (wk = 0) or odd columns k; past the end nothing is
    // stored
    float* pb = part + z * stride + n0 + wn * (BN / 2) + fr;
#pragma unroll
    for (int u = 0; u < UT; ++u)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int k = k0 + 2 * (32 * t + 8 * (r >> 2) + 4 * fh + (r & 3)) + wk;
                if (k < sh.KKC && n0 + wn * (BN / 2) + 32 * u + fr < sh.Cout)
                    pb[(size_t)k * sh.Cout + 32 * u] = acc[t][u][r];
            }
    if (summing) {
        // the two halves of the rows, in order (the tile loop left LDS behind its barrier)
        float* l = reinterpret_cast<float*>(lds);
        if (dput) l[tid] = bs;
        __syncthreads();
        if (tid < BN && n0 + tid < sh.Cout) sums[z * stride + n0 + tid] = l[tid] + l[tid + BN];
    }
}

// out[i] = part[0][i] + part[1][i] + ... (split order), n elements a split, of
// which those from nw on (the column sums of dY, where they were asked for) go
// to gb.
__global__ __launch_bounds__(256) void wgrad_reduce(float* __restrict__ gW, float* __restrict__ gb,
    const float* __restrict__ part, int S, long long n, long long nw) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    // kB slices in flight, added in slice order
    constexpr int kB = 8;
    float t = part[i];
    int z = 1;
    for (; z + kB <= S; z += kB) {
        float v[kB];
#pragma unroll
        for (int u = 0; u < kB; ++u) v[u] = part[(size_t)(z + u) * n + i];
#pragma unroll
        for (int u = 0; u < kB; ++u) t += v[u];
    }
    for (; z < S; ++z) t += part[(size_t)z * n + i];
    if (i < nw) gW[i] = t;
    else gb[i - nw] = t;
}

// The same for many slices (S beyond kTallS) of few elements (up to kTallN): 16
// waves share the slices of 64 elements, eight in flight each, and add their
// sums in order.  [27, 64] in 512 slices: 32 -> 5 us; at [1152, 128] in 56 the
// elements alone fill the device, 7.6 us against 10.6.
constexpr int kTallS = 24;
constexpr long long kTallN = 32768;
__global__ __launch_bounds__(1024) void wgrad_reduce_tall(float* __restrict__ gW, float* __restrict__ gb,
    const float* __restrict__ part, int S, long long n, long long nw) {
    __shared__ float l[16][kWave];
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    const long long i = (long long)blockIdx.x * kWave + lane;
    float t = 0.0f;
    if (i < n) {
        constexpr int kB = 8;
        int z = wid;
        for (; z + (kB - 1) * 16 < S; z += kB * 16) {
            float v[kB];
#pragma unroll
            for (int u = 0; u < kB; ++u) v[u] = part[(size_t)(z + 16 * u) * n + i];
#pragma unroll
            for (int u = 0; u < kB; ++u) t += v[u];
        }
        for (; z < S; z += 16) t += part[(size_t)z * n + i];
    }
    l[wid][lane] = t;
    __syncthreads();
    if (wid == 0 && i < n) {
        float a = l[0][lane];
#pragma unroll
        for (int w = 1; w < 16; ++w) a += l[w][lane];
        if (i < nw) gW[i] = a;
        else gb[i - nw] = a;
    }
}

struct WgradPlan {
    int S, rows;
};

// 128 columns a workgroup above 64: a tile of 64 takes more than half as long.
inline int tile_n(int Cout) { return Cout > 64 ? 128 : 64; }

// At most as many splits as one round of resident workgroups holds (two per CU
// on 256 CUs), of kWgM rows at least.  A plan may have fewer, its rows being
// multiples of kWgM, so the splits do not grow with M (3x3 64 -> 64: 52 at
// 3300 rows, 100 at 3200); this bound does, and sizes the workspaces, which
// serve every smaller batch.
inline int wgrad_most_splits(int M, int KKC, int Cout) {
    const int tiles = ((KKC + 127) / 128) * ((Cout + tile_n(Cout) - 1) / tile_n(Cout));
    const int S = tiles >= 512 ? 1 : 512 / tiles, smax = (M + kWgM - 1) / kWgM;
    return S > smax ? smax : S;
}

inline WgradPlan wgrad_plan(int M, int KKC, int Cout) {
    const int S = wgrad_most_splits(M, KKC, Cout);
    int rows = (M + S - 1) / S;
    rows = (rows + kWgM - 1) / kWgM * kWgM;
    WgradPlan p;
    p.rows = rows;
    p.S = (M + rows - 1) / rows;
    return p;
}

// Whether the small tiles beat the tiled kernel, by times in us that fit the
// sweep of conv_tile: the small tiles are bound by round trips or by their
// vector work, the tiled kernel takes a time for every 32 rows of a split, then
// the sum of the splits.  For example [8, 7 x 7, 128 -> 128]: small 8.2, tiled 17
// us; dense [128, 512 -> 512]: 4.9, 14; [8, 28 x 28, 32 -> 32]: 59, 19; [16, 16 x
// 16, 256 -> 256]: 113, 50.
inline bool wgrad_small_wins(const ConvShape& sh) {
    if (sh.Cout >= kMostChannels) return true;
    const double steps = (sh.M + 15) / 16, cells = (double)((sh.KKC + 31) / 32) * ((sh.Cout + 31) / 32);
    const double waves = waves_for((int)steps);
    const bool dense = sh.K == 1 && sh.stride == 1 && sh.pad == 0;  // no pixels to decode
    const double trips = (dense ? 0.9 : 2.3) * ceil(steps / waves), work = (dense ? 0.0005 : 0.00078) * cells * steps;
    const WgradPlan p = wgrad_plan(sh.M, sh.KKC, sh.Cout);
    const double stage = tile_n(sh.Cout) == 128 ? 3.0 : 2.0;
    return 4.0 + (trips > work ? trips : work) < 12.0 + stage * (p.rows / kWgM);
}

// Floats of partial sums that the tiled kernel leaves, 0 where it writes the result.
inline size_t wgrad_scratch(const ConvShape& sh, bool sums) {
    const WgradPlan p = wgrad_plan(sh.M, sh.KKC, sh.Cout);
    return p.S > 1 ? (size_t)p.S * ((size_t)sh.KKC * sh.Cout + (sums ? sh.Cout : 0)) : 0;
}

// The tiled weight gradient of a checked, non-empty shape, and with gb non-null
// the column sums of dY.
inline void wgrad_run(const char* what, float* gW, float* gb, const float* X, const float* dY, const ConvShape& sh,
    float* workspace, hipStream_t s, ConvPick pick = {}) {
    const WgradPlan p = wgrad_plan(sh.M, sh.KKC, sh.Cout);
    const long long nw = (long long)sh.KKC * sh.Cout, n = nw + (gb ? sh.Cout : 0);
    float *part = gW, *sums = gb;
    bool pooled = false;
    if (p.S > 1) {
        if (workspace) {
            part = workspace;
        } else {
            part = nnk_scratch_acquire((size_t)p.S * n, s, what);
            if (!part) return;
            pooled = true;
        }
        if (gb) sums = part + nw;
    }
    const int BN = tile_n(sh.Cout);
    const dim3 grid((unsigned)((sh.KKC + 127) / 128) * (unsigned)((sh.Cout + BN - 1) / BN) * (unsigned)p.S);
    const int own = sh.Cin % 2 || (uintptr_t)X % 8 ? kSingles : sh.Wo % 4 ? kPairs : kQuads;
    const int loads = own > pick.staging ? own : pick.staging;
    const size_t lds = (size_t)3 * kPlanes * (128 + BN) * kStage4 * sizeof(uint4);
    bool ok = false;
#define NNK_WGRAD(BN_, LOADS_)                                                                                 \
    do {                                                                                                       \
        static std::atomic<unsigned long long> done;                                                           \
        if (!(ok = lds_raised((const void*)igemm_wgrad<BN_, LOADS_>, done, what))) break;                      \
        igemm_wgrad<BN_, LOADS_><<<grid, kTpb, lds, s>>>(part, sums, (size_t)n, X, dY, sh, p.rows);            \
    } while (0)
#define NNK_WGRAD_LOADS(BN_)                            \
    do {                                                \
        if (loads == kQuads) NNK_WGRAD(BN_, kQuads);    \
        else if (loads == kPairs) NNK_WGRAD(BN_, kPairs); \
        else NNK_WGRAD(BN_, kSingles);                  \
    } while (0)
    if (BN == 128) NNK_WGRAD_LOADS(128);
    else NNK_WGRAD_LOADS(64);
#undef NNK_WGRAD_LOADS
#undef NNK_WGRAD
    if (ok && p.S > 1) {
        if (p.S > kTallS && n <= kTallN)
            wgrad_reduce_tall<<<(unsigned)((n + kWave - 1) / kWave), 1024, 0, s>>>(gW, gb, part, p.S, n, nw);
        else wgrad_reduce<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(gW, gb, part, p.S, n, nw);
    }
    if (pooled) nnk_scratch_release(part, s);
}

inline void wgrad_launch(const char* what, float* gW, const float* X, const float* dY, int batch, int H, int W, int C_in,
    int C_out, int K, int stride, int pad, int H_out, int W_out, float* workspace, hipStream_t s) {
    ConvShape sh;
    if (wgrad_setup(what, gW, X, dY, batch, H, W, C_in, C_out, K, stride, pad, H_out, W_out, s, sh) <= 0) return;
    if (wgrad_small_wins(sh)) nnk_wgrad_small(gW, nullptr, X, dY, sh, s);
    else wgrad_run(what, gW, nullptr, X, dY, sh, workspace, s);
    nnk_after_launch(what, s);
}

}  // namespace

