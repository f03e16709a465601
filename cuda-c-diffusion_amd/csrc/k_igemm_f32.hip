// k_igemm_f32.hip -- the convolutions of the weight-normalised conv2d modules
// (magnitude-preserving, with a gain) on the fp32 matrix cores
// (v_mfma_f32_32x32x2f32): forward, stride-1 input gradient and weight gradient as
// implicit GEMMs, the same sums as k_igemm.hip's (src/conv2d.c:17-66).
//
// Why not the bf16 planes, which are faster and closer to 64 bits: these modules
// train a gain by sum_j <Wn_j, gW_j>, a sum of terms of either sign.  What is left of
// it can be a hundredth of what was added, and another summation order of the
// products is then a visibly other number: in the [128, 32, 32, 128] residual block
// (12 inputs, sums of deviation 1.7) the planes' gain gradients are 0.8e-6 from 64
// bits and these 1.7e-6, and for 2 of the 12 the two differ by more than 2e-5 of the
// number itself.  A training run that is compared with an earlier one, or goes on
// from its checkpoint, has to find the gradients that it had.  What it costs: 3x3,
// 128 -> 128 at [128, 32, 32] forward 320 us against 184, input gradient 317 against
// 188, weight gradient 337 against 227.
//
// The im2col matrix is never written: each workgroup gathers its A tile from X
// directly (a k-slice of 32 channels of one (kh, kw) is 128 contiguous bytes
// of one input pixel).  The weight is read in the reference's layout too, with
// no transposed or flipped copy: the forward stages its [32 k][BN n] slice as
// it lies in Wt and reads the B operand 32 bits at a time; the input
// gradient's operand B[ci][(kh, kw, co)] = Wt[((K-1-kh) K + (K-1-kw)) C_in +
// ci][co] is k-contiguous and is staged like A.
//
// Workgroup tile 128 (m) x BN (n, 128 or 64), k in slices of 32; 4 waves of
// 64 x BN/2, each a 2 x BN/64 grid of 32 x 32 MFMA accumulators.  Per slice a
// thread loads 4 float4 of A and up to 4 of the weight into registers, the
// slice before it computes from LDS, then the registers go to the other LDS
// buffer (two buffers of 2 x 16 KB; two workgroups fit a CU).  A tiles (and
// the input gradient's B) are [128 rows][8 float4 chunks of 4 k] with the
// chunk index xor-swizzled by the row (slot()), so the 128-bit fragment reads
// of a wave (32 rows, one chunk per half-wave) and the tile writes are free of
// bank conflicts.  The forward's B tile is [32 k][BN n], each row rotated by
// 32 n on alternate groups of 4 rows (kslot()), so the two half-waves of a
// 32-bit fragment read (rows k and k + 4, 32 consecutive n each) use
// disjoint banks.
//
// Lane layout of v_mfma_f32_32x32x2f32 (checked on the device): lane l supplies
// A[l % 32][l / 32] and B[l / 32][l % 32]; accumulator register r of lane l
// holds D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32].  A 128-bit fragment read
// gives a lane 4 consecutive k of its row; component c feeds the c-th MFMA,
// which pairs k = 4h + c of the two half-waves h: any pairing of k is the same
// sum, as long as A and B use the same one.
//
// Summation order: each output is a fixed-order fp32 sum (per slice, pairs of k in
// MFMA order, slices in k order).
#include "conv_api.h"
#include "conv_common.h"

namespace {

using namespace nnk;
using namespace nnk::conv;

constexpr int kTpb = 256;

// float4 slot of (row, chunk) in a [128][8] tile.  The xor spreads any 8
// consecutive rows of one chunk over the 8 chunk positions, and any 16
// consecutive rows over distinct (row parity, position) pairs, so 128-bit
// accesses whose lane groups cover 128 or 256 bytes of banks do not conflict.
__device__ __forceinline__ int slot(int row, int chunk) {
    return row * 8 + (chunk ^ (row & 7) ^ ((row >> 3) & 1));
}

// float offset of (k, n) in a [32][BN] B tile: rows 4..7 of every 8 rotated by 32
template <int BN>
__device__ __forceinline__ int kslot(int k, int n) {
    return k * BN + ((n + 32 * ((k >> 2) & 1)) & (BN - 1));
}

// Y[m, n] = gain[0] sum_k A[m, k] B[k, n], then the fused neighbour (activation:
// MP-SiLU).  FLIP: as conv_x3's (igemm.h).
template <int BN, bool FLIP, int XE>
__global__ __launch_bounds__(kTpb, 2) void conv_f32(float* __restrict__ Y, const float* __restrict__ X,
    const float* __restrict__ Wt, ConvShape sh, ConvEpi ep) {
    constexpr int UT = BN / 64;  // 32-column accumulator tiles per wave
    // weight float4 loaded per thread: a 4 x 4 block (forward) or BN / 32
    // rows of one chunk (flipped)
    constexpr int BQ = !FLIP ? 4 : BN / 32;
    constexpr int NQ = BN / 4;   // forward: n quads of the tile
    __shared__ float4 As[2][kBM * 8];
    __shared__ float4 Bs[2][BN * 8];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wm = w >> 1, wn = w & 1;
    const int m0 = blockIdx.x * kBM, n0 = blockIdx.y * BN;
    // loader role: chunk ch of rows r0 + 32 q
    const int ch = tid & 7, r0 = tid >> 3;
    int pix[4], ihb[4], iwb[4];
    bool rok[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int m = m0 + r0 + 32 * q;
        rok[q] = m < sh.M;
        const int mm = rok[q] ? m : 0;
        uint32_t t, ow, b, oh;
        sh.wo.divmod((uint32_t)mm, t, ow);
        sh.ho.divmod(t, b, oh);
        pix[q] = (int)b * sh.H * sh.W;
        ihb[q] = (int)oh * sh.stride - sh.pad;
        iwb[q] = (int)ow * sh.stride - sh.pad;
    }
    // forward weight roles: n quad n4, k rows 4 kq .. 4 kq + 3 of the slice
    // (with BN = 64 the second half of the workgroup repeats the first's
    // loads and stores nothing: every lane loads, see below)
    const int n4 = tid % NQ, kq = (tid / NQ) % 8;
    const bool bput = NQ * 8 >= kTpb || tid < NQ * 8;
    const float* wq = Wt + (size_t)(4 * kq) * sh.Cout + n0 + 4 * n4;
    // flipped weight: row n0 + r0 + 32 q of the tap's [C_in][C_out] block
    const float* wrow = Wt + (size_t)(n0 + r0) * sh.Cin + ch * 4;
    const int KK = sh.K * sh.K;

    // Every lane loads (a padding position reads channel ci of pixel 0 and is
    // zeroed when stored): a branch around a load would make the compiler's
    // later waits drain the whole vector-memory counter, i.e. wait for the
    // next slice's loads before the current slice's MFMAs.
    // Two register sets: the slice two ahead is loaded while the next one is
    // written to LDS, so a load has two slices of MFMA work to arrive.
    struct Regs {
        float4 a[4], b[BQ];
        bool ok[4];
    };
    Regs R0, R1;
    auto load = [&](int kt, Regs& R) {
        const int k0 = kt * kBK;
        const int khw = k0 / sh.Cin, cs = k0 - khw * sh.Cin, ci = cs + ch * 4;
        const int kh = khw / sh.K, kw = khw - kh * sh.K;
        // flipped weight: the slice's channels cs.. of tap KK-1-khw, a
        // uniform offset from each lane's row (held in a scalar register)
        const int wfo = __builtin_amdgcn_readfirstlane((KK - 1 - khw) * sh.Cout * sh.Cin + cs);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int ih = ihb[q] + kh, iw = iwb[q] + kw;
            R.ok[q] = rok[q] & ((unsigned)ih < (unsigned)sh.H) & ((unsigned)iw < (unsigned)sh.W);
            const int p = R.ok[q] ? pix[q] + ih * sh.W + iw : 0;
            R.a[q] = ld4(X + (size_t)p * sh.Cin + ci);
            if constexpr (!FLIP) R.b[q] = ld4(wq + (size_t)(k0 + q) * sh.Cout);
            else if (q < BQ) R.b[q] = ld4(wrow + wfo + 32 * q * sh.Cin);
        }
    };
    // Padding is zeroed by masking the bits (a select of whole float4 values
    // becomes a select of their addresses, which puts them in scratch memory).
    auto store = [&](int buf, const Regs& R) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const unsigned mk = R.ok[q] ? 0xffffffffu : 0u;
            const float4 a = R.a[q];
            float4 v;
            v.x = __uint_as_float(__float_as_uint(a.x) & mk);
            v.y = __uint_as_float(__float_as_uint(a.y) & mk);
            v.z = __uint_as_float(__float_as_uint(a.z) & mk);
            v.w = __uint_as_float(__float_as_uint(a.w) & mk);
            As[buf][slot(r0 + 32 * q, ch)] = v;
            if constexpr (FLIP) {
                if (q < BQ) Bs[buf][slot(r0 + 32 * q, ch)] = R.b[q];
            }
        }
        // forward: k rows 4 kq + i, n 4 n4 .. 4 n4 + 3, as loaded
        if constexpr (!FLIP) {
            if (bput) {
                float* bs = reinterpret_cast<float*>(&Bs[buf][0]);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    *reinterpret_cast<float4*>(bs + kslot<BN>(4 * kq + i, 4 * n4)) = R.b[i];
            }
        }
    };

    f32x16 acc[2][UT];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int u = 0; u < UT; ++u) acc[t][u] = (f32x16){};
    const int nk = sh.KKC / kBK;
    const int fr = lane & 31, fh = lane >> 5;
    const float g = ep.gain[0];
    // Fragments of a k quarter (8 k: one 128-bit read per row tile) and the
    // 16 MFMAs on them.  The next quarter's reads are issued before the
    // current quarter's MFMAs (two fragment register sets; the scheduling
    // barriers keep the compiler from sinking the reads below the MFMAs, which
    // would leave the matrix core idle for the LDS latency of every quarter).
    auto frag = [&](int buf, int kq, float4 (&a)[2], float4 (&b)[UT]) {
        const int c = 2 * kq + fh;
#pragma unroll
        for (int t = 0; t < 2; ++t) a[t] = As[buf][slot(wm * 64 + 32 * t + fr, c)];
        if constexpr (!FLIP) {
            // component j of b[u] = B[k = 4 c + j][n]: rows 8 kq + 4 fh + j
            const float* bs = reinterpret_cast<const float*>(&Bs[buf][0]);
#pragma unroll
            for (int u = 0; u < UT; ++u) {
                const int n = wn * (BN / 2) + 32 * u + fr;
                b[u].x = bs[kslot<BN>(4 * c + 0, n)];
                b[u].y = bs[kslot<BN>(4 * c + 1, n)];
                b[u].z = bs[kslot<BN>(4 * c + 2, n)];
                b[u].w = bs[kslot<BN>(4 * c + 3, n)];
            }
        } else {
#pragma unroll
            for (int u = 0; u < UT; ++u) b[u] = Bs[buf][slot(wn * (BN / 2) + 32 * u + fr, c)];
        }
    };
    auto mfmas = [&](const float4 (&a)[2], const float4 (&b)[UT]) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int u = 0; u < UT; ++u) acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t].x, b[u].x, acc[t][u], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int u = 0; u < UT; ++u) acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t].y, b[u].y, acc[t][u], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int u = 0; u < UT; ++u) acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t].z, b[u].z, acc[t][u], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int u = 0; u < UT; ++u) acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t].w, b[u].w, acc[t][u], 0, 0, 0);
    };
    auto compute = [&](int buf) {
        float4 a0[2], b0[UT], a1[2], b1[UT];
        frag(buf, 0, a0, b0);
        frag(buf, 1, a1, b1);
        __builtin_amdgcn_sched_barrier(0);
        mfmas(a0, b0);
        __builtin_amdgcn_sched_barrier(0);
        frag(buf, 2, a0, b0);
        __builtin_amdgcn_sched_barrier(0);
        mfmas(a1, b1);
        __builtin_amdgcn_sched_barrier(0);
        frag(buf, 3, a1, b1);
        __builtin_amdgcn_sched_barrier(0);
        mfmas(a0, b0);
        __builtin_amdgcn_sched_barrier(0);
        mfmas(a1, b1);
    };
    // Slices: prologue, a branch-free steady loop over pairs of slices (slice
    // kt computes from LDS buffer kt % 2 while R[kt % 2] receives slice kt + 2
    // and R[(kt + 1) % 2] goes to the other buffer; the second load of a pair
    // is clamped to the last slice, a harmless reload), then the one or two
    // slices left.
    load(0, R0);
    if (nk > 1) load(1, R1);
    store(0, R0);
    __syncthreads();
    int kt = 0;
    for (; kt + 2 < nk; kt += 2) {
        load(kt + 2, R0);
        compute(0);
        store(1, R1);
        __syncthreads();
        load(min(kt + 3, nk - 1), R1);
        compute(1);
        store(0, R0);
        __syncthreads();
    }
    // Fused epilogue operands: all of a lane's are loaded at the start of the
    // epilogue, one round trip (the main loop's registers are free by then).
    // A row past M reads row M - 1 (harmless) and stores nothing.  Offsets are
    // 32-bit (the launcher bounds the tensors below 2^31 elements).
    const int mrow = m0 + wm * 64 + 4 * fh, ncol = n0 + wn * (BN / 2) + fr;
    const int rowlim = sh.M - 1 - mrow;
    const uint32_t lofs = (uint32_t)(mrow * sh.Cout + ncol);
    float e1[UT][2][16], e2[UT][2][16];
    auto fetch = [&](int u) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int d = min(32 * t + 8 * (r >> 2) + (r & 3), rowlim);
                const uint32_t off = lofs + (uint32_t)(d * sh.Cout + 32 * u);
                if constexpr ((XE & kXeRes) != 0) e1[u][t][r] = ep.res[off];
                if constexpr ((XE & kXeActG) != 0) e2[u][t][r] = ep.xa[off];
                if constexpr ((XE & kXeMod) != 0) {
                    uint32_t bb, q;
                    ep.hw.divmod((uint32_t)(mrow + d), bb, q);
                    e2[u][t][r] = ep.cond[bb * (uint32_t)sh.Cout + (uint32_t)(ncol + 32 * u)];
                }
            }
    };
    compute(0);
    if (kt + 1 < nk) {
        store(1, R1);
        __syncthreads();
        compute(1);
    }

    // epilogue: lanes 0-31 and 32-63 each write 32 consecutive outputs of a
    // row.  A full row tile stores with no per-row test (a branch per store
    // would make every store wait for all earlier ones).
    auto out = [&](int t, int u, int r) { return acc[t][u][r] * g; };
    float* yb = Y + (size_t)(m0 + wm * 64 + 4 * fh) * sh.Cout + n0 + wn * (BN / 2) + fr;
    if constexpr (XE != kXeNone) {
#pragma unroll
        for (int u = 0; u < UT; ++u) fetch(u);
#pragma unroll
        for (int u = 0; u < UT; ++u) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int dm = 32 * t + 8 * (r >> 2) + (r & 3);
                    if (mrow + dm >= sh.M) continue;
                    float v = out(t, u, r);
                    if constexpr ((XE & kXeActG) != 0) v = v * act_grad<ACT_MP_SILU, false>(e2[u][t][r]);
                    if constexpr ((XE & kXeRes) != 0) v = ep.wa * e1[u][t][r] + ep.wb * v;
                    yb[(size_t)dm * sh.Cout + 32 * u] = v;
                    if constexpr ((XE & kXeMod) != 0)
                        ep.y2[(size_t)(mrow + dm) * sh.Cout + ncol + 32 * u] =
                            act_fwd<ACT_MP_SILU, false>(v * (e2[u][t][r] + 1.0f));
                }
        }
    } else if (m0 + kBM <= sh.M) {
#pragma unroll
        for (int u = 0; u < UT; ++u)
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    yb[(size_t)(32 * t + 8 * (r >> 2) + (r & 3)) * sh.Cout + 32 * u] = out(t, u, r);
    } else {
#pragma unroll
        for (int u = 0; u < UT; ++u)
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int dm = 32 * t + 8 * (r >> 2) + (r & 3);
                    if (m0 + wm * 64 + 4 * fh + dm < sh.M) yb[(size_t)dm * sh.Cout + 32 * u] = out(t, u, r);
                }
    }
}

// ---------------------------------------------------------------------------
// Weight gradient: gW[k, n] = sum_m A[m, k] dY[m, n], A gathered from X as in the
// forward.  The m reduction (B * Ho * Wo rows) is split over S workgroups per 128 x
// BN output tile; split z writes its fixed-order partial tile to part[z], and a
// second launch adds the S partials in split order.
//
// Per stage a workgroup stages 32 pixel rows m of A (its 128 k columns) and
// of dY (its BN n columns) in LDS transposed: per column, 8 float4 chunks of
// 4 consecutive m (tslot).  A lane's MFMA operands then run along the pixel
// reduction in one 128-bit read: in quad Q of the stage, lane l reads pixels
// 8 Q + 4 (l / 32) .. + 3 of its column (k, or n, = l % 32 of a 32-column
// block), and component c feeds the c-th MFMA, which pairs pixels 8 Q + c and
// 8 Q + 4 + c of the two half-waves (any pairing gives the same sum, as long
// as A and dY use the same one; this one is fixed).  Each loader thread
// gathers 4 consecutive pixel rows of one 4-column chunk (one pixel decode,
// then steps along the output row) and transposes them in registers into 4
// chunk writes.
// ---------------------------------------------------------------------------
// float4 slot of (column, chunk of 4 m) in a [columns][8] transposed tile.
// The xor with (col ^ col / 8) mod 8 puts the 16 columns that a 16-lane group
// reads (consecutive columns, one chunk) on 16 distinct bank quads, and the
// columns 4 ch + i that a loader instruction writes (ch = 16 consecutive
// lanes) on at most two lanes per quad.
__device__ __forceinline__ int tslot(int col, int mc) { return col * 8 + (mc ^ ((col ^ (col >> 3)) & 7)); }

template <int BN>
__global__ __launch_bounds__(kTpb, 2) void wgrad_f32(float* __restrict__ part, const float* __restrict__ X,
    const float* __restrict__ dY, ConvShape sh, int rows_per_split) {
    constexpr int UT = BN / 64;               // 32-column accumulator tiles per wave
    constexpr int DCH = BN / 4;               // float4 chunks per dY row
    constexpr int DTHR = DCH * (kWgM / 4);    // dY loader threads: (n chunk, group of 4 rows)
    static_assert(kWgM == 32 && DTHR <= kTpb && kTpb == 32 * (kWgM / 4), "loader roles");
    __shared__ float4 As[2][128 * 8];
    __shared__ float4 Ds[2][BN * 8];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wk = w >> 1, wn = w & 1;
    // tile (k tile, n tile, split z), k tile fastest, in XCD-aware order
    const int KT = (sh.KKC + 127) / 128, NT = sh.Cout / BN;
    const int tl = xcd_order((int)blockIdx.x, (int)gridDim.x);
    const int k0 = (tl % KT) * 128, n0 = ((tl / KT) % NT) * BN, z = tl / (KT * NT);
    const int mbeg = z * rows_per_split;
    const int mend = min(sh.M, mbeg + rows_per_split);
    // loader roles: A chunk ch (k = k0 + 4 ch .. + 3) of the stage's pixel rows
    // 4 g .. 4 g + 3; dY chunk dch (n = n0 + 4 dch .. + 3) of rows 4 dg .. + 3
    const int ch = tid & 31, g = tid >> 5;
    const int dch = tid % DCH, dg = tid / DCH;
    const bool dld = tid < DTHR;
    const int kc = k0 + 4 * ch;
    const bool kok = kc < sh.KKC;
    const int tap = kok ? kc / sh.Cin : 0, ci = kok ? kc - tap * sh.Cin : 0;
    const int kh = tap / sh.K, kw = tap - kh * sh.K;
    const float* dcol = dY + n0 + 4 * dch;
    const uint32_t Wo = (uint32_t)sh.Wo, Ho = (uint32_t)sh.Ho;

    // Two register sets: the stage two ahead is loaded while the next one is
    // written to LDS, so a load has two stages of MFMA work to arrive.  Every
    // lane loads (rows past the end, padding and the idle dY loaders of a
    // 64-column tile read a valid address and are zeroed when stored): a
    // branch around a load would make the compiler's later waits drain the
    // whole vector-memory counter.
    struct Regs {
        float4 a[4], d[4];
        bool aok[4], dok[4];
    };
    Regs R0, R1;
    auto load = [&](int ms, Regs& R) {
        // decode the first of the 4 rows once, then step along the output row
        const int m0 = ms + 4 * g;
        uint32_t t, ow, b, oh;
        sh.wo.divmod((uint32_t)(m0 < sh.M ? m0 : 0), t, ow);
        sh.ho.divmod(t, b, oh);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int ih = (int)oh * sh.stride - sh.pad + kh, iw = (int)ow * sh.stride - sh.pad + kw;
            R.aok[q] = (m0 + q < mend) & kok & ((unsigned)ih < (unsigned)sh.H) & ((unsigned)iw < (unsigned)sh.W);
            const int p = R.aok[q] ? ((int)b * sh.H + ih) * sh.W + iw : 0;
            // 32-bit element offsets (the host bounds x and dy below 2^31
            // elements): 346.5 -> 343.7 us at [128, 32, 32, 128 -> 128]
            // against 64-bit products; the forward's loader measured slower with the same change
            R.a[q] = ld4(X + (uint32_t)(p * sh.Cin + ci));
            if (++ow == Wo) {
                ow = 0;
                if (++oh == Ho) {
                    oh = 0;
                    ++b;
                }
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int m = ms + 4 * dg + q;
            R.dok[q] = dld & (m < mend);
            R.d[q] = ld4(dcol + (uint32_t)((R.dok[q] ? m : 0) * sh.Cout));
        }
    };
    auto mask4 = [](float4 v, bool ok) {
        const unsigned mk = ok ? 0xffffffffu : 0u;
        v.x = __uint_as_float(__float_as_uint(v.x) & mk);
        v.y = __uint_as_float(__float_as_uint(v.y) & mk);
        v.z = __uint_as_float(__float_as_uint(v.z) & mk);
        v.w = __uint_as_float(__float_as_uint(v.w) & mk);
        return v;
    };
    // 4 rows x 4 columns in registers -> 4 column chunks (rows 4 gg .. + 3)
    auto put = [&](float4* tile, int col0, int gg, const float4 (&v)[4], const bool (&ok)[4]) {
        const float4 r0 = mask4(v[0], ok[0]), r1 = mask4(v[1], ok[1]), r2 = mask4(v[2], ok[2]),
                     r3 = mask4(v[3], ok[3]);
        tile[tslot(col0 + 0, gg)] = make_float4(r0.x, r1.x, r2.x, r3.x);
        tile[tslot(col0 + 1, gg)] = make_float4(r0.y, r1.y, r2.y, r3.y);
        tile[tslot(col0 + 2, gg)] = make_float4(r0.z, r1.z, r2.z, r3.z);
        tile[tslot(col0 + 3, gg)] = make_float4(r0.w, r1.w, r2.w, r3.w);
    };
    auto store = [&](int buf, const Regs& R) {
        put(As[buf], 4 * ch, g, R.a, R.aok);
        if (dld) put(Ds[buf], 4 * dch, dg, R.d, R.dok);
    };
    f32x16 acc[2][UT];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int u = 0; u < UT; ++u) acc[t][u] = (f32x16){};
    const int fr = lane & 31, fh = lane >> 5;
    // Operands of quad Q (pixels 8 Q .. 8 Q + 7) and their MFMAs.  Two operand
    // register sets: the reads of quad Q + 2 are issued right after the MFMAs
    // of quad Q (the scheduling barriers keep them there), so each quad's
    // reads have the next quad's 4 x 2 x UT MFMAs to arrive.
    auto qfrag = [&](int buf, int Q, float4 (&a)[2], float4 (&d)[UT]) {
        const int mc = 2 * Q + fh;
#pragma unroll
        for (int t = 0; t < 2; ++t) a[t] = As[buf][tslot(wk * 64 + 32 * t + fr, mc)];
#pragma unroll
        for (int u = 0; u < UT; ++u) d[u] = Ds[buf][tslot(wn * (BN / 2) + 32 * u + fr, mc)];
    };
    // component-major: the 2 x UT accumulators in turn, so consecutive MFMAs
    // never wait for each other's result
    auto qmfma = [&](const float4 (&a)[2], const float4 (&d)[UT]) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int u = 0; u < UT; ++u) acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t].x, d[u].x, acc[t][u], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int u = 0; u < UT; ++u) acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t].y, d[u].y, acc[t][u], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int u = 0; u < UT; ++u) acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t].z, d[u].z, acc[t][u], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int u = 0; u < UT; ++u) acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t].w, d[u].w, acc[t][u], 0, 0, 0);
    };
    auto compute = [&](int buf) {
        float4 a0[2], d0[UT], a1[2], d1[UT];
        qfrag(buf, 0, a0, d0);
        qfrag(buf, 1, a1, d1);
        __builtin_amdgcn_sched_barrier(0);
        qmfma(a0, d0);
        __builtin_amdgcn_sched_barrier(0);
        qfrag(buf, 2, a0, d0);
        __builtin_amdgcn_sched_barrier(0);
        qmfma(a1, d1);
        __builtin_amdgcn_sched_barrier(0);
        qfrag(buf, 3, a1, d1);
        __builtin_amdgcn_sched_barrier(0);
        qmfma(a0, d0);
        __builtin_amdgcn_sched_barrier(0);
        qmfma(a1, d1);
        __builtin_amdgcn_sched_barrier(0);
    };
    // Stages: prologue, a branch-free steady loop over pairs of stages (stage
    // st computes from LDS buffer st % 2 while R[st % 2] receives stage st + 2
    // and R[(st + 1) % 2] goes to the other buffer; the second load of a pair
    // is clamped to the last stage, a harmless reload), then the one or two
    // stages left.
    const int nst = (mend - mbeg + kWgM - 1) / kWgM;
    if (nst > 0) {
        load(mbeg, R0);
        if (nst > 1) load(mbeg + kWgM, R1);
        store(0, R0);
        __syncthreads();
        int st = 0;
        for (; st + 2 < nst; st += 2) {
            load(mbeg + (st + 2) * kWgM, R0);
            compute(0);
            store(1, R1);
            __syncthreads();
            load(mbeg + min(st + 3, nst - 1) * kWgM, R1);
            compute(1);
            store(0, R0);
            __syncthreads();
        }
        compute(0);
        if (st + 1 < nst) {
            store(1, R1);
            __syncthreads();
            compute(1);
        }
    }
    // partial tile: D[k][n], rows k = k0 + wk 64 + 32 t + 8 (r / 4) + 4 h + r % 4
    float* pb = part + (size_t)z * sh.KKC * sh.Cout + (size_t)(k0 + wk * 64 + 4 * fh) * sh.Cout + n0 + wn * (BN / 2) + fr;
#pragma unroll
    for (int u = 0; u < UT; ++u)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int dk = 32 * t + 8 * (r >> 2) + (r & 3);
                if (k0 + wk * 64 + 4 * fh + dk < sh.KKC) pb[(size_t)dk * sh.Cout + 32 * u] = acc[t][u][r];
            }
}


// out[i] = part[0][i] + part[1][i] + ... (split order), eight splits in flight.
__global__ __launch_bounds__(kTpb) void sum_splits(float* __restrict__ gW, const float* __restrict__ part, int S,
    long long n) {
    const long long i = (long long)blockIdx.x * kTpb + threadIdx.x;
    if (i >= n) return;
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
    gW[i] = t;
}

int tile_n(int Cout) { return Cout % 128 == 0 ? 128 : 64; }

// One round of resident workgroups (two per CU on 256 CUs), and a split for every
// 32 rows at most.  The splits of a batch may be fewer, its rows being whole
// stages, so they do not grow with the batch; this bound does.
int most_splits(int M, int KKC, int Cout) {
    const int tiles = ((KKC + 127) / 128) * (Cout / tile_n(Cout));
    const int S = tiles >= 512 ? 1 : 512 / tiles, smax = (M + kWgM - 1) / kWgM;
    return S > smax ? smax : S;
}

template <bool FLIP, int XE>
void launch(float* Y, const float* X, const float* Wt, const ConvShape& sh, const ConvEpi& ep, hipStream_t s) {
    const int BN = tile_n(sh.Cout);
    const dim3 grid((unsigned)((sh.M + kBM - 1) / kBM), (unsigned)(sh.Cout / BN));
    if (BN == 128) conv_f32<128, FLIP, XE><<<grid, kTpb, 0, s>>>(Y, X, Wt, sh, ep);
    else conv_f32<64, FLIP, XE><<<grid, kTpb, 0, s>>>(Y, X, Wt, sh, ep);
}

}  // namespace

extern "C" {

void nnk_conv_f32_forward(float* y, const float* x, const float* w, const float* gain, int batch, int H, int W,
    int C_in, int C_out, int K, int stride, int pad, int H_out, int W_out, const NnConvFusion* f, hipStream_t s) {
    const char* what = "conv2d forward";
    ConvShape sh;
    if (fwd_setup(what, y, x, w, nullptr, gain, batch, H, W, C_in, C_out, K, stride, pad, H_out, W_out, sh) <= 0)
        return;
    ConvEpi ep{};
    ep.gain = gain;
    if (f && f->res) {
        ep.res = f->res;
        ep.wa = f->res_w;
        ep.wb = f->out_w;
        launch<false, kXeRes>(y, x, w, sh, ep, s);
    } else if (f) {
        ep.cond = f->cond;
        ep.y2 = f->y2;
        ep.hw = FastDiv((uint32_t)(H_out * W_out));
        launch<false, kXeMod>(y, x, w, sh, ep, s);
    } else {
        launch<false, kXeNone>(y, x, w, sh, ep, s);
    }
    nnk_after_launch(what, s);
}

void nnk_conv_f32_input_grad(float* dx, const float* dy, const float* w, const float* gain, int batch, int H, int W,
    int C_in, int C_out, int K, int pad, const NnConvFusion* f, hipStream_t s) {
    const char* what = "conv2d input gradient";
    ConvShape sh;
    if (dgrad_setup(what, dx, dy, w, batch, H, W, C_in, C_out, K, pad, sh) <= 0) return;
    ConvEpi ep{};
    ep.gain = gain;
    if (f) {
        ep.res = f->res;
        ep.xa = f->act_in;
        ep.wa = f->res_w;
        ep.wb = f->out_w;
        launch<true, kXeActG | kXeRes>(dx, dy, w, sh, ep, s);
    } else {
        launch<true, kXeNone>(dx, dy, w, sh, ep, s);
    }
    nnk_after_launch(what, s);
}

size_t nnk_conv_f32_weight_grad_workspace(int batch, int C_in, int C_out, int K, int H_out, int W_out) {
    const long long M = (long long)batch * H_out * W_out;
    if (M <= 0 || M >= (1LL << 31) || !nnhip_conv2d_wgrad_implicit_supported(C_in, C_out)) return 0;
    const int S = most_splits((int)M, K * K * C_in, C_out);
    return S > 1 ? (size_t)S * K * K * C_in * C_out : 0;
}

void nnk_conv_f32_weight_grad(float* gw, const float* x, const float* dy, int batch, int H, int W, int C_in,
    int C_out, int K, int stride, int pad, int H_out, int W_out, float* workspace, hipStream_t s) {
    const char* what = "conv2d weight gradient";
    ConvShape sh;
    if (wgrad_setup(what, gw, x, dy, batch, H, W, C_in, C_out, K, stride, pad, H_out, W_out, s, sh) <= 0) return;
    int S = most_splits(sh.M, sh.KKC, sh.Cout);
    const int rows = ((sh.M + S - 1) / S + kWgM - 1) / kWgM * kWgM;
    S = (sh.M + rows - 1) / rows;
    NNK_REQUIRE(S == 1 || workspace, what, "%s: null workspace", what);
    float* part = S > 1 ? workspace : gw;
    const int BN = tile_n(sh.Cout);
    const dim3 grid((unsigned)((sh.KKC + 127) / 128) * (unsigned)(sh.Cout / BN) * (unsigned)S);
    if (BN == 128) wgrad_f32<128><<<grid, kTpb, 0, s>>>(part, x, dy, sh, rows);
    else wgrad_f32<64><<<grid, kTpb, 0, s>>>(part, x, dy, sh, rows);
    if (S > 1) {
        const long long n = (long long)sh.KKC * sh.Cout;
        sum_splits<<<(unsigned)((n + kTpb - 1) / kTpb), kTpb, 0, s>>>(gw, part, S, n);
    }
    nnk_after_launch(what, s);
}

}  // extern "C"
