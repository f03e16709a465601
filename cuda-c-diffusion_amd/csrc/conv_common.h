// conv_common.h -- what the matrix-core convolution kernels share: the shape and
// epilogue descriptions, the split of fp32 operands into bf16 planes and the
// products of planes.  Design notes and the MFMA lane layout: k_igemm.hip.
#pragma once
#include "nn_hip_rt.h"
#include "nnk_common.h"

namespace nnk {
namespace conv {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kBM = 128, kBK = 32;  // rows and k slices of the tiled kernels
constexpr int kBNmin = 64;          // columns that the launchers of nn_hip.h need
constexpr int kWgM = 32;            // rows that a split of the weight gradient is made of

struct ConvShape {
    int B, H, W, Cin, Cout, K, stride, pad, Ho, Wo;
    int M;    // B * Ho * Wo
    int KKC;  // K * K * Cin
    FastDiv wo, ho;  // output pixel decode m -> (b, oh, ow)
};

// The tiled kernels address up to 31 rows of a weight, or 15 of dY, by 32-bit byte
// offsets from the first: below this many channels in and out.  Wider shapes
// take the small tiles (launchers of nn_hip.h) or the library's products (modules).
constexpr int kMostChannels = 1 << 24;
// Rows, channels and k that leave room in 32 bits for a tile past the end.
constexpr long long kMostIndex = (1LL << 31) - 4096;

// XCD-aware tile order.  Workgroups are dispatched round-robin over the
// device's 8 XCDs (workgroup L on XCD L % 8), each with its own L2.  Tile
// L' = xcd_order(L) gives XCD x a contiguous range of tiles, so tiles that
// read the same activations run in the same L2 instead of on different XCDs.  A bijection of [0, total) for any total.
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_order(int L, int total) {
    const int x = L % kXcds, j = L / kXcds, q = total / kXcds, r = total % kXcds;
    return x * q + min(x, r) + j;
}

// ---------------------------------------------------------------------------
// fp32 operands on the bf16 matrix cores.  v = p0 + p1 + p2 with p0 = bf16(v),
// p1 = bf16(v - p0), p2 = v - p0 - p1: 8 + 8 + 8 significand bits, so the sum
// is exact for every v of 2^-103 and above (below it p2 may lie under the
// smallest normal number).  a b is then the sum of the products p_i q_j; the
// six with i + j <= 2 are taken, the other three are each below 2^-25 |a b|, below
// 2^-24 together.  Each product of two bf16 is exact and the matrix core adds in
// fp32.  What smaller operands lose: split_failed.
// ---------------------------------------------------------------------------
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
constexpr int kPlanes = 3;

// the planes of (a, b), a in the low half
__device__ __forceinline__ void split2(float a, float b, uint32_t (&p)[kPlanes]) {
#pragma unroll
    for (int i = 0; i < kPlanes; ++i) {
        const f32x2 v = {a, b};
        p[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
        if (i + 1 < kPlanes) {
            a = a - __uint_as_float(p[i] << 16);
            b = b - __uint_as_float(p[i] & 0xffff0000u);
        }
    }
}

// the planes of 8 consecutive k
__device__ __forceinline__ void split8(const float (&v)[8], uint4 (&p)[kPlanes]) {
    uint32_t d[4][kPlanes];
#pragma unroll
    for (int i = 0; i < 4; ++i) split2(v[2 * i], v[2 * i + 1], d[i]);
#pragma unroll
    for (int i = 0; i < kPlanes; ++i) p[i] = make_uint4(d[0][i], d[1][i], d[2][i], d[3][i]);
}
__device__ __forceinline__ float keep(float v, bool ok) { return __uint_as_float(__float_as_uint(v) & (ok ? ~0u : 0u)); }

// d += a b over the k of a fragment of 8 k a lane: 16 k and a tile of 32 x 32
// (lane l: row l % 32, k 8 (l / 32) .. + 7), or 32 k and 16 x 16 (row l % 16, k 8
// (l / 16) .. + 7).
__device__ __forceinline__ void mfma(const uint4& a, const uint4& b, f32x16& d) {
    d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), d, 0, 0, 0);
}
__device__ __forceinline__ void mfma(const uint4& a, const uint4& b, f32x4& d) {
    d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), d, 0, 0, 0);
}

// A wave's products over a fragment's k: T x U accumulators from the planes of
// its row tiles' fragments.  The
// matrix core cuts off what an addend has below the last place of the largest
// one, towards minus infinity.  p0 q0 products lie on a coarse grid and lose
// next to nothing; the five small products, added to the same accumulator,
// would lose enough to shift every output by -6e-8 of its root mean square at
// K = 1152, which sums over many outputs (a bias gradient, a norm's) show.  So
// they have an accumulator of their own, `cor`, 2^-8 as large: error against
// 64 bits 2.0e-7 (mean 2e-10) of the root mean square at K = 1152 with standard
// normal operands, against 5.2e-7 (mean -6e-8) with one accumulator and 6.1e-7
// with the fp32 MFMA.  Each product runs over all T x U accumulators, so
// consecutive MFMAs rarely wait for each other's result.
template <int T, int U, class V>
__device__ __forceinline__ void products(const uint4 (&a)[kPlanes][T], const uint4 (&b)[kPlanes][U], V (&acc)[T][U],
    V (&cor)[T][U]) {
    constexpr int PI[6] = {0, 2, 0, 1, 1, 0}, PJ[6] = {0, 0, 2, 1, 0, 1};
#pragma unroll
    for (int x = 0; x < 6; ++x)
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int u = 0; u < U; ++u) mfma(a[PI[x]][t], b[PJ[x]][u], x ? cor[t][u] : acc[t][u]);
}

// Whether a wave's results must be formed again from the unsplit operands.  Not
// finite: an infinite or NaN operand, or one that rounds to infinity in bf16,
// splits into NaN planes.  Small: an operand below 2^-103 may lose up to 2^-126, so
// n products with operands up to b lose up to 2^-126 n b of a result.  A result
// below 2^-80 is formed again, which leaves 2^-24 of a result for n b up to 2^22; so
// is a row or column of the tile that has none of 2^-55, as one has whose operands
// are all that small: 2^-24 of the row's largest for n b up to 2^47.  What is left
// is an operand below 2^-103 in sums with some of 2^47 / n and above.  A zero is
// taken for one (a masked row, an operand of zeros), also where all operands of a
// sum lie below 2^-126.
template <int T, int U, class V>
__device__ __forceinline__ bool split_failed(const V (&acc)[T][U]) {
    constexpr int N = (int)(sizeof(V) / sizeof(float)), L = N == 16 ? 32 : 16;  // L lanes to a row
    constexpr float kElement = 0x1p-80f, kLine = 0x1p-55f;
    // of the bits of |v|, and of those less one, which leaves zeros out (a wave whose
    // taps lie outside the image has many)
    uint32_t most = 0, least = ~0u;
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int r = 0; r < N; ++r) {
                const float v = acc[t][u][r];
                const uint32_t b = __float_as_uint(v) & 0x7fffffffu;
                most = max(most, b);
                least = min(least, b - 1);
            }
    bool bad = most >= 0x7f800000u;
    if (!__any(bad || least < __float_as_uint(kLine) - 1)) return false;
    auto small = [](float v, float limit) { return v > 0.0f && v < limit; };
    float column[U];
#pragma unroll
    for (int u = 0; u < U; ++u) column[u] = 0.0f;
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int r = 0; r < N; ++r) {
            float row = 0.0f;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float v = fabsf(acc[t][u][r]);
                bad |= small(v, kElement);
                row = fmaxf(row, v);
                column[u] = fmaxf(column[u], v);
            }
#pragma unroll
            for (int o = 1; o < L; o <<= 1) row = fmaxf(row, __shfl_xor(row, o, kWave));
            bad |= small(row, kLine);
        }
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int o = L; o < kWave; o <<= 1) column[u] = fmaxf(column[u], __shfl_xor(column[u], o, kWave));
        bad |= small(column[u], kLine);
    }
    return __any(bad);
}

// Fused neighbours of the forward / input-gradient kernel (bit flags), with v
// the output after bias or gain:
//   kXeRes : y = wa * res[m, n] + wb * v            (launch_weighted_sum(y, res, v, wa, wb))
//   kXeActG: v = v * act'(xa[m, n]) first            (launch_activation_backward)
//   kXeMod : y = v and y2 = act(v * (cond[b, n] + 1)) (launch_spatial_modulate_act_forward)
// each with the operation order of the pass it replaces, so the results are
// those of the separate passes bit for bit.
enum { kXeNone = 0, kXeRes = 1, kXeActG = 2, kXeMod = 4 };
struct ConvEpi {
    const float* bias;  // + bias[n], or null
    const float* gain;  // * gain[0], or null
    const float* res;   // kXeRes: [M][C_out]
    const float* xa;    // kXeActG: [M][C_out]
    const float* cond;  // kXeMod: [B][C_out]
    float* y2;          // kXeMod: [M][C_out]
    float wa, wb;       // kXeRes weights
    int mp;             // the activation is MP-SiLU (SiLU otherwise)
    FastDiv hw;         // kXeMod: output pixels per sample
};

// v with bias or gain, then the fused neighbours in xe, at output (m, n)
// (offset o).  The act' operand and the residual are read here.
__device__ __forceinline__ void epilogue_store(float* __restrict__ Y, float v, int xe, uint32_t o, uint32_t co,
    const ConvEpi& ep, float bias, float gain) {
    if (ep.bias) v = v + bias;
    else if (ep.gain) v = v * gain;
    if (xe & kXeActG) {
        const float d = act_grad<ACT_SILU, false>(ep.xa[o]);
        v = v * (ep.mp ? d * kMpSiluScale : d);
    }
    if (xe & kXeRes) v = ep.wa * ep.res[o] + ep.wb * v;
    Y[o] = v;
    if (xe & kXeMod) {
        const float z = act_fwd<ACT_SILU, false>(v * (ep.cond[co] + 1.0f));
        ep.y2[o] = ep.mp ? z * kMpSiluScale : z;
    }
}

// Checks shared by the forward launchers (plain and fused): -1 after
// recording an error, 0 when there is nothing to do (batch 0), 1 with `sh`
// filled in.
inline int fwd_setup(const char* what, const float* Y, const float* X, const float* Wt, const float* bias,
    const float* gain, int batch, int H, int W, int C_in, int C_out, int K, int stride, int pad, int H_out,
    int W_out, ConvShape& sh) {
    NNK_REQUIRE_RET(batch >= 0 && H > 0 && W > 0 && K > 0 && stride > 0 && pad >= 0, -1, what,
        "%s: bad geometry", what);
    NNK_REQUIRE_RET(nnhip_conv2d_implicit_supported(C_in, C_out), -1, what,
        "%s: needs C_in %% %d == 0 and C_out %% %d == 0 (C_in=%d C_out=%d)", what, kBK, kBNmin, C_in, C_out);
    NNK_REQUIRE_RET(H_out == (H + 2 * pad - K) / stride + 1 && W_out == (W + 2 * pad - K) / stride + 1 &&
                        H_out > 0 && W_out > 0,
        -1, what, "%s: output size %dx%d does not match the geometry", what, H_out, W_out);
    NNK_REQUIRE_RET((long long)batch * H * W * C_in < (1LL << 31) &&
                        (long long)batch * H_out * W_out * C_out < (1LL << 31),
        -1, what, "%s: tensor exceeds the 32-bit index range", what);
    NNK_REQUIRE_RET(!(bias && gain), -1, what, "%s: bias and gain are exclusive", what);
    if (batch == 0) return 0;
    NNK_REQUIRE_RET(Y && X && Wt, -1, what, "%s: null pointer", what);
    NNK_REQUIRE_RET(aligned16(X) && aligned16(Wt), -1, what, "%s: x and the weight must be 16-byte aligned", what);
    sh = ConvShape{batch, H, W, C_in, C_out, K, stride, pad, H_out, W_out, batch * H_out * W_out, K * K * C_in,
        FastDiv((uint32_t)W_out), FastDiv((uint32_t)H_out)};
    return 1;
}

// Checks shared by the input-gradient launchers; `sh` is then the stride-1
// convolution of dy (Ho x Wo x C_out) with the flipped kernel and padding
// K-1-pad, whose output is H x W x C_in.
inline int dgrad_setup(const char* what, const float* dX, const float* dY, const float* Wt, int batch, int H, int W,
    int C_in, int C_out, int K, int pad, ConvShape& sh) {
    NNK_REQUIRE_RET(batch >= 0 && H > 0 && W > 0 && K > 0 && pad >= 0, -1, what, "%s: bad geometry", what);
    NNK_REQUIRE_RET(nnhip_conv2d_input_grad_implicit_supported(C_in, C_out, K, 1, pad), -1, what,
        "%s: needs pad <= K - 1, C_out %% %d == 0 and C_in %% %d == 0 (C_in=%d C_out=%d K=%d pad=%d)", what, kBK,
        kBNmin, C_in, C_out, K, pad);
    const int Ho = H + 2 * pad - K + 1, Wo = W + 2 * pad - K + 1;
    NNK_REQUIRE_RET(Ho > 0 && Wo > 0, -1, what, "%s: empty output for this geometry", what);
    NNK_REQUIRE_RET((long long)batch * H * W * C_in < (1LL << 31) && (long long)batch * Ho * Wo * C_out < (1LL << 31) &&
                        (long long)K * K * C_in * C_out < (1LL << 31),
        -1, what, "%s: tensor exceeds the 32-bit index range", what);
    if (batch == 0) return 0;
    NNK_REQUIRE_RET(dX && dY && Wt, -1, what, "%s: null pointer", what);
    NNK_REQUIRE_RET(aligned16(dY) && aligned16(Wt), -1, what, "%s: dy and the weight must be 16-byte aligned", what);
    sh = ConvShape{batch, Ho, Wo, C_out, C_in, K, 1, K - 1 - pad, H, W, batch * H * W, K * K * C_out,
        FastDiv((uint32_t)W), FastDiv((uint32_t)H)};
    return 1;
}

// Checks of the weight-gradient launchers; batch 0 clears gW.
inline int wgrad_setup(const char* what, float* gW, const float* X, const float* dY, int batch, int H, int W, int C_in,
    int C_out, int K, int stride, int pad, int H_out, int W_out, hipStream_t s, ConvShape& sh) {
    NNK_REQUIRE_RET(batch >= 0 && H > 0 && W > 0 && K > 0 && stride > 0 && pad >= 0, -1, what, "%s: bad geometry", what);
    NNK_REQUIRE_RET(nnhip_conv2d_wgrad_implicit_supported(C_in, C_out), -1, what,
        "%s: needs C_in %% 4 == 0 and C_out %% %d == 0 (C_in=%d C_out=%d)", what, kBNmin, C_in, C_out);
    NNK_REQUIRE_RET(H_out == (H + 2 * pad - K) / stride + 1 && W_out == (W + 2 * pad - K) / stride + 1 && H_out > 0 &&
                        W_out > 0,
        -1, what, "%s: output size %dx%d does not match the geometry", what, H_out, W_out);
    NNK_REQUIRE_RET((long long)batch * H * W * C_in < (1LL << 31) &&
                        (long long)batch * H_out * W_out * C_out < (1LL << 31),
        -1, what, "%s: tensor exceeds the 32-bit index range", what);
    NNK_REQUIRE_RET(gW && (batch == 0 || (X && dY)), -1, what, "%s: null pointer", what);
    const int KKC = K * K * C_in;
    if (batch == 0) {
        nnhip_fill_f32(gW, 0.0f, (size_t)KKC * C_out, s);
        return 0;
    }
    NNK_REQUIRE_RET(aligned16(X) && aligned16(dY), -1, what, "%s: X and dY must be 16-byte aligned", what);
    sh = ConvShape{batch, H, W, C_in, C_out, K, stride, pad, H_out, W_out, batch * H_out * W_out, KKC,
        FastDiv((uint32_t)W_out), FastDiv((uint32_t)H_out)};
    return 1;
}

// Waves of a small tile by its steps: one or two steps each.
inline int waves_for(int steps) { return steps <= 4 ? 4 : steps <= 16 ? 8 : 16; }

// The time of the small tiles of t x t outputs, in us, as fitted to the sweep of
// conv_tile.  Tiles of 16 take 32 k a step and spread over four times the
// workgroups, so they win while a wave's round trips of loads count, and lose
// with twice the vector work per output where that does.  32 / 16 measured:
// forward [8, 7 x 7, 128 -> 128] 9.3 / 6.2, its input gradient 11.6 / 6.9; [1, 8 x
// 8, 448 -> 448] 22 / 14; dense [128, 512 -> 512] 6.2 / 4.9, [1024, 256 -> 256] 5.2
// / 6.7; [8, 28 x 28, 32 -> 32] 5.4 / 6.4; [4, 16 x 16, 256 -> 256] 16 / 25; 5x5
// input gradient 320 -> 4 at [22, 5, 8] 37 / 21.
inline double small_us(const ConvShape& sh, bool flip, int t) {
    const bool t32 = t == 32;
    const int sk = 512 / t, steps = sh.K * sh.K * ((sh.Cin + sk - 1) / sk);
    const double cells = (double)((sh.M + t - 1) / t) * ((sh.Cout + t - 1) / t);
    const double trips = (t32 ? 1.15 : flip ? 1.3 : 1.2) * ((steps + waves_for(steps) - 1) / waves_for(steps));
    double step = flip ? t32 ? 0.00045 : 0.00040 : t32 ? 0.00036 : 0.00031;
    if (sh.Cin % 8) step *= 1.8;  // one element a load
    const double work = cells * (steps * step + (t32 ? 0.005 : 0.0015));
    return (t32 ? 3.8 : 3.5) + (trips > work ? trips : work);
}

}  // namespace conv
}  // namespace nnk

// Which form of a kernel runs, where a caller names it: columns a workgroup (0: the
// small tiles) and the staging (conv_x3's MODE, igemm_wgrad's LOADS; a more special
// one than the shape allows is not taken).  Negative: by the rules.
struct ConvPick {
    int columns = -1, staging = -1;
};

// Few output tiles: 32 x 32 outputs a workgroup, the k range split over its
// waves (k_conv_small.hip).  `flip`, `xe`: as conv_x3's parameters.
void nnk_conv_small(bool flip, int xe, float* Y, const float* X, const float* Wt, const nnk::conv::ConvShape& sh,
    const nnk::conv::ConvEpi& ep, hipStream_t s);
// gW (overwritten), and with gb non-null the column sums of dY, in one launch.
void nnk_wgrad_small(float* gW, float* gb, const float* X, const float* dY, const nnk::conv::ConvShape& sh,
    hipStream_t s);
// The tiled kernels with a neighbour folded in, of checked shapes (k_igemm_fused.hip).
void nnk_conv_forward_fused(float* Y, const float* X, const float* Wt, const nnk::conv::ConvShape& sh,
    nnk::conv::ConvEpi ep, const NnConvFusion& f, hipStream_t s, ConvPick pick = {});
void nnk_conv_input_grad_fused(float* dX, const float* dY, const float* Wt, const nnk::conv::ConvShape& sh,
    nnk::conv::ConvEpi ep, const NnConvFusion& f, hipStream_t s, ConvPick pick = {});
