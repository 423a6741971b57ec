// The dw-striding subsampling of 128 mel bins at 256 channels in three kernels, channels last, with everything that is a
// contraction on the FP16 matrix cores at FP32 accuracy (kea_split.h):
//   1. conv 3x3/2 (1 -> 256) + ReLU + depthwise 3x3/2 + pointwise 256 -> 256 + ReLU     [B][128][T] -> [B][T2][32][256]
//   2. depthwise 3x3/2 + pointwise 256 -> 256 + ReLU, split            [B][T2][32][256] -> [B][T3][hi, lo][16 x 256]
//   3. the output linear 4096 -> d (and a sum over its K slices)                                     -> [B][T3][d]
// A workgroup of 1 and 2 makes all 256 channels of its positions, so a pointwise convolution's input never leaves LDS,
// where the same layers as separate kernels (kea_subsample_front, a library GEMM, kea_dwconv2d_s2, a library GEMM,
// kea_bias_relu_flatten) write and read [B][256][T2][32] three times and the FP32 GEMMs run at 1/16 of the FP16 rate.
// The first convolution is itself one matrix product: its 9 taps times the three products of a split operand are 27 of a
// 32-deep MFMA's terms. Kernel 2 makes whole rows of the output linear's input, so it can split them with a row's scale.
// Tiles whose inputs have no such form (infinities, sizes too far apart) take the same sums in FP32, the first convolutions
// on the vector unit with a thread per channel, the pointwise product on the FP32 matrix instruction: eight 10-second clips
// with a large value in every tile 191 us against 113 (one thread per channel throughout took 2180).
//
// Measured on eight 10-second clips (T = 1000): 50 + 26 + 34 us, where five launches and a library GEMM take 53 + 90 +
// 25 + 27 + 25 + 70 us; one clip 15 + 15 + 17 us.
// Kernel 1 executes 1845 vector instructions and 232 MFMAs a wave, which at 2.4 GHz take 25 and 12 us of its 50 and hardly
// overlap; LDS takes 11, and the waves wait for 38% of their time. Two rows of 32 positions to a workgroup, two workgroups to
// a CU, is the split that measured best: four rows (one workgroup to a CU, half the weight reads) take 60 and, for one
// clip, 25 us. Kernel 2 is latency: the weights (256 KB a workgroup) and its input from L2; half the rows to a workgroup
// take 37 us, as the weights are read twice as often. Kernel 3 is bound by L2: 268 MB of operands in 26 us, then 16 MB of
// partial sums out and in again; larger tiles would halve the operands and double the partial sums.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <type_traits>

#include "kea_internal.h"
#include "kea_split.h"
#include "../../include/kea_encoder.h"

namespace {

using kea::exponent_of;
using kea::kInfBits;
using kea::mfma_f16;
using kea::mfma_split;
using kea::pow2;
using kea::split1;
using kea::v4f;
using kea::v8h;

constexpr int kC = 256, kF = 128, kF2 = 32, kF3 = 16;
constexpr int kWaves = 8, kThreads = 64 * kWaves;

// max(x, 0) of an x that is not a NaN, on the bits (fmaxf would canonicalise an MFMA's result first).
__device__ __forceinline__ float relu(float x) { return __builtin_bit_cast(float, max(__builtin_bit_cast(int, x), 0)); }

// The pointwise product of a tile of positions: D[n][m] = sum_k W[n][k] x[m][k] over the LDS tile x (hi and lo planes
// [MT * 16][256], 16-byte units XOR-swizzled by row), wave w taking output channels 32 w .. 32 w + 31. W: the fragments
// [n-tile][k-step][plane][lane][8] of split weights, read from L2 two k-steps ahead of their products (the first two
// before the tile is complete). acc[nt][mt]: rows n = 4 (lane / 16) + r, column m = lane % 16.
struct Weights {
    const _Float16 *at;
    v8h f[3][2][2];  // [k-step % 3][n-tile][plane]
    __device__ __forceinline__ void load(int ks) {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
            for (int p = 0; p < 2; ++p) f[ks % 3][nt][p] = *(const v8h *)(at + ((nt * 8 + ks) * 2 + p) * 64 * 8);
    }
    __device__ __forceinline__ void start(const _Float16 *w, int wave, int lane) {
        at = w + ((long long)(2 * wave) * 8 * 2 * 64 + lane) * 8;
        load(0);
        load(1);
    }
};
template <int MT>
__device__ __forceinline__ void pointwise(const _Float16 *tile, Weights &w, int lane, v4f (&acc)[2][MT]) {
    const int i = lane & 15, g = lane >> 4;
    constexpr int PLANE = MT * 16 * kC;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
        if (ks + 2 < 8) w.load(ks + 2);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const _Float16 *p = tile + (mt * 16 + i) * kC + (((4 * ks + g) ^ i) * 8);
            const v8h hi = *(const v8h *)p, lo = *(const v8h *)(p + PLANE);
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
                acc[nt][mt] = mfma_split(w.f[ks % 3][nt][0], w.f[ks % 3][nt][1], hi, lo, acc[nt][mt]);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The same product of FP32 operands on the FP32 matrix instruction, for tiles that are not split: x in LDS ([MT * 16][256],
// 16-byte units XOR-swizzled by row), W [256][256] from L2. Element 16 s + 4 g + e of a row is step (s, e).
__device__ __forceinline__ int fp32_at(int row, int k) { return row * kC + (((k >> 2) ^ (row & 15)) << 2) + (k & 3); }
template <int MT>
__device__ __forceinline__ void pointwise_fp32(const float *tile, const float *w, int wave, int lane, v4f (&acc)[2][MT]) {
    typedef float v4f_any __attribute__((ext_vector_type(4), aligned(4)));
    const int i = lane & 15, g = lane >> 4;
    const float *const row = w + (long long)(32 * wave + i) * kC + 4 * g;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = (v4f){0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < kC / 16; ++s) {
        const v4f a0 = *(const v4f_any *)(row + 16 * s), a1 = *(const v4f_any *)(row + 16 * kC + 16 * s);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const v4f x = *(const v4f *)(tile + fp32_at(16 * mt + i, 16 * s + 4 * g));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                acc[0][mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[e], x[e], acc[0][mt], 0, 0, 0);
                acc[1][mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1[e], x[e], acc[1][mt], 0, 0, 0);
            }
        }
    }
}

// 3x3/2 taps of output position (r, c) read input rows 2 r - 1 + ky and columns 2 c - 1 + kx (padding 1).

// Kernel 1: a workgroup = one clip's output rows t2 = 2 blockIdx.x and + 1, all 32 columns and 256 channels.
constexpr int kMinExponent = -50, kHalfOne = 0x3c00;  // (FP16 bits of 1, 2^-14 of the scale's lower end)
constexpr float kLeastTap = 0x1p-102f;               // (2^24 times the smallest normal number)
constexpr int kRows2 = 2, kPos1 = kRows2 * kF2;              // positions of a tile: 64, m = 32 q + f2
constexpr int kRows1 = 2 * kRows2 + 1, kPatchR = 2 * kRows1 + 1, kPatchC = kF + 2;
constexpr int kPatch = kPatchR * kPatchC;                    // input rows 4 t2 - 3 .., columns -1 .. 128
constexpr int kTile1 = 2 * kPos1 * kC * 2;                   // bytes of the split tile (the first convolution's operand
                                                             // fragments, kRows1 x 4 KB, lie there before it)
constexpr int kLds1Patch = kTile1, kLds1Max = kLds1Patch + (2 * kPatch + 8) * 2 / 16 * 16 + 16;
constexpr int kLds1Scale = kLds1Max + kWaves * kPos1 * 4, kLds1Bytes = kLds1Scale + kPos1 * 4 + 32;

__global__ void __launch_bounds__(kThreads, 4)
subsample1_kernel(const float *x, int T, int T1, int T2, const _Float16 *w1f, const float *w1m, const float *w1,
                  const float *b1, const float *w2, const float *b2, const _Float16 *w3f, const float *w3m, const float *w3,
                  const float *b3, float *y) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), i = lane & 15, g = lane >> 4;
    const int b = blockIdx.y, t2a = blockIdx.x * kRows2, r0 = 4 * t2a - 3;
    const float *xb = x + (long long)b * kF * T;
    _Float16 *const tile = (_Float16 *)lds, *const patch = (_Float16 *)(lds + kLds1Patch);
    float *const pmax = (float *)(lds + kLds1Max), *const pscale = (float *)(lds + kLds1Scale);
    int *const top = (int *)(lds + kLds1Scale + kPos1 * 4);

    // the weights of the wave's 32 channels, two per lane (32 wave + 2 i + e)
    const int ch2 = 32 * wave + 2 * i;
    const v8h wf[2] = {*(const v8h *)(w1f + (2 * wave * 64 + lane) * 8), *(const v8h *)(w1f + ((2 * wave + 1) * 64 + lane) * 8)};
    const float2 m1 = *(const float2 *)(w1m + ch2), first = *(const float2 *)(b1 + ch2), second = *(const float2 *)(b2 + ch2);
    float2 taps[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) taps[k] = *(const float2 *)(w2 + k * kC + ch2);

    // the input patch, split with one scale for the tile
    constexpr int PN = (kPatch + kThreads - 1) / kThreads;
    float px[PN];
    float m = 0.f;
    bool plain = false;
#pragma unroll
    for (int u = 0; u < PN; ++u) {
        const int e = u * kThreads + tid, c = e / kPatchR, r = e - c * kPatchR, t = r0 + r;  // time runs fastest in x
        px[u] = e < kPatch && t >= 0 && t < T && c >= 1 && c <= kF ? xb[(long long)(c - 1) * T + t] : 0.f;
        m = kea::max_abs2(px[u], 0.f, m);
        plain = plain || px[u] != px[u];
    }
    const int wtop = kea::wave_max_bits(m);
    if (lane == 0) top[wave] = wtop;
    __syncthreads();
    int bits = top[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) bits = max(bits, top[w]);
    // a tile of values below the smallest scale is summed in FP32, as NaNs and infinities are, and as one is where the scale
    // of its largest value costs others their accuracy: a value that both planes lose (below 2^-39 of it), or a window of 3x3
    // inputs without one above 2^-14 of it (held to 2^-25 of the window's largest from there on). The output rows of a tile do
    // not all see that largest value.
    const int xe = bits == 0 ? 0 : max(exponent_of(bits), kMinExponent);
    plain = plain || bits >= kInfBits || (bits != 0 && exponent_of(bits) < kMinExponent);
#pragma unroll
    for (int u = 0; u < PN; ++u) {
        const int e = u * kThreads + tid, c = e / kPatchR, r = e - c * kPatchR;
        _Float16 hi, lo;
        split1(px[u], pow2(14 - xe), hi, lo);
        plain = plain || (px[u] != 0.f && hi == (_Float16)0.f);
        if (e < kPatch) {
            patch[r * kPatchC + c] = hi;
            patch[kPatch + r * kPatchC + c] = lo;
        }
    }
    if (tid == 0) patch[2 * kPatch] = (_Float16)0.f;
    __syncthreads();
    // operand fragments [row t1][16 columns f1] of the first convolution: term k = 8 g + j of a lane is tap k % 9 of
    // x hi (k < 9, against the weights' hi), x lo (< 18, hi) and x hi (< 27, against lo)
    {
        int at[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int k = 8 * g + j, part = k / 9, tap = k - 9 * part;
            at[j] = k < 27 ? (part == 1 ? kPatch : 0) + tap / 3 * kPatchC + tap % 3 : -1;
        }
        for (int f = wave; f < kRows1 * 4; f += kWaves) {
            const int base = 2 * (f >> 2) * kPatchC + 2 * (16 * (f & 3) + i);
            v8h v;
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = patch[at[j] < 0 ? 2 * kPatch : base + at[j]];
            *(v8h *)(tile + (f * 64 + lane) * 8) = v;
            // the window's largest: its nine hi values are terms 0 .. 7 of group 0 and term 0 of group 1
            typedef uint16_t v8u __attribute__((ext_vector_type(8)));
            const v8u size = __builtin_bit_cast(v8u, v) & (uint16_t)0x7fff;
            int top9 = g == 0 ? __builtin_reduce_max(size) : g == 1 ? size[0] : 0;
            top9 = max(top9, __shfl_xor(top9, 16, 64));
            plain = plain || (g == 0 && top9 > 0 && top9 < kHalfOne);
        }
    }
    __syncthreads();

    // the first convolution's rows in order, each accumulated into the depthwise outputs it belongs to. o[e][q][j][s]: row t2a + q, column 8 j + 2 g + s.
    // The first convolution stays in the units of its operands, m1 * 2^(xe - 14): its bias is divided by them, the
    // depthwise weights multiplied.
    float o[2][kRows2][4][2], dw[2][9], bias1[2];
    const float mul[2] = {m1.x * pow2(xe - 14), m1.y * pow2(xe - 14)};
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        dw[0][k] = taps[k].x * mul[0];
        dw[1][k] = taps[k].y * mul[1];
    }
    // (weights that these units make too small for 24 bits: FP32 as well)
    float tap[2] = {kea::max_abs2(taps[8].x, 0.f, 0.f), kea::max_abs2(taps[8].y, 0.f, 0.f)};
#pragma unroll
    for (int k = 0; k < 8; k += 2) {
        tap[0] = kea::max_abs2(taps[k].x, taps[k + 1].x, tap[0]);
        tap[1] = kea::max_abs2(taps[k].y, taps[k + 1].y, tap[1]);
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        plain = plain || (tap[e] > 0.f && tap[e] * mul[e] < kLeastTap);
        bias1[e] = (e ? first.y : first.x) * __builtin_amdgcn_rcpf(e ? m1.y : m1.x) * pow2(14 - xe);  // (m1: powers of two)
#pragma unroll
        for (int q = 0; q < kRows2; ++q)
#pragma unroll
            for (int j = 0; j < 4; ++j) o[e][q][j][0] = o[e][q][j][1] = e ? second.y : second.x;
    }
#pragma unroll
    for (int rr = 0; rr < kRows1; ++rr) {
        const int t1 = 2 * t2a - 1 + rr;
        v8h xf[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) xf[j] = *(const v8h *)(tile + ((rr * 4 + j) * 64 + lane) * 8);
        if (t1 >= 0 && t1 < T1) {  // the same for the whole workgroup; a row of the padding adds nothing
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                float v[4][4], before[4], turned[4];  // columns 16 j + 4 g + r, and the column before each four
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const v4f d = mfma_f16(xf[j], wf[e], (v4f){bias1[e], bias1[e], bias1[e], bias1[e]});
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[j][r] = relu(d[r]);
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) turned[j] = __shfl(v[j][3], (lane + 48) & 63, 64);  // group g - 1's last column
#pragma unroll
                for (int j = 0; j < 4; ++j) before[j] = g > 0 ? turned[j] : j > 0 ? turned[j - 1] : 0.f;
#pragma unroll
                for (int q = 0; q < kRows2; ++q) {
                    const int dy = rr - 2 * q;
                    if (dy < 0 || dy > 2) continue;
                    const float a = dw[e][3 * dy], c = dw[e][3 * dy + 1], d = dw[e][3 * dy + 2];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        float u0 = o[e][q][j][0], u1 = o[e][q][j][1];
                        u0 = __builtin_fmaf(d, v[j][1], __builtin_fmaf(c, v[j][0], __builtin_fmaf(a, before[j], u0)));
                        u1 = __builtin_fmaf(d, v[j][3], __builtin_fmaf(c, v[j][2], __builtin_fmaf(a, v[j][1], u1)));
                        o[e][q][j][0] = u0;
                        o[e][q][j][1] = u1;
                    }
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // each position's largest magnitude over the channels: 16 lanes here, the waves through LDS
#pragma unroll
    for (int q = 0; q < kRows2; ++q)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const float top16 = kea::max16(kea::max_abs2(o[0][q][j][s], o[1][q][j][s], 0.f));
                if (i == 0) pmax[wave * kPos1 + 32 * q + 8 * j + 2 * g + s] = top16;
            }
    __syncthreads();
    int big = 0;
    if (tid < kPos1) {
#pragma unroll
        for (int w = 0; w < kWaves; ++w) big = max(big, __builtin_bit_cast(int, pmax[w * kPos1 + tid]));
        pscale[tid] = pow2(14 - exponent_of(big));
    }
    plain = __syncthreads_or(plain || big >= kInfBits) != 0;
    const int rows = min(kRows2, T2 - t2a);
    float *const yb = y + ((long long)b * T2 + t2a) * kF2 * kC;
    v4f acc[2][kPos1 / 16];
    if (plain) {  // the same sums in FP32: a thread takes a channel of one output row
        float *const xs = (float *)patch, *const h = (float *)lds;  // the patch (all waves are past the split one), [kPos1][256]
        static_assert(kThreads == kRows2 * kC, "a thread per channel and row");
#pragma unroll
        for (int u = 0; u < PN; ++u) {
            const int e = u * kThreads + tid, c = e / kPatchR, r = e - c * kPatchR;
            if (e < kPatch) xs[r * kPatchC + c] = px[u];
        }
        __syncthreads();
        const int c = tid & (kC - 1), q = tid / kC, t1 = 2 * (t2a + q) - 1;
        float wa[9], wb[9], before[3] = {0.f, 0.f, 0.f};  // before: the first convolution's column 2 f2 - 1
        const float ba = b1[c], bb = b2[c];
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            wa[k] = w1[k * kC + c];
            wb[k] = w2[k * kC + c];
        }
        for (int f2 = 0; f2 < kF2; ++f2) {
            const float *const x0 = xs + 4 * q * kPatchC + 4 * f2;
            float sum = bb;
#pragma unroll
            for (int dy = 0; dy < 3; ++dy) {
                float v[2];
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    float a = ba;
#pragma unroll
                    for (int k = 0; k < 9; ++k) a = __builtin_fmaf(wa[k], x0[(2 * dy + k / 3) * kPatchC + 2 * s + k % 3], a);
                    v[s] = t1 + dy >= 0 && t1 + dy < T1 ? fmaxf(a, 0.f) : 0.f;
                }
                sum = __builtin_fmaf(wb[3 * dy], before[dy], sum);
                sum = __builtin_fmaf(wb[3 * dy + 1], v[0], sum);
                sum = __builtin_fmaf(wb[3 * dy + 2], v[1], sum);
                before[dy] = v[1];
            }
            h[fp32_at(32 * q + f2, c)] = sum;
        }
        __syncthreads();
        pointwise_fp32<kPos1 / 16>(h, w3, wave, lane, acc);
    } else {
        Weights weights;
        weights.start(w3f, wave, lane);
        // the split tile (all waves are past the fragments): two channels of a position are one word
#pragma unroll
        for (int q = 0; q < kRows2; ++q)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const int p = 32 * q + 8 * j + 2 * g + s, ch = 32 * wave + 2 * i;
                    const float sf = pscale[p];
                    typedef _Float16 v2h __attribute__((ext_vector_type(2)));
                    _Float16 h0, l0, h1, l1;
                    split1(o[0][q][j][s], sf, h0, l0);
                    split1(o[1][q][j][s], sf, h1, l1);
                    _Float16 *dst = tile + p * kC + (((ch >> 3) ^ (p & 15)) * 8) + (ch & 7);
                    *(v2h *)dst = (v2h){h0, h1};
                    *(v2h *)(dst + kPos1 * kC) = (v2h){l0, l1};
                }
        __syncthreads();
        pointwise<kPos1 / 16>(tile, weights, lane, acc);
    }
    // D[n][m]: a lane holds four consecutive output channels of a position
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
        const int n = 32 * wave + 16 * nt + 4 * g;
        const float4 bias = *(const float4 *)(b3 + n), wm = plain ? make_float4(1.f, 1.f, 1.f, 1.f) : *(const float4 *)(w3m + n);
#pragma unroll
        for (int mt = 0; mt < kPos1 / 16; ++mt) {
            const int p = 16 * mt + i;
            const float pm = plain ? 1.f : 1.0f / pscale[p];  // (powers of two: exact)
            const v4f d = acc[nt][mt];
            // (the product of both scales may leave the range that the result stays in)
            if (p < rows * kF2)
                *(float4 *)(yb + p * kC + n) = make_float4(fmaxf(__builtin_fmaf(d[0] * wm.x, pm, bias.x), 0.f),
                                                           fmaxf(__builtin_fmaf(d[1] * wm.y, pm, bias.y), 0.f),
                                                           fmaxf(__builtin_fmaf(d[2] * wm.z, pm, bias.z), 0.f),
                                                           fmaxf(__builtin_fmaf(d[3] * wm.w, pm, bias.w), 0.f));
        }
    }
}

// Kernel 2: a workgroup = one clip's output rows t3 = 4 blockIdx.x .. + 3, all 16 columns and 256 channels; a lane
// takes four channels.
constexpr int kRows3 = 4, kPos2 = kRows3 * kF3, kCols3 = kPos2 / kWaves;  // 64 positions, 8 to a wave's depthwise
constexpr int kTile2 = 2 * kPos2 * kC * 2, kLds2Top = kTile2 + kPos2 * 4;
constexpr int kLds2Bytes = kLds2Top + kWaves * kRows3 * 4;
constexpr int kOutK = kF3 * kC;  // the output linear's inputs

__global__ void __launch_bounds__(kThreads)
subsample2_kernel(const float *x, int T2, int T3, const float *w5, const float *b5, const _Float16 *w6f, const float *w6m,
                  const float *w6, const float *b6, _Float16 *y, float *ys) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), i = lane & 15, g = lane >> 4;
    const int b = blockIdx.y, t3a = blockIdx.x * kRows3;
    const float *xb = x + (long long)b * T2 * kF2 * kC;
    _Float16 *const tile = (_Float16 *)lds;
    float *const pscale = (float *)(lds + kTile2);
    int *const tops = (int *)(lds + kLds2Top);
    float4 wt[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) wt[k] = *(const float4 *)(w5 + k * kC + 4 * lane);
    const float4 bias = *(const float4 *)(b5 + 4 * lane);
    // depthwise: columns f0 .. f0 + kCols3 - 1 of row q; every input column is loaded once
    const int q = wave / (kF3 / kCols3), f0 = kCols3 * (wave % (kF3 / kCols3)), t3 = t3a + q;
    bool plain = false;
    float o[kCols3][4];
#pragma unroll
    for (int c = 0; c < kCols3; ++c) {
        o[c][0] = bias.x, o[c][1] = bias.y, o[c][2] = bias.z, o[c][3] = bias.w;
    }
#pragma unroll
    for (int dy = 0; dy < 3; ++dy) {
        const int t2 = 2 * t3 - 1 + dy;
        const bool row = t2 >= 0 && t2 < T2;
        const float *src = xb + ((long long)(row ? t2 : 0) * kF2) * kC + 4 * lane;
        float4 v[2 * kCols3 + 1];
#pragma unroll
        for (int c = 0; c < 2 * kCols3 + 1; ++c) {  // input columns 2 f0 - 1 + c
            const int f2 = 2 * f0 - 1 + c;
            v[c] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (row && f2 >= 0) v[c] = *(const float4 *)(src + f2 * kC);
        }
#pragma unroll
        for (int c = 0; c < kCols3; ++c)
#pragma unroll
            for (int dx = 0; dx < 3; ++dx) {
                const float4 a = v[2 * c + dx];
                const float4 w = wt[3 * dy + dx];
                o[c][0] = __builtin_fmaf(w.x, a.x, o[c][0]);
                o[c][1] = __builtin_fmaf(w.y, a.y, o[c][1]);
                o[c][2] = __builtin_fmaf(w.z, a.z, o[c][2]);
                o[c][3] = __builtin_fmaf(w.w, a.w, o[c][3]);
            }
    }
#pragma unroll
    for (int c = 0; c < kCols3; ++c) {
        const int p = 16 * q + f0 + c;
        const int bits = kea::wave_max_bits(kea::max_abs<4>(o[c]));
        plain = plain || bits >= kInfBits;
        const int e = exponent_of(bits);
        typedef _Float16 v4h __attribute__((ext_vector_type(4)));
        v4h hi, lo;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            _Float16 h, l;
            split1(o[c][k], pow2(14 - e), h, l);
            hi[k] = h;
            lo[k] = l;
        }
        _Float16 *dst = tile + p * kC + (((lane >> 1) ^ (p & 15)) * 8) + (lane & 1) * 4;
        *(v4h *)dst = hi;
        *(v4h *)(dst + kPos2 * kC) = lo;
        if (lane == 0) pscale[p] = pow2(e - 14);
    }
    Weights weights;
    weights.start(w6f, wave, lane);
    plain = __syncthreads_or(plain) != 0;
    const int rows = min(kRows3, T3 - t3a);
    const long long row0 = (long long)b * T3 + t3a;
    typedef _Float16 v4h __attribute__((ext_vector_type(4)));
    // four values of a row, split with its scale; of a row with an infinity only the infinities count
    auto store = [&](int r, int k, v4f v, float sf, bool inf) {
        v4h hi, lo;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            _Float16 h, l;
            split1(v[e], sf, h, l);
            hi[e] = h;
            lo[e] = inf ? (_Float16)0.f : l;
        }
        _Float16 *dst = y + (row0 + r) * 2 * kOutK + k;
        *(v4h *)dst = hi;
        *(v4h *)(dst + kOutK) = lo;
    };
    auto row_scale = [&](int r) {  // of row r's largest magnitude (all waves' parts are in tops)
        int big = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) big = max(big, tops[w * kRows3 + r]);
        return big;
    };
    // A copy for each form: where their sums met in one, the compiler moved them (26.1 against 25.1 us; in kernel 1 the copies
    // are the slower ones).
    auto epilogue = [&](auto split_tag, v4f (&acc)[2][kPos2 / 16]) {
        constexpr bool SPLIT = decltype(split_tag)::value;
#pragma unroll
        for (int mt = 0; mt < kPos2 / 16; ++mt) {  // m-tile = output row, m = its column
            const float pm = SPLIT ? pscale[16 * mt + i] : 1.f;
            float m = 0.f;
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) {
                const int n = 32 * wave + 16 * nt + 4 * g;
                const v4f bs = *(const v4f *)(b6 + n), wm = SPLIT ? *(const v4f *)(w6m + n) : (v4f){1.f, 1.f, 1.f, 1.f};
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[nt][mt][r] = fmaxf(__builtin_fmaf(acc[nt][mt][r] * wm[r], pm, bs[r]), 0.f);
                m = kea::max_abs2(acc[nt][mt][0], acc[nt][mt][1], m);
                m = kea::max_abs2(acc[nt][mt][2], acc[nt][mt][3], m);
            }
            const int t = kea::wave_max_bits(m);
            if (lane == 0) tops[wave * kRows3 + mt] = t;
        }
        __syncthreads();
#pragma unroll
        for (int mt = 0; mt < kPos2 / 16; ++mt) {
            if (mt >= rows) continue;
            const int big = row_scale(mt), e = exponent_of(big);
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
                store(mt, i * kC + 32 * wave + 16 * nt + 4 * g, acc[nt][mt], pow2(14 - e), big >= kInfBits);
            if (tid == 0) ys[row0 + mt] = big >= kInfBits ? __builtin_inff() : pow2(e - 14);
        }
    };
    v4f acc[2][kPos2 / 16];
    if (plain) {  // an infinity: the same sums in FP32
        float *const h = (float *)lds;  // [kPos2][256]
#pragma unroll
        for (int c = 0; c < kCols3; ++c)
            *(float4 *)(h + fp32_at(16 * q + f0 + c, 4 * lane)) = make_float4(o[c][0], o[c][1], o[c][2], o[c][3]);
        __syncthreads();
        pointwise_fp32<kPos2 / 16>(h, w6, wave, lane, acc);
        epilogue(std::false_type{}, acc);
    } else {
        pointwise<kPos2 / 16>(tile, weights, lane, acc);
        epilogue(std::true_type{}, acc);
    }
}

// Kernel 3, the output linear: y[m][n] = sum_k x[m][k] w[n][k] + bias[n] over the 4096 split inputs of a row, 128 x 128
// tiles. Both operands come by direct copies to LDS in MFMA operand order (the weights laid out so, the inputs by
// their rows), two k-steps of 32 a stage, two stages; waves 0 - 3 (64 x 64 each) take the stage's first
// k-step, waves 4 - 7 the second, and their sums meet in LDS at the end. A wave holds the next stage's operands in
// registers while it multiplies this one's, so a stage's buffer is refilled a stage and a half before it is read.
constexpr int kBlk = 128, kStage = 2 * 2 * kBlk * 32 * 2 * 2, kLds3Bytes = 2 * kStage;  // 64 KB a stage

typedef __attribute__((address_space(1))) const void *gptr_t;
typedef __attribute__((address_space(3))) void *lptr_t;
template <int VM, int LGKM>
__device__ __forceinline__ void wait_counts() { __builtin_amdgcn_s_waitcnt((VM & 15) | ((VM >> 4) << 14) | (7 << 4) | (LGKM << 8)); }
__device__ __forceinline__ void stage_barrier() {  // without the wait for the copies in flight that __syncthreads makes
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// One output row's four columns: scaled sums, or for a row with infinities those alone (w: [n][256 x 16] FP32).
__device__ __forceinline__ void finish(const _Float16 *x, const float *xs, const float *wm, const float *w, float gain,
                                       const float *bias, long long m, int n, int N, v4f v, float *y) {
    const float s = xs[m];
    const v4f b = *(const v4f *)(bias + n), sc = *(const v4f *)(wm + n);
    v4f r;
    if (s == __builtin_inff()) {
        v = (v4f){0.f, 0.f, 0.f, 0.f};
        for (int k = 0; k < kOutK; ++k)
            if ((float)x[m * 2 * kOutK + k] == __builtin_inff())
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[e] += w[(long long)(n + e) * kOutK + (k % kC) * kF3 + k / kC] * gain * __builtin_inff();
        r = v + b;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] = __builtin_fmaf(v[e] * sc[e], s, b[e]);
    }
    *(v4f *)(y + m * N + n) = r;
}

__global__ void __launch_bounds__(kThreads)
subsample3_kernel(const _Float16 *x, const float *xs, long long M, int N, int S, const _Float16 *wf, const float *wm,
                  const float *w, float gain, const float *bias, float *part, float *y) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), i = lane & 15, g = lane >> 4;
    // an XCD (workgroups go round them) takes neighbouring tiles of one K slice
    const int total = gridDim.x, id = blockIdx.x;
    const int v = total % 8 == 0 ? (id & 7) * (total / 8) + (id >> 3) : id;
    const int tiles_n = N / kBlk, nt0 = v % tiles_n, rest = v / tiles_n, tiles_m = (int)((M + kBlk - 1) / kBlk);
    const long long m0 = (long long)(rest % tiles_m) * kBlk;
    const int slice = rest / tiles_m, n0 = nt0 * kBlk;
    const int steps = kOutK / 64 / S;  // stages of this slice: 4 to 64
    // A stage: [x][16-row tile][plane][16 rows][64 inputs], 16-byte pieces XOR-swizzled by row, then [w][k-step][16-row
    // tile][plane][64 lanes][8]; this wave copies its tile of x, whole 128-byte lines of eight rows at a time, and of w.
    const int r8 = lane >> 3, piece = (lane & 7) ^ r8;
    const long long row = m0 + 16 * wave + r8;
    const _Float16 *xa = x + min(row, M - 1) * 2 * kOutK + slice * (kOutK / S) + 8 * piece;
    const _Float16 *xb = x + min(row + 8, M - 1) * 2 * kOutK + slice * (kOutK / S) + 8 * piece;
    const _Float16 *wa = wf + (((long long)(n0 / 16 + wave) * (kOutK / 32) + slice * (kOutK / 32 / S)) * 2 * 64 + lane) * 8;
    auto copy = [&](int p) {
        char *dst = lds + (p & 1) * kStage;
#pragma unroll
        for (int pl = 0; pl < 2; ++pl) {
            __builtin_amdgcn_global_load_lds((gptr_t)(xa + pl * kOutK + p * 64), (lptr_t)(dst + (wave * 2 + pl) * 2048), 16, 0, 0);
            __builtin_amdgcn_global_load_lds((gptr_t)(xb + pl * kOutK + p * 64),
                                             (lptr_t)(dst + (wave * 2 + pl) * 2048 + 1024), 16, 0, 0);
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
                __builtin_amdgcn_global_load_lds((gptr_t)(wa + ((2 * p + kk) * 2 + pl) * 512),
                                                 (lptr_t)(dst + 32768 + kk * 16384 + (wave * 2 + pl) * 1024), 16, 0, 0);
        }
    };
    const int kg = wave >> 2, wm4 = 4 * ((wave >> 1) & 1), wn4 = 4 * (wave & 1);
    struct Operands {
        v8h x[4][2], w[4][2];
    };
    auto read = [&](int p, Operands &o) {
        const char *src = lds + (p & 1) * kStage, *sx = src + i * 128 + (((4 * kg + g) ^ (i & 7)) * 16),
                   *sw = src + 32768 + kg * 16384 + lane * 16;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int pl = 0; pl < 2; ++pl) {
                o.x[t][pl] = *(const v8h *)(sx + ((wm4 + t) * 2 + pl) * 2048);
                o.w[t][pl] = *(const v8h *)(sw + ((wn4 + t) * 2 + pl) * 1024);
            }
    };
    v4f acc[4][4];  // [n-tile][m-tile]
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[a][c] = (v4f){0.f, 0.f, 0.f, 0.f};
    auto step = [&](int p, const Operands &now, Operands &next) {
        if (p + 2 < steps)
            wait_counts<8, 15>();  // stage p + 1 has landed, p + 2 may be in flight
        else
            wait_counts<0, 15>();
        stage_barrier();
        if (p + 1 < steps) read(p + 1, next);
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[a][c] = mfma_split(now.w[a][0], now.w[a][1], now.x[c][0], now.x[c][1], acc[a][c]);
        wait_counts<63, 0>();  // the reads are done: the buffer can be refilled
        stage_barrier();
        if (p + 3 < steps) copy(p + 3);
    };
    Operands even, odd;
    copy(0);
    copy(1);
    wait_counts<8, 15>();
    stage_barrier();
    read(0, even);
    wait_counts<63, 0>();
    stage_barrier();
    copy(2);
    for (int p = 0; p < steps; p += 2) {
        step(p, even, odd);
        step(p + 1, odd, even);
    }
    // waves 4 - 7 hand their sums over
    v4f *const hand = (v4f *)lds + (wave & 3) * 16 * 64 + lane;
    if (kg == 1) {
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int c = 0; c < 4; ++c) hand[(a * 4 + c) * 64] = acc[a][c];
    }
    __syncthreads();
    if (kg == 1) return;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const long long m = m0 + 16 * (wm4 + c) + i;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const int n = n0 + 16 * (wn4 + a) + 4 * g;
            const v4f sum = acc[a][c] + hand[(a * 4 + c) * 64];
            if (m < M) {
                if (S > 1)
                    *(v4f *)(part + ((long long)slice * M + m) * N + n) = sum;
                else
                    finish(x, xs, wm, w, gain, bias, m, n, N, sum, y);
            }
        }
    }
}

// The K slices of kernel 3 added up in order.
template <int S>
__global__ void __launch_bounds__(256)
subsample_sum_kernel(const _Float16 *x, const float *xs, long long M, int N, const float *wm, const float *w,
                     float gain, const float *bias, const float *part, float *y) {
    const long long e = ((long long)blockIdx.x * 256 + threadIdx.x) * 4;
    if (e >= M * N) return;
    v4f t[S];
#pragma unroll
    for (int s = 0; s < S; ++s) t[s] = *(const v4f *)(part + s * M * N + e);
    v4f sum = t[0];
#pragma unroll
    for (int s = 1; s < S; ++s) sum += t[s];
    const long long m = e / N;
    finish(x, xs, wm, w, gain, bias, m, (int)(e - m * N), N, sum, y);
}

// K slices: enough workgroups for the 256 CUs, at least four stages to a slice.
int slices(long long M, int N) {
    const long long tiles = (M + kBlk - 1) / kBlk * (N / kBlk);
    int s = 1;
    while (s < 16 && tiles * s * 2 <= 256) s *= 2;
    return s;
}

int launched(const char *what) {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? KEA_OK : kea::fail((int)e, std::string(what) + " launch failed: " + hipGetErrorString(e));
}
template <class Fn>
int allow_lds(Fn fn, int bytes) {
    const hipError_t e = hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    return e == hipSuccess ? KEA_OK : kea::fail((int)e, std::string("LDS attribute refused: ") + hipGetErrorString(e));
}

}  // namespace

extern "C" int kea_subsample_stage1(const float *x, int64_t batch, int64_t t, const void *w1f, const float *w1m,
                                    const float *w1, const float *b1, const float *w2, const float *b2, const void *w3f,
                                    const float *w3m, const float *w3, const float *b3, float *y, void *stream) {
    if (batch < 0 || batch > 65535 || t < 1 || t > INT32_MAX / 4) return kea::fail(KEA_EINVAL, "bad sizes");
    if (batch == 0) return KEA_OK;
    if (!x || !w1f || !w1m || !w1 || !b1 || !w2 || !b2 || !w3f || !w3m || !w3 || !b3 || !y)
        return kea::fail(KEA_EINVAL, "null pointer");
    if (((uintptr_t)w1f | (uintptr_t)w1m | (uintptr_t)b1 | (uintptr_t)w2 | (uintptr_t)b2 | (uintptr_t)w3f | (uintptr_t)w3m | (uintptr_t)b3 | (uintptr_t)y) & 15)
        return kea::fail(KEA_EALIGN, "every operand but x, w1 and w3 must be 16-byte aligned");
    const int t1 = (int)((t - 1) / 2 + 1), t2 = (t1 - 1) / 2 + 1;
    if (const int rc = allow_lds(subsample1_kernel, kLds1Bytes)) return rc;
    hipLaunchKernelGGL(subsample1_kernel, dim3((unsigned)((t2 + kRows2 - 1) / kRows2), (unsigned)batch), dim3(kThreads),
                       kLds1Bytes, (hipStream_t)stream, x, (int)t, t1, t2, (const _Float16 *)w1f, w1m, w1, b1, w2, b2,
                       (const _Float16 *)w3f, w3m, w3, b3, y);
    return launched("subsample stage 1");
}

extern "C" int kea_subsample_stage2(const float *x, int64_t batch, int64_t t2, const float *w5, const float *b5,
                                    const void *w6f, const float *w6m, const float *w6, const float *b6, void *y,
                                    float *ys, void *stream) {
    if (batch < 0 || batch > 65535 || t2 < 1 || t2 > INT32_MAX / 4) return kea::fail(KEA_EINVAL, "bad sizes");
    if (batch == 0) return KEA_OK;
    if (!x || !w5 || !b5 || !w6f || !w6m || !w6 || !b6 || !y || !ys) return kea::fail(KEA_EINVAL, "null pointer");
    if (((uintptr_t)x | (uintptr_t)w5 | (uintptr_t)b5 | (uintptr_t)w6f | (uintptr_t)w6m | (uintptr_t)b6 | (uintptr_t)y) & 15)
        return kea::fail(KEA_EALIGN, "every operand but w6 and ys must be 16-byte aligned");
    const int t3 = (int)((t2 - 1) / 2 + 1);
    if (const int rc = allow_lds(subsample2_kernel, kLds2Bytes)) return rc;
    hipLaunchKernelGGL(subsample2_kernel, dim3((unsigned)((t3 + kRows3 - 1) / kRows3), (unsigned)batch), dim3(kThreads),
                       kLds2Bytes, (hipStream_t)stream, x, (int)t2, t3, w5, b5, (const _Float16 *)w6f, w6m, w6, b6,
                       (_Float16 *)y, ys);
    return launched("subsample stage 2");
}

extern "C" int64_t kea_subsample_out_workspace(int64_t m, int64_t n) {
    if (m < 1 || n < kBlk || n % kBlk) return 0;
    const int s = slices(m, (int)n);
    return s > 1 ? s * m * n * (int64_t)sizeof(float) : 0;
}

extern "C" int kea_subsample_out(const void *x, const float *xs, int64_t m, int64_t n, const void *wf, const float *wm,
                                 const float *w, float gain, const float *bias, float *y, void *workspace,
                                 int64_t workspace_bytes, void *stream) {
    if (m < 0 || n < kBlk || n % kBlk || n > 65536) return kea::fail(KEA_EINVAL, "bad sizes: n must be a multiple of 128");
    if (m == 0) return KEA_OK;
    const long long tiles = (m + kBlk - 1) / kBlk * (n / kBlk);
    if (tiles > (1 << 20)) return kea::fail(KEA_EINVAL, "too many rows");
    if (!x || !xs || !wf || !wm || !w || !bias || !y) return kea::fail(KEA_EINVAL, "null pointer");
    if (((uintptr_t)x | (uintptr_t)wf | (uintptr_t)wm | (uintptr_t)bias | (uintptr_t)y | (uintptr_t)workspace) & 15)
        return kea::fail(KEA_EALIGN, "every operand but xs and w must be 16-byte aligned");
    const int s = slices(m, (int)n);
    if (s > 1 && (!workspace || workspace_bytes < kea_subsample_out_workspace(m, n)))
        return kea::fail(KEA_ESPACE, "workspace too small");
    if (const int rc = allow_lds(subsample3_kernel, kLds3Bytes)) return rc;
    hipLaunchKernelGGL(subsample3_kernel, dim3((unsigned)(tiles * s)), dim3(kThreads), kLds3Bytes, (hipStream_t)stream,
                       (const _Float16 *)x, xs, (long long)m, (int)n, s, (const _Float16 *)wf, wm, w, gain, bias,
                       (float *)workspace, y);
    if (const int rc = launched("subsample output linear")) return rc;
    if (s == 1) return KEA_OK;
    const auto sum = s == 2 ? subsample_sum_kernel<2> : s == 4 ? subsample_sum_kernel<4> : s == 8 ? subsample_sum_kernel<8>
                                                                                            : subsample_sum_kernel<16>;
    hipLaunchKernelGGL(sum, dim3((unsigned)((m * n / 4 + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       (const _Float16 *)x, xs, (long long)m, (int)n, wm, w, gain, bias, (const float *)workspace, y);
    return launched("subsample output sum");
}
