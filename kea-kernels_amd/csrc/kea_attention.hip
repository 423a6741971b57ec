// Relative-position self-attention over sequences of any length for MI355X (gfx950): key blocks with an online softmax
// on the FP16 matrix cores at FP32 accuracy.
//
//   s[i][j] = ((q_i + u) . k_j + (q_i + v) . p_{T-1-i+j}) * scale,  out_i = sum_j softmax_j(s)[i][j] v_j
//
// Arithmetic. The FP32 matrix instruction runs at 1/16 of the FP16 rate, so operands are pairs of FP16 values and a
// product is three FP16 MFMAs (kea_split.h), with one power of two per query row, per four rows of K and P and per value
// row. Against FP64 the result is closer than the FP32 forms (fewer roundings of the accumulator). Where the inputs hold an
// infinity, or rows whose elements differ so much in size that the pairs would lose what FP32 keeps (kScores, kLowPairs), a
// workgroup takes an FP32 form on the FP32 matrix instruction instead (NaNs propagate by themselves). That form reads its
// operands from global memory and computes the scores twice: T = 200 batch 8 130 us, T = 750 batch 2 370.
//
// Two launches. split_kernel writes K, V and P once as hi / lo planes in the order the LDS of the second kernel holds
// them, 64 rows to a block; relpos_tiled_kernel then copies blocks straight to LDS (global_load_lds) and spends no
// vector instruction on them. (Splitting inside the attention kernel, every 64-query workgroup for itself, took a third
// of its time: T = 750, batch 2 67 us, when the two launches took 58.)
//
// Layout of the work. A workgroup is 4 x 2 waves on 64 queries of one (clip, head); it walks the keys in blocks of 64,
// wave (qg, ks) taking queries 16 qg .. and keys 32 ks .. of a block with its own online softmax; the two partial
// results of a query group are merged through LDS at the end. Scores are formed transposed (D[key][query] = K Q^T), so
// a lane owns one query, the row maximum is two cross-lane steps, and its eight probabilities of a 32-key step are
// already the B operand of O^T = V^T P^T: the contraction order over keys is chosen to match (group g of a wave's
// keys: 4 g + r of both 16-key tiles), and V is stored transposed in that order. The position scores of a wave are the
// band of 47 relative rows its 16 x 32 tile needs (three 16-row tiles), read back along the diagonal from LDS. The
// band of a workgroup is 127 rows, two blocks of P, which are cut so that every workgroup's band starts at a block:
// each key block needs one new block of P. Rows are unpadded with XOR-swizzled 16-byte units, so 16 rows read at one
// unit are conflict-free. K and the new P block are copied while the softmax and the P.V products run, V while the
// next scores do.
//
// Bound by the phases' barriers: of the second kernel's 45 us at T = 750, batch 2 (192 workgroups, one to a CU; hardware
// counters) the MFMAs of a SIMD's two waves take 13, their vector instructions 12 and the CU's LDS 12, and the waves wait
// for 48% of their time. Measured on MI355X, graph-timed, both launches, against what served these
// lengths before (T <= 256 an FP32 vector kernel, above it PyTorch operators on [T, 2T] score matrices): T = 200 batch 8
// 32 / 173 us, T = 250 batch 1 24 / 28, T = 375 batch 2 33 / 146, T = 750 batch 2 51 / 285, T = 750 batch 8 154 / 890. Up to
// 128 frames the FP32 matrix-core kernels of kea_encoder.hip, one pass without a workspace, are the faster ones: T = 125
// batch 8 19 against 24 us, batch 1 11 against 17; at T = 129 batch 1 it is 20 against 20.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <type_traits>

#include "kea_internal.h"
#include "kea_split.h"
#include "kea_wave.h"
#include "../../include/kea_encoder.h"

namespace {

constexpr int kDK = 128;
constexpr float kLog2e = 1.4426950408889634f;

using kea::exponent_of;
using kea::kInfBits;
using kea::max_abs;
using kea::pow2;
using kea::split1;
using kea::split8;
using kea::v4f;
using kea::v8h;
using kea::wave_max_bits;

constexpr int kQG = 4, kKS = 2;                 // query groups and key halves: one wave each
constexpr int kNW = kQG * kKS, kRows = 64;      // rows of a block of K, V or P; queries of a workgroup
static_assert(kKS == 2 && 16 * kQG == kRows && 32 * kKS == kRows, "queries, keys and P rows advance by the same block");
constexpr int kPlane = kRows * kDK;             // elements of one plane of a block
constexpr int kBlockBytes = 2 * kPlane * 2;     // hi and lo planes
// Rows that the split form would not hold to FP32's accuracy go to the FP32 form. A value row's elements are held to 2^-31 of
// the row's largest (with their probabilities): a wave's 16 rows with nonzero pairs of elements 2^10 below their row's largest
// in kLowPairs or more of the 64 columns of pairs are not split (a normal pair is that small once in 10^5, four of the 1024
// once in 10^10). An element of Q, K or P is held to 2^-39
// of its row's largest (K and P: of four rows'), which costs a score at most 2^-31 of the largest query element times the
// largest of K and P times the scale, and that if every element of the rows is so small: up to kScores, 2^-25 measured,
// what FP32 rounds off a score of ordinary rows.
constexpr int kLowPairs = 4;
constexpr float kScores = 4096.f;
constexpr int kBandStride = 52;                 // band scores of a query in LDS (floats): 47 used

// The split operands in the workspace.
//   K, V: block (b, h, kb), keys 64 kb ..;  P: block (h, pb), relative rows T - 64 + 64 (pb + 1 - tiles) ..: the two
//   planes, in LDS order;  Q: block (b, h, tile): for both biases (u, v) the two planes of four 16-query groups as MFMA
//   operands [s][lane][8] (lane: query lane % 16, elements 32 s + 8 (lane / 16) .. + 7).
//   Multipliers 2^(e - 14): km, pm one for four rows, qm [bias][query]; ve: the exponent e of each of the 64 value rows.
//   top: the bits of the largest magnitude, kt for K, pt for P, qt for Q; vt: an infinity's bits where the block's value rows
//   are not to be split, or zero.
struct SplitOperands {
    char *q, *k, *v, *p;
    float *qm, *km, *pm;
    int32_t *ve, *qt, *kt, *vt, *pt;
    int tiles, pblocks;  // 64-row tiles of the sequence; blocks of P per head
};
constexpr int kQBlockBytes = 2 * kBlockBytes;
inline long long split_layout(SplitOperands *s, char *ws, long long batch, int heads, long long t) {
    const long long tiles = (t + kRows - 1) / kRows, kv = batch * heads * tiles, np = 2 * tiles * heads;
    long long off = 0;
    auto take = [&](auto &field, long long bytes) {
        field = (std::remove_reference_t<decltype(field)>)(ws + off);
        off += (bytes + 15) / 16 * 16;
    };
    take(s->q, kv * kQBlockBytes);
    take(s->k, kv * kBlockBytes);
    take(s->v, kv * kBlockBytes);
    take(s->p, np * kBlockBytes);
    take(s->qm, kv * 2 * kRows * 4);
    take(s->km, kv * 16 * 4);
    take(s->pm, np * 16 * 4);
    take(s->ve, kv * kRows * 4);
    take(s->qt, kv * 4);
    take(s->kt, kv * 4);
    take(s->vt, kv * 4);
    take(s->pt, np * 4);
    s->tiles = (int)tiles;
    s->pblocks = (int)(2 * tiles);
    return off;
}

// One workgroup (256 threads) splits one block: blockIdx.x < kv a block of V, then kv blocks of Q, kv of K, then P. Bound by
// the bytes at large sizes (4 read and 4, Q: 8, written an element) and by one block's chain of loads, maxima and stores at
// small ones: K and V by one workgroup, one after the other, were 0.9 us slower at T = 175, batch 2.
__global__ void __launch_bounds__(256)
split_kernel(const float *qkv, long long ld, const float *pos, long long ldp, const float *bias_u, const float *bias_v,
             int T, int H, int kv, SplitOperands so) {
    __shared__ __attribute__((aligned(16))) _Float16 vt[2 * kPlane];
    __shared__ int top[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;
    int seen = 0;
    // 64 rows of a [rows][stride] matrix from row `first` (zeros outside [0, count)): four rows a wave and step, 16
    // lanes a row
    auto rows = [&](const float *src, long long stride, int first, int count, _Float16 *dst, float *mul) {
        float x[4][8];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int row = first + 16 * u + 4 * wave + g;
            float4 a = make_float4(0.f, 0.f, 0.f, 0.f), d = a;
            if (row >= 0 && row < count) {
                const float *p = src + (long long)row * stride + 8 * n;
                a = *(const float4 *)p;
                d = *(const float4 *)(p + 4);
            }
            x[u][0] = a.x; x[u][1] = a.y; x[u][2] = a.z; x[u][3] = a.w; x[u][4] = d.x; x[u][5] = d.y; x[u][6] = d.z; x[u][7] = d.w;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int row = 16 * u + 4 * wave + g;
            const int bits = wave_max_bits(max_abs<8>(x[u])), e = exponent_of(bits);
            seen = max(seen, bits);
            v8h hi, lo;
            split8(x[u], pow2(14 - e), hi, lo);
            _Float16 *p = dst + row * kDK + ((n ^ (row & 15)) * 8);
            *(v8h *)p = hi;
            *(v8h *)(p + kPlane) = lo;
            if (lane == 0) mul[4 * u + wave] = pow2(e - 14);
        }
    };
    auto finish = [&](int32_t *word) {  // the block's largest magnitude
        if (lane == 0) top[wave] = seen;
        __syncthreads();
        if (tid == 0) *word = max(max(top[0], top[1]), max(top[2], top[3]));
    };
    if ((int)blockIdx.x >= 3 * kv) {
        const int id = blockIdx.x - 3 * kv, h = id / so.pblocks, pb = id - h * so.pblocks;
        rows(pos + (long long)h * kDK, ldp, T - kRows + kRows * (pb + 1 - so.tiles), 2 * T - 1,
             (_Float16 *)(so.p + (long long)id * kBlockBytes), so.pm + (long long)id * 16);
        finish(so.pt + id);
        return;
    }
    const int part = (int)blockIdx.x / kv, id = (int)blockIdx.x - part * kv;
    const int kb = id % so.tiles, bh = id / so.tiles, h = bh % H, b = bh / H, j0 = kb * kRows;
    const float *qbase = qkv + (long long)b * T * ld + (long long)h * kDK;
    if (part == 2) {
        rows(qbase + (long long)H * kDK, ld, j0, T, (_Float16 *)(so.k + (long long)id * kBlockBytes), so.km + (long long)id * 16);
        finish(so.kt + id);
        return;
    }
    if (part == 1) {  // queries: wave = 16-query group, a lane per query and quarter of each 32-element step
        const int i = j0 + 16 * wave + n;
        float x[2][4][8];
        const float *q = qbase + (long long)min(i, T - 1) * ld + 8 * g;
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int c = 0; c < 8; c += 4) {
                const int at = h * kDK + 8 * g + 32 * s + c;
                const float4 a = *(const float4 *)(q + 32 * s + c), u = *(const float4 *)(bias_u + at),
                             v = *(const float4 *)(bias_v + at);
                x[0][s][c] = a.x + u.x; x[0][s][c + 1] = a.y + u.y; x[0][s][c + 2] = a.z + u.z; x[0][s][c + 3] = a.w + u.w;
                x[1][s][c] = a.x + v.x; x[1][s][c + 1] = a.y + v.y; x[1][s][c + 2] = a.z + v.z; x[1][s][c + 3] = a.w + v.w;
            }
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            float m = max_abs<32>(&x[w][0][0]);
            m = fmaxf(m, __shfl_xor(m, 16, 64));
            m = fmaxf(m, __shfl_xor(m, 32, 64));
            seen = max(seen, wave_max_bits(m));
            const int e = exponent_of(__builtin_bit_cast(int, m));
            if (g == 0) so.qm[((long long)id * 2 + w) * kRows + 16 * wave + n] = pow2(e - 14);
            char *dst = so.q + (long long)id * kQBlockBytes + w * kBlockBytes + wave * 4096 + lane * 16;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                v8h hi, lo;
                split8(x[w][s], pow2(14 - e), hi, lo);
                *(v8h *)(dst + s * 1024) = hi;
                *(v8h *)(dst + s * 1024 + kPlane * 2) = lo;
            }
        }
        finish(so.qt + id);
        return;
    }
    const float *vbase = qbase + 2LL * H * kDK;
    float v[2][8][2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int grp = 4 * u + wave;  // keys 32 (grp / 4) + 16 t + 4 (grp % 4) + r, t = 0, 1, r = 0..3
            const int j = j0 + 32 * (grp >> 2) + 16 * (e >> 2) + 4 * (grp & 3) + (e & 3);
            float2 w = make_float2(0.f, 0.f);
            if (j < T) w = *(const float2 *)(vbase + (long long)j * ld + 2 * lane);
            v[u][e][0] = w.x;
            v[u][e][1] = w.y;
        }
    // A scale per key: its row may be any size beside the others'. Key index x + 4 y: the exponents are formed in the lanes of
    // row y and the scales read from there (16 of each in scalar instructions took half a microsecond).
    float pair[16], most[4], sf[16];
    int ex[4];
#pragma unroll
    for (int k = 0; k < 16; ++k) pair[k] = max_abs<2>(v[k >> 3][k & 7]);
    kea::wave_max_rows(pair, most);
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        ex[x] = exponent_of(__builtin_bit_cast(int, most[x]));
#pragma unroll
        for (int y = 0; y < 4; ++y) sf[x + 4 * y] = kea::lane_value(pow2(14 - ex[x]), 16 * y);
    }
    if (n == 0) *(int4 *)(so.ve + (long long)id * kRows + 16 * g + 4 * wave) = make_int4(ex[0], ex[1], ex[2], ex[3]);
    bool low = false;  // (a row's largest is scaled to [2^14, 2^15))
#pragma unroll
    for (int k = 0; k < 16; ++k) low = low || (pair[k] != 0.f && pair[k] * sf[k] < 16.f);
    const bool infinite = fmaxf(fmaxf(most[0], most[1]), fmaxf(most[2], most[3])) >= __builtin_inff();
    if (__any(infinite) || __popcll(__ballot(low)) >= kLowPairs) seen = kInfBits;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int grp = 4 * u + wave;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            v8h hi, lo;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                _Float16 h, l;
                split1(v[u][k][c], sf[8 * u + k], h, l);
                hi[k] = h;
                lo[k] = l;
            }
            _Float16 *p = vt + (2 * lane + c) * kRows + ((grp ^ (lane & 7)) * 8);  // row d = 2 lane + c, unit ^ (d / 2 % 8)
            *(v8h *)p = hi;
            *(v8h *)(p + kPlane) = lo;
        }
    }
    finish(so.vt + id);
    v8h *dst = (v8h *)(so.v + (long long)id * kBlockBytes);
#pragma unroll
    for (int u = 0; u < 2 * kPlane / 8 / 256; ++u) dst[u * 256 + tid] = ((const v8h *)vt)[u * 256 + tid];
}

typedef __attribute__((address_space(1))) const void *gptr_t;
typedef __attribute__((address_space(3))) void *lptr_t;

// A block from the workspace to LDS, by all waves of the workgroup: four 16-byte copies a lane.
__device__ __forceinline__ void copy_block(const char *src, char *dst, int wave, int lane) {
#pragma unroll
    for (int u = 0; u < kBlockBytes / (kNW * 1024); ++u) {
        const int off = (u * kNW + wave) * 1024;
        __builtin_amdgcn_global_load_lds((gptr_t)(src + off + lane * 16), (lptr_t)(dst + off), 16, 0, 0);
    }
}
// Every copy (and load) of this wave has landed; then all waves' (no fence: only LDS copies and reads are ordered here).
// The wait is the builtin so that the compiler counts it: after an inline one it waits again at the first use of a
// loaded value, and with that for the copies issued since.
__device__ __forceinline__ void landed_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

constexpr int kLdsK = 0, kLdsP = kLdsK + kBlockBytes, kLdsV = kLdsP + 2 * kBlockBytes, kLdsBand = kLdsV + kBlockBytes;
constexpr int kLdsPlain = kLdsBand + kNW * 16 * kBandStride * 4, kTiledLds = kLdsPlain + kNW * 4;

__global__ void __launch_bounds__(kNW * 64)
relpos_tiled_kernel(const float *qkv, long long ld, const float *pos, long long ldp, const float *bias_u,
                    const float *bias_v, float *out, long long ldo, int T, int H, float scale, SplitOperands so) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4, qg = wave / kKS, ks = wave % kKS;
    // blockIdx.x is the head: consecutive workgroups go to different XCDs, so one XCD's L2 serves a head's K, V and P
    const int h = blockIdx.x, iq0 = blockIdx.y, b = blockIdx.z, tiles = so.tiles;
    const long long bh = (long long)b * H + h;
    const char *kblk = so.k + bh * tiles * kBlockBytes, *vblk = so.v + bh * tiles * kBlockBytes;
    // the band starts at P block tiles - iq0 - 1; key block kb uses it and the next, advanced by kb
    const long long pfirst = (long long)h * so.pblocks + tiles - iq0 - 1;
    const char *pblk = so.p + pfirst * kBlockBytes;
    _Float16 *const Kh = (_Float16 *)(lds + kLdsK), *const Ph = (_Float16 *)(lds + kLdsP), *const Vh = (_Float16 *)(lds + kLdsV);
    float *const bd = (float *)(lds + kLdsBand) + wave * 16 * kBandStride;
    int *const plain = (int *)(lds + kLdsPlain);  // a word per wave, written by every wave before the first barrier

    copy_block(kblk, lds + kLdsK, wave, lane);
    copy_block(pblk, lds + kLdsP, wave, lane);
    copy_block(pblk + kBlockBytes, lds + kLdsP + kBlockBytes, wave, lane);
    copy_block(vblk, lds + kLdsV, wave, lane);
    // the wave's queries as MFMA operands; their multipliers with the softmax scale and the change to base 2
    v8h qu[2][4], qv[2][4];
    const char *qblk = so.q + (bh * tiles + iq0) * kQBlockBytes + qg * 4096 + lane * 16;
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            qu[p][s] = *(const v8h *)(qblk + p * (kPlane * 2) + s * 1024);
            qv[p][s] = *(const v8h *)(qblk + kBlockBytes + p * (kPlane * 2) + s * 1024);
        }
    const int iq = iq0 * kRows + 16 * qg + n;
    const float *qm = so.qm + (bh * tiles + iq0) * 2 * kRows + 16 * qg + n;
    const float mqu = qm[0] * (scale * kLog2e), mqv = qm[kRows] * (scale * kLog2e);
    const int qtop = so.qt[bh * tiles + iq0];
    int top = 0;
    for (int i = tid; i < tiles; i += kNW * 64)
        top = max(max(max(top, so.kt[bh * tiles + i]), so.vt[bh * tiles + i]), max(so.pt[pfirst + i], so.pt[pfirst + i + 1]));
    const float most = __builtin_bit_cast(float, qtop) * __builtin_bit_cast(float, top) * fabsf(scale * kLog2e);
    const bool wave_plain = __any(max(qtop, top) >= kInfBits || most > kScores) != 0;
    if (lane == 0) plain[wave] = wave_plain;
    // multipliers of the wave's band tiles (rows 48 - 16 qg + 32 ks + 16 t of the two blocks), keys and V groups
    const int band0 = 48 - 16 * qg + 32 * ks;
    const float *pmp = so.pm + pfirst * 16 + band0 / 4 + g, *kmp = so.km + bh * tiles * 16 + 8 * ks + g;
    const int32_t *vep = so.ve + bh * tiles * kRows + 32 * ks + 4 * g;
    float pmul[3], kmul[2];
    int4 ev[2];  // exponents of the lane's eight value rows
    auto load_multipliers = [&](int kb) {
#pragma unroll
        for (int t = 0; t < 3; ++t) pmul[t] = pmp[kb * 16 + 4 * t];
#pragma unroll
        for (int t = 0; t < 2; ++t) kmul[t] = kmp[kb * 16 + 4 * t];
#pragma unroll
        for (int t = 0; t < 2; ++t) ev[t] = *(const int4 *)(vep + kb * kRows + 16 * t);
    };
    load_multipliers(0);
    landed_barrier();

    // Online softmax in base 2 with lazy references: probabilities are 2^(s - m_ref) with the integer m_ref raised only when
    // a score passes it by more than 8. A key's contribution to its query is its probability times 2^(exponent of its value
    // row); 2^em is their size for this lane's query, raised (and the sums rescaled) only when one passes it by a factor of
    // 2^8, so most blocks accumulate in the MFMA. The probabilities are split at 2^6 of that: what a query's output is
    // made of holds its 22 bits whatever the value rows of other keys are, and a contribution is held to 2^-31 of the
    // query's largest. (em of a step's largest value row instead, whatever its probability, lost the rest of the row to a
    // large value under a suppressed key: 4e-5 of it at 2^16, 1e-2 at 2^24.)
    constexpr int kLazy = 8, kProbExp = 6;
    float m_ref = -INFINITY, l_run = 0.f;  // l_run: this lane's keys only
    int em = -1000;
    v4f o[8];
#pragma unroll
    for (int d = 0; d < 8; ++d) o[d] = (v4f){0.f, 0.f, 0.f, 0.f};

    int any_plain = 0;
#pragma unroll
    for (int w = 0; w < kNW; ++w) any_plain |= plain[w];
    any_plain = __builtin_amdgcn_readfirstlane(any_plain);
    if (__builtin_expect(any_plain, 0)) {
        // The FP32 form, on the FP32 matrix instruction: the same tiles and lanes, operands straight from global memory, the
        // exact two-pass softmax. Element 16 s + 4 g + e of a row is step (s, e) of the contraction.
        const float *qp = qkv + ((long long)b * T + min(iq, T - 1)) * ld + (long long)h * kDK + 4 * g;
        const float *kbase = qkv + (long long)b * T * ld + (long long)(H + h) * kDK + 4 * g, *pbase = pos + (long long)h * kDK + 4 * g;
        const float *vbase = qkv + (long long)b * T * ld + (long long)(2 * H + h) * kDK + n;
        v4f fu[8], fv[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const v4f q = *(const v4f *)(qp + 16 * s);
            fu[s] = q + *(const v4f *)(bias_u + h * kDK + 4 * g + 16 * s);
            fv[s] = q + *(const v4f *)(bias_v + h * kDK + 4 * g + 16 * s);
        }
        auto product = [&](const float *row, const v4f (&q)[8]) {
            v4f c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const v4f x = *(const v4f *)(row + 16 * s);
#pragma unroll
                for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], q[s][e], c, 0, 0, 0);
            }
            return c;
        };
        auto scores = [&](int jw, float (&p)[8]) {
            const int first = T - 16 - (iq0 * kRows + 16 * qg) + jw;  // the band's first relative row
            v4f c[2], r[3];
#pragma unroll
            for (int t = 0; t < 3; ++t) r[t] = product(pbase + (long long)min(max(first + 16 * t + n, 0), 2 * T - 2) * ldp, fv);
#pragma unroll
            for (int t = 0; t < 2; ++t) c[t] = product(kbase + (long long)min(jw + 16 * t + n, T - 1) * ld, fu);
            asm volatile("" ::: "memory");  // (a wave's LDS accesses stay in order)
#pragma unroll
            for (int t = 0; t < 3; ++t) *(v4f *)(bd + n * kBandStride + 16 * t + 4 * g) = r[t];
            asm volatile("" ::: "memory");
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int jj = 16 * t + 4 * g + e;
                    p[4 * t + e] = jw + jj < T ? (c[t][e] + bd[n * kBandStride + 15 - n + jj]) * scale : -INFINITY;
                }
            asm volatile("" ::: "memory");
        };
        float p[8];
        for (int jw = 32 * ks; jw < T; jw += kRows) {
            scores(jw, p);
#pragma unroll
            for (int e = 0; e < 8; ++e) m_ref = fmaxf(m_ref, p[e]);
        }
        m_ref = fmaxf(m_ref, __shfl_xor(m_ref, 16, 64));
        m_ref = fmaxf(m_ref, __shfl_xor(m_ref, 32, 64));
        float *const maxima = (float *)(lds + kLdsV);  // (nothing else lies there from here on)
        if (g == 0) maxima[wave * 16 + n] = m_ref;
        __syncthreads();
        m_ref = fmaxf(m_ref, maxima[(wave ^ 1) * 16 + n]);
        for (int jw = 32 * ks; jw < T; jw += kRows) {
            scores(jw, p);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int j = jw + 16 * (e >> 2) + 4 * g + (e & 3);
                p[e] = j < T ? expf(p[e] - m_ref) : 0.f;
                l_run = l_run + p[e];
                const float *v = vbase + (long long)min(j, T - 1) * ld;
#pragma unroll
                for (int d = 0; d < 8; ++d)
                    o[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(j < T ? v[16 * d] : 0.f, p[e], o[d], 0, 0, 0);
            }
        }
        em = 14 + kProbExp;
    }
    for (int kb = 0; kb < tiles && !any_plain; ++kb) {
        const int jw = kb * kRows + 32 * ks;  // this wave's first key
        int pbase[3];  // element offset of each band tile in the two-block ring
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const int row = band0 + 16 * t;
            pbase[t] = ((kb + row / kRows) & 1) * 2 * kPlane + (row % kRows + n) * kDK;
        }
        v4f sc[2], sp[3];
#pragma unroll
        for (int t = 0; t < 2; ++t) sc[t] = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 3; ++t) sp[t] = (v4f){0.f, 0.f, 0.f, 0.f};
        if (jw < T) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int c = ((4 * s + g) ^ n) * 8;  // tiles start at multiples of 16 rows: row & 15 = n
#pragma unroll
                for (int t = 0; t < 3; ++t) {
                    const _Float16 *p = Ph + pbase[t] + c;
                    const v8h hi = *(const v8h *)p, lo = *(const v8h *)(p + kPlane);
                    sp[t] = kea::mfma_split(hi, lo, qv[0][s], qv[1][s], sp[t]);
                }
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const _Float16 *p = Kh + (32 * ks + 16 * t + n) * kDK + c;
                    const v8h hi = *(const v8h *)p, lo = *(const v8h *)(p + kPlane);
                    sc[t] = kea::mfma_split(hi, lo, qu[0][s], qu[1][s], sc[t]);
                }
            }
            // the band scores of query n at relative positions 16 t + 4 g + r; key jj of the wave is position jj + 15 - n.
            // Stored before the next copies go out: the compiler lets an LDS store wait for every copy in flight.
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                const float mul = pmul[t] * mqv;
                *(float4 *)(bd + n * kBandStride + 16 * t + 4 * g) =
                    make_float4(sp[t][0] * mul, sp[t][1] * mul, sp[t][2] * mul, sp[t][3] * mul);
            }
        }
        landed_barrier();  // K and the older P block are free; V has landed
        if (kb + 1 < tiles) {
            copy_block(kblk + (long long)(kb + 1) * kBlockBytes, lds + kLdsK, wave, lane);
            copy_block(pblk + (long long)(kb + 2) * kBlockBytes, lds + kLdsP + (kb & 1) * kBlockBytes, wave, lane);
        }
        if (jw < T) {
            float p[8], mx = -INFINITY;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const float mul = kmul[t] * mqu;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    p[4 * t + r] = __builtin_fmaf(sc[t][r], mul, bd[n * kBandStride + 15 - n + 16 * t + 4 * g + r]);
            }
            if (jw + 32 > T) {  // the last keys' tile
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (jw + 16 * (e >> 2) + 4 * g + (e & 3) >= T) p[e] = -INFINITY;
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) mx = fmaxf(mx, p[e]);
            if (__any(mx > m_ref + kLazy)) {  // the sums keep their values: 2^em falls by what the reference rises
                mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
                mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
                const bool above = mx > m_ref + kLazy;
                const float m_new = above ? ceilf(mx) : m_ref, rise = above ? m_new - m_ref : 0.f;
                l_run = l_run * __builtin_amdgcn_exp2f(-rise);
                em -= (int)fminf(rise, 1e6f);
                m_ref = m_new;
            }
            const int ek[8] = {ev[0].x, ev[0].y, ev[0].z, ev[0].w, ev[1].x, ev[1].y, ev[1].z, ev[1].w};
            float w[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                p[e] = __builtin_amdgcn_exp2f(p[e] - m_ref);
                l_run = l_run + p[e];
                w[e] = __builtin_amdgcn_ldexpf(p[e], ek[e] - em + kProbExp);
            }
            if (__any(max_abs<8>(w) >= (float)(2 << (kLazy + kProbExp)))) {
                // the largest contribution's exponent (a probability of zero has none, however large its value row is)
                int size = -3000000;
#pragma unroll
                for (int e = 0; e < 8; ++e) size = max(size, p[e] > 0.f ? __builtin_amdgcn_frexp_expf(p[e]) + ek[e] : size);
                size = max(size, __shfl_xor(size, 16, 64));
                size = max(size, __shfl_xor(size, 32, 64)) - 1;
                const int en = size > em + kLazy ? size : em;
                const float f = pow2(max(em - en, -127));
                em = en;
#pragma unroll
                for (int d = 0; d < 8; ++d)
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[d][r] = o[d][r] * f;
#pragma unroll
                for (int e = 0; e < 8; ++e) w[e] = __builtin_amdgcn_ldexpf(p[e], ek[e] - em + kProbExp);
            }
            v8h ph, pl;
            split8(w, 1.f, ph, pl);
#pragma unroll
            for (int d = 0; d < 8; ++d) {
                const _Float16 *vp = Vh + (16 * d + n) * kRows + (((4 * ks + g) ^ (n >> 1)) * 8);
                const v8h hi = *(const v8h *)vp, lo = *(const v8h *)(vp + kPlane);
                o[d] = kea::mfma_split(hi, lo, ph, pl, o[d]);
            }
        }
        if (kb + 1 < tiles) load_multipliers(kb + 1);
        landed_barrier();  // V is free; the next K and P have landed
        if (kb + 1 < tiles) copy_block(vblk + (long long)(kb + 1) * kBlockBytes, lds + kLdsV, wave, lane);
    }
    l_run = l_run + __shfl_xor(l_run, 16, 64);
    l_run = l_run + __shfl_xor(l_run, 32, 64);
    em -= 14 + kProbExp;  // the sums are in units of 2^em now

    // the two partial results of a query group meet in wave ks = 0
    constexpr int kLane = 36;  // floats per lane: 32 outputs, m, l, em
    float *const mb = (float *)lds + (qg * 64 + lane) * kLane;
    if (ks > 0) {
#pragma unroll
        for (int d = 0; d < 8; ++d) *(float4 *)(mb + 4 * d) = make_float4(o[d][0], o[d][1], o[d][2], o[d][3]);
        mb[32] = m_ref;
        mb[33] = l_run;
        mb[34] = __builtin_bit_cast(float, em);
    }
    __syncthreads();
    if (ks > 0) return;
    const float m1 = mb[32], mm = fmaxf(m_ref, m1);
    const float a0 = __builtin_amdgcn_exp2f(m_ref - mm), a1 = __builtin_amdgcn_exp2f(m1 - mm);
    const float inv = 1.0f / __builtin_fmaf(mb[33], a1, l_run * a0);
    // each half times 2^(em + m - mm) / l, their common exponent last: nothing leaves FP32's range before the result does
    const int e0 = em + (int)fmaxf(m_ref - mm, -1e6f), e1 = __builtin_bit_cast(int, mb[34]) + (int)fmaxf(m1 - mm, -1e6f);
    const int et = max(e0, e1);
    const float f0 = pow2(max(e0 - et, -127)) * inv, f1 = pow2(max(e1 - et, -127)) * inv;
    if (iq < T) {
        float *dst = out + ((long long)b * T + iq) * ldo + (long long)h * kDK + 4 * g;
#pragma unroll
        for (int d = 0; d < 8; ++d) {
            const float4 w = *(const float4 *)(mb + 4 * d);
            auto sum = [&](float x0, float x1) { return __builtin_amdgcn_ldexpf(__builtin_fmaf(x1, f1, x0 * f0), et); };
            *(float4 *)(dst + 16 * d) = make_float4(sum(o[d][0], w.x), sum(o[d][1], w.y), sum(o[d][2], w.z), sum(o[d][3], w.w));
        }
    }
}

int64_t tiled_workspace(int64_t batch, int64_t t, int heads) {
    SplitOperands so;
    return split_layout(&so, nullptr, batch, heads, t);
}

// The largest sequence: 65535 query tiles of a launch.
constexpr int64_t kMaxRows = 65535 * kRows;

}  // namespace

extern "C" int64_t kea_relpos_attention_tiled_workspace(int64_t batch, int64_t t, int heads) {
    if (batch < 1 || t < 1 || heads < 1 || t > kMaxRows) return 0;
    return tiled_workspace(batch, t, heads);
}

extern "C" int kea_relpos_attention_tiled(const float *qkv, int64_t ld, const float *pos, int64_t ldp,
                                          const float *bias_u, const float *bias_v, float *out, int64_t ldo,
                                          int64_t batch, int64_t t, int heads, int head_dim, float scale,
                                          void *workspace, int64_t workspace_bytes, void *stream) {
    if (batch < 0 || t < 1 || heads < 1 || head_dim != kDK || batch > 65535 || heads > 65535 || t > kMaxRows)
        return kea::fail(KEA_EINVAL, "bad sizes (head_dim must be 128)");
    if (batch == 0) return KEA_OK;
    if (!qkv || !pos || !bias_u || !bias_v || !out) return kea::fail(KEA_EINVAL, "null pointer");
    if (ld < 3LL * heads * head_dim || ldp < (int64_t)heads * head_dim || ldo < (int64_t)heads * head_dim)
        return kea::fail(KEA_EINVAL, "leading dimension too small");
    if (((uintptr_t)qkv | (uintptr_t)pos | (uintptr_t)out | (uintptr_t)bias_u | (uintptr_t)bias_v) & 15 ||
        (ld | ldp | ldo) & 3)
        return kea::fail(KEA_EALIGN, "qkv, pos, out and the biases need 16-byte aligned rows");
    const int64_t need = tiled_workspace(batch, t, heads);
    if (!workspace || workspace_bytes < need)
        return kea::fail(KEA_ESPACE, "attention workspace too small: need " + std::to_string(need) + " bytes");
    if ((uintptr_t)workspace & 15) return kea::fail(KEA_EALIGN, "attention workspace must be 16-byte aligned");
    SplitOperands so;
    split_layout(&so, (char *)workspace, batch, heads, t);
    const int64_t kv = batch * heads * so.tiles, blocks = 3 * kv + (int64_t)heads * so.pblocks;
    if (!kea::fits_dispatch(blocks, 256)) return kea::fail(KEA_EINVAL, "too large for one launch: split the batch");
    hipError_t e = hipFuncSetAttribute((const void *)relpos_tiled_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kTiledLds);
    if (e != hipSuccess) return kea::fail((int)e, std::string("LDS attribute refused: ") + hipGetErrorString(e));
    hipLaunchKernelGGL(split_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, qkv, (long long)ld, pos,
                       (long long)ldp, bias_u, bias_v, (int)t, heads, (int)kv, so);
    e = hipGetLastError();
    if (e != hipSuccess) return kea::fail((int)e, std::string("attention split launch failed: ") + hipGetErrorString(e));
    hipLaunchKernelGGL(relpos_tiled_kernel, dim3((unsigned)heads, (unsigned)so.tiles, (unsigned)batch), dim3(kNW * 64),
                       kTiledLds, (hipStream_t)stream, qkv, (long long)ld, pos, (long long)ldp, bias_u, bias_v, out,
                       (long long)ldo, (int)t, heads, scale, so);
    e = hipGetLastError();
    if (e != hipSuccess) return kea::fail((int)e, std::string("attention launch failed: ") + hipGetErrorString(e));
    return KEA_OK;
}
