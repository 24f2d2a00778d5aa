// gdn_batch.hip -- multi-stream decode: up to 64 independent token streams,
// each with its own recurrent and conv state, advanced one token per stream
// per step.  The reference decodes a single stream (README.md:75-77); this
// path keeps its per-stream arithmetic and moves the projections onto the
// matrix cores.
//
// Arithmetic.  Every operator outside the projections is the BF16W_FP32S
// arithmetic of the batch-1 engine (the same device functions): embedding
// import, residual adds and RMSNorms in chunk order, the tiny a/b rows in
// FP32 products, conv + SiLU with the tail shift, beta/decay, the recurrence
// on an FP32 state, the output norm * gate, SwiGLU, FP32 logits and the
// strict-'>' argmax.  The projections take the same BF16 operands (weights
// and activations at their BF16 rounding points, subnormals flushed) but form
// exact products and accumulate them in FP32 on v_mfma_f32_16x16x32_bf16, in
// the matrix cores' order instead of the reference's tree16 + four banks.
// Results therefore agree with the batch-1 engine to rounding, not bit for
// bit; outputs are rounded to BF16 at the same points.
//
// Layout.  A projection W [N][K] is stored as MFMA A-operand tiles (16 rows x
// 32 columns, gdn_tile_bf16; gate/up in k_bgu's 44-row blocks, tile_gu).  The activations of all streams enter as the B
// operand: X [64 streams][K] BF16 in tiles of 32 columns x 16 streams, lane l
// holding stream l % 16 and columns 8 (l / 16) .. + 7.  Stream s of a GEMM
// output is column s of D = W X^T, so streams never mix.
//
// Per layer (8 launches):
//   k_bgemm<QKVG>  q,k,v,g rows; epilogue: BF16 rounding, conv + SiLU with
//                  each stream's tails, gate and sigmoid(gate)
//   k_brecur       the recurrence per (head, stream, 64 columns), state in registers
//   k_bonorm       per (head, stream) output RMSNorm * gate -> X
//   k_bgemm<RAW>   o_proj in 4 K splits -> split sums
//   k_bnorm        h = R(h + R(y)), MLP RMSNorm -> X
//   k_bgu          gate/up, 22 channels per workgroup, SwiGLU -> X (K = 5632)
//   k_bgemm<RAW>   down in 4 K splits -> split sums
//   k_bnorm        h = R(h + R(y)), next attention RMSNorm (or the final norm)
//                  -> X; with the next layer's a/b rows and beta/decay it runs
//                  four workgroups per stream, two heads' rows each
// plus the embedding norm before layer 0, the LM head with a per-workgroup
// argmax, and the per-stream argmax merge.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <type_traits>
#include <vector>

#include "gdn_amd.h"
#include "gdn_device.h"
#include "gdn_internal.h"
#include "gdn_scan.h"

namespace gdn {
namespace bt {

constexpr int kMaxB = GDN_MAX_STREAMS;  // streams = the 64 B-operand columns
static_assert(kMaxB == 64, "four 16-stream groups per MFMA B operand");
constexpr int kRecCols = 64;  // state columns per multi-stream recurrence workgroup
constexpr int kSplitO = 4;              // K splits of o_proj (16 k tiles each)
constexpr int kSplitDown = 4;           // K splits of the down projection (44 k tiles each)
constexpr int kRtO = 2;                 // 16-row tiles per o_proj workgroup
constexpr int kRtDown = 2;              // 16-row tiles per down workgroup
constexpr int kKtH = kH / 32;           // k tiles of a K = 2048 projection
constexpr int kKtI = kI / 32;           // k tiles of the down projection
constexpr size_t kLayerState = (size_t)kNH * kHD * kHD;  // floats per (layer, stream)
constexpr size_t kStreamTails = (size_t)3 * 3 * kH;      // floats per (layer, stream)

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

enum { EPI_RAW = 0, EPI_QKVG = 2, EPI_LM = 4 };

// BF16 bits of a value already at a BF16 rounding point, subnormals flushed
// to a signed zero (the reference's products treat them as zero).
__device__ __forceinline__ uint32_t bf16_daz_bits(float v) {
    const uint32_t b = f2u(v);
    return ((b & 0x7f800000u) == 0u) ? ((b >> 16) & 0x8000u) : (b >> 16);
}

// Offset (BF16 elements) of (stream or token m, column k) in an X tile
// buffer of K columns: blocks of 64 streams (a step has one; a prefill
// segment one per 64 tokens), each [k tile][16-stream group][64 lanes][8].
__device__ __forceinline__ size_t xt_index(int m, int k, int K = kH) {
    const int kt = k >> 5, kk = k & 31, mm = m & 63;
    return (size_t)(m >> 6) * 64 * K +
           (size_t)((((kt * 4 + (mm >> 4)) * 64 + ((kk >> 3) << 4) + (mm & 15)) << 3) + (kk & 7));
}

// Eight consecutive columns k..k+7 (k % 8 == 0) of stream m in a K = kH X
// tile buffer, one 16-byte store.
__device__ __forceinline__ void store_x8(uint16_t *x, int m, int k, const float *v) {
    u32x4 w;
    w.x = bf16_daz_bits(v[0]) | (bf16_daz_bits(v[1]) << 16);
    w.y = bf16_daz_bits(v[2]) | (bf16_daz_bits(v[3]) << 16);
    w.z = bf16_daz_bits(v[4]) | (bf16_daz_bits(v[5]) << 16);
    w.w = bf16_daz_bits(v[6]) | (bf16_daz_bits(v[7]) << 16);
    *reinterpret_cast<u32x4 *>(x + xt_index(m, k)) = w;
}

// ------------------------------------------------------------ the GEMM

struct BEpi {
    int n_streams;
    int n_rows;          // N: row stride of y / logits
    float *y;            // EPI_RAW: [splits][y_rows][N]
    int y_rows;          // rows of one split's plane (64 in a step)
    float *qkv;          // EPI_QKVG: [64][3][kH] after conv + SiLU
    float *gate;         // [64][kH] R(g)
    float *sgate;        // [64][kH] sigmoid(R(g))
    uint16_t *tails;     // this layer's [n_streams][3][3][kH], BF16 bits (the values are BF16)
    const float *conv_w; // [3][kH][4]
    float *logits;       // EPI_LM: [64][N]
    float *part_val;     // [gridDim.x][64]
    int *part_idx;
};

// D[rows][64 streams] = W[rows][K] X^T for 16 * RT rows per workgroup and
// KT / S k tiles (split S of the K range: grid (N / (16 RT), S)).  The NW
// waves split the workgroup's k tiles (wave w takes tiles w, w + NW, ...),
// keep up to four tiles of operands in flight, and the per-wave sums are
// added in wave order through LDS; the epilogue then runs on the reduced
// tile.  Split partial sums (EPI_RAW with S > 1) are added in split order by
// the consumer.  With EPI_RAW the grid's z dimension is the 64-token block of
// a prefill segment.  G: the 16-stream groups that are formed (four, or as
// many as hold the step's streams); a group's sums do not depend on the
// others.
template <int RT, int KT, int NW, int S, int EPI, int G = 4>
__global__ __launch_bounds__(NW * 64) void k_bgemm(const u32x4 *__restrict__ W, const u32x4 *__restrict__ X,
                                                   BEpi ep) {
    constexpr int KTS = KT / S, KTW = KTS / NW, GT = NW * 64;
    static_assert(KT % S == 0 && KTS % NW == 0, "whole k tiles per wave");
    static_assert(S == 1 || EPI == EPI_RAW, "split sums leave the GEMM unrounded");
    constexpr int D = KTW < 4 ? KTW : 4;
    constexpr size_t WSTEP = (size_t)NW * RT * 64, XSTEP = (size_t)NW * 4 * 64;
    __shared__ f32x4 red[NW * RT * G * 64];
    __shared__ float lm_v[RT * 4][16 * G];
    __shared__ int lm_i[RT * 4][16 * G];
    __shared__ uint64_t exp2_lds[EPI == EPI_QKVG ? 32 : 1];  // expf's table for the epilogue
    __shared__ f32x4 conv_lds[EPI == EPI_QKVG ? RT * 16 : 1];  // the conv taps of the workgroup's channels
    if constexpr (EPI == EPI_QKVG) fill_exp2_lds_imm(exp2_lds);
    // QKVG: consecutive row blocks on one XCD (workgroups are dealt to the 8
    // XCDs round-robin), so the two 64-byte halves of a conv-tail line are
    // fetched into one XCD's L2 once instead of into two
    const int rb = (EPI == EPI_QKVG && (gridDim.x & 7) == 0)
                       ? (int)((blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3))
                       : (int)blockIdx.x;
    const int t = threadIdx.x, w = t >> 6, l = t & 63, sp = blockIdx.y;
    const int kt0 = sp * KTS + w;
    const u32x4 *wp = W + ((size_t)rb * KT + kt0) * (RT * 64) + l;
    const int zb = EPI == EPI_RAW ? (int)blockIdx.z : 0;
    const u32x4 *xp = X + ((size_t)zb * KT + kt0) * (4 * 64) + l;

    // QKVG epilogue tasks: four consecutive channels of one stream per
    // thread and pass (4-channel group g of the workgroup's RT * 4, stream
    // q / (RT * 4)), so tails, q/k/v and gate move as 8- and 16-byte
    // accesses.  Each stream's conv tails (three taps of BF16 bits per
    // channel) and the workgroup's taps (into LDS) are read ahead of the
    // weight stream.
    constexpr int CG = RT * 4;
    constexpr int QE = (EPI == EPI_QKVG) ? (16 * G * CG + GT - 1) / GT : 1;
    const int which = (rb * 16 * RT) / kH, c0 = rb * 16 * RT - which * kH;  // q, k, v, g section
    uint2 qtl[QE][3];
    if constexpr (EPI == EPI_QKVG) {
        if (which < 3 && t < RT * 16)
            conv_lds[t] = *reinterpret_cast<const f32x4 *>(ep.conv_w + ((size_t)which * kH + c0 + t) * 4);
#pragma unroll
        for (int j = 0; j < QE; ++j) {
            const int q = t + GT * j, m = q / CG, c = c0 + 4 * (q % CG);
#pragma unroll
            for (int k = 0; k < 3; ++k) qtl[j][k] = make_uint2(0u, 0u);
            if (which < 3 && m < ep.n_streams) {
                const uint16_t *tl = ep.tails + ((size_t)m * 3 + which) * 3 * kH + c;
#pragma unroll
                for (int k = 0; k < 3; ++k) qtl[j][k] = *reinterpret_cast<const uint2 *>(tl + k * kH);
            }
        }
    }

    f32x4 acc[RT][G];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int g = 0; g < G; ++g) acc[r][g] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    u32x4 a[D][RT], b[D][G];
#pragma unroll
    for (int i = 0; i < D; ++i) {
#pragma unroll
        for (int r = 0; r < RT; ++r) a[i][r] = wp[i * WSTEP + r * 64];
#pragma unroll
        for (int g = 0; g < G; ++g) b[i][g] = xp[i * XSTEP + g * 64];
    }
    // the scheduler keeps every prefetch where it is issued: D k tiles stay
    // in flight instead of one
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < KTW; ++i) {
        const int s = i % D;
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int g = 0; g < G; ++g)
                acc[r][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[s][r]),
                                                                    __builtin_bit_cast(bf16x8, b[s][g]),
                                                                    acc[r][g], 0, 0, 0);
        if (i + D < KTW) {
#pragma unroll
            for (int r = 0; r < RT; ++r) a[s][r] = wp[(i + D) * WSTEP + r * 64];
#pragma unroll
            for (int g = 0; g < G; ++g) b[s][g] = xp[(i + D) * XSTEP + g * 64];
        }
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int g = 0; g < G; ++g) red[((w * RT + r) * G + g) * 64 + l] = acc[r][g];
    __syncthreads();

    // Task (rt, nq, m): rows rt * 16 + nq * 4 + 0..3 of stream m, held by lane
    // nq * 16 + m % 16 of stream group m / 16 in every wave's D tile.  Every
    // epilogue takes whole tasks (the four rows as one f32x4).
    auto red_index = [&](int rt, int nq, int m) { return (rt * G + (m >> 4)) * 64 + nq * 16 + (m & 15); };
    auto reduced = [&](int rt, int nq, int m) {
        const int idx = red_index(rt, nq, m);
        f32x4 v = red[idx];
#pragma unroll
        for (int ww = 1; ww < NW; ++ww) v = v + red[ww * RT * G * 64 + idx];
        return v;
    };
    if constexpr (EPI == EPI_RAW || EPI == EPI_LM) {
#pragma unroll
        for (int q = t; q < RT * 4 * 16 * G; q += GT) {
            const int m = q % (16 * G), nq = (q / (16 * G)) & 3, rt = q / (64 * G);
            const f32x4 v = reduced(rt, nq, m);
            const int row = rb * 16 * RT + rt * 16 + nq * 4;
            if constexpr (EPI == EPI_LM) {
                *reinterpret_cast<f32x4 *>(ep.logits + (size_t)m * ep.n_rows + row) = v;
                float best = -3.402823466e38f;
                int idx = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (v[e] > best) {
                        best = v[e];
                        idx = row + e;
                    }
                lm_v[rt * 4 + nq][m] = best;
                lm_i[rt * 4 + nq][m] = idx;
            } else {
                *reinterpret_cast<f32x4 *>(ep.y + ((size_t)sp * ep.y_rows + zb * 64 + m) * ep.n_rows + row) = v;
            }
        }
    } else if constexpr (EPI == EPI_QKVG) {
#pragma unroll
        for (int j = 0; j < QE; ++j) {
            const int q = t + GT * j, g = q % CG, m = q / CG, c = c0 + 4 * g;
            if (m >= ep.n_streams) continue;
            // channels c..c+3 are rows 4 (g % 4) .. of row tile g / 4
            const f32x4 v = reduced(g >> 2, g & 3, m);
            const float raw[4] = {rne_bf16(v.x), rne_bf16(v.y), rne_bf16(v.z), rne_bf16(v.w)};
            if (which < 3) {
                // gdn_depthwise_conv_silu_head_kind, gdn_model.cpp:1543-1667
                uint16_t *tl = ep.tails + ((size_t)m * 3 + which) * 3 * kH + c;
                const uint32_t tw[3][2] = {{qtl[j][0].x, qtl[j][0].y}, {qtl[j][1].x, qtl[j][1].y},
                                           {qtl[j][2].x, qtl[j][2].y}};
                float o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int sh = 16 * (e & 1);
                    const f32x4 cw = conv_lds[4 * g + e];
                    const float t0 = bf16_bits_to_f32((uint16_t)(tw[0][e >> 1] >> sh));
                    const float t1 = bf16_bits_to_f32((uint16_t)(tw[1][e >> 1] >> sh));
                    const float t2 = bf16_bits_to_f32((uint16_t)(tw[2][e >> 1] >> sh));
                    const float sum = t0 * cw.x + t1 * cw.y + t2 * cw.z + raw[e] * cw.w;
                    o[e] = rne_bf16(silu_ref(sum, Exp2Lds{exp2_lds}));
                }
                // the tails shift by one tap: (t1, t2, raw)
                *reinterpret_cast<uint2 *>(tl) = qtl[j][1];
                *reinterpret_cast<uint2 *>(tl + kH) = qtl[j][2];
                *reinterpret_cast<uint2 *>(tl + 2 * kH) =
                    make_uint2((uint32_t)bf16_hi(raw[0]) | ((uint32_t)bf16_hi(raw[1]) << 16),
                               (uint32_t)bf16_hi(raw[2]) | ((uint32_t)bf16_hi(raw[3]) << 16));
                *reinterpret_cast<f32x4 *>(ep.qkv + ((size_t)m * 3 + which) * kH + c) =
                    (f32x4){o[0], o[1], o[2], o[3]};
            } else {
                *reinterpret_cast<f32x4 *>(ep.gate + (size_t)m * kH + c) = (f32x4){raw[0], raw[1], raw[2], raw[3]};
                *reinterpret_cast<f32x4 *>(ep.sgate + (size_t)m * kH + c) =
                    (f32x4){sigmoid_ref(raw[0], Exp2Lds{exp2_lds}), sigmoid_ref(raw[1], Exp2Lds{exp2_lds}),
                            sigmoid_ref(raw[2], Exp2Lds{exp2_lds}), sigmoid_ref(raw[3], Exp2Lds{exp2_lds})};
            }
        }
    }
    if constexpr (EPI == EPI_LM) {
        __syncthreads();
        if (t < 16 * G) {
            // row quads in index order: strict '>' keeps the lowest index of
            // equal maxima (NaN never wins)
            float best = lm_v[0][t];
            int idx = lm_i[0][t];
#pragma unroll
            for (int q = 1; q < RT * 4; ++q)
                if (lm_v[q][t] > best) {
                    best = lm_v[q][t];
                    idx = lm_i[q][t];
                }
            ep.part_val[(size_t)rb * 64 + t] = best;
            ep.part_idx[(size_t)rb * 64 + t] = idx;
        }
    }
}

// ------------------------------------------------------------ gate/up
//
// 5632 channels over 256 workgroups, one per CU: workgroup b owns channels
// 22 b .. 22 b + 21, i.e. 44 rows in three row tiles: the gate rows of its
// first 16 channels, their up rows, and a 12-row tile with the gate then the
// up rows of the last 6 (rows 12..15 of that tile stay zero).  Whole 16-row
// pairs (32 rows per workgroup) give 352 workgroups, i.e. two on some CUs,
// and every workgroup reads all 64 streams' activations beside its rows.
constexpr int kGuCh = 22;                // channels per gate/up workgroup
constexpr int kGuWgs = kI / kGuCh;       // 256
constexpr int kGuTail2 = 2 * (kGuCh - 16);     // rows of the third tile (12)
constexpr int kGuTileU4 = 128 + 4 * kGuTail2;  // 16-byte entries per k tile
constexpr int kGuWaves = 4;                    // waves per gate/up workgroup
static_assert(kGuWgs * kGuCh == kI && kGuCh > 16 && kGuCh <= 24 && (kGuCh % 2) == 0, "gate/up split");

// One k tile of the layout: tile 0 lane l = (row l % 16, columns 8 (l / 16)..),
// tile 1 likewise, the 12-row tile's entry (quarter kq, row r) at 128 + kq * 12 + r.
// The NW waves split the 64 k tiles as k_bgemm's do (wave w: w, w + NW, ...)
// and the per-wave sums are added in wave order, so each channel's sums are
// those of k_bgemm's 16-channel pairing with the same NW.
template <int NW, int G = 4>
__global__ __launch_bounds__(NW * 64) void k_bgu(const u32x4 *__restrict__ W, const u32x4 *__restrict__ X,
                                                 uint16_t *__restrict__ x_next, int n_streams) {
    // grid y: the 64-token block of a prefill segment of n_streams tokens
    constexpr int RT = 3, KT = kKtH, KTW = KT / NW, GT = NW * 64;
    static_assert(KT % NW == 0, "whole k tiles per wave");
    constexpr int D = KTW < 4 ? KTW : 4;
    constexpr size_t WSTEP = (size_t)NW * kGuTileU4, XSTEP = (size_t)NW * 4 * 64;
    __shared__ f32x4 red[NW * RT * G * 64];
    __shared__ uint64_t exp2_lds[32];  // expf's table for the SwiGLU epilogue
    const int t = threadIdx.x, w = t >> 6, l = t & 63, rb = blockIdx.x;
    fill_exp2_lds_imm(exp2_lds);
    // the 12-row tile: lanes of rows 12..15 read entry 0 (in bounds) and
    // zero it
    const bool p2 = (l & 15) < kGuTail2;
    const int o2 = 128 + (p2 ? (l >> 4) * kGuTail2 + (l & 15) : 0);
    const u32x4 *wp = W + ((size_t)rb * KT + w) * kGuTileU4;
    const int mb = (int)blockIdx.y * kMaxB;
    const u32x4 *xp = X + ((size_t)blockIdx.y * KT + w) * (4 * 64) + l;
    const u32x4 zero = {0u, 0u, 0u, 0u};

    f32x4 acc[RT][G];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int g = 0; g < G; ++g) acc[r][g] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    u32x4 a[D][RT], b[D][G];
#pragma unroll
    for (int i = 0; i < D; ++i) {
        a[i][0] = wp[i * WSTEP + l];
        a[i][1] = wp[i * WSTEP + 64 + l];
        a[i][2] = wp[i * WSTEP + o2];
#pragma unroll
        for (int g = 0; g < G; ++g) b[i][g] = xp[i * XSTEP + g * 64];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < KTW; ++i) {
        const int s = i % D;
        if (!p2) a[s][2] = zero;
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int g = 0; g < G; ++g)
                acc[r][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[s][r]),
                                                                    __builtin_bit_cast(bf16x8, b[s][g]),
                                                                    acc[r][g], 0, 0, 0);
        if (i + D < KTW) {
            a[s][0] = wp[(i + D) * WSTEP + l];
            a[s][1] = wp[(i + D) * WSTEP + 64 + l];
            a[s][2] = wp[(i + D) * WSTEP + o2];
#pragma unroll
            for (int g = 0; g < G; ++g) b[s][g] = xp[(i + D) * XSTEP + g * 64];
        }
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int g = 0; g < G; ++g) red[((w * RT + r) * G + g) * 64 + l] = acc[r][g];
    __syncthreads();

    // rows 4 nq .. 4 nq + 3 of tile r for stream m: lane nq * 16 + m % 16 of
    // stream group m / 16 in every wave's tile, the waves added in order
    auto val4 = [&](int r, int nq, int m) {
        const int idx = (r * G + (m >> 4)) * 64 + nq * 16 + (m & 15);
        f32x4 v = red[idx];
#pragma unroll
        for (int ww = 1; ww < NW; ++ww) v = v + red[ww * RT * G * 64 + idx];
        return v;
    };
    // gemv32_store SwiGLU branch, gdn_model.cpp:4751-4767, for one channel
    // (its gate g and up u as the GEMM left them)
    auto swiglu = [&](float g, float u) {
        return bf16_daz_bits(rne_bf16(silu_ref(rne_bf16(g), Exp2Lds{exp2_lds}) * rne_bf16(u)));
    };
    static_assert(kGuCh == 22 && GT == 256, "16 + 6 channels; 256 + 192 tasks over four waves");
    // channels 4 nq .. 4 nq + 3 (gate rows of tile 0, up rows of tile 1):
    // task (stream m, nq), thread 4 m + nq
    if (t < 64 * G) {
        const int m = t >> 2, nq = t & 3;
        if (mb + m < n_streams) {
            const f32x4 g = val4(0, nq, m), u = val4(1, nq, m);
            const uint32_t lo = swiglu(g.x, u.x) | (swiglu(g.y, u.y) << 16);
            const uint32_t hi = swiglu(g.z, u.z) | (swiglu(g.w, u.w) << 16);
            const int k0 = rb * kGuCh + 4 * nq;  // even: pairs never straddle an 8-column group
            if ((k0 & 3) == 0) {
                *reinterpret_cast<uint2 *>(x_next + xt_index(mb + m, k0, kI)) = make_uint2(lo, hi);
            } else {
                *reinterpret_cast<uint32_t *>(x_next + xt_index(mb + m, k0, kI)) = lo;
                *reinterpret_cast<uint32_t *>(x_next + xt_index(mb + m, k0 + 2, kI)) = hi;
            }
        }
    }
    // channels 16 + 2 p, 17 + 2 p (gate rows 2 p, 2 p + 1 and up rows
    // 2 p + 6, 2 p + 7 of tile 2): task (stream m, p), thread 64 + 3 m + p
    if (t >= 64 && t < 64 + 48 * G) {
        const int q = t - 64, m = q / 3, p = q - 3 * m;
        if (mb + m < n_streams) {
            const int rg = 2 * p, ru = 2 * p + 6;
            const f32x4 gv = val4(2, rg >> 2, m), uv = val4(2, ru >> 2, m);
            const float g0 = (rg & 3) ? gv.z : gv.x, g1 = (rg & 3) ? gv.w : gv.y;
            const float u0 = (ru & 3) ? uv.z : uv.x, u1 = (ru & 3) ? uv.w : uv.y;
            *reinterpret_cast<uint32_t *>(x_next + xt_index(mb + m, rb * kGuCh + 16 + 2 * p, kI)) =
                swiglu(g0, u0) | (swiglu(g1, u1) << 16);
        }
    }
}

// Per-stream merge of the LM head's per-workgroup results (in index order):
// strict '>' within a thread's increasing blocks, then larger value / lower
// index across threads -- the reference's first-maximum scan.
__global__ __launch_bounds__(kT) void k_bargmax(const float *__restrict__ part_val,
                                                const int *__restrict__ part_idx, int n_blocks,
                                                int *__restrict__ tok_out) {
    __shared__ float bv[4];
    __shared__ int bi[4];
    const int m = blockIdx.x, t = threadIdx.x;
    float best = -3.402823466e38f;
    int idx = 0;
    for (int i = t; i < n_blocks; i += kT) {
        const float v = part_val[(size_t)i * 64 + m];
        if (v > best) {
            best = v;
            idx = part_idx[(size_t)i * 64 + m];
        }
    }
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
        const float ov = __shfl_xor(best, s);
        const int oi = __shfl_xor(idx, s);
        if (ov > best || (ov == best && oi < idx)) {
            best = ov;
            idx = oi;
        }
    }
    if ((t & 63) == 0) {
        bv[t >> 6] = best;
        bi[t >> 6] = idx;
    }
    __syncthreads();
    if (t == 0) {
        for (int i = 1; i < 4; ++i)
            if (bv[i] > best || (bv[i] == best && bi[i] < idx)) {
                best = bv[i];
                idx = bi[i];
            }
        tok_out[m] = idx;
    }
}

// ------------------------------------------------------ per-stream kernels

struct BNorm {
    const float *h_in;     // [64][kH] residual stream
    float *h_out;          // h_in, or (AB, several workgroups per stream) the other residual buffer
    const float *y;        // [splits][y_rows][kH] partial sums: h = R(h + R(sum)) first
    int y_rows;
    const uint16_t *emb;   // embedding rows (BF16): h = R(emb[tok[m]]) (EMBED)
    const int *tok;
    const float *w;        // norm weight [kH]
    uint16_t *x_out;       // X tiles of the next projection
    float *xn_out;         // optional [64][kH] copy of the normalized vector
    const float *ab_w;     // a_proj (8 x kH) then b_proj (8 x kH) (AB)
    const float *a_log;
    const float *dt_bias;
    float *bd;             // [64][16]: beta, decay per head
    float eps;
};

// beta and decay (head_scalars) of TOK tokens x HEADS heads of a workgroup:
// wave 0's threads form the betas, wave 1's the decays, so the two serial
// evaluations of the reference's transcendentals run side by side.  The
// heads' parameters are requested at the kernel's start (read), where they
// were loaded behind the a/b chains.
struct HeadParams {
    float a_log = 0.0f, dt_bias = 0.0f;
    template <int HEADS>
    __device__ __forceinline__ void read(int t, int h0, const float *__restrict__ al, const float *__restrict__ dt) {
        if ((t >> 6) == 1) {
            const int hd = h0 + (t & 63) % HEADS;
            a_log = al[hd];
            dt_bias = dt[hd];
        }
    }
    // abv[token][row]: the a rows, then the b rows; bd[token][16]
    template <int HEADS, int TOK>
    __device__ __forceinline__ void write(int t, int h0, int n, const float *abv, int rows, float *__restrict__ bd,
                                          const Exp2Lds &tab) const {
        static_assert(HEADS * TOK <= 64, "one wave");
        const int i = t & 63, m = i / HEADS, hh = i % HEADS;
        if (i >= HEADS * TOK || m >= n) return;
        float *out = bd + m * 16 + 2 * (h0 + hh);
        if ((t >> 6) == 0)
            out[0] = sigmoid_ref(abv[m * rows + HEADS + hh], tab);
        else if ((t >> 6) == 1)
            out[1] = exp_ref(-exp_ref(a_log, tab) * softplus_ref(abv[m * rows + hh] + dt_bias, tab), tab);
    }
};
constexpr int kAbSplit = 4;
constexpr int kAbHeads = kNH / kAbSplit;  // heads per a/b workgroup
static_assert(kNH % kAbSplit == 0 && (2 * kAbHeads * kH) % (4 * kT) == 0 && 2 * kAbHeads <= kT,
              "whole heads per a/b workgroup, whole 16-byte row pieces per thread");
// Per stream: the residual add (or embedding import), the RMSNorm in chunk
// order (gdn_rmsnorm_rows_bf16 / gdn_residual_rmsnorm_bf16,
// gdn_model.cpp:1394-1474, :3351-3450) and, before an attention block, the
// tiny a/b rows and beta/decay (gdn_gemv_tiny_ab :1501-1536, :2461-2465).
// Thread t holds elements 8t..8t+7; a 16-element chunk is the sequential sum
// of thread 2c's eight squares continued by thread 2c + 1.  SPLITS partial
// sums of the preceding projection are added in split order (1: its rounded
// sums as BF16 bits; 0: no residual add; EMBED: the embedding row instead).
// Without AB one workgroup per stream updates the residual in place.  With AB, grid (streams, kAbSplit):
// workgroup j repeats the norm and runs the a/b rows of heads
// kNH / kAbSplit * j .. (a 32 KB slice of the 128 KB of rows, requested
// before the norm's first wait on memory); workgroup 0 alone writes the
// residual, to h_out != h_in, and the X tiles.
template <int SPLITS, bool EMBED, bool AB>
__global__ __launch_bounds__(kT) void k_bnorm(BNorm p) {
    constexpr int ABR = 2 * kAbHeads;  // a/b rows per workgroup: a rows, then b rows
    __shared__ __attribute__((aligned(16))) float xs[kH];
    __shared__ __attribute__((aligned(16))) float cs[kH / 16];
    __shared__ __attribute__((aligned(16))) float tab[ABR][64][2];
    __shared__ float abv[ABR];
    __shared__ float scale_s;
    __shared__ uint64_t exp2_lds[AB ? 32 : 1];  // expf's table for beta and decay
    const int m = blockIdx.x, t = threadIdx.x, e0 = 8 * t;
    const int j = AB ? (int)blockIdx.y : 0;
    const bool writer = j == 0;
    HeadParams hp;
    if constexpr (AB) {
        fill_exp2_lds_imm(exp2_lds);
        hp.read<kAbHeads>(t, kAbHeads * j, p.a_log, p.dt_bias);
    }
    const f32x4 *w4 = reinterpret_cast<const f32x4 *>(p.w + e0);
    const f32x4 wa = w4[0], wb = w4[1];
    float hv[8];
    if constexpr (EMBED) {
        const u32x4 raw = *reinterpret_cast<const u32x4 *>(p.emb + (size_t)p.tok[m] * kH + e0);
        const uint32_t wv[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            hv[2 * j] = rne_bf16(u2f(wv[j] << 16));
            hv[2 * j + 1] = rne_bf16(u2f(wv[j] & 0xffff0000u));
        }
    } else {
        const f32x4 *h4 = reinterpret_cast<const f32x4 *>(p.h_in + (size_t)m * kH + e0);
        const f32x4 a0 = h4[0], a1 = h4[1];
        hv[0] = a0.x; hv[1] = a0.y; hv[2] = a0.z; hv[3] = a0.w;
        hv[4] = a1.x; hv[5] = a1.y; hv[6] = a1.z; hv[7] = a1.w;
        if constexpr (SPLITS == 1) {
            // the projection's sums, rounded by its kernel
            const u32x4 y = *reinterpret_cast<const u32x4 *>(reinterpret_cast<const uint16_t *>(p.y) +
                                                             (size_t)m * kH + e0);
            const uint32_t yw[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                hv[2 * i] = rne_bf16(hv[2 * i] + u2f(yw[i] << 16));
                hv[2 * i + 1] = rne_bf16(hv[2 * i + 1] + u2f(yw[i] & 0xffff0000u));
            }
        } else if constexpr (SPLITS > 0) {
            // the projection's split sums in split order, then its rounding
            f32x4 yp[SPLITS][2];
#pragma unroll
            for (int sp = 0; sp < SPLITS; ++sp) {
                const f32x4 *y4 = reinterpret_cast<const f32x4 *>(p.y + ((size_t)sp * p.y_rows + m) * kH + e0);
                yp[sp][0] = y4[0];
                yp[sp][1] = y4[1];
            }
            f32x4 y0 = yp[0][0], y1 = yp[0][1];
#pragma unroll
            for (int sp = 1; sp < SPLITS; ++sp) {
                y0 = y0 + yp[sp][0];
                y1 = y1 + yp[sp][1];
            }
            const float yv[8] = {y0.x, y0.y, y0.z, y0.w, y1.x, y1.y, y1.z, y1.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) hv[e] = rne_bf16(hv[e] + rne_bf16(yv[e]));
        }
    }
    // the a/b rows are requested behind the operands of the norm (loads
    // return in order)
    // local row r: a row of head kAbHeads j + r (r < kAbHeads), else the b
    // row of head kAbHeads j + r - kAbHeads
    auto ab_row = [&](int r) { return r < kAbHeads ? kAbHeads * j + r : kNH + kAbHeads * j + r - kAbHeads; };
    constexpr int ABN = AB ? ABR * kH / (4 * kT) : 1;
    f32x4 wq[ABN];
    if constexpr (AB) {
#pragma unroll
        for (int i = 0; i < ABN; ++i) {
            const int q = t + kT * i, grp = q >> 3, sub = q & 7;
            wq[i] = *reinterpret_cast<const f32x4 *>(p.ab_w + (size_t)ab_row(grp >> 6) * kH + 32 * (grp & 63) +
                                                     4 * sub);
        }
    }
    if ((EMBED || SPLITS > 0) && writer) {
        f32x4 *d = reinterpret_cast<f32x4 *>(p.h_out + (size_t)m * kH + e0);
        d[0] = (f32x4){hv[0], hv[1], hv[2], hv[3]};
        d[1] = (f32x4){hv[4], hv[5], hv[6], hv[7]};
    }
    // chunk sums: the even thread's partial continues in the odd thread
    float part = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) part += hv[e] * hv[e];
    const float lead = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(part), 0xB1, 0xf, 0xf, false));
    if (t & 1) {
        float s = lead;
#pragma unroll
        for (int e = 0; e < 8; ++e) s += hv[e] * hv[e];
        cs[t >> 1] = s;
    }
    __syncthreads();
    if (t == 0) {
        // every chunk sum read ahead of the sequential adds
        float v[kH / 16];
#pragma unroll
        for (int c = 0; c < kH / 64; ++c) {
            const f32x4 q = reinterpret_cast<const f32x4 *>(cs)[c];
            v[4 * c] = q.x;
            v[4 * c + 1] = q.y;
            v[4 * c + 2] = q.z;
            v[4 * c + 3] = q.w;
        }
        float sum = 0.0f;
#pragma unroll
        for (int c = 0; c < kH / 16; ++c) sum += v[c];
        scale_s = 1.0f / __builtin_sqrtf(sum / (float)kH + p.eps);
    }
    __syncthreads();
    const float sc = scale_s;
    const float wv[8] = {wa.x, wa.y, wa.z, wa.w, wb.x, wb.y, wb.z, wb.w};
    float xv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) xv[e] = rne_bf16(hv[e] * sc * wv[e]);
    if (writer) store_x8(p.x_out, m, e0, xv);
    if (p.xn_out && writer) {
        f32x4 *d = reinterpret_cast<f32x4 *>(p.xn_out + (size_t)m * kH + e0);
        d[0] = (f32x4){xv[0], xv[1], xv[2], xv[3]};
        d[1] = (f32x4){xv[4], xv[5], xv[6], xv[7]};
    }
    if constexpr (AB) {
        {
            f32x4 *d = reinterpret_cast<f32x4 *>(xs + e0);
            d[0] = (f32x4){xv[0], xv[1], xv[2], xv[3]};
            d[1] = (f32x4){xv[4], xv[5], xv[6], xv[7]};
        }
        __syncthreads();
        // Eight lanes per (local row, 32-column beat), four products each:
        // lanes 0-3 form tree16 of the lower half, lanes 4-7 of the upper
        // (pairs, then lane pairs, then lane quads), so a wave's loads cover
        // eight consecutive beats of one row.
#pragma unroll
        for (int i = 0; i < ABN; ++i) {
            const int q = t + kT * i, grp = q >> 3, sub = q & 7;
            const f32x4 xq = *reinterpret_cast<const f32x4 *>(xs + 32 * (grp & 63) + 4 * sub);
            const f32x4 w = wq[i];
            float s = (xq.x * w.x + xq.y * w.y) + (xq.z * w.z + xq.w * w.w);
            s = quad_sum(s);
            if ((sub & 3) == 0) tab[grp >> 6][grp & 63][sub >> 2] = s;
        }
        __syncthreads();
        if (t < ABR) {
            float v[128];
#pragma unroll
            for (int i = 0; i < 32; ++i) {
                const f32x4 q = reinterpret_cast<const f32x4 *>(&tab[t][0][0])[i];
                v[4 * i] = q.x;
                v[4 * i + 1] = q.y;
                v[4 * i + 2] = q.z;
                v[4 * i + 3] = q.w;
            }
            float acc = 0.0f;
#pragma unroll
            for (int bt = 0; bt < 64; ++bt) acc = (acc + v[2 * bt]) + v[2 * bt + 1];
            abv[t] = rne_bf16(acc);
        }
        __syncthreads();
        hp.write<kAbHeads, 1>(t, kAbHeads * j, 1, abv, ABR, p.bd + m * 16, Exp2Lds{exp2_lds});
    }
}

// The a/b rows and beta/decay of kPabTok tokens per workgroup, from their
// normalised inputs (the prefill's split of k_bnorm's AB part, whose
// workgroups each re-read their 32 KB of rows): grid (kAbSplit, ceil(n /
// kPabTok)).  Workgroup j loads its four rows once.  Per token the thread
// tasks, products, quad sums, the 64-beat chains and the head scalars are
// k_bnorm's, so every value is the step's.
constexpr int kPabTok = 16;
constexpr int kPabRow = 128 + 4;
__global__ __launch_bounds__(kT) void k_pab(const float *__restrict__ xn, int n, const float *__restrict__ ab_w,
                                            const float *__restrict__ a_log, const float *__restrict__ dt_bias,
                                            float *__restrict__ bd) {
    constexpr int ABR = 2 * kAbHeads, ABN = ABR * kH / (4 * kT);
    static_assert(kPabTok * ABR <= kT, "one chain thread per (token, row)");
    // a row's 128 sums 132 apart: the chains' 64 lanes read 16 bytes of a row
    // each, all from the same four banks if the rows were 128 apart (25.0 ->
    // 24.0 us at 4096 tokens, 11.0 -> 10.3 at 70)
    __shared__ __attribute__((aligned(16))) float tab[kPabTok][ABR][kPabRow];
    __shared__ float abv[kPabTok][ABR];
    __shared__ uint64_t exp2_lds[32];
    const int j = blockIdx.x, m0 = (int)blockIdx.y * kPabTok, t = threadIdx.x;
    fill_exp2_lds_imm(exp2_lds);
    HeadParams hp;
    hp.read<kAbHeads>(t, kAbHeads * j, a_log, dt_bias);
    // local row r: the a row of head kAbHeads j + r (r < kAbHeads), else the
    // b row of head kAbHeads j + r - kAbHeads
    auto ab_row = [&](int r) { return r < kAbHeads ? kAbHeads * j + r : kNH + kAbHeads * j + r - kAbHeads; };
    f32x4 wq[ABN];
#pragma unroll
    for (int i = 0; i < ABN; ++i) {
        const int q = t + kT * i, grp = q >> 3, sub = q & 7;
        wq[i] = *reinterpret_cast<const f32x4 *>(ab_w + (size_t)ab_row(grp >> 6) * kH + 32 * (grp & 63) + 4 * sub);
    }
    // PG tokens' inputs requested together (a token past the segment's end
    // re-reads its last one, unused), then their products
    constexpr int PG = 4;
    static_assert(kPabTok % PG == 0, "whole token groups");
    for (int mg = 0; mg < kPabTok && m0 + mg < n; mg += PG) {
        f32x4 xq[PG][ABN];
#pragma unroll
        for (int g = 0; g < PG; ++g) {
            const int m = m0 + mg + g < n ? m0 + mg + g : n - 1;
            const float *x = xn + (size_t)m * kH;
#pragma unroll
            for (int i = 0; i < ABN; ++i) {
                const int q = t + kT * i, grp = q >> 3, sub = q & 7;
                xq[g][i] = *reinterpret_cast<const f32x4 *>(x + 32 * (grp & 63) + 4 * sub);
            }
        }
#pragma unroll
        for (int g = 0; g < PG; ++g) {
#pragma unroll
            for (int i = 0; i < ABN; ++i) {
                const int q = t + kT * i, grp = q >> 3, sub = q & 7;
                const f32x4 w = wq[i], x = xq[g][i];
                float s = (x.x * w.x + x.y * w.y) + (x.z * w.z + x.w * w.w);
                s = quad_sum(s);
                if ((sub & 3) == 0) tab[mg + g][grp >> 6][2 * (grp & 63) + (sub >> 2)] = s;
            }
        }
    }
    __syncthreads();
    if (t < kPabTok * ABR) {
        const int mt = t / ABR, r = t % ABR;
        if (m0 + mt < n) {
            float v[128];
#pragma unroll
            for (int i = 0; i < 32; ++i) {
                const f32x4 q = reinterpret_cast<const f32x4 *>(tab[mt][r])[i];
                v[4 * i] = q.x;
                v[4 * i + 1] = q.y;
                v[4 * i + 2] = q.z;
                v[4 * i + 3] = q.w;
            }
            float acc = 0.0f;
#pragma unroll
            for (int bt = 0; bt < 64; ++bt) acc = (acc + v[2 * bt]) + v[2 * bt + 1];
            abv[mt][r] = rne_bf16(acc);
        }
    }
    __syncthreads();
    hp.write<kAbHeads, kPabTok>(t, kAbHeads * j, n - m0, &abv[0][0], ABR, bd + m0 * 16, Exp2Lds{exp2_lds});
}

// Per (head, stream): the output RMSNorm times the gate and sigmoid(gate)
// (gdn_output_norm_and_gate, gdn_model.cpp:3226-3349) into X tiles, for
// streams (or prefill tokens) PT y .. PT y + PT - 1 of n: every input of
// the workgroup's PT streams is requested at its start (a stream past n
// re-reads stream n - 1, unused), so they share one memory latency.  RAW: gate
// is the g section of the projection's rounded sums ([token][4 kH] BF16 bits)
// and the sigmoid is formed here: 4 bytes less to read a value, and 8 less
// for the conv kernel to write.
template <int PT, bool RAW>
__global__ __launch_bounds__(kT) void k_bonorm(const float *__restrict__ attn, const void *__restrict__ gate,
                                               const float *__restrict__ sgate, const float *__restrict__ w,
                                               float eps, uint16_t *__restrict__ x_out, int n) {
    static_assert(PT * (kHD / 8) <= kT && kT == kHD, "a thread per channel; one X store task per thread");
    __shared__ float as[PT][kHD];
    __shared__ float cs[PT][kHD / 16];
    __shared__ float xs[PT][kHD];
    __shared__ float scale_s[PT];
    __shared__ uint64_t exp2_lds[RAW ? 32 : 1];  // expf's table for the sigmoid
    if constexpr (RAW) fill_exp2_lds_imm(exp2_lds);
    const int h = blockIdx.x, m0 = (int)blockIdx.y * PT, t = threadIdx.x, c = h * kHD + t;
    float a[PT], gt[PT], sg[PT];
#pragma unroll
    for (int i = 0; i < PT; ++i) {
        const size_t m = m0 + i < n ? m0 + i : n - 1;
        a[i] = attn[m * kH + c];
        if constexpr (RAW) {
            gt[i] = bf16_bits_to_f32(static_cast<const uint16_t *>(gate)[m * 4 * kH + 3 * kH + c]);
        } else {
            gt[i] = static_cast<const float *>(gate)[m * kH + c];
            sg[i] = sgate[m * kH + c];
        }
    }
    const float wt = w[t];
#pragma unroll
    for (int i = 0; i < PT; ++i) as[i][t] = a[i];
    __syncthreads();
    if constexpr (RAW) {
#pragma unroll
        for (int i = 0; i < PT; ++i) sg[i] = sigmoid_ref(gt[i], Exp2Lds{exp2_lds});
    }
    if (t < PT * (kHD / 16)) {
        const int i = t / (kHD / 16), r = t % (kHD / 16);
        float s = 0.0f;
#pragma unroll
        for (int kk = 0; kk < 16; ++kk) {
            const float v = as[i][16 * r + kk];
            s += v * v;
        }
        cs[i][r] = s;
    }
    __syncthreads();
    if (t < PT) {
        float v[kHD / 16];
#pragma unroll
        for (int i = 0; i < kHD / 16; ++i) v[i] = cs[t][i];
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < kHD / 16; ++i) sum += v[i];
        scale_s[t] = 1.0f / __builtin_sqrtf(sum / (float)kHD + eps);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PT; ++i) xs[i][t] = rne_bf16(a[i] * scale_s[i] * wt * gt[i] * sg[i]);
    __syncthreads();
    if (t < PT * (kHD / 8)) {
        const int i = t / (kHD / 8), j = t % (kHD / 8);
        if (m0 + i < n) store_x8(x_out, m0 + i, h * kHD + 8 * j, xs[i] + 8 * j);
    }
}
constexpr int kOnTok = 4;  // prefill tokens per output-norm workgroup

// The recurrence of one (head, stream, 64-column group) per workgroup of 256
// threads, with the batch-1 arithmetic (gdn_island_prep / read / update,
// gdn_model.cpp:2376-2933).  Wave w owns state rows 64 w .. + 63 of the
// group's columns (a column per lane), held in registers from load to store.
// Every wave forms its products S[j][i] kn[j] and S[j][i] qn[j] as its rows
// arrive; only the adds of the chains, in the reference's order j = 0..255,
// go from wave to wave: in turn s wave s continues the r chain, wave s - 1 the
// p chain behind it, the partial sums through LDS.  Then every wave forms
// delta (the last one o) and writes its rows of S' = decay * S + kn (x) delta.
// The norms and alpha are each wave's own (four values per lane, then the
// lanes: the batch-1 tree), so nothing waits for a barrier before the chains.
// What bounds it: at 64 streams the state's read and write (268 MB, 5.5 TB/s);
// at few streams the latency of load, chains and store.  In 128-column groups
// whose waves multiplied inside the chains: 10.7 -> 5.3 us at one stream, 17.3
// -> 13.4 at 16, 55.7 -> 49.2 at 64 (21.4 -> 22.4 at 24, where 768 workgroups
// fill the 512 places one and a half times).
__global__ __launch_bounds__(kT, 2) void k_brecur(const float *__restrict__ qkv, const float *__restrict__ bd,
                                                  float *__restrict__ state, float *__restrict__ attn) {
    constexpr int RW = kHD / 4;  // rows per wave
    __shared__ __attribute__((aligned(16))) float kq[4][2][kHD];  // each wave's kn, qn
    __shared__ float rs[kRecCols], ps[kRecCols];
    const int cg = blockIdx.x % (kHD / kRecCols), h = blockIdx.x / (kHD / kRecCols), m = blockIdx.y;
    const int t = threadIdx.x, w = t >> 6, lane = t & 63, col = cg * kRecCols + lane;
    const float *qp = qkv + (size_t)m * 3 * kH + h * kHD;
    const f32x4 q4 = *reinterpret_cast<const f32x4 *>(qp + 4 * lane);
    const f32x4 k4 = *reinterpret_cast<const f32x4 *>(qp + kH + 4 * lane);
    float *S = state + (size_t)m * kLayerState + (size_t)h * kHD * kHD + (size_t)(RW * w) * kHD + col;
    float sv[RW];
#pragma unroll
    for (int j = 0; j < RW; ++j) sv[j] = S[(size_t)j * kHD];
    const float beta = bd[m * 16 + 2 * h], decay = bd[m * 16 + 2 * h + 1], v = qp[2 * kH + col];
    auto tree = [](f32x4 x, f32x4 y) { return wave_tree64((x.x * y.x + x.y * y.y) + (x.z * y.z + x.w * y.w)); };
    const float q_inv = 1.0f / __builtin_sqrtf(tree(q4, q4) + 1e-6f);
    const float k_inv = 1.0f / __builtin_sqrtf(tree(k4, k4) + 1e-6f);
    const f32x4 qn = {q4.x * q_inv, q4.y * q_inv, q4.z * q_inv, q4.w * q_inv};
    const f32x4 kn = {k4.x * k_inv, k4.y * k_inv, k4.z * k_inv, k4.w * k_inv};
    const float alpha = tree(qn, kn);
    *reinterpret_cast<f32x4 *>(&kq[w][0][4 * lane]) = kn;
    *reinterpret_cast<f32x4 *>(&kq[w][1][4 * lane]) = qn;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float pr[RW], pp[RW];
#pragma unroll
    for (int j = 0; j < RW; j += 4) {
        const f32x4 kv = *reinterpret_cast<const f32x4 *>(&kq[w][0][RW * w + j]);
        const f32x4 qv = *reinterpret_cast<const f32x4 *>(&kq[w][1][RW * w + j]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            pr[j + e] = sv[j + e] * kv[e];
            pp[j + e] = sv[j + e] * qv[e];
            // formed here, not sunk into the chains' branches
            asm volatile("" : "+v"(pr[j + e]), "+v"(pp[j + e]));
        }
    }
#pragma unroll
    for (int s = 0; s < 5; ++s) {
        if (w == s) {
            float r = s ? rs[lane] : 0.0f;
#pragma unroll
            for (int j = 0; j < RW; ++j) r = r + pr[j];
            rs[lane] = r;
        } else if (w == s - 1) {
            float p = s > 1 ? ps[lane] : 0.0f;
#pragma unroll
            for (int j = 0; j < RW; ++j) p = p + pp[j];
            ps[lane] = p;
        }
        if (s < 4) __syncthreads();
    }
    const float d = beta * (v - decay * rs[lane]);
    if (w == 3) attn[(size_t)m * kH + h * kHD + col] = rne_bf16(0.0625f * (decay * ps[lane] + alpha * d));
#pragma unroll
    for (int j = 0; j < RW; j += 4) {
        const f32x4 kv = *reinterpret_cast<const f32x4 *>(&kq[w][0][RW * w + j]);
#pragma unroll
        for (int e = 0; e < 4; ++e) S[(size_t)(j + e) * kHD] = decay * sv[j + e] + kv[e] * d;
    }
}

// ---------------------------------------------------------------- prefill
//
// A prompt runs through one stream's state in segments, layer by layer, the
// tokens taking the place of the streams: each layer's projections take the
// whole segment (the step's sums in the step's order, see "prefill
// projections"), the causal conv reads its taps from the neighbouring tokens,
// and the recurrence runs over the segment's tokens in one launch, in order
// with the state in registers (k_pscan) or in the chunked form (k_wy_seq).  In
// order, every token sees the arithmetic of a multi-stream step, so a prefill
// of n tokens equals n steps bit for bit.

// The causal conv of one 64-channel block over 64 tokens of a segment of n:
// grid (4 kH / 64, ceil(n / 64)), with B16 (3 kH / 64, ..), the gate left to
// k_bonorm; thread 16 r + j on channels 4 j .. 4 j + 3 of the block and tokens
// r, r + 16, r + 32, r + 48 (16-byte loads and stores; the four loads in
// flight together).  raw is [n][4 kH]: the unrounded q, k, v, g sums, or (B16)
// their roundings R(raw); the tails are the prefilled stream's for this layer,
// [q,k,v][3 oldest..newest][kH].  Token m's window is (s[m], s[m+1],
// s[m+2]) and its input s[m+3] in the sequence s = tails ++ R(raw[0..n));
// the new tails are s[n], s[n+1], s[n+2].  Only the first token block reads
// the old tails, and it writes the new ones after that read.
constexpr int kConvT = 256;                  // threads per conv workgroup
constexpr int kConvR = 16 * kMaxB / kConvT;  // tokens per thread
template <bool B16>
__global__ __launch_bounds__(kConvT) void k_pconv(const void *__restrict__ raw, int n, uint16_t *__restrict__ tails,
                                                  const float *__restrict__ conv_w, float *__restrict__ qkv,
                                                  float *__restrict__ gate, float *__restrict__ sgate) {
    static_assert(kConvR * kConvT == 16 * kMaxB && kConvT >= 64, "16 lanes of 4 channels x kMaxB tokens");
    constexpr int MS = kConvT / 16;  // token stride between a thread's tokens
    __shared__ __attribute__((aligned(16))) float xs[kMaxB + 3][64];
    __shared__ uint64_t exp2_lds[32];  // expf's table, read per SiLU / sigmoid
    const int row0 = blockIdx.x * 64, t = threadIdx.x, mr = t >> 4, c4 = 4 * (t & 15);
    const int m0 = (int)blockIdx.y * kMaxB, nb = n - m0 < kMaxB ? n - m0 : kMaxB;
    fill_exp2_lds_imm(exp2_lds);
    const Exp2Lds tab{exp2_lds};
    const int which = row0 / kH, cb = row0 - which * kH;  // section and its first channel
    // tokens m0 + mr + MS i: raw sums of channels cb + c4 .. + 3.  Tokens
    // past the segment load its last token (in bounds, unused), so every
    // load is unconditional and all are in flight at once.
    auto one = [&](int m) {  // R(raw) of token m, channel row0 + t
        const size_t o = (size_t)m * 4 * kH + row0 + t;
        if constexpr (B16) return bf16_bits_to_f32(static_cast<const uint16_t *>(raw)[o]);
        else return rne_bf16(static_cast<const float *>(raw)[o]);
    };
    f32x4 rr[kConvR];
#pragma unroll
    for (int i = 0; i < kConvR; ++i) {
        const int m = mr + MS * i < nb ? mr + MS * i : nb - 1;
        const size_t o = (size_t)(m0 + m) * 4 * kH + row0 + c4;
        if constexpr (B16) {
            const u32x2 r = *reinterpret_cast<const u32x2 *>(static_cast<const uint16_t *>(raw) + o);
            rr[i] = (f32x4){u2f(r.x << 16), u2f(r.x & 0xffff0000u), u2f(r.y << 16), u2f(r.y & 0xffff0000u)};
        } else {
            const f32x4 r = *reinterpret_cast<const f32x4 *>(static_cast<const float *>(raw) + o);
            rr[i] = (f32x4){rne_bf16(r.x), rne_bf16(r.y), rne_bf16(r.z), rne_bf16(r.w)};
        }
    }
    if (B16 || which < 3) {
        uint16_t *tl = tails + (size_t)which * 3 * kH + cb;
        const f32x4 *cw4 = reinterpret_cast<const f32x4 *>(conv_w + ((size_t)which * kH + cb + c4) * 4);
        const f32x4 cw[4] = {cw4[0], cw4[1], cw4[2], cw4[3]};
        if (t < 64) {
            if (m0 == 0) {
                xs[0][t] = bf16_bits_to_f32(tl[t]);
                xs[1][t] = bf16_bits_to_f32(tl[kH + t]);
                xs[2][t] = bf16_bits_to_f32(tl[2 * kH + t]);
            } else {
#pragma unroll
                for (int i = 0; i < 3; ++i) xs[i][t] = one(m0 - 3 + i);
            }
        }
#pragma unroll
        for (int i = 0; i < kConvR; ++i)
            if (mr + MS * i < nb) *reinterpret_cast<f32x4 *>(&xs[3 + mr + MS * i][c4]) = rr[i];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kConvR; ++i) {
            const int m = mr + MS * i;
            if (m >= nb) break;
            // gdn_depthwise_conv_silu_head_kind, gdn_model.cpp:1543-1667
            const f32x4 x0 = *reinterpret_cast<const f32x4 *>(&xs[m][c4]);
            const f32x4 x1 = *reinterpret_cast<const f32x4 *>(&xs[m + 1][c4]);
            const f32x4 x2 = *reinterpret_cast<const f32x4 *>(&xs[m + 2][c4]);
            const f32x4 x3 = *reinterpret_cast<const f32x4 *>(&xs[m + 3][c4]);
            f32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float sum = x0[e] * cw[e].x + x1[e] * cw[e].y + x2[e] * cw[e].z + x3[e] * cw[e].w;
                o[e] = rne_bf16(silu_ref(sum, tab));
            }
            *reinterpret_cast<f32x4 *>(qkv + ((size_t)(m0 + m) * 3 + which) * kH + cb + c4) = o;
        }
        if (t < 64 && m0 == 0) {
            if (n <= kMaxB) {
                tl[t] = bf16_hi(xs[n][t]);
                tl[kH + t] = bf16_hi(xs[n + 1][t]);
                tl[2 * kH + t] = bf16_hi(xs[n + 2][t]);
            } else {
#pragma unroll
                for (int i = 0; i < 3; ++i) tl[i * kH + t] = bf16_hi(one(n - 3 + i));
            }
        }
    } else {
        __syncthreads();  // expf's table
#pragma unroll
        for (int i = 0; i < kConvR; ++i) {
            const int m = mr + MS * i;
            if (m >= nb) break;
            const size_t o = (size_t)(m0 + m) * kH + cb + c4;
            *reinterpret_cast<f32x4 *>(gate + o) = rr[i];
            *reinterpret_cast<f32x4 *>(sgate + o) =
                (f32x4){sigmoid_ref(rr[i].x, tab), sigmoid_ref(rr[i].y, tab), sigmoid_ref(rr[i].z, tab),
                        sigmoid_ref(rr[i].w, tab)};
        }
    }
}

// Per (head, token): the q/k L2 norms and alpha of the recurrence, in the
// batch-1 tree order, for tokens kQkTok y .. + kQkTok - 1 of n, their loads
// requested together (a token past n re-reads token n - 1, unused).
constexpr int kQkTok = 4;
__global__ __launch_bounds__(kT) void k_pqk(const float *__restrict__ qkv, int n, float *__restrict__ qn_out,
                                            float *__restrict__ kn_out, float *__restrict__ alpha_out) {
    static_assert(kT == kHD, "a thread per head channel");
    __shared__ float red[kQkTok][8], red2[kQkTok][4];
    const int h = blockIdx.x, m0 = (int)blockIdx.y * kQkTok, t = threadIdx.x, w = t >> 6, lane = t & 63;
    float q[kQkTok], k[kQkTok];
#pragma unroll
    for (int i = 0; i < kQkTok; ++i) {
        const float *qp = qkv + (size_t)(m0 + i < n ? m0 + i : n - 1) * 3 * kH + h * kHD;
        q[i] = qp[t];
        k[i] = qp[kH + t];
    }
#pragma unroll
    for (int i = 0; i < kQkTok; ++i) {
        const float qs = wave_tree64(q[i] * q[i]), ks = wave_tree64(k[i] * k[i]);
        if (lane == 0) {
            red[i][w] = qs;
            red[i][4 + w] = ks;
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kQkTok; ++i) {
        const int m = m0 + i;
        const float q_sq = (red[i][0] + red[i][1]) + (red[i][2] + red[i][3]);
        const float k_sq = (red[i][4] + red[i][5]) + (red[i][6] + red[i][7]);
        const float qv = q[i] * (1.0f / __builtin_sqrtf(q_sq + 1e-6f));
        const float kv = k[i] * (1.0f / __builtin_sqrtf(k_sq + 1e-6f));
        if (m < n) {
            qn_out[(size_t)m * kH + h * kHD + t] = qv;
            kn_out[(size_t)m * kH + h * kHD + t] = kv;
        }
        const float qk = wave_tree64(qv * kv);
        if (lane == 0) red2[i][w] = qk;
    }
    __syncthreads();
    if (t < kQkTok && m0 + t < n) alpha_out[(m0 + t) * kNH + h] = (red2[t][0] + red2[t][1]) + (red2[t][2] + red2[t][3]);
}

// The recurrence over a segment's n_total tokens in token order, one launch
// per layer: grid (kHD / kScanWgCols, kNH), scan_block with the normalised
// q and k of k_pqk.  Each value is formed as the decode step's k_brecur forms
// it.
struct SegScalars {
    const float *bd, *alpha;  // [token][16] beta, decay per head; [token][kNH]
    int h;
    __device__ __forceinline__ f32x4 get(int m) const {
        return (f32x4){bd[m * 16 + 2 * h], bd[m * 16 + 2 * h + 1], alpha[m * kNH + h], 0.0f};
    }
};
__global__ __launch_bounds__(kT) void k_pscan(const float *__restrict__ qkv, const float *__restrict__ qn_seg,
                                               const float *__restrict__ kn_seg, const float *__restrict__ alpha_seg,
                                               const float *__restrict__ bd_seg, int n_total, float *__restrict__ state,
                                               float *__restrict__ attn_seg) {
    __shared__ ScanLds lds;
    const int h = blockIdx.y, c0 = blockIdx.x * kScanWgCols;
    ScanArgs a;
    a.k = kn_seg + h * kHD;
    a.q = qn_seg + h * kHD;
    a.v = qkv + 2 * kH + h * kHD + c0;
    a.o = attn_seg + h * kHD + c0;
    a.ldq = a.ldo = kH;
    a.ldv = 3 * kH;
    a.n = n_total;
    scan_block<kBf16w, false>(a, SegScalars{bd_seg, alpha_seg, h}, state + (size_t)h * kHD * kHD + c0, lds);
}

// ---------------------------------------------------- chunked prefill (WY form)
//
// The chunk's recurrence in the chunk-parallel form of the gated delta rule
// (chunk.py:616-686 computes the same quantities with a WY representation).
// With the state S (key row j, value column i) before the chunk, per-token
// decay a_m, cumulative log decay G_m = sum_{s<=m} log a_m (so a_{s+1} ...
// a_m = exp(G_m - G_s)), and normalised k_m, q_m:
//   L[m][s]  = beta_m exp(G_m - G_s) (k_m . k_s)      s < m
//   Mq[m][s] = exp(G_m - G_s) (q_m . k_s)             s <= m
//   delta_m  = beta_m (v_m - exp(G_m) S^T k_m) - sum_{s<m} L[m][s] delta_s,
//              i.e. delta = T b with T = (I + L)^-1 (formed per chunk by
//              k_wy_prep, chunk.py's solve of the same triangular system)
//   o_m      = (exp(G_m) S^T q_m + sum_{s<=m} Mq[m][s] delta_s) / 16
//   S'       = exp(G_{n-1}) S + sum_s exp(G_{n-1} - G_s) k_s delta_s^T
// which is the per-token recurrence of the decode step unrolled over the
// chunk (delta_m is the step's beta (v - decay S_{m-1}^T k), o_m its
// S_m^T q / 16).  The sums are associated differently from the step's
// sequential chains, so this mode matches the scan within a tolerance, not
// bit for bit; o is rounded to BF16 as the step rounds it.

//
// q and k are BF16 values before their normalisation, so every product with
// them runs on the BF16 matrix cores without loss: k_m . k_s and q_m . k_s
// as they are, with the two inverse norms as factors of the sum, and
// products with an FP32 operand (the state, the deltas) after that operand
// is split into three BF16 terms whose sum it is (8 + 8 + 8 significand
// bits).  v_mfma_f32_16x16x32_bf16 forms exact products and FP32 sums at
// 16 times the rate of v_mfma_f32_16x16x4_f32, so three (or, between two
// split operands, six) of them still take a fifth (three eighths) of its
// time.

__device__ __forceinline__ f32x4 mfma_bf16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
}

// x as three BF16 terms: p[0] + p[1] + p[2] = x (each rounded to nearest, the
// differences exact), four values packed in two words.  The first term is
// held to the largest finite BF16 value, so every finite x of 2^-110 and more
// is its terms' sum (rounded up to an infinity, that term would leave
// infinity - infinity behind); below, the last terms are BF16 subnormals.  An
// infinite or NaN x has a NaN term.
__device__ __forceinline__ void split3(const f32x4 x, u32x2 (&p)[3]) {
    constexpr float kMax = 0x1.fep127f;
    auto held = [](float v) { return __builtin_amdgcn_fmed3f(v, -kMax, kMax); };
    f32x4 r = x;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        p[i].x = i == 0 ? cvt_pk(held(r.x), held(r.y)) : cvt_pk(r.x, r.y);
        p[i].y = i == 0 ? cvt_pk(held(r.z), held(r.w)) : cvt_pk(r.z, r.w);
        if (i < 2) {
            r.x = r.x - u2f(p[i].x << 16);
            r.y = r.y - u2f(p[i].x & 0xffff0000u);
            r.z = r.z - u2f(p[i].y << 16);
            r.w = r.w - u2f(p[i].y & 0xffff0000u);
        }
    }
}

// The product of two split operands over one 32-wide k step, smallest terms
// first (the three terms below 2^-24 of the product are left out).
__device__ __forceinline__ f32x4 mfma_split(const u32x4 (&a)[3], const u32x4 (&b)[3], f32x4 c) {
    c = mfma_bf16(a[2], b[0], c);
    c = mfma_bf16(a[0], b[2], c);
    c = mfma_bf16(a[1], b[1], c);
    c = mfma_bf16(a[1], b[0], c);
    c = mfma_bf16(a[0], b[1], c);
    return mfma_bf16(a[0], b[0], c);
}

// One (chunk, head)'s operands of k_wy_seq, written by k_wy_prep: MFMA A
// fragments (64 lanes x 8 BF16 values, 1 KB), grouped by the wave that reads
// them.
//   kf, qf  [wave w][16-token tile][k step t]: token 16 tile + l % 16, keys
//           64 w + 32 t + 4 (l / 16) + {0..3, 16..19} (the keys a lane of
//           k_wy_seq holds of the state, so the state is the B operand as
//           it lies in registers)
//   ktf     [w][16-key tile][t]: key 64 w + 16 tile + l % 16, tokens
//           32 t + 8 (l / 16) .. + 7
//   tf, mf  [w][t][term]: T and Mq, row 16 w + l % 16, columns
//           32 t + 8 (l / 16) .. + 7, the three BF16 terms
//   sc      [token]: exp(G_m) / |k_m|, beta_m, exp(G_m) / |q_m|,
//           exp(G_{n-1} - G_m) / |k_m|
//   dn      exp(G_{n-1})
struct WyOps {
    u32x4 kf[4][4][2][64], qf[4][4][2][64], ktf[4][4][2][64];
    u32x4 tf[4][2][3][64], mf[4][2][3][64];
    f32x4 sc[kMaxB];
    float dn, pad[3];
};
static_assert(sizeof(WyOps) % 16 == 0, "16-byte fragments of every (chunk, head)");

// The operands of one (head, chunk): grid (kNH, chunks).  q and k come as
// the conv left them ([token][3][kH], BF16 values); each row is scaled by a
// power of two to the size of a unit vector (exact, so the sums of raw
// products cannot overflow where the normalised ones would not) and that
// power is taken back in its inverse norm.  T = (I + L)^-1 is formed in 16 x
// 16 blocks: the diagonal blocks by forward substitution (a lane per column),
// then T[I][J] = -T[I][I] sum_{J <= K < I} L[I][K] T[K][J] by distance from
// the diagonal on v_mfma_f32_16x16x4_f32.  One wave substituting all 64 rows
// took 24 us a launch; with the norms (k_pqk) and the FP32 gram kernel this
// launch replaces, 108 us per layer of a 4096-token prefill.
constexpr int kWyRow = kHD + 8;    // padded BF16 row of a token (528 bytes)
constexpr int kWyMat = kMaxB + 4;  // padded FP32 row of a chunk matrix
__global__ __launch_bounds__(kT) void k_wy_prep(const float *__restrict__ qkv_seg, const float *__restrict__ bd_seg,
                                                int n_total, WyOps *__restrict__ ops_seg) {
    constexpr int kRows = kMaxB * kWyRow * 2, kMats = 2 * kMaxB * kWyMat * 4;
    // q rows, later L and Mq; k rows, later T
    __shared__ __attribute__((aligned(16))) unsigned char mem_q[kMats > kRows ? kMats : kRows];
    __shared__ __attribute__((aligned(16))) unsigned char mem_k[kRows];
    __shared__ double glog[kMaxB];
    __shared__ float ikn[kMaxB], iqn[kMaxB], bet[kMaxB];
    uint16_t(*qr)[kWyRow] = reinterpret_cast<uint16_t(*)[kWyRow]>(mem_q);
    uint16_t(*kr)[kWyRow] = reinterpret_cast<uint16_t(*)[kWyRow]>(mem_k);
    float(*lm)[kWyMat] = reinterpret_cast<float(*)[kWyMat]>(mem_q);
    float(*mm)[kWyMat] = lm + kMaxB;
    float(*tm)[kWyMat] = reinterpret_cast<float(*)[kWyMat]>(mem_k);
    static_assert(kMaxB * kWyMat * 4 <= kRows, "T fits the k rows");
    const int h = blockIdx.x, ch = blockIdx.y, t = threadIdx.x, w = t >> 6, lane = t & 63;
    const int li = lane & 15, kk = lane >> 4;
    const int n = n_total - kMaxB * ch < kMaxB ? n_total - kMaxB * ch : kMaxB;
    const float *qkv = qkv_seg + (size_t)ch * kMaxB * 3 * kH + h * kHD + 4 * lane;
    const float *bd = bd_seg + (size_t)ch * kMaxB * 16;
    WyOps &ops = ops_seg[(size_t)ch * kNH + h];

    // wave w: tokens 16 w .. + 15, four channels per lane; a token past the
    // chunk's end re-reads its last one and is stored as zeros
    f32x4 x[2][16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int m = 16 * w + i < n ? 16 * w + i : n - 1;
#pragma unroll
        for (int j = 0; j < 2; ++j) x[j][i] = *reinterpret_cast<const f32x4 *>(qkv + ((size_t)m * 3 + j) * kH);
    }
    if (t < kMaxB) {
        // G: inclusive prefix sum of log(decay) over the chunk (a decay that
        // underflowed to 0 is taken as 1e-30: the products it enters are 0
        // to FP32 either way, and G stays finite).  In FP64: the weights are
        // exponentials of differences of G, whose FP32 rounding alone was
        // most of this mode's distance from the scan.
        double v = t < n ? log((double)fmaxf(bd[t * 16 + 2 * h + 1], 1e-30f)) : 0.0;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const double o = __shfl_up(v, d);
            if (lane >= d) v += o;
        }
        glog[t] = v;
        bet[t] = t < n ? bd[t * 16 + 2 * h] : 0.0f;
    }
    // lane 2 i + j: |x[j][i]|^2 in gdn_tree_reduce_256's order, as the scan has
    // it, so one square root and division serve the wave's 32 rows (each row's
    // own, in every lane, was a fifth of the kernel's instructions: 17.8 -> 14.9
    // us at 70 tokens, 33.6 -> 30.4 at 4096)
    float sq = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const f32x4 v = x[j][i];
            const float r = wave_tree64((v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w));
            sq = lane == 2 * i + j ? r : sq;
        }
    const float inv = 1.0f / __builtin_sqrtf(sq + 1e-6f);
    // 2^e of 1 / |x|; both factors normal numbers
    uint32_t pw = f2u(inv) & 0x7f800000u;
    pw = pw < 0x01000000u ? 0x01000000u : pw;
    if (lane < 32) (lane & 1 ? ikn : iqn)[16 * w + (lane >> 1)] = inv * u2f(0x7f000000u - pw);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int m = 16 * w + i;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const f32x4 v = x[j][i];
            const float up = u2f((uint32_t)__builtin_amdgcn_readlane((int)pw, 2 * i + j));
            u32x2 pk;
            pk.x = m < n ? cvt_pk(v.x * up, v.y * up) : 0u;
            pk.y = m < n ? cvt_pk(v.z * up, v.w * up) : 0u;
            *reinterpret_cast<u32x2 *>(&(j ? kr : qr)[m][4 * lane]) = pk;
        }
    }
    __syncthreads();
    if (t < kMaxB) {
        const float g = __expf((float)glog[t]);
        ops.sc[t] = (f32x4){g * ikn[t], bet[t], g * iqn[t], __expf((float)(glog[n - 1] - glog[t])) * ikn[t]};
        if (t == 0) ops.dn = __expf((float)glog[n - 1]);
    }
    // A fragments for k_wy_seq's wave w
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int key = 64 * w + 32 * ks + 4 * kk;
            const u32x2 k0 = *reinterpret_cast<const u32x2 *>(&kr[16 * mt + li][key]);
            const u32x2 k1 = *reinterpret_cast<const u32x2 *>(&kr[16 * mt + li][key + 16]);
            ops.kf[w][mt][ks][lane] = (u32x4){k0.x, k0.y, k1.x, k1.y};
            const u32x2 q0 = *reinterpret_cast<const u32x2 *>(&qr[16 * mt + li][key]);
            const u32x2 q1 = *reinterpret_cast<const u32x2 *>(&qr[16 * mt + li][key + 16]);
            ops.qf[w][mt][ks][lane] = (u32x4){q0.x, q0.y, q1.x, q1.y};
            uint32_t kt[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) kt[e] = kr[32 * ks + 8 * kk + e][64 * w + 16 * mt + li];
            ops.ktf[w][mt][ks][lane] = (u32x4){kt[0] | (kt[1] << 16), kt[2] | (kt[3] << 16), kt[4] | (kt[5] << 16),
                                               kt[6] | (kt[7] << 16)};
        }
    // rows 16 w .. + 15 of K K^T and Q K^T, the tiles on or below the diagonal
    f32x4 gk[4], gq[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) gk[s] = gq[s] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int g = 0; g < kHD / 32; ++g) {
        const u32x4 ka = *reinterpret_cast<const u32x4 *>(&kr[16 * w + li][32 * g + 8 * kk]);
        const u32x4 qa = *reinterpret_cast<const u32x4 *>(&qr[16 * w + li][32 * g + 8 * kk]);
#pragma unroll
        for (int s = 0; s < 4; ++s)
            if (s <= w) {
                const u32x4 kb = *reinterpret_cast<const u32x4 *>(&kr[16 * s + li][32 * g + 8 * kk]);
                gk[s] = mfma_bf16(ka, kb, gk[s]);
                gq[s] = mfma_bf16(qa, kb, gq[s]);
            }
    }
    __syncthreads();  // q and k rows read; L, Mq and T take their place
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int c = 16 * s + li;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = 16 * w + 4 * kk + r;
            float lv = 0.0f, mv = 0.0f;
            if (m < n && c <= m) {
                const float ratio = __expf((float)(glog[m] - glog[c])) * ikn[c];
                if (c < m) lv = bet[m] * (ratio * ikn[m]) * gk[s][r];
                mv = (ratio * iqn[m]) * gq[s][r];
            }
            lm[m][c] = lv;
            mm[m][c] = mv;
            tm[m][c] = 0.0f;
        }
    }
    __syncthreads();
    auto write_terms = [&](const float(*src)[kWyMat], u32x4(&dst)[4][2][3][64], int tile) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            u32x2 a[3], b[3];
            split3(*reinterpret_cast<const f32x4 *>(&src[16 * tile + li][32 * ks + 8 * kk]), a);
            split3(*reinterpret_cast<const f32x4 *>(&src[16 * tile + li][32 * ks + 8 * kk + 4]), b);
#pragma unroll
            for (int p = 0; p < 3; ++p) dst[tile][ks][p][lane] = (u32x4){a[p].x, a[p].y, b[p].x, b[p].y};
        }
    };
    if (w == 0) {
        // lane 16 B + j: column j of the inverse of diagonal block B
        const int b0 = 16 * kk;
        float tc[16];
#pragma unroll
        for (int m = 0; m < 16; ++m) {
            float acc = m == li ? 1.0f : 0.0f;
#pragma unroll
            for (int s4 = 0; s4 < (m + 3) / 4; ++s4) {
                const f32x4 lv = *reinterpret_cast<const f32x4 *>(&lm[b0 + m][b0 + 4 * s4]);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (4 * s4 + e < m) acc = __builtin_fmaf(lv[e], -tc[4 * s4 + e], acc);
            }
            tc[m] = acc;
        }
#pragma unroll
        for (int m = 0; m < 16; ++m) tm[b0 + m][b0 + li] = tc[m];
    } else {
        write_terms(mm, ops.mf, w);
        if (w == 1) write_terms(mm, ops.mf, 0);
    }
    __syncthreads();
#pragma unroll
    for (int d = 1; d < 4; ++d) {
        if (w + d < 4) {
            const int I = w + d, J = w;
            f32x4 y = {0.0f, 0.0f, 0.0f, 0.0f}, z = y;
            for (int K = J; K < I; ++K) {
                const f32x4 a = *reinterpret_cast<const f32x4 *>(&lm[16 * I + li][16 * K + 4 * kk]);
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    y = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q], tm[16 * K + 4 * kk + q][16 * J + li], y, 0, 0, 0);
            }
            // y's rows 4 kk + r are the B operand's k = 4 kk + q as they lie
            const f32x4 a = *reinterpret_cast<const f32x4 *>(&tm[16 * I + li][16 * I + 4 * kk]);
#pragma unroll
            for (int q = 0; q < 4; ++q) z = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q], y[q], z, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) tm[16 * I + 4 * kk + r][16 * J + li] = -z[r];
        }
        __syncthreads();
    }
    write_terms(tm, ops.tf, w);
}

// One head's recurrence over a segment's chunks for 16 state columns: grid
// 8 x 16 workgroups of eight waves, workgroup b on head b % 8 (so an XCD's L2
// serves one head's operands to its sixteen workgroups).
// Waves 0..3, the sequential path: wave w holds state rows 64 w .. + 63 in
// registers from the first chunk to the last, as the accumulator tiles of
// its updates (lane l: rows 16 tile + 4 (l / 16) + r, column l % 16).  Per
// chunk: its keys' share of K S for all 64 tokens, summed over the waves
// through LDS; b = beta (v - exp(G) S^T k) for its 16 tokens; delta = T b;
// S' = exp(G_{n-1}) S + sum_s k_s (exp(G_{n-1} - G_s) delta_s)^T on its rows.
// Waves 4..7, beside them: the same keys' share of Q S (the state's terms
// through LDS) and o for 16 tokens.
// Three barriers a chunk.  Every operand but b, delta, the terms and the
// partial sums comes straight from global memory into registers, a chunk
// ahead.  What bounds it, from cycle stamps of each phase: the latencies of
// the sequential path's three dependent products and their barriers (about
// 4200 cycles a chunk), and the issue of the operand loads (about 1700: 128 KB
// per CU and chunk against a SIMD's limit of some 16 loads in flight); with
// the Q products, or two thirds of the state products, left out it ran only
// 10 % shorter.  At 4096 tokens a launch takes 180 to 190 us on different
// boxes (2.8 to 3.0 us a chunk); where it took 180, the o path on the same four
// waves took 192, and FP32 MFMAs with the state and operands through LDS and
// seven barriers a chunk 520 (8.0 a chunk).
constexpr int kWyCols = 16;
constexpr int kWyTok = kMaxB + 8;  // padded token stride of b and delta (BF16)
constexpr int kWyWaves = 8;

struct WyLds {
    f32x4 ksp[4][4][64], qsp[4][4][64];  // [wave][token tile][lane]
    u32x4 sb[4][3][2][64];               // the state's terms: [wave][term][k step][lane]
    uint16_t bt[3][kWyCols][kWyTok];     // b's terms, [column][token]
    uint16_t dt[3][kWyCols][kWyTok];     // delta's
    uint16_t ft[3][kWyCols][kWyTok];     // the scaled delta's
};

// part[i], component r: token 16 i + 4 (lane / 16) + r, column lane % 16
__device__ __forceinline__ void wy_state_product(const u32x4 (&xf)[4][2], const u32x4 (&sb)[3][2], f32x4 (&part)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) part[i] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int i = 0; i < 4; ++i) part[i] = mfma_bf16(xf[i][ks], sb[p][ks], part[i]);
}
__device__ __forceinline__ void wy_read_terms(const uint16_t (&src)[3][kWyCols][kWyTok], int li, int kk,
                                              u32x4 (&b)[2][3]) {
#pragma unroll
    for (int i = 0; i < 6; ++i)
        b[i / 3][i % 3] = *reinterpret_cast<const u32x4 *>(&src[i % 3][li][32 * (i / 3) + 8 * kk]);
}
__device__ __forceinline__ void wy_write_terms(uint16_t (&dst)[3][kWyCols][kWyTok], int li, int tok, const f32x4 v) {
    u32x2 p[3];
    split3(v, p);
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x2 *>(&dst[i][li][tok]) = p[i];
}
__device__ __forceinline__ f32x4 wy_sum4(const f32x4 (&part)[4][4][64], int tile, int lane) {
    return (part[0][tile][lane] + part[1][tile][lane]) + (part[2][tile][lane] + part[3][tile][lane]);
}
__device__ __forceinline__ void wy_load8(const u32x4 (&src)[4][2][64], int lane, u32x4 (&dst)[4][2]) {
#pragma unroll
    for (int i = 0; i < 8; ++i) dst[i >> 1][i & 1] = src[i >> 1][i & 1][lane];
}
__device__ __forceinline__ void wy_load6(const u32x4 (&src)[2][3][64], int lane, u32x4 (&dst)[2][3]) {
#pragma unroll
    for (int i = 0; i < 6; ++i) dst[i / 3][i % 3] = src[i / 3][i % 3][lane];
}

__global__ __launch_bounds__(kWyWaves * 64) void k_wy_seq(const float *__restrict__ qkv,
                                                          const WyOps *__restrict__ ops_seg, int n_total,
                                                          float *__restrict__ state, float *__restrict__ attn) {
    __shared__ __attribute__((aligned(16))) WyLds lds;
    const int h = blockIdx.x & 7, c0 = (blockIdx.x >> 3) * kWyCols;
    const int t = threadIdx.x, w = (t >> 6) & 3, lane = t & 63, li = lane & 15, kk = lane >> 4;
    const int tok = 16 * w + 4 * kk;  // this lane's four tokens of a chunk
    const int chunks = (n_total + kMaxB - 1) / kMaxB;
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    auto ops = [&](int c) -> const WyOps & { return ops_seg[(size_t)c * kNH + h]; };

    if (t < 256) {
        float *S = state + (size_t)h * kHD * kHD + (size_t)(64 * w + 4 * kk) * kHD + c0 + li;
        const float *vp = qkv + 2 * kH + h * kHD + c0 + li;
        u32x4 kf[4][2], ktf[4][2], tf[2][3];
        f32x4 scn[4], st[4];
        float vn[4], dnn;
        auto load_sv = [&](int c) __attribute__((always_inline)) {
            dnn = vector_load(&ops(c).dn);  // a scalar load's wait would also wait for LDS, and LDS's for it
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = kMaxB * c + tok + r;
                scn[r] = ops(c).sc[tok + r];
                vn[r] = vp[(size_t)(m < n_total ? m : n_total - 1) * 3 * kH];
            }
        };
        load_sv(0);
        wy_load8(ops(0).kf[w], lane, kf);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) st[i][r] = S[(size_t)(16 * i + r) * kHD];
        wy_load6(ops(0).tf[w], lane, tf);
        wy_load8(ops(0).ktf[w], lane, ktf);
        for (int c = 0; c < chunks; ++c) {
            // the next chunk's operands (the last chunk re-reads its own, unused)
            const int cn = c + 1 < chunks ? c + 1 : c;
            f32x4 sc[4], part[4];
            float vv[4];
            const float dn = dnn;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                sc[r] = scn[r];
                vv[r] = vn[r];
            }
            load_sv(cn);
            u32x4 sb[3][2];
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                u32x2 a[3], b[3];
                split3(st[2 * ks], a);
                split3(st[2 * ks + 1], b);
#pragma unroll
                for (int p = 0; p < 3; ++p) sb[p][ks] = (u32x4){a[p].x, a[p].y, b[p].x, b[p].y};
            }
            wy_state_product(kf, sb, part);
#pragma unroll
            for (int i = 0; i < 6; ++i) lds.sb[w][i >> 1][i & 1][lane] = sb[i >> 1][i & 1];
#pragma unroll
            for (int i = 0; i < 4; ++i) lds.ksp[w][i][lane] = part[i];
            wy_load8(ops(cn).kf[w], lane, kf);
            __syncthreads();
            {
                const f32x4 d = wy_sum4(lds.ksp, w, lane);
                f32x4 b;
#pragma unroll
                for (int r = 0; r < 4; ++r) b[r] = sc[r].y * (vv[r] - sc[r].x * d[r]);
                wy_write_terms(lds.bt, li, tok, b);
            }
            __syncthreads();
            // delta = T b (T is the identity and b zero from the chunk's
            // length on; T is zero above the diagonal, so the first two
            // waves' second k step is)
            {
                u32x4 b[2][3];
                wy_read_terms(lds.bt, li, kk, b);
                f32x4 d = mfma_split(tf[0], b[0], zero);
                if (w >= 2) d = mfma_split(tf[1], b[1], zero) + d;
                wy_write_terms(lds.ft, li, tok,
                               (f32x4){sc[0].w * d[0], sc[1].w * d[1], sc[2].w * d[2], sc[3].w * d[3]});
                wy_write_terms(lds.dt, li, tok, d);
                wy_load6(ops(cn).tf[w], lane, tf);
            }
            __syncthreads();
            u32x4 f[2][3];
            wy_read_terms(lds.ft, li, kk, f);
            f32x4 up[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) up[i] = zero;
#pragma unroll
            for (int p = 0; p < 3; ++p)
#pragma unroll
                for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                    for (int i = 0; i < 4; ++i) up[i] = mfma_bf16(ktf[i][ks], f[ks][p], up[i]);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) st[i][r] = __builtin_fmaf(dn, st[i][r], up[i][r]);
            wy_load8(ops(cn).ktf[w], lane, ktf);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) S[(size_t)(16 * i + r) * kHD] = st[i][r];
    } else {
        float *op = attn + h * kHD + c0 + li;
        u32x4 qf[4][2], mf[2][3];
        float cq[4], cqn[4];
        auto load_cq = [&](int c) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < 4; ++r) cqn[r] = ops(c).sc[tok + r].z;
        };
        load_cq(0);
        wy_load8(ops(0).qf[w], lane, qf);
        wy_load6(ops(0).mf[w], lane, mf);
        for (int c = 0; c < chunks; ++c) {
            const int cn = c + 1 < chunks ? c + 1 : c;
#pragma unroll
            for (int r = 0; r < 4; ++r) cq[r] = cqn[r];
            load_cq(cn);
            __syncthreads();
            {
                u32x4 sb[3][2];
                f32x4 part[4];
#pragma unroll
                for (int i = 0; i < 6; ++i) sb[i >> 1][i & 1] = lds.sb[w][i >> 1][i & 1][lane];
                wy_state_product(qf, sb, part);
#pragma unroll
                for (int i = 0; i < 4; ++i) lds.qsp[w][i][lane] = part[i];
                wy_load8(ops(cn).qf[w], lane, qf);
            }
            __syncthreads();
            __syncthreads();
            // o_m = (exp(G_m) S^T q_m + sum_{s<=m} Mq[m][s] delta_s) / 16, rounded
            u32x4 b[2][3];
            wy_read_terms(lds.dt, li, kk, b);
            f32x4 d = mfma_split(mf[0], b[0], zero);
            if (w >= 2) d = mfma_split(mf[1], b[1], zero) + d;
            const f32x4 q = wy_sum4(lds.qsp, w, lane);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = kMaxB * c + tok + r;
                if (m < n_total) op[(size_t)m * kH] = rne_bf16(0.0625f * (cq[r] * q[r] + d[r]));
            }
            wy_load6(ops(cn).mf[w], lane, mf);
        }
    }
}

// ------------------------------------------------ prefill projections
//
// A prefill segment runs layer by layer, so each layer's projection weights
// are read once per segment instead of once per 64 tokens.  k_pgemm (and
// k_pgemm_a, below) and k_pgu form the segment's projections as GEMMs: one workgroup per 128 rows
// (four 32-row blocks of the weight layout; gate/up: two channel groups) x
// 128 tokens (two 64-token X tile blocks), eight waves of 64 rows x 32
// tokens, the k tile's fragments staged once through LDS (double buffer,
// two k tiles of loads in flight per thread).  Every output element is
// formed with the step's operations in the step's order: the same
// v_mfma_f32_16x16x32_bf16 fragments; the k tiles of class c (c, c + NW,
// ... within a split) chained from zero in increasing order, as wave c of
// k_bgemm / k_bgu chains them; the classes added in order, as k_bgemm adds
// its waves' sums; and the splits' sums added in split order, as the
// step's norm adds k_bgemm's split partials.  A prefill therefore still
// equals the steps bit for bit.
constexpr int kPgD = 2;      // k tiles of operand loads in flight per thread
constexpr int kPgTok = 128;  // tokens per workgroup (2 X tile blocks)
constexpr int kSegDefault = 4096;  // prefill tokens per segment by default
constexpr int kSegMax = 32768;     // largest segment (k_pqk's grid.y holds it)
constexpr int kStepTok = 256;      // longest segment whose q/k/v/g take the step's kernel (and gate buffers)

// The j-th k tile in class order: split s, class c, i-th tile of the class.
template <int KT, int NW, int S>
__device__ __forceinline__ int pg_tile(int j) {
    constexpr int KTS = KT / S, KTW = KTS / NW;
    const int s = j / KTS, r = j - s * KTS, c = r / KTW, i = r - c * KTW;
    return s * KTS + c + NW * i;
}

// The workgroup's (row tile, token tile).  Workgroups are dealt to the 8
// XCDs round robin in launch order; when the grid allows, the 32 that one
// XCD runs together cover 4 row tiles x 8 token tiles (a "super tile"), so
// that XCD's L2 serves each weight tile to 8 of them and each activation
// tile to 4.  The super tiles that are left over when their number is no
// multiple of 8 are cut in equal parts over the XCDs (or run in order).
// Otherwise the plain (blockIdx.x, blockIdx.y).
__device__ __forceinline__ void pg_place(int &rt, int &tt) {
    const int R = gridDim.x, C = gridDim.y, L = blockIdx.x + R * blockIdx.y;
    if (R % 4 == 0 && C % 8 == 0) {
        const int gr = R / 4, ns = gr * (C / 8), whole = ns & ~7, rem = ns & 7;
        int u, q;
        if (L < whole * 32) {
            u = 8 * ((L >> 3) >> 5) + (L & 7);
            q = (L >> 3) & 31;
        } else {
            const int r = L - whole * 32;
            if (rem == 1 || rem == 2 || rem == 4) {
                const int parts = 8 / rem, x = r & 7;
                u = whole + x / parts;
                q = (x % parts) * (32 / parts) + (r >> 3);
            } else {
                u = whole + (r >> 5);
                q = r & 31;
            }
        }
        rt = 4 * (u % gr) + (q & 3);
        tt = 8 * (u / gr) + (q >> 2);
    } else {
        rt = blockIdx.x;
        tt = blockIdx.y;
    }
}

// Class bookkeeping after k tile j: the class chain joins the split's sum
// (the first class is taken as it is).  Returns true when the tile closes a
// split (its sum is complete in part).
template <int KT, int NW, int S, int NB>
__device__ __forceinline__ bool pg_close(int j, f32x4 (&chain)[NB], f32x4 (&part)[NB]) {
    constexpr int KTS = KT / S, KTW = KTS / NW;
    if ((j + 1) % KTW != 0) return false;
    const int cls = ((j + 1) / KTW - 1) % NW;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        part[b] = cls == 0 ? chain[b] : part[b] + chain[b];
        chain[b] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    }
    return cls == NW - 1;
}

// y[m][row] for rows 128 rt .. +127 and tokens 128 tt .. +127 (pg_place):
// the sum k_bgemm<2, KT, NW, S, EPI_RAW> forms for the row (S = 1), or one of
// its S split partials.  W in the 32-row block layout ([row block][k tile][2
// tiles][64 lanes]); X in 64-token X tile blocks; y has the padded token
// count's rows.
// Waves per workgroup: 8 of 64 rows x 32 tokens (about 100 VGPRs, four
// waves per SIMD) measured 98.4k against 95.9k prefill tokens/s for 4 of
// 64 x 64 (two per SIMD), with twice the LDS fragment reads.
constexpr int kPgW = 8;

// PLANES: grid z is the split; a workgroup forms one split's sum and writes
// it to that split's plane of y (y_rows tokens), which the consumer adds in
// split order, as it adds the step's: S times the workgroups of a kernel that
// adds the splits itself, for segments whose tiles leave CUs idle.
// B16: the sums are written rounded, as BF16 bits (the step rounds them before
// anything else reads them), half the bytes for this kernel and its reader.
__device__ __forceinline__ void pg_store(float *y, size_t o, const f32x4 v, bool b16) {
    if (b16)
        *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(y) + o) =
            make_uint2((f2u(rne_bf16(v.x)) >> 16) | f2u(rne_bf16(v.y)), (f2u(rne_bf16(v.z)) >> 16) | f2u(rne_bf16(v.w)));
    else
        *reinterpret_cast<f32x4 *>(y + o) = v;
}
template <int KT, int NW, int S, bool PLANES, bool B16>
__global__ __launch_bounds__(kPgW * 64) void k_pgemm(const u32x4 *__restrict__ W, const u32x4 *__restrict__ X,
                                                     float *__restrict__ y, int n_rows, int y_rows) {
    constexpr int NT = PLANES ? KT / S : KT;  // k tiles of this workgroup
    static_assert(NT % kPgD == 0, "whole groups of kPgD k tiles");
    static_assert(S == 1 || PLANES, "one split's sum per workgroup");
    const int jb = PLANES ? (int)blockIdx.z * NT : 0;
    if constexpr (PLANES) y += (size_t)blockIdx.z * y_rows * n_rows;
    constexpr int GT = kPgW * 64, AU = 4 * 2 * 64, BU = 2 * 4 * 64, PT = (AU + BU) / GT;
    constexpr int TG = 2;                 // 16-token groups per wave
    constexpr int NB = 4 * TG;            // 16 x 16 blocks per wave
    static_assert(KT % kPgD == 0 && kPgD % 2 == 0, "whole groups of kPgD k tiles");
    __shared__ u32x4 stg[2][AU + BU];
    const int t = threadIdx.x, w = t >> 6, l = t & 63, wr = w & 1, wt = w >> 1;
    int rt, tt;
    pg_place(rt, tt);
    // entry q = t + GT i: A (row block q / 128, entry q % 128) below AU,
    // else B (token block, entry)
    const u32x4 *src[PT];
    int stride[PT];
#pragma unroll
    for (int i = 0; i < PT; ++i) {
        const int q = t + GT * i;
        if (q < AU) {
            src[i] = W + (size_t)(4 * rt + q / 128) * KT * 128 + (q % 128);
            stride[i] = 128;
        } else {
            src[i] = X + (size_t)(2 * tt + (q - AU) / 256) * KT * 256 + ((q - AU) % 256);
            stride[i] = 256;
        }
    }
    auto fetch = [&](u32x4 (&r)[PT], int kt) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < PT; ++i) r[i] = src[i][(size_t)kt * stride[i]];
    };
    f32x4 chain[NB], part[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) chain[b] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    // row tile f: rows 128 rt + 64 wr + 16 f + 4 (l / 16) .. +3; token
    // group g of the wave: token 128 tt + 16 (TG wt + g) + l % 16
    const int row = 128 * rt + 64 * wr + 4 * (l >> 4);
    const int m = kPgTok * tt + 16 * TG * wt + (l & 15);
    u32x4 rg[kPgD][PT];
#pragma unroll
    for (int d = 0; d < kPgD; ++d) fetch(rg[d], pg_tile<KT, NW, S>(jb + d));
    for (int j0 = 0; j0 < NT; j0 += kPgD) {
#pragma unroll
        for (int d = 0; d < kPgD; ++d) {
            const int j = j0 + d, sb = d & 1;
#pragma unroll
            for (int i = 0; i < PT; ++i) stg[sb][t + GT * i] = rg[d][i];
            // issued on every pass (the last passes re-read the final tile,
            // unused): a conditional load would make the compiler's wait
            // for the next stage a wait for every load in flight
            fetch(rg[d], pg_tile<KT, NW, S>(jb + (j + kPgD < NT ? j + kPgD : NT - 1)));
            __syncthreads();
            u32x4 fa[4], fb[TG];
#pragma unroll
            for (int f = 0; f < 4; ++f) fa[f] = stg[sb][256 * wr + 64 * f + l];
#pragma unroll
            for (int g = 0; g < TG; ++g) fb[g] = stg[sb][AU + 64 * (TG * wt + g) + l];
#pragma unroll
            for (int f = 0; f < 4; ++f)
#pragma unroll
                for (int g = 0; g < TG; ++g)
                    chain[TG * f + g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf16x8, fa[f]), __builtin_bit_cast(bf16x8, fb[g]), chain[TG * f + g], 0,
                        0, 0);
            if (pg_close<KT, NW, S, NB>(j, chain, part)) {
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    pg_store(y, (size_t)(m + 16 * (b % TG)) * n_rows + row + 16 * (b / TG), part[b], B16);
            }
        }
    }
}

// k_pgemm with the weights streamed straight into registers: one workgroup
// per 32 kPgW rows (a 32-row block per wave) x 128 tokens, wave w owning
// rows 32 w .. 32 w + 31 of them for all 128 tokens, so no two waves need the same
// weight fragment and only the tokens' fragments (8 KB per k tile) pass
// through LDS.  The k loop runs one class of one split per trip (its KTW
// tiles unrolled, the next kPaD tiles' operands in flight across trips):
// a loop of fixed shape, whose waits on memory the compiler keeps exact,
// where a loop of kPgD tiles with a data-dependent class close waited for
// every load in flight at its top.  A class starts from a zero operand of its
// first MFMAs, the first class of a split in the split's sum itself: 64 adds
// per further class are all that its close costs (145 -> 131 us for 4096
// tokens' q/k/v/g against cleared chains and a select of the first class).
// A tile's fragments are read from LDS under the second half of the tile
// before it, the barrier in the middle of that tile's products: at 4096
// tokens gate/up 239 -> 223 us, o_proj 42 -> 41, q/k/v/g 140 and down 90 as
// they were (4 waves of 64 rows, half the LDS reads at one wave per SIMD: 279,
// 56, 160, 111).  The total over the splits stays in LDS, each thread's own
// elements: through the output tile, as k_pgemm's splits once had it, o_proj
// at 4096 tokens took 84 us (now 41, 0.84 PFLOP/s) and down 123 (now 90, 1.05).
// What bounds it: the LDS reads of the tokens' fragments (64 KB per k tile and
// CU), as long as the products themselves, and one barrier per k tile.
// Same fragments, chains, class order and split order as the step's kernels,
// so the same sums bit for bit.  PLANES: as k_pgemm's.
constexpr int kPaW = 8;             // waves per workgroup
constexpr int kPaRows = 32 * kPaW;  // rows per workgroup
constexpr int kPaD = 2;             // k tiles of operands in flight

// The i-th of the 16 channels of k_pgu_a's block b: eight of 11 blocks are the
// first 16 channels of a 22-channel group (whole tiles of its weights), three
// the last six of those eight groups.  Channels i and i + 1 (i even) are
// neighbours.
__device__ __forceinline__ int gu_channel(int b, int i) {
    constexpr int kTail = kGuCh - 16;
    static_assert(8 * kTail == 3 * 16 && kGuWgs % 8 == 0 && kTail % 2 == 0, "three blocks of tails per eight groups");
    const int g0 = 8 * (b / 11), q = b % 11;
    if (q < 8) return (g0 + q) * kGuCh + i;
    const int t = 16 * (q - 8) + i;
    return (g0 + t / kTail) * kGuCh + 16 + t % kTail;
}
template <int KT, int NW, int S, bool SWIGLU, bool PLANES, bool B16>
__device__ __forceinline__ void pgemm_a_block(const u32x4 *__restrict__ W, const u32x4 *__restrict__ X,
                                              float *__restrict__ y, uint16_t *__restrict__ x_next, int n_rows,
                                              int n_tok) {
    constexpr bool TOTAL = S > 1 && !PLANES;  // the splits are added here
    constexpr int R = kPaRows / 16 / kPaW;  // 16-row tiles per wave
    constexpr int T = kPgTok / 16;          // 16-token groups per wave
    constexpr int GT = kPaW * 64, BU = T * 64, PB = BU / GT;
    constexpr int NB = R * T, KTS = KT / S, KTW = KTS / NW;
    static_assert(R == 2 && BU % GT == 0 && KT % S == 0 && KTS % NW == 0, "row and token tiles per workgroup");
    __shared__ u32x4 stg[2][BU];
    __shared__ f32x4 tot[TOTAL ? NB : 1][TOTAL ? GT : 1];  // each thread's own sums
    __shared__ uint64_t exp2_lds[SWIGLU ? 32 : 1];  // expf's table for the SwiGLU epilogue
    // the first k tile in class order, and the one past the last
    const int jb = PLANES ? (int)blockIdx.z * KTS : 0, je = PLANES ? jb + KTS : KT;
    if constexpr (SWIGLU) fill_exp2_lds_imm(exp2_lds);
    const int t = threadIdx.x, w = t >> 6, l = t & 63;
    int rt, tt;
    pg_place(rt, tt);
    // wave w's rows: 32-row block kPaW rt + w of the weight layout (its two
    // tiles at entries 0..63 and 64..127 of each k tile), or the gate and up
    // rows of the 16 channels gu_channel names, in k_bgu's 44-row groups
    constexpr int AS = SWIGLU ? kGuTileU4 : 128;  // entries per k tile
    const u32x4 *ap[R];
#pragma unroll
    for (int f = 0; f < R; ++f) {
        if constexpr (SWIGLU) {
            const int c = gu_channel(kPaW * rt + w, l & 15), g = c / kGuCh, r = c % kGuCh;
            ap[f] = W + (size_t)g * KT * AS +
                    (r < 16 ? 64 * f + l : 128 + (l >> 4) * kGuTail2 + (r - 16) + f * (kGuCh - 16));
        } else {
            ap[f] = W + (size_t)(kPaW * rt + w) * KT * AS + 64 * f + l;
        }
    }
    // B entry q of a k tile: token group q / 64 (of 8), lane q % 64
    const u32x4 *bp[PB];
#pragma unroll
    for (int i = 0; i < PB; ++i) {
        const int q = t + GT * i;
        bp[i] = X + (size_t)(2 * tt + (q >> 8)) * KT * 256 + (q & 255);
    }
    f32x4 chain[NB], part[NB];
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    // ra[d]: the weights of tile j + d; rb[d]: the tokens of tile j + 1 + d
    u32x4 ra[kPaD + 1][R], rb[kPaD][PB], fb[T];
    auto load_a = [&](u32x4(&r)[R], int j) __attribute__((always_inline)) {
        const int kt = pg_tile<KT, NW, S>(j < je ? j : je - 1);
#pragma unroll
        for (int f = 0; f < R; ++f) r[f] = ap[f][(size_t)kt * AS];
    };
    auto load_b = [&](u32x4(&r)[PB], int j) __attribute__((always_inline)) {
        const int kt = pg_tile<KT, NW, S>(j < je ? j : je - 1);
#pragma unroll
        for (int i = 0; i < PB; ++i) r[i] = bp[i][(size_t)kt * 256];
    };
    {
        u32x4 r0[PB];
        load_b(r0, jb);
#pragma unroll
        for (int d = 0; d < kPaD; ++d) {
            load_a(ra[d], jb + d);
            load_b(rb[d], jb + 1 + d);
        }
#pragma unroll
        for (int q = 0; q < PB; ++q) stg[jb & 1][t + GT * q] = r0[q];
        __syncthreads();
#pragma unroll
        for (int g = 0; g < T; ++g) fb[g] = stg[jb & 1][64 * g + l];
    }
    // row tile f: rows kPaRows rt + 32 w + 16 f + 4 (l / 16) .. +3; token group
    // g: token 128 tt + 16 g + l % 16
    const int row = kPaRows * rt + 32 * w + 4 * (l >> 4);
    const int m = kPgTok * tt + (l & 15);
    // the k tiles of class c, chained in acc from zero
    auto run_class = [&](int c, f32x4(&acc)[NB]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < KTW; ++i) {
            const int j = c * KTW + i, sb = (j + 1) & 1;
            u32x4 fn[T];
            // issued on every tile (the last ones re-read the final tile,
            // unused), so the loop's shape stays fixed
            load_a(ra[kPaD], j + kPaD);
            // the buffer's fragments of tile j - 1 were read before the
            // barrier of tile j - 1
#pragma unroll
            for (int q = 0; q < PB; ++q) stg[sb][t + GT * q] = rb[0][q];
#pragma unroll
            for (int d = 0; d + 1 < kPaD; ++d)
#pragma unroll
                for (int q = 0; q < PB; ++q) rb[d][q] = rb[d + 1][q];
            load_b(rb[kPaD - 1], j + 1 + kPaD);
            auto mm = [&](int g) __attribute__((always_inline)) {
#pragma unroll
                for (int f = 0; f < R; ++f)
                    acc[T * f + g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf16x8, ra[0][f]), __builtin_bit_cast(bf16x8, fb[g]),
                        i == 0 ? zero : acc[T * f + g], 0, 0, 0);
            };
#pragma unroll
            for (int g = 0; g < T / 2; ++g) mm(g);
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
#pragma unroll
            for (int g = 0; g < T; ++g) fn[g] = stg[sb][64 * g + l];
#pragma unroll
            for (int g = T / 2; g < T; ++g) mm(g);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int g = 0; g < T; ++g) fb[g] = fn[g];
#pragma unroll
            for (int d = 0; d < kPaD; ++d)
#pragma unroll
                for (int f = 0; f < R; ++f) ra[d][f] = ra[d + 1][f];
        }
    };
    // a split's first class chains in part itself, the others in chain and
    // join it; the split's sum joins the total in split order
#pragma unroll 1
    for (int s = PLANES ? (int)blockIdx.z : 0, se = PLANES ? s + 1 : S; s < se; ++s) {
        run_class(s * NW, part);
#pragma unroll 1
        for (int c = 1; c < NW; ++c) {
            run_class(s * NW + c, chain);
#pragma unroll
            for (int b = 0; b < NB; ++b) part[b] = part[b] + chain[b];
        }
        if constexpr (TOTAL) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if (s) part[b] = tot[b][t] + part[b];
                if (s + 1 < S) tot[b][t] = part[b];
            }
        }
    }
    if constexpr (!SWIGLU) {
#pragma unroll
        for (int f = 0; f < R; ++f)
#pragma unroll
            for (int g = 0; g < T; ++g)
                pg_store(y, (size_t)(m + 16 * g) * n_rows + row + 16 * f, part[T * f + g], B16);
    } else {
        // row tile 0: the gate rows of the wave's 16 channels, tile 1 their
        // up rows, so a lane holds both of the wave's channels 4 (l / 16) .. + 3
        // (gemv32_store SwiGLU branch, gdn_model.cpp:4751-4767)
        // channels of a pair are neighbours, pairs need not be (gu_channel)
        const int k0 = gu_channel(kPaW * rt + w, 4 * (l >> 4)), k2 = gu_channel(kPaW * rt + w, 4 * (l >> 4) + 2);
        // one token group per trip, the next ones moved down (unrolled, the
        // eight groups' SiLUs are 50 KB of code)
#pragma unroll 1
        for (int g = 0; g < T; ++g) {
            uint32_t hv[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                hv[e] = bf16_daz_bits(rne_bf16(silu_ref(rne_bf16(part[0][e]), Exp2Lds{exp2_lds}) *
                                               rne_bf16(part[T][e])));
            if (m + 16 * g < n_tok) {
                *reinterpret_cast<uint32_t *>(x_next + xt_index(m + 16 * g, k0, kI)) = hv[0] | (hv[1] << 16);
                *reinterpret_cast<uint32_t *>(x_next + xt_index(m + 16 * g, k2, kI)) = hv[2] | (hv[3] << 16);
            }
#pragma unroll
            for (int i = 0; i + 1 < T; ++i) {
                part[i] = part[i + 1];
                part[T + i] = part[T + i + 1];
            }
        }
    }
}
template <int KT, int NW, int S, bool PLANES, bool B16>
__global__ __launch_bounds__(kPaW * 64) void k_pgemm_a(const u32x4 *__restrict__ W, const u32x4 *__restrict__ X,
                                                       float *__restrict__ y, int n_rows, int y_rows) {
    if constexpr (PLANES) y += (size_t)blockIdx.z * y_rows * n_rows;
    pgemm_a_block<KT, NW, S, false, PLANES, B16>(W, X, y, nullptr, n_rows, 0);
}

// Gate/up + SwiGLU on the same kernel, over the step's weights: a wave takes
// 16 channels' gate rows and their up rows out of k_bgu's 44-row groups, classes
// as k_bgu's, so the sums are the step's; the first n_tok tokens are written.
// All rows carry weights, where the 44-row groups of k_pgu leave 4 of 48 empty,
// and a wave reads 8 fragments from LDS per 16 MFMAs where k_pgu's reads 5 per 6.
// A copy of the weights in 32-row blocks of 16 channels in order (46 MB a layer)
// took 205-208 us at 4096 tokens and 73 at 1000 where this takes 212-214 and 75,
// and 42 at 400 to 640 tokens where this takes 40; channels in order out of the
// groups, 224, 76 and 41.
__global__ __launch_bounds__(kPaW * 64) void k_pgu_a(const u32x4 *__restrict__ W, const u32x4 *__restrict__ X,
                                                     uint16_t *__restrict__ x_next, int n_tok) {
    pgemm_a_block<kKtH, kGuWaves, 1, true, false, false>(W, X, nullptr, x_next, 2 * kI, n_tok);
}

// Gate/up + SwiGLU for channel groups 2 rt, +1 (k_bgu's layout and sums:
// four classes of 16 k tiles) and tokens 128 tt .. +127 (pg_place; the
// first n_tok are written).  Wave w: group w & 1, token block w >> 1.
__global__ __launch_bounds__(kPgW * 64) void k_pgu(const u32x4 *__restrict__ W, const u32x4 *__restrict__ X,
                                                   uint16_t *__restrict__ x_next, int n_tok) {
    constexpr int KT = kKtH, NW = kGuWaves, GT = kPgW * 64;
    constexpr int AU = 2 * kGuTileU4, BU = 2 * 4 * 64, PT = (AU + BU + GT - 1) / GT;
    constexpr int TG = 2;                 // 16-token groups per wave
    constexpr int NB = 3 * TG;            // 16 x 16 blocks per wave
    static_assert(KT % kPgD == 0 && kPgD % 2 == 0, "whole groups of kPgD k tiles");
    __shared__ u32x4 stg[2][AU + BU];
    __shared__ f32x4 red[kPgW][NB * 64];
    __shared__ uint64_t exp2_lds[32];  // expf's table for the SwiGLU epilogue
    const int t = threadIdx.x, w = t >> 6, l = t & 63, wg = w & 1, wt = w >> 1;
    int rt, tt;
    pg_place(rt, tt);
    const int gb = 2 * rt;
    fill_exp2_lds_imm(exp2_lds);
    // entry q = t + GT i: A (group q / kGuTileU4) below AU, else B
    const u32x4 *src[PT];
    int stride[PT];
    bool live[PT];
#pragma unroll
    for (int i = 0; i < PT; ++i) {
        const int q = t + GT * i;
        live[i] = q < AU + BU;
        // entries past the end re-read B entry 0 (loaded, not stored), so
        // every load is unconditional
        if (q < AU) {
            src[i] = W + (size_t)(gb + q / kGuTileU4) * KT * kGuTileU4 + (q % kGuTileU4);
            stride[i] = kGuTileU4;
        } else {
            const int qb = live[i] ? q - AU : 0;
            src[i] = X + (size_t)(2 * tt + qb / 256) * KT * 256 + (qb % 256);
            stride[i] = 256;
        }
    }
    auto fetch = [&](u32x4 (&r)[PT], int kt) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < PT; ++i) r[i] = src[i][(size_t)kt * stride[i]];
    };
    const bool p2 = (l & 15) < kGuTail2;
    const int o2 = 128 + (p2 ? (l >> 4) * kGuTail2 + (l & 15) : 0);
    const u32x4 zero = {0u, 0u, 0u, 0u};
    f32x4 chain[NB], part[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) chain[b] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    u32x4 rg[kPgD][PT];
#pragma unroll
    for (int d = 0; d < kPgD; ++d) fetch(rg[d], pg_tile<KT, NW, 1>(d));
    for (int j0 = 0; j0 < KT; j0 += kPgD) {
#pragma unroll
        for (int d = 0; d < kPgD; ++d) {
            const int j = j0 + d, sb = d & 1;
#pragma unroll
            for (int i = 0; i < PT; ++i)
                if (live[i]) stg[sb][t + GT * i] = rg[d][i];
            fetch(rg[d], pg_tile<KT, NW, 1>(j + kPgD < KT ? j + kPgD : KT - 1));
            __syncthreads();
            u32x4 fa[3], fb[TG];
            fa[0] = stg[sb][wg * kGuTileU4 + l];
            fa[1] = stg[sb][wg * kGuTileU4 + 64 + l];
            fa[2] = p2 ? stg[sb][wg * kGuTileU4 + o2] : zero;
#pragma unroll
            for (int g = 0; g < TG; ++g) fb[g] = stg[sb][AU + 64 * (TG * wt + g) + l];
#pragma unroll
            for (int f = 0; f < 3; ++f)
#pragma unroll
                for (int g = 0; g < TG; ++g)
                    chain[TG * f + g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf16x8, fa[f]), __builtin_bit_cast(bf16x8, fb[g]), chain[TG * f + g], 0,
                        0, 0);
            (void)pg_close<KT, NW, 1, NB>(j, chain, part);
        }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) red[w][b * 64 + l] = part[b];
    // the wave reads only its own sums
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // row rr of tile r, token m of the wave: lane (rr / 4) * 16 + m % 16 of
    // token group m / 16, component rr % 4 (k_bgu's val)
    auto val = [&](int r, int rr, int m) {
        return reinterpret_cast<const float *>(red[w])[4 * ((r * TG + (m >> 4)) * 64 + (rr >> 2) * 16 + (m & 15)) +
                                                       (rr & 3)];
    };
    const int mb = kPgTok * tt + 16 * TG * wt;
    for (int q = l; q < 16 * TG * (kGuCh / 2); q += 64) {
        const int m = q / (kGuCh / 2), cp = q - m * (kGuCh / 2);
        if (mb + m >= n_tok) continue;
        uint32_t packed = 0;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int cc = 2 * cp + e;
            const float g = rne_bf16(cc < 16 ? val(0, cc, m) : val(2, cc - 16, m));
            const float u = rne_bf16(cc < 16 ? val(1, cc, m) : val(2, cc - 16 + (kGuCh - 16), m));
            packed |= bf16_daz_bits(rne_bf16(silu_ref(g, Exp2Lds{exp2_lds}) * u)) << (16 * e);
        }
        *reinterpret_cast<uint32_t *>(x_next + xt_index(mb + m, (gb + wg) * kGuCh + 2 * cp, kI)) = packed;
    }
}

}  // namespace bt
}  // namespace gdn

// ===================================================================== engine

using namespace gdn;
using namespace gdn::bt;

struct GDNBatchEngine {
    int layers = 0, vocab = 0, streams = 0;
    float eps = 1e-6f;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    void *wmem = nullptr;
    const u32x4 *w_qkvg[kMaxLayers] = {}, *w_o[kMaxLayers] = {}, *w_gu[kMaxLayers] = {},
                *w_down[kMaxLayers] = {}, *w_lm = nullptr;
    uint16_t *emb = nullptr;
    float *aux = nullptr;      // [layers][kAuxLayer] + final_norm[kH]
    float *state = nullptr;    // [layers][streams][kNH][kHD][kHD]
    uint16_t *tails = nullptr; // [layers][streams][3][3][kH], BF16 bits
    float *act = nullptr;
    float *h = nullptr, *qkv = nullptr, *gate = nullptr, *sgate = nullptr, *bd = nullptr,
          *attn = nullptr, *ypart = nullptr, *xn = nullptr, *logits = nullptr, *part_val = nullptr;
    int *part_idx = nullptr;
    uint16_t *x_h = nullptr, *x_o = nullptr, *x_d = nullptr;  // X tiles, K = 2048 / 2048 / 5632
    int *tok_host = nullptr;  // pinned, mapped, coherent: [0..64) tokens in, [64..128) argmaxes out
    int *tok_map = nullptr;   // the device's address of tok_host (the step's tokens)
    // prefill: the last token block's logits and argmax tokens (buffers of
    // their own, so a prefill leaves the other streams' last step readable)
    float *p_logits = nullptr;
    int *p_tok = nullptr;
    int prefill_mode = GDN_PREFILL_SCAN;
    // prefill segment buffers, allocated at the first prefill for seg_cap
    // tokens (per token: residual ping-pong, projection sums, q/k/v,
    // beta/decay, attention output, alpha, the norms' copy; X tiles of three
    // widths; gate and sigmoid(gate) for kStepTok tokens).  s_wy, the chunked
    // mode's operands, shares its memory with s_qn and s_kn, the scan's
    // normalised q and k
    int seg_tokens = kSegDefault, seg_cap = 0;
    void *seg_mem = nullptr;
    float *s_h = nullptr, *s_y = nullptr, *s_qkv = nullptr, *s_gate = nullptr, *s_sgate = nullptr, *s_bd = nullptr,
          *s_attn = nullptr, *s_qn = nullptr, *s_kn = nullptr, *s_alpha = nullptr, *s_xn = nullptr;
    WyOps *s_wy = nullptr;
    uint16_t *s_xh = nullptr, *s_xo = nullptr, *s_xd = nullptr;
    int *s_tok = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    bool use_graph = true;
};

namespace {

float *b_aux(GDNBatchEngine *e, int l) { return e->aux + (size_t)l * kAuxLayer; }
uint16_t *b_tails(GDNBatchEngine *e, int l) { return e->tails + (size_t)l * e->streams * kStreamTails; }
float *b_state(GDNBatchEngine *e, int l) { return e->state + (size_t)l * e->streams * kLayerState; }
// The LM head takes 64 rows per workgroup (half the activation re-reads of
// 32: 35.1 -> 28.8 us for the 32000-row head, same sums) where the vocabulary
// allows, else 32; its weights are tiled to match.
int lm_rt(const GDNBatchEngine *e) { return (e->vocab % 64) == 0 ? 4 : 2; }
int lm_wgs(const GDNBatchEngine *e) { return e->vocab / (16 * lm_rt(e)); }
// The step's GEMM on as many 16-stream groups as hold n streams (or prefill
// tokens).  Every workgroup reads the activations of the groups it forms
// beside its rows, two bytes for each weight byte at four groups.  Measured
// with four groups / as many as needed, us per launch: q/k/v/g 13.1 / 10.0 at
// one stream, 13.1 / 11.5 at 16, 14.1 / 12.8 at 32; gate/up 14.7 / 12.6, 15.6 /
// 13.6, 16.2 / 14.8; down 8.1 / 5.6, 8.1 / 6.3, 8.5 / 7.1; LM head 29 / 25,
// 32 / 27, 35 / 31.
template <int RT, int KT, int NW, int S, int EPI>
void launch_bgemm(int n, dim3 grid, const u32x4 *w, const void *x, const BEpi &ep, hipStream_t s) {
    const u32x4 *x4 = reinterpret_cast<const u32x4 *>(x);
    const dim3 block(NW * 64);
    if (n <= 16)
        hipLaunchKernelGGL((k_bgemm<RT, KT, NW, S, EPI, 1>), grid, block, 0, s, w, x4, ep);
    else if (n <= 32)
        hipLaunchKernelGGL((k_bgemm<RT, KT, NW, S, EPI, 2>), grid, block, 0, s, w, x4, ep);
    else if (n <= 48)
        hipLaunchKernelGGL((k_bgemm<RT, KT, NW, S, EPI, 3>), grid, block, 0, s, w, x4, ep);
    else
        hipLaunchKernelGGL((k_bgemm<RT, KT, NW, S, EPI, 4>), grid, block, 0, s, w, x4, ep);
}
void launch_lm_gemm(GDNBatchEngine *e, const BEpi &ep, const void *x, hipStream_t s) {
    const dim3 grid(lm_wgs(e));
    if (lm_rt(e) == 4) launch_bgemm<4, kKtH, 4, 1, EPI_LM>(ep.n_streams, grid, e->w_lm, x, ep, s);
    else launch_bgemm<2, kKtH, 4, 1, EPI_LM>(ep.n_streams, grid, e->w_lm, x, ep, s);
}

// Gate/up for n streams or tokens in `blocks` blocks of 64.
void launch_bgu(int n, int blocks, const u32x4 *w, const u32x4 *x, uint16_t *x_next, hipStream_t s) {
    const dim3 grid(kGuWgs, blocks), block(kGuWaves * 64);
    if (n <= 16) hipLaunchKernelGGL((k_bgu<kGuWaves, 1>), grid, block, 0, s, w, x, x_next, n);
    else if (n <= 32) hipLaunchKernelGGL((k_bgu<kGuWaves, 2>), grid, block, 0, s, w, x, x_next, n);
    else if (n <= 48) hipLaunchKernelGGL((k_bgu<kGuWaves, 3>), grid, block, 0, s, w, x, x_next, n);
    else hipLaunchKernelGGL((k_bgu<kGuWaves, 4>), grid, block, 0, s, w, x, x_next, n);
}

int b_check_shape(const GDNWeightHeader *c) {
    if (c->hidden_size != (uint32_t)kH || c->num_heads != (uint32_t)kNH || c->num_v_heads != (uint32_t)kNH ||
        c->head_dim != (uint32_t)kHD || c->intermediate_size != (uint32_t)kI || c->conv_size != 4u) {
        gdn_error("gdn: the engine is specialised for hidden 2048, 8x256 heads, intermediate 5632, conv 4");
        return -1;
    }
    if (c->num_layers < 1 || c->num_layers > (uint32_t)kMaxLayers) {
        gdn_error("gdn: num_layers must be 1..24");
        return -1;
    }
    if (c->vocab_size == 0 || (c->vocab_size % 32) != 0) {
        gdn_error("gdn: the multi-stream engine needs a vocabulary that is a multiple of 32");
        return -1;
    }
    return 0;
}

// BF16 bits (subnormals flushed) of n BF16-exact floats.
void to_bf16(const float *src, size_t n, std::vector<uint16_t> &dst) {
    dst.resize(n);
    float mn, mx;
    int bad;
    gdn_pack_bf16_daz(src, dst.data(), n, &mn, &mx, &bad);
}

int upload_tiled(const std::vector<uint16_t> &rows, size_t n_rows, size_t k, int rt, char *&p,
                 const u32x4 *&out) {
    std::vector<uint16_t> tiled(n_rows * k);
    gdn_tile_bf16(rows.data(), n_rows, k, rt, tiled.data());
    GDN_HIP(hipMemcpy(p, tiled.data(), tiled.size() * 2, hipMemcpyHostToDevice));
    out = reinterpret_cast<const u32x4 *>(p);
    p += tiled.size() * 2;
    return 0;
}

// Gate [kI][kH] and up [kI][kH] BF16 rows in k_bgu's layout: per workgroup b
// and k tile, gate rows 22 b .. + 15 and up rows 22 b .. + 15 as A-operand
// tiles, then the 12-row tile (gate rows 22 b + 16 .. + 21, up rows likewise)
// as (quarter, row) entries.
void tile_gu(const uint16_t *g, const uint16_t *u, uint16_t *dst) {
    const size_t K = kH;
#pragma omp parallel for schedule(static)
    for (int b = 0; b < kGuWgs; ++b)
        for (int kt = 0; kt < kKtH; ++kt) {
            uint16_t *tile = dst + ((size_t)b * kKtH + kt) * kGuTileU4 * 8;
            const size_t col = (size_t)kt * 32;
            for (int l = 0; l < 64; ++l) {
                const size_t ch = (size_t)b * kGuCh + l % 16, c8 = col + 8 * (l / 16);
                std::memcpy(tile + l * 8, g + ch * K + c8, 16);
                std::memcpy(tile + (64 + l) * 8, u + ch * K + c8, 16);
            }
            constexpr int kTail = kGuCh - 16;
            for (int kq = 0; kq < 4; ++kq)
                for (int r = 0; r < kGuTail2; ++r) {
                    const size_t ch = (size_t)b * kGuCh + 16 + (r % kTail);
                    std::memcpy(tile + (128 + kq * kGuTail2 + r) * 8, (r < kTail ? g : u) + ch * K + col + 8 * kq,
                                16);
                }
        }
}

int b_upload(GDNBatchEngine *e, const GDNModel *m) {
    const size_t H = kH, I = kI, V = (size_t)e->vocab, L = (size_t)e->layers;
    const size_t per_layer = 4 * H * H + H * H + 2 * I * H + H * I;
    GDN_HIP(hipMalloc(&e->wmem, (L * per_layer + V * H) * 2));
    char *p = static_cast<char *>(e->wmem);
    std::vector<uint16_t> rows, part;
    for (size_t l = 0; l < L; ++l) {
        const GDNLayerWeights &w = m->layers[l];
        rows.resize(4 * H * H);
        const float *src[4] = {w.q_proj, w.k_proj, w.v_proj, w.g_proj};
        for (int s = 0; s < 4; ++s) {
            to_bf16(src[s], H * H, part);
            std::memcpy(rows.data() + s * H * H, part.data(), H * H * 2);
        }
        if (upload_tiled(rows, 4 * H, H, 2, p, e->w_qkvg[l])) return -1;
        to_bf16(w.o_proj, H * H, rows);
        if (upload_tiled(rows, H, H, kRtO, p, e->w_o[l])) return -1;
        std::vector<uint16_t> g16, u16;
        to_bf16(w.mlp_gate_proj, I * H, g16);
        to_bf16(w.mlp_up_proj, I * H, u16);
        rows.resize(2 * I * H);
        tile_gu(g16.data(), u16.data(), rows.data());
        GDN_HIP(hipMemcpy(p, rows.data(), rows.size() * 2, hipMemcpyHostToDevice));
        e->w_gu[l] = reinterpret_cast<const u32x4 *>(p);
        p += rows.size() * 2;
        to_bf16(w.mlp_down_proj, H * I, rows);
        if (upload_tiled(rows, H, I, kRtDown, p, e->w_down[l])) return -1;
    }
    to_bf16(m->lm_head, V * H, rows);
    if (upload_tiled(rows, V, H, lm_rt(e), p, e->w_lm)) return -1;
    // embeddings keep their top 16 bits (the batch-1 engine's import)
    std::vector<uint16_t> emb(V * H);
    for (size_t i = 0; i < V * H; ++i) {
        uint32_t b;
        std::memcpy(&b, m->embeddings + i, 4);
        emb[i] = (uint16_t)(b >> 16);
    }
    GDN_HIP(hipMalloc(&e->emb, emb.size() * 2));
    GDN_HIP(hipMemcpy(e->emb, emb.data(), emb.size() * 2, hipMemcpyHostToDevice));

    std::vector<float> aux(L * kAuxLayer + H, 0.0f);
    for (size_t l = 0; l < L; ++l) {
        const GDNLayerWeights &w = m->layers[l];
        float *a = aux.data() + l * kAuxLayer;
        std::memcpy(a + kAuxAttnNorm, w.attn_norm, H * 4);
        std::memcpy(a + kAuxMlpNorm, w.mlp_norm, H * 4);
        std::memcpy(a + kAuxONorm, w.o_norm, kHD * 4);
        std::memcpy(a + kAuxALog, w.a_log, kNH * 4);
        std::memcpy(a + kAuxDtBias, w.dt_bias, kNH * 4);
        std::memcpy(a + kAuxAB, w.a_proj, kNH * H * 4);
        std::memcpy(a + kAuxAB + kNH * H, w.b_proj, kNH * H * 4);
        std::memcpy(a + kAuxConv, w.q_conv, H * 4 * 4);
        std::memcpy(a + kAuxConv + H * 4, w.k_conv, H * 4 * 4);
        std::memcpy(a + kAuxConv + 2 * H * 4, w.v_conv, H * 4 * 4);
    }
    std::memcpy(aux.data() + L * kAuxLayer, m->final_norm, H * 4);
    GDN_HIP(hipMalloc(&e->aux, aux.size() * 4));
    GDN_HIP(hipMemcpy(e->aux, aux.data(), aux.size() * 4, hipMemcpyHostToDevice));
    return 0;
}

int b_alloc(GDNBatchEngine *e) {
    const size_t L = (size_t)e->layers, B = (size_t)e->streams, V = (size_t)e->vocab;
    GDN_HIP(hipMalloc(&e->state, L * B * kLayerState * 4));
    GDN_HIP(hipMemset(e->state, 0, L * B * kLayerState * 4));
    GDN_HIP(hipMalloc(&e->tails, L * B * kStreamTails * 2));
    GDN_HIP(hipMemset(e->tails, 0, L * B * kStreamTails * 2));
    const size_t G = (size_t)lm_wgs(e);
    const size_t act = kMaxB * (2 * kH + 3 * kH + kH + kH + 16 + kH + kSplitDown * kH + kH + V) + G * kMaxB;
    GDN_HIP(hipMalloc(&e->act, act * 4));
    GDN_HIP(hipMemset(e->act, 0, act * 4));
    float *p = e->act;
    e->h = p; p += 2 * kMaxB * kH;  // residual ping-pong (layer parity)
    e->qkv = p; p += kMaxB * 3 * kH;
    e->gate = p; p += kMaxB * kH;
    e->sgate = p; p += kMaxB * kH;
    e->bd = p; p += kMaxB * 16;
    e->attn = p; p += kMaxB * kH;
    e->ypart = p; p += (size_t)kSplitDown * kMaxB * kH;
    e->xn = p; p += kMaxB * kH;
    e->logits = p; p += kMaxB * V;
    e->part_val = p; p += G * kMaxB;
    GDN_HIP(hipMalloc(&e->part_idx, G * kMaxB * sizeof(int)));
    // X tiles: streams beyond n_streams stay zero
    GDN_HIP(hipMalloc(&e->x_h, (size_t)kMaxB * kH * 2));
    GDN_HIP(hipMalloc(&e->x_o, (size_t)kMaxB * kH * 2));
    GDN_HIP(hipMalloc(&e->x_d, (size_t)kMaxB * kI * 2));
    GDN_HIP(hipMemset(e->x_h, 0, (size_t)kMaxB * kH * 2));
    GDN_HIP(hipMemset(e->x_o, 0, (size_t)kMaxB * kH * 2));
    GDN_HIP(hipMemset(e->x_d, 0, (size_t)kMaxB * kI * 2));
    GDN_HIP(hipMalloc(&e->p_logits, (size_t)kMaxB * V * 4));
    GDN_HIP(hipMalloc(&e->p_tok, (size_t)kMaxB * sizeof(int)));
    // a step reads its tokens from and writes its argmaxes to host memory
    // directly
    GDN_HIP(hipHostMalloc(&e->tok_host, 2 * kMaxB * sizeof(int), hipHostMallocMapped | hipHostMallocCoherent));
    std::memset(e->tok_host, 0, 2 * kMaxB * sizeof(int));
    GDN_HIP(hipHostGetDevicePointer(reinterpret_cast<void **>(&e->tok_map), e->tok_host, 0));
    GDN_HIP(hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking));
    GDN_HIP(hipEventCreate(&e->ev0));
    GDN_HIP(hipEventCreate(&e->ev1));
    GDN_HIP(hipDeviceSynchronize());
    return 0;
}

// The residual entering layer l's attention block lives in buffer l & 1: the
// MLP norm updates it in place and the split a/b norm after the down
// projection writes the next layer's buffer.
float *b_resid(GDNBatchEngine *e, int l) { return e->h + (size_t)(l & 1) * kMaxB * kH; }

BNorm bnorm(GDNBatchEngine *e, const float *y, const float *w, uint16_t *x_out, int ab_layer, int l_in,
            int l_out) {
    BNorm p{};
    p.h_in = b_resid(e, l_in);
    p.h_out = b_resid(e, l_out);
    p.y = y;
    p.y_rows = kMaxB;
    p.w = w;
    p.x_out = x_out;
    p.eps = e->eps;
    if (ab_layer >= 0) {
        float *a = b_aux(e, ab_layer);
        p.ab_w = a + kAuxAB;
        p.a_log = a + kAuxALog;
        p.dt_bias = a + kAuxDtBias;
        p.bd = e->bd;
    }
    return p;
}

// Kernel kinds of gdn_batch_profile_kernels, in output order.
enum { KB_EMBED, KB_QKVG, KB_RECUR, KB_ONORM, KB_O, KB_NORM, KB_GU, KB_DOWN, KB_LM, KB_ARGMAX, KB_KINDS };

void launch_embed(GDNBatchEngine *e, hipStream_t s) {
    BNorm p = bnorm(e, nullptr, b_aux(e, 0) + kAuxAttnNorm, e->x_h, 0, 0, 0);
    p.emb = e->emb;
    p.tok = e->tok_map;
    hipLaunchKernelGGL((k_bnorm<0, true, true>), dim3(e->streams, kAbSplit), dim3(kT), 0, s, p);
}
void launch_qkvg(GDNBatchEngine *e, int l, hipStream_t s) {
    BEpi ep{};
    ep.n_streams = e->streams;
    ep.n_rows = 4 * kH;
    ep.qkv = e->qkv;
    ep.gate = e->gate;
    ep.sgate = e->sgate;
    ep.tails = b_tails(e, l);
    ep.conv_w = b_aux(e, l) + kAuxConv;
    launch_bgemm<2, kKtH, 8, 1, EPI_QKVG>(e->streams, dim3(4 * kH / 32), e->w_qkvg[l], e->x_h, ep, s);
}
void launch_recur(GDNBatchEngine *e, int l, hipStream_t s) {
    hipLaunchKernelGGL(k_brecur, dim3(kNH * (kHD / kRecCols), e->streams), dim3(kT), 0, s, e->qkv, e->bd,
                       b_state(e, l), e->attn);
}
void launch_onorm(GDNBatchEngine *e, int l, hipStream_t s) {
    hipLaunchKernelGGL((k_bonorm<1, false>), dim3(kNH, e->streams), dim3(kT), 0, s, e->attn, e->gate, e->sgate,
                       b_aux(e, l) + kAuxONorm, e->eps, e->x_o, e->streams);
}
void launch_o(GDNBatchEngine *e, int l, hipStream_t s) {
    BEpi ep{};
    ep.n_streams = e->streams;
    ep.n_rows = kH;
    ep.y = e->ypart;
    ep.y_rows = kMaxB;
    launch_bgemm<kRtO, kKtH, 4, kSplitO, EPI_RAW>(e->streams, dim3(kH / (16 * kRtO), kSplitO), e->w_o[l], e->x_o, ep, s);
}
void launch_mlp_norm(GDNBatchEngine *e, int l, hipStream_t s) {
    const BNorm p = bnorm(e, e->ypart, b_aux(e, l) + kAuxMlpNorm, e->x_h, -1, l, l);
    hipLaunchKernelGGL((k_bnorm<kSplitO, false, false>), dim3(e->streams), dim3(kT), 0, s, p);
}
void launch_gu(GDNBatchEngine *e, int l, hipStream_t s) {
    launch_bgu(e->streams, 1, e->w_gu[l], reinterpret_cast<const u32x4 *>(e->x_h), e->x_d, s);
}
void launch_down(GDNBatchEngine *e, int l, hipStream_t s) {
    BEpi ep{};
    ep.n_streams = e->streams;
    ep.n_rows = kH;
    ep.y = e->ypart;
    ep.y_rows = kMaxB;
    launch_bgemm<kRtDown, kKtI, 4, kSplitDown, EPI_RAW>(e->streams, dim3(kH / (16 * kRtDown), kSplitDown),
                                                        e->w_down[l], e->x_d, ep, s);
}
// After layer l's down projection: h = R(h + y), then the next layer's
// attention norm with its a/b rows, or the final norm.
void launch_layer_norm(GDNBatchEngine *e, int l, hipStream_t s) {
    if (l + 1 < e->layers) {
        const BNorm p = bnorm(e, e->ypart, b_aux(e, l + 1) + kAuxAttnNorm, e->x_h, l + 1, l, l + 1);
        hipLaunchKernelGGL((k_bnorm<kSplitDown, false, true>), dim3(e->streams, kAbSplit), dim3(kT), 0, s, p);
    } else {
        BNorm p = bnorm(e, e->ypart, e->aux + (size_t)e->layers * kAuxLayer, e->x_h, -1, l, l);
        p.xn_out = e->xn;
        hipLaunchKernelGGL((k_bnorm<kSplitDown, false, false>), dim3(e->streams), dim3(kT), 0, s, p);
    }
}
void launch_lm(GDNBatchEngine *e, hipStream_t s) {
    BEpi ep{};
    ep.n_streams = e->streams;
    ep.n_rows = e->vocab;
    ep.logits = e->logits;
    ep.part_val = e->part_val;
    ep.part_idx = e->part_idx;
    launch_lm_gemm(e, ep, e->x_h, s);
}
void launch_argmax(GDNBatchEngine *e, hipStream_t s) {
    hipLaunchKernelGGL(k_bargmax, dim3(e->streams), dim3(kT), 0, s, e->part_val, e->part_idx, lm_wgs(e),
                       e->tok_map + kMaxB);
}

void b_enqueue_step(GDNBatchEngine *e, hipStream_t s) {
    launch_embed(e, s);
    for (int l = 0; l < e->layers; ++l) {
        launch_qkvg(e, l, s);
        launch_recur(e, l, s);
        launch_onorm(e, l, s);
        launch_o(e, l, s);
        launch_mlp_norm(e, l, s);
        launch_gu(e, l, s);
        launch_down(e, l, s);
        launch_layer_norm(e, l, s);
    }
    launch_lm(e, s);
    launch_argmax(e, s);
}

int b_ensure_graph(GDNBatchEngine *e) {
    if (e->exec) return 0;
    GDN_HIP(hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal));
    b_enqueue_step(e, e->stream);
    GDN_HIP(hipStreamEndCapture(e->stream, &e->graph));
    GDN_HIP(hipGraphInstantiate(&e->exec, e->graph, nullptr, nullptr, 0));
    return 0;
}

// tokens[n_streams] in (host) -> step -> next tokens out (host).
int b_run_step(GDNBatchEngine *e, const int32_t *tokens, int32_t *next, float *inner_ms) {
    for (int i = 0; i < e->streams; ++i) {
        if (tokens[i] < 0 || tokens[i] >= e->vocab) {
            gdn_error("token id out of range");
            return -1;
        }
    }
    if (e->use_graph && b_ensure_graph(e) != 0) return -1;
    std::memcpy(e->tok_host, tokens, (size_t)e->streams * sizeof(int));  // read through tok_map
    if (inner_ms) GDN_HIP(hipEventRecord(e->ev0, e->stream));
    if (e->use_graph) {
        GDN_HIP(hipGraphLaunch(e->exec, e->stream));
    } else {
        b_enqueue_step(e, e->stream);
        GDN_HIP(hipGetLastError());
    }
    if (inner_ms) GDN_HIP(hipEventRecord(e->ev1, e->stream));
    GDN_HIP(hipStreamSynchronize(e->stream));  // k_bargmax wrote tok_host[kMaxB..]
    if (next) std::memcpy(next, e->tok_host + kMaxB, (size_t)e->streams * sizeof(int));
    if (inner_ms) GDN_HIP(hipEventElapsedTime(inner_ms, e->ev0, e->ev1));
    return 0;
}

// Prefill segment buffers for e->seg_tokens tokens (kept while the segment
// length stays).
int seg_alloc(GDNBatchEngine *e) {
    if (e->seg_cap == e->seg_tokens && e->seg_mem) return 0;
    GDN_HIP(hipStreamSynchronize(e->stream));
    (void)hipFree(e->seg_mem);
    e->seg_mem = nullptr;
    e->seg_cap = 0;
    const size_t T = (size_t)e->seg_tokens, chunks = T / kMaxB;
    const size_t TG = std::min(T, (size_t)kStepTok);  // longer ones leave the gate in s_y
    // normalised q and k (scan) or k_wy_seq's operands (chunked)
    const size_t qk = std::max(T * 2 * kH, chunks * kNH * sizeof(WyOps) / sizeof(float));
    const size_t floats = T * (2 * kH + 4 * kH + 3 * kH + 16 + kH + kNH + kH) + TG * 2 * kH + qk;
    const size_t halves = T * (kH + kH + kI);
    const size_t bytes = floats * 4 + halves * 2 + T * sizeof(int);
    GDN_HIP(hipMalloc(&e->seg_mem, bytes));
    // X tiles of padded tokens are read by the GEMMs (their sums unused):
    // start them at zero, on the engine's stream (a plain hipMemset may
    // return before it completes, and the non-blocking stream would not
    // wait for it)
    GDN_HIP(hipMemsetAsync(e->seg_mem, 0, bytes, e->stream));
    float *p = static_cast<float *>(e->seg_mem);
    e->s_h = p; p += 2 * T * kH;
    e->s_y = p; p += 4 * T * kH;
    e->s_qkv = p; p += 3 * T * kH;
    e->s_gate = p; p += TG * kH;
    e->s_sgate = p; p += TG * kH;
    e->s_bd = p; p += T * 16;
    e->s_attn = p; p += T * kH;
    e->s_qn = p;
    e->s_kn = p + T * kH;
    e->s_wy = reinterpret_cast<WyOps *>(p);
    p += qk;
    e->s_alpha = p; p += T * kNH;
    e->s_xn = p; p += T * kH;
    uint16_t *q = reinterpret_cast<uint16_t *>(p);
    e->s_xh = q; q += T * kH;
    e->s_xo = q; q += T * kH;
    e->s_xd = q; q += T * kI;
    e->s_tok = reinterpret_cast<int *>(q);
    e->seg_cap = e->seg_tokens;
    return 0;
}

// A segment's norm: the residual of layer l's attention block in buffer
// l & 1 (as in the step), segment-sized.
BNorm seg_norm(GDNBatchEngine *e, const float *y, const float *w, uint16_t *x_out, int ab_layer, int l_in,
               int l_out) {
    BNorm p{};
    p.h_in = e->s_h + (size_t)(l_in & 1) * e->seg_cap * kH;
    p.h_out = e->s_h + (size_t)(l_out & 1) * e->seg_cap * kH;
    p.y = y;
    p.y_rows = e->seg_cap;
    p.w = w;
    p.x_out = x_out;
    p.eps = e->eps;
    if (ab_layer >= 0) {
        float *a = b_aux(e, ab_layer);
        p.ab_w = a + kAuxAB;
        p.a_log = a + kAuxALog;
        p.dt_bias = a + kAuxDtBias;
        p.bd = e->s_bd;
    }
    return p;
}

// The prefill's projections over n tokens (X in 64-token tile blocks, padded
// to whole 128-token tiles), by a rule on n; every choice forms the same sums.
enum PRoute {
    P_STEP,        // the decode step's kernels, a grid plane per 64-token block
    P_TILE,        // k_pgemm / k_pgu, 128 tokens per workgroup (q/k/v/g, gate/up)
    P_PLANES,      // k_pgemm with a workgroup per split (o_proj, down)
    P_WIDE,        // k_pgemm_a / k_pgu_a, 256 rows x 128 tokens per workgroup
    P_WIDE_PLANES  // k_pgemm_a with a workgroup per split (down)
};
// Where the lines lie, us per launch with the weights in cache, the stores as
// the engine takes them (the step's kernels re-read the weights per 64 tokens;
// the others leave CUs idle on short segments).  At 64 tokens, in a prefill:
// q/k/v/g step 12, tile 30; o_proj 5 / planes 11; down 9 / 20; gate/up 15 / 30.
//   tokens         256 384 512 640 768 896 1024 1152 1280 1408 1536 2048 2560 3072 4096
//   q/k/v/g  step   27  39  51  62  74  84   96  107  118  129  141  186    -    -    -
//            tile   25  27  28  43  44  45   47   63   64   66   67   87  110  131  173
//            wide   27  28  31  31  33  34   35   57   56   59   60   65   92   98  141
//   o_proj   step    9  12  15  19  22  25   28   32   35   37   40   53    -    -    -
//            planes 11  12  14  18  19  19   20   26   27   27   28   35   43   49   63
//            wide   30  31  31  32  32  32   32   33   34   34   34   36   37   39   41
//   down     step   17  24  31  36  43  50   57   62   69   76   83  110    -    -    -
//            planes 21  23  25  34  35  36   38   51   52   54   55   68   85   98  127
//       wide planes 21  23  25  26  27  28   29   45   46   47   49   53   75   77   97
//            wide   67  67  68  69  70  70   70   71   72   72   73   76   79   82   88
//   gate/up  step   29  41  54  66  78  91  103  116  128  140  152  202    -    -    -
//            tile   31  44  46  64  68  83   86  102  105  121  124  162  199  237  313
//            wide   40  40  41  42  70  75   78   76   78   79  108  115  150  182  222
// The lines were drawn from fewer sizes than these; what the table would move
// (wide for q/k/v/g from 640 tokens and gate/up at 896, wide planes for down at
// 1025 to 1280) is 5 to 12 us a launch.  A norm behind four planes costs more
// than behind one sum: 8.3 against 6.8 us at 512 tokens, 12.6 / 9.7 at 1024,
// 19 / 13 at 1536, 25 / 18 at 2048, 30 / 21 at 2560, 37 / 24 at 3072.
int p_tiles(int n) { return (n + kPgTok - 1) / kPgTok; }
bool pa_fills(int rows, int n) { return rows % kPaRows == 0 && (rows / kPaRows) * p_tiles(n) >= 256; }
PRoute route_qkvg(int rows, int n) { return n <= kStepTok ? P_STEP : pa_fills(rows, n) ? P_WIDE : P_TILE; }
PRoute route_o(int n) { return n <= 256 ? P_STEP : n <= 1536 ? P_PLANES : P_WIDE; }
// down's wide planes take whole rounds of 256 workgroups (eight tiles, about
// 26 us), its planes about 4.4 us a tile and 4.
PRoute route_down(int n) {
    if (n <= 256) return P_STEP;
    if (n > 2560) return P_WIDE;
    return 65 * ((p_tiles(n) + 7) / 8) <= 11 * p_tiles(n) + 10 ? P_WIDE_PLANES : P_PLANES;
}
// k_pgu_a takes whole rounds of 256 workgroups (one per CU, 44 per 128 tokens),
// about 37 us each; k_pgu (two per CU) about 8.5 us per 128 tokens and 14.
bool pgu_a_pays(int n) {
    const int rounds = (2 * kI / kPaRows * p_tiles(n) + 255) / 256;
    return 76 * rounds <= 17 * p_tiles(n) + 22;
}
PRoute route_gu(int n) { return n <= 192 ? P_STEP : pgu_a_pays(n) ? P_WIDE : P_TILE; }

// A projection in 32-row blocks of KT k tiles, NW classes and S splits:
// returns the planes of y (y_rows tokens each) that its consumer adds: S, or
// 1 (the total).  P_WIDE and P_TILE write rounded sums as BF16 bits with B16
// (without, the test of the sums reads them whole); the others FP32.
template <int KT, int NW, int S, bool B16>
int launch_p_gemm(PRoute route, const u32x4 *w, const u32x4 *x, float *y, int rows, int n, int y_rows,
                  hipStream_t s) {
    const int blocks = (n + kMaxB - 1) / kMaxB, tiles = p_tiles(n);
    if (route == P_STEP) {
        BEpi ep{};
        ep.n_streams = kMaxB;
        ep.n_rows = rows;
        ep.y = y;
        ep.y_rows = y_rows;
        launch_bgemm<2, KT, NW, S, EPI_RAW>(n, dim3(rows / 32, S, blocks), w, x, ep, s);
        return S;
    }
    if (route == P_WIDE) {
        hipLaunchKernelGGL((k_pgemm_a<KT, NW, S, false, B16>), dim3(rows / kPaRows, tiles), dim3(kPaW * 64), 0, s, w, x, y,
                           rows, 0);
        return 1;
    }
    if constexpr (S > 1) {
        if constexpr (KT == kKtI) {
            if (route == P_WIDE_PLANES) {
                hipLaunchKernelGGL((k_pgemm_a<KT, NW, S, true, false>), dim3(rows / kPaRows, tiles, S),
                                   dim3(kPaW * 64), 0, s, w, x, y, rows, y_rows);
                return S;
            }
        }
        hipLaunchKernelGGL((k_pgemm<KT, NW, S, true, false>), dim3(rows / 128, tiles, S), dim3(kPgW * 64), 0, s, w, x,
                           y, rows, y_rows);
        return S;
    } else {
        hipLaunchKernelGGL((k_pgemm<KT, NW, 1, false, B16>), dim3(rows / 128, tiles), dim3(kPgW * 64), 0, s, w, x, y, rows,
                           0);
        return 1;
    }
}
static_assert(kRtO == 2 && kRtDown == 2, "o_proj and down in 32-row blocks");

// Gate/up on the step's layout.
void launch_p_gu(PRoute route, const u32x4 *w, const u32x4 *x, uint16_t *x_next, int n, hipStream_t s) {
    const int tiles = (n + kPgTok - 1) / kPgTok;
    if (route == P_STEP)
        launch_bgu(n, (n + kMaxB - 1) / kMaxB, w, x, x_next, s);
    else if (route == P_WIDE)
        hipLaunchKernelGGL(k_pgu_a, dim3(2 * kI / kPaRows, tiles), dim3(kPaW * 64), 0, s, w, x, x_next, n);
    else
        hipLaunchKernelGGL(k_pgu, dim3(kGuWgs / 2, tiles), dim3(kPgW * 64), 0, s, w, x, x_next, n);
}

// The residual add and norm after o_proj or down.
void launch_p_norm(const BNorm &p, int planes, int n, hipStream_t s) {
    static_assert(kSplitO == kSplitDown, "one norm kernel for both");
    if (planes == 1)
        hipLaunchKernelGGL((k_bnorm<1, false, false>), dim3(n), dim3(kT), 0, s, p);
    else
        hipLaunchKernelGGL((k_bnorm<kSplitO, false, false>), dim3(n), dim3(kT), 0, s, p);
}

// One prefill segment of n tokens (already in s_tok[0..n)) through stream
// `slot`'s state, layer by layer: the step's kernels with the tokens as the
// streams (the projections by route, k_bnorm + k_pab in place of the split
// a/b norm; same sums), the conv across the segment (k_pconv), and the
// recurrence over all its tokens: in token order (k_pqk, k_pscan) or in the WY
// form (k_wy_prep over every 64-token chunk at once, then k_wy_seq over the
// chunks in order).
void enqueue_prefill_segment(GDNBatchEngine *e, int slot, int n, bool last, hipStream_t s) {
    const int blocks = (n + kMaxB - 1) / kMaxB;
    const int pab_blocks = (n + kPabTok - 1) / kPabTok;
    // a norm's a/b rows and beta/decay, from its normalised copy in s_xn
    auto launch_ab = [&](int l_ab) {
        const float *a = b_aux(e, l_ab);
        hipLaunchKernelGGL(k_pab, dim3(kAbSplit, pab_blocks), dim3(kT), 0, s, e->s_xn, n, a + kAuxAB, a + kAuxALog,
                           a + kAuxDtBias, e->s_bd);
    };
    BNorm p0 = seg_norm(e, nullptr, b_aux(e, 0) + kAuxAttnNorm, e->s_xh, -1, 0, 0);
    p0.emb = e->emb;
    p0.tok = e->s_tok;
    p0.xn_out = e->s_xn;
    hipLaunchKernelGGL((k_bnorm<0, true, false>), dim3(n), dim3(kT), 0, s, p0);
    launch_ab(0);
    const u32x4 *xh = reinterpret_cast<const u32x4 *>(e->s_xh), *xo = reinterpret_cast<const u32x4 *>(e->s_xo),
                *xd = reinterpret_cast<const u32x4 *>(e->s_xd);
    const PRoute r_qkvg = route_qkvg(4 * kH, n);
    for (int l = 0; l < e->layers; ++l) {
        float *st = b_state(e, l) + (size_t)slot * kLayerState;
        uint16_t *tl = b_tails(e, l) + (size_t)slot * kStreamTails;
        launch_p_gemm<kKtH, 8, 1, true>(r_qkvg, e->w_qkvg[l], xh, e->s_y, 4 * kH, n, e->seg_cap, s);
        hipLaunchKernelGGL(r_qkvg == P_STEP ? k_pconv<false> : k_pconv<true>,
                           dim3((r_qkvg == P_STEP ? 4 : 3) * kH / 64, blocks), dim3(kConvT), 0, s, e->s_y, n, tl, b_aux(e, l) + kAuxConv, e->s_qkv, e->s_gate, e->s_sgate);
        if (e->prefill_mode == GDN_PREFILL_CHUNKED) {
            hipLaunchKernelGGL(k_wy_prep, dim3(kNH, blocks), dim3(kT), 0, s, e->s_qkv, e->s_bd, n, e->s_wy);
            hipLaunchKernelGGL(k_wy_seq, dim3(kNH * (kHD / kWyCols)), dim3(kWyWaves * 64), 0, s, e->s_qkv, e->s_wy, n, st,
                               e->s_attn);
        } else {
            hipLaunchKernelGGL(k_pqk, dim3(kNH, (n + kQkTok - 1) / kQkTok), dim3(kT), 0, s, e->s_qkv, n, e->s_qn,
                               e->s_kn, e->s_alpha);
            hipLaunchKernelGGL(k_pscan, dim3(kHD / kScanWgCols, kNH), dim3(kT), 0, s, e->s_qkv, e->s_qn, e->s_kn,
                               e->s_alpha, e->s_bd, n, st, e->s_attn);
        }
        const bool raw = r_qkvg != P_STEP;
        hipLaunchKernelGGL((raw ? k_bonorm<kOnTok, true> : k_bonorm<kOnTok, false>),
                           dim3(kNH, (n + kOnTok - 1) / kOnTok), dim3(kT), 0, s, e->s_attn,
                           raw ? e->s_y : e->s_gate, e->s_sgate, b_aux(e, l) + kAuxONorm, e->eps, e->s_xo, n);
        const int po = launch_p_gemm<kKtH, 4, kSplitO, true>(route_o(n), e->w_o[l], xo, e->s_y, kH, n, e->seg_cap, s);
        launch_p_norm(seg_norm(e, e->s_y, b_aux(e, l) + kAuxMlpNorm, e->s_xh, -1, l, l), po, n, s);
        launch_p_gu(route_gu(n), e->w_gu[l], xh, e->s_xd, n, s);
        const int pd =
            launch_p_gemm<kKtI, 4, kSplitDown, true>(route_down(n), e->w_down[l], xd, e->s_y, kH, n, e->seg_cap, s);
        if (l + 1 < e->layers) {
            BNorm pa = seg_norm(e, e->s_y, b_aux(e, l + 1) + kAuxAttnNorm, e->s_xh, -1, l, l + 1);
            pa.xn_out = e->s_xn;
            launch_p_norm(pa, pd, n, s);
            launch_ab(l + 1);
        } else {
            BNorm pf = seg_norm(e, e->s_y, e->aux + (size_t)e->layers * kAuxLayer, e->s_xh, -1, l, l);
            pf.xn_out = e->s_xn;
            launch_p_norm(pf, pd, n, s);
        }
    }
    if (!last) return;
    // the LM head over the last token block
    const int lb = blocks - 1, nl = n - lb * kMaxB;
    BEpi lm{};
    lm.n_streams = nl;
    lm.n_rows = e->vocab;
    lm.logits = e->p_logits;
    lm.part_val = e->part_val;
    lm.part_idx = e->part_idx;
    launch_lm_gemm(e, lm, e->s_xh + (size_t)lb * kMaxB * kH, s);
    hipLaunchKernelGGL(k_bargmax, dim3(nl), dim3(kT), 0, s, e->part_val, e->part_idx, lm_wgs(e), e->p_tok);
}

int b_prefill(GDNBatchEngine *e, int slot, const int32_t *prompt, uint32_t n_tokens, int32_t *seed) {
    for (uint32_t i = 0; i < n_tokens; ++i) {
        if (prompt[i] < 0 || prompt[i] >= e->vocab) {
            gdn_error("token id out of range");
            return -1;
        }
    }
    if (seg_alloc(e)) return -1;
    const uint32_t seg = (uint32_t)e->seg_cap;
    int n = 0;
    for (uint32_t off = 0; off < n_tokens; off += seg) {
        n = (int)std::min<uint32_t>(seg, n_tokens - off);
        GDN_HIP(hipMemcpyAsync(e->s_tok, prompt + off, (size_t)n * sizeof(int), hipMemcpyHostToDevice, e->stream));
        enqueue_prefill_segment(e, slot, n, off + (uint32_t)n == n_tokens, e->stream);
        GDN_HIP(hipGetLastError());
    }
    // the last position's logits, final hidden vector and token into the
    // stream's rows of the step buffers
    const int nl = n - ((n - 1) / kMaxB) * kMaxB;
    GDN_HIP(hipMemcpyAsync(e->logits + (size_t)slot * e->vocab, e->p_logits + (size_t)(nl - 1) * e->vocab,
                           (size_t)e->vocab * 4, hipMemcpyDeviceToDevice, e->stream));
    GDN_HIP(hipMemcpyAsync(e->xn + (size_t)slot * kH, e->s_xn + (size_t)(n - 1) * kH, (size_t)kH * 4,
                           hipMemcpyDeviceToDevice, e->stream));
    GDN_HIP(hipMemcpyAsync(e->tok_host + kMaxB + slot, e->p_tok + (nl - 1), sizeof(int), hipMemcpyDeviceToHost,
                           e->stream));
    GDN_HIP(hipStreamSynchronize(e->stream));
    if (seed) *seed = e->tok_host[kMaxB + slot];
    return 0;
}

void b_destroy(GDNBatchEngine *e) {
    if (!e) return;
    if (e->exec) (void)hipGraphExecDestroy(e->exec);
    if (e->graph) (void)hipGraphDestroy(e->graph);
    if (e->ev0) (void)hipEventDestroy(e->ev0);
    if (e->ev1) (void)hipEventDestroy(e->ev1);
    if (e->stream) (void)hipStreamDestroy(e->stream);
    (void)hipFree(e->wmem);
    (void)hipFree(e->emb);
    (void)hipFree(e->aux);
    (void)hipFree(e->state);
    (void)hipFree(e->tails);
    (void)hipFree(e->act);
    (void)hipFree(e->part_idx);
    (void)hipFree(e->x_h);
    (void)hipFree(e->x_o);
    (void)hipFree(e->x_d);
    (void)hipFree(e->p_logits);
    (void)hipFree(e->p_tok);
    (void)hipFree(e->seg_mem);
    if (e->tok_host) (void)hipHostFree(e->tok_host);
    delete e;
}

GDNBatchEngine *engine_of(const GDNBatchState *s) {
    if (!s || !s->engine) gdn_error("gdn: multi-stream state not initialised");
    return s ? s->engine : nullptr;
}

// Copy between one stream's [layers][per] block and the strided device array.
int stream_copy(float *dev, size_t per, int streams, int layers, uint32_t stream, float *host, bool to_dev) {
    const size_t width = per * 4, dpitch = (size_t)streams * per * 4;
    float *d = dev + (size_t)stream * per;
    if (to_dev)
        GDN_HIP(hipMemcpy2D(d, dpitch, host, width, width, (size_t)layers, hipMemcpyHostToDevice));
    else
        GDN_HIP(hipMemcpy2D(host, width, d, dpitch, width, (size_t)layers, hipMemcpyDeviceToHost));
    return 0;
}

// The conv tails of one stream: FP32 words on the host (the .gdnstate
// section layout), BF16 bits on the device.  Loading requires BF16-exact
// values, as the reference's head buffer does.
int tails_copy(uint16_t *dev, int streams, int layers, uint32_t stream, float *host, bool to_dev) {
    const size_t n = (size_t)layers * kStreamTails;
    std::vector<uint16_t> bits(n);
    const size_t width = kStreamTails * 2, dpitch = (size_t)streams * kStreamTails * 2;
    uint16_t *d = dev + (size_t)stream * kStreamTails;
    if (to_dev) {
        const size_t bad = gdn_first_non_bf16(host, n);
        if (bad != n) {
            gdn_report_non_bf16("multi-stream conv tail", host, bad);
            return -1;
        }
        for (size_t i = 0; i < n; ++i) {
            uint32_t u;
            std::memcpy(&u, host + i, 4);
            bits[i] = (uint16_t)(u >> 16);
        }
        GDN_HIP(hipMemcpy2D(d, dpitch, bits.data(), width, width, (size_t)layers, hipMemcpyHostToDevice));
    } else {
        GDN_HIP(hipMemcpy2D(bits.data(), width, d, dpitch, width, (size_t)layers, hipMemcpyDeviceToHost));
        for (size_t i = 0; i < n; ++i) {
            const uint32_t u = (uint32_t)bits[i] << 16;
            std::memcpy(host + i, &u, 4);
        }
    }
    return 0;
}

}  // namespace

// ================================================================== C ABI

extern "C" {

int gdn_batch_init(GDNBatchState *state, const GDNModel *model, uint32_t n_streams) {
    std::memset(state, 0, sizeof(*state));
    if (n_streams == 0 || n_streams > (uint32_t)kMaxB) {
        gdn_error("gdn: n_streams must be 1..64");
        return -1;
    }
    if (b_check_shape(&model->config) != 0) return -1;
    if (gdn_validate_bf16_exact_weights(model->weight_data, &model->config) != 0) {
        gdn_error("gdn: the multi-stream engine needs a BF16-exact checkpoint");
        return -1;
    }
    GDNBatchEngine *e = new GDNBatchEngine();
    e->layers = (int)model->config.num_layers;
    e->vocab = (int)model->config.vocab_size;
    e->streams = (int)n_streams;
    e->eps = model->config.norm_eps;
    if (b_alloc(e) != 0 || b_upload(e, model) != 0) {
        b_destroy(e);
        return -1;
    }
    state->engine = e;
    state->n_streams = n_streams;
    return 0;
}

void gdn_batch_free(GDNBatchState *state) {
    b_destroy(state->engine);
    std::memset(state, 0, sizeof(*state));
}

int gdn_batch_set_graph_mode(GDNBatchState *state, int use_graph) {
    GDNBatchEngine *e = engine_of(state);
    if (!e) return -1;
    e->use_graph = use_graph != 0;
    return 0;
}

int gdn_batch_decode_step(GDNBatchState *state, const int32_t *tokens, int32_t *next_tokens) {
    GDNBatchEngine *e = engine_of(state);
    if (!e) return -1;
    if (tokens == nullptr || next_tokens == nullptr) {
        gdn_error("gdn_batch_decode_step: tokens and next_tokens are required");
        return -1;
    }
    return b_run_step(e, tokens, next_tokens, nullptr);
}

int gdn_batch_read_tokens(const GDNBatchState *state, int32_t *tokens) {
    GDNBatchEngine *e = engine_of(state);
    if (!e) return -1;
    GDN_HIP(hipStreamSynchronize(e->stream));
    std::memcpy(tokens, e->tok_host + kMaxB, (size_t)e->streams * sizeof(int));
    return 0;
}

int gdn_batch_read_logits(const GDNBatchState *state, uint32_t stream, float *logits, size_t count) {
    GDNBatchEngine *e = engine_of(state);
    if (!e || stream >= (uint32_t)e->streams || count > (size_t)e->vocab) return -1;
    GDN_HIP(hipMemcpy(logits, e->logits + (size_t)stream * e->vocab, count * 4, hipMemcpyDeviceToHost));
    return 0;
}

int gdn_batch_read_final_hidden(const GDNBatchState *state, uint32_t stream, float *hidden, size_t count) {
    GDNBatchEngine *e = engine_of(state);
    if (!e || stream >= (uint32_t)e->streams || count > (size_t)kH) return -1;
    GDN_HIP(hipMemcpy(hidden, e->xn + (size_t)stream * kH, count * 4, hipMemcpyDeviceToHost));
    return 0;
}

int gdn_batch_load_stream_state(GDNBatchState *state, uint32_t stream, const float *recurrent,
                                size_t recurrent_floats, const float *conv_tails, size_t conv_floats) {
    GDNBatchEngine *e = engine_of(state);
    if (!e || stream >= (uint32_t)e->streams) return -1;
    if (recurrent && recurrent_floats != (size_t)e->layers * kLayerState) return -1;
    if (conv_tails && conv_floats != (size_t)e->layers * kStreamTails) return -1;
    // the tails first: they are checked (BF16-exact) before anything is written
    if (conv_tails && tails_copy(e->tails, e->streams, e->layers, stream, const_cast<float *>(conv_tails), true))
        return -1;
    if (recurrent && stream_copy(e->state, kLayerState, e->streams, e->layers, stream,
                                 const_cast<float *>(recurrent), true))
        return -1;
    return 0;
}

int gdn_batch_save_stream_state(const GDNBatchState *state, uint32_t stream, float *recurrent,
                                size_t recurrent_floats, float *conv_tails, size_t conv_floats) {
    GDNBatchEngine *e = engine_of(state);
    if (!e || stream >= (uint32_t)e->streams) return -1;
    if (recurrent && recurrent_floats != (size_t)e->layers * kLayerState) return -1;
    if (conv_tails && conv_floats != (size_t)e->layers * kStreamTails) return -1;
    if (recurrent && stream_copy(e->state, kLayerState, e->streams, e->layers, stream, recurrent, false)) return -1;
    if (conv_tails && tails_copy(e->tails, e->streams, e->layers, stream, conv_tails, false)) return -1;
    return 0;
}

int gdn_batch_set_prefill_mode(GDNBatchState *state, int mode) {
    GDNBatchEngine *e = engine_of(state);
    if (!e || (mode != GDN_PREFILL_SCAN && mode != GDN_PREFILL_CHUNKED)) return -1;
    e->prefill_mode = mode;
    return 0;
}

int gdn_batch_set_prefill_segment(GDNBatchState *state, uint32_t tokens) {
    GDNBatchEngine *e = engine_of(state);
    if (!e) return -1;
    if (tokens < (uint32_t)kPgTok || tokens > (uint32_t)kSegMax || tokens % kPgTok != 0) {
        gdn_error("gdn: a prefill segment is a multiple of 128 tokens, 128..32768");
        return -1;
    }
    e->seg_tokens = (int)tokens;
    return 0;
}

int gdn_batch_prefill(GDNBatchState *state, uint32_t stream, const int32_t *prompt, uint32_t n_tokens,
                      int32_t *seed_token) {
    GDNBatchEngine *e = engine_of(state);
    if (!e || stream >= (uint32_t)e->streams || n_tokens == 0 || !prompt) return -1;
    return b_prefill(e, (int)stream, prompt, n_tokens, seed_token);
}

int gdn_batch_run_teacher_forced(GDNBatchState *state, const int32_t *tokens, uint32_t n_steps,
                                 int32_t *argmax_out, float *inner_ms, float *outer_ms) {
    GDNBatchEngine *e = engine_of(state);
    if (!e) return -1;
    if (tokens == nullptr && n_steps > 0) {
        gdn_error("gdn_batch_run_teacher_forced: no tokens");
        return -1;
    }
    const size_t B = (size_t)e->streams;
    std::vector<int32_t> next(B);
    for (uint32_t i = 0; i < n_steps; ++i) {
        const auto t0 = std::chrono::steady_clock::now();
        if (b_run_step(e, tokens + (size_t)i * B, next.data(), inner_ms ? inner_ms + i : nullptr) != 0) return -1;
        const auto t1 = std::chrono::steady_clock::now();
        if (outer_ms) outer_ms[i] = std::chrono::duration<float, std::milli>(t1 - t0).count();
        if (argmax_out) std::memcpy(argmax_out + (size_t)i * B, next.data(), B * sizeof(int32_t));
    }
    return 0;
}

int gdn_batch_profile_kernels(GDNBatchState *state, uint32_t rounds, float *avg_us, uint32_t n_kinds) {
    GDNBatchEngine *e = engine_of(state);
    if (!e) return -1;
    for (uint32_t id = 0; id < n_kinds && id < (uint32_t)KB_KINDS; ++id) {
        GDN_HIP(hipStreamSynchronize(e->stream));
        GDN_HIP(hipEventRecord(e->ev0, e->stream));
        uint32_t launches = 0;
        for (uint32_t r = 0; r < rounds; ++r) {
            const int per_layer = (id == KB_EMBED || id == KB_LM || id == KB_ARGMAX) ? 1 : e->layers;
            for (int l = 0; l < per_layer; ++l, ++launches) {
                switch (id) {
                case KB_EMBED: launch_embed(e, e->stream); break;
                case KB_QKVG: launch_qkvg(e, l, e->stream); break;
                case KB_RECUR: launch_recur(e, l, e->stream); break;
                case KB_ONORM: launch_onorm(e, l, e->stream); break;
                case KB_O: launch_o(e, l, e->stream); break;
                case KB_NORM: launch_layer_norm(e, l, e->stream); break;
                case KB_GU: launch_gu(e, l, e->stream); break;
                case KB_DOWN: launch_down(e, l, e->stream); break;
                case KB_LM: launch_lm(e, e->stream); break;
                default: launch_argmax(e, e->stream); break;
                }
            }
        }
        GDN_HIP(hipEventRecord(e->ev1, e->stream));
        GDN_HIP(hipEventSynchronize(e->ev1));
        GDN_HIP(hipGetLastError());
        float ms = 0.0f;
        GDN_HIP(hipEventElapsedTime(&ms, e->ev0, e->ev1));
        avg_us[id] = launches ? 1000.0f * ms / (float)launches : 0.0f;
    }
    return 0;
}

int gdn_test_batch_gemm(const float *W, const float *X, uint32_t N, uint32_t K, float *Y) {
    const bool k_hidden = K == (uint32_t)kH;
    const uint32_t rows = 16u * (uint32_t)(k_hidden ? kRtO : kRtDown);  // rows per workgroup
    if (!(k_hidden || K == (uint32_t)kI) || N == 0 || (N % rows) != 0) {
        gdn_error("gdn_test_batch_gemm: K must be 2048 or 5632 and N a multiple of the workgroup's rows");
        return -1;
    }
    // the production configurations: o_proj's for K = 2048, down's for 5632
    const int splits = k_hidden ? kSplitO : kSplitDown;
    std::vector<uint16_t> wb, wt((size_t)N * K), xb;
    to_bf16(W, (size_t)N * K, wb);
    gdn_tile_bf16(wb.data(), N, K, k_hidden ? kRtO : kRtDown, wt.data());
    // X [64][K] in B-operand tiles: the A tiling of 64 rows in 4 row tiles
    to_bf16(X, (size_t)kMaxB * K, xb);
    std::vector<uint16_t> xt((size_t)kMaxB * K);
    gdn_tile_bf16(xb.data(), kMaxB, K, 4, xt.data());
    void *dw = nullptr, *dx = nullptr;
    float *dy = nullptr;
    GDN_HIP(hipMalloc(&dw, wt.size() * 2));
    GDN_HIP(hipMalloc(&dx, xt.size() * 2));
    GDN_HIP(hipMalloc(&dy, (size_t)splits * kMaxB * N * 4));
    GDN_HIP(hipMemcpy(dw, wt.data(), wt.size() * 2, hipMemcpyHostToDevice));
    GDN_HIP(hipMemcpy(dx, xt.data(), xt.size() * 2, hipMemcpyHostToDevice));
    BEpi ep{};
    ep.n_streams = kMaxB;
    ep.n_rows = (int)N;
    ep.y = dy;
    ep.y_rows = kMaxB;
    if (k_hidden)
        hipLaunchKernelGGL((k_bgemm<kRtO, kKtH, 4, kSplitO, EPI_RAW>), dim3(N / rows, kSplitO), dim3(kT), 0, 0,
                           static_cast<const u32x4 *>(dw), static_cast<const u32x4 *>(dx), ep);
    else
        hipLaunchKernelGGL((k_bgemm<kRtDown, kKtI, 4, kSplitDown, EPI_RAW>), dim3(N / rows, kSplitDown), dim3(kT),
                           0, 0, static_cast<const u32x4 *>(dw), static_cast<const u32x4 *>(dx), ep);
    GDN_HIP(hipGetLastError());
    std::vector<float> parts((size_t)splits * kMaxB * N);
    GDN_HIP(hipMemcpy(parts.data(), dy, parts.size() * 4, hipMemcpyDeviceToHost));
    // split sums in split order, as the consumers add them
    for (size_t i = 0; i < (size_t)kMaxB * N; ++i) {
        float v = parts[i];
        for (int sp = 1; sp < splits; ++sp) v = v + parts[(size_t)sp * kMaxB * N + i];
        Y[i] = v;
    }
    (void)hipFree(dw);
    (void)hipFree(dx);
    (void)hipFree(dy);
    return 0;
}

int gdn_test_prefill_gemm(int kind, const float *W, const float *X, uint32_t N, uint32_t T, float *Y,
                          float *Y_step) {
    // kind 0: q/k/v/g configuration (K 2048, 8 classes); 1: o_proj (K 2048,
    // 4 classes, 4 splits); 2: down (K 5632, 4 classes, 4 splits); 3:
    // gate/up + SwiGLU (W = gate then up rows, N = 5632)
    if (kind < 0 || kind > 3 || T == 0 || T > (uint32_t)kSegMax || N == 0 ||
        (kind < 3 && (N % 128) != 0) || (kind == 3 && N != (uint32_t)kI)) {
        gdn_error("gdn_test_prefill_gemm: kind 0..3, N a multiple of 128 (5632 for gate/up), T 1..32768");
        return -1;
    }
    const uint32_t K = kind == 2 ? (uint32_t)kI : (uint32_t)kH;
    const uint32_t blocks = (T + kMaxB - 1) / kMaxB, tp = (T + kPgTok - 1) / kPgTok * kPgTok;
    const size_t wn = (kind == 3 ? 2 : 1) * (size_t)N * K;
    std::vector<uint16_t> wb, wt(wn), xb, xt((size_t)tp * K, 0);
    to_bf16(W, wn, wb);
    if (kind == 3) tile_gu(wb.data(), wb.data() + (size_t)N * K, wt.data());
    else gdn_tile_bf16(wb.data(), N, K, 2, wt.data());
    std::vector<float> xpad((size_t)blocks * kMaxB * K, 0.0f);
    std::memcpy(xpad.data(), X, (size_t)T * K * 4);
    to_bf16(xpad.data(), xpad.size(), xb);
    for (uint32_t b = 0; b < blocks; ++b)
        gdn_tile_bf16(xb.data() + (size_t)b * kMaxB * K, kMaxB, K, 4, xt.data() + (size_t)b * kMaxB * K);
    const size_t out_elems = kind == 3 ? (size_t)tp * kI : (size_t)kSplitDown * tp * N;
    void *dw = nullptr, *dx = nullptr, *dy = nullptr, *dr = nullptr;
    GDN_HIP(hipMalloc(&dw, wt.size() * 2));
    GDN_HIP(hipMalloc(&dx, xt.size() * 2));
    GDN_HIP(hipMalloc(&dy, out_elems * 4));
    GDN_HIP(hipMalloc(&dr, out_elems * 4));
    GDN_HIP(hipMemset(dr, 0, out_elems * 4));
    GDN_HIP(hipMemcpy(dw, wt.data(), wt.size() * 2, hipMemcpyHostToDevice));
    GDN_HIP(hipMemcpy(dx, xt.data(), xt.size() * 2, hipMemcpyHostToDevice));
    const u32x4 *w4 = static_cast<const u32x4 *>(dw), *x4 = static_cast<const u32x4 *>(dx);
    // one route into out (floats of a zeroed buffer's planes added in order,
    // or the X tiles' halves)
    const int rows = (int)N, toks = (int)T, pad = (int)tp;
    auto launch_route = [&](PRoute route, auto b16) {
        constexpr bool B16 = decltype(b16)::value;
        float *y = static_cast<float *>(dy);
        if (kind == 0) return launch_p_gemm<kKtH, 8, 1, B16>(route, w4, x4, y, rows, toks, pad, nullptr);
        if (kind == 1) return launch_p_gemm<kKtH, 4, kSplitO, B16>(route, w4, x4, y, rows, toks, pad, nullptr);
        return launch_p_gemm<kKtI, 4, kSplitDown, B16>(route, w4, x4, y, rows, toks, pad, nullptr);
    };
    auto run_route = [&](PRoute route, std::vector<float> &out, std::vector<uint16_t> &tiles16) -> int {
        GDN_HIP(hipMemset(dy, 0, out_elems * 4));
        int planes = 1;
        if (kind < 3)
            planes = launch_route(route, std::false_type{});
        else
            launch_p_gu(route, w4, x4, static_cast<uint16_t *>(dy), toks, nullptr);
        GDN_HIP(hipGetLastError());
        GDN_HIP(hipDeviceSynchronize());
        if (kind == 3) {
            tiles16.resize((size_t)tp * kI);
            GDN_HIP(hipMemcpy(tiles16.data(), dy, tiles16.size() * 2, hipMemcpyDeviceToHost));
            return 0;
        }
        std::vector<float> a(out_elems);
        GDN_HIP(hipMemcpy(a.data(), dy, a.size() * 4, hipMemcpyDeviceToHost));
        out.resize((size_t)T * N);
        for (size_t i = 0; i < out.size(); ++i) {
            float v = a[i];
            for (int sp = 1; sp < planes; ++sp) v = v + a[(size_t)sp * tp * N + i];
            out[i] = v;
        }
        return 0;
    };
    // the 128-token kernels give the result; every other kernel that a
    // segment of some length runs on has to agree with it bit for bit
    std::vector<PRoute> routes = {P_STEP, kind == 1 || kind == 2 ? P_PLANES : P_TILE};
    const bool wide = kind == 3 || N % kPaRows == 0;
    if (wide) routes.insert(routes.begin(), P_WIDE);
    else std::swap(routes[0], routes[1]);
    if (wide && kind == 2) routes.push_back(P_WIDE_PLANES);
    std::vector<float> first, other;
    std::vector<uint16_t> first16, other16;
    if (run_route(routes[0], first, first16)) return -1;
    for (size_t r = 1; r < routes.size(); ++r) {
        if (run_route(routes[r], other, other16)) return -1;
        const size_t bytes = kind == 3 ? first16.size() * 2 : first.size() * 4;
        if (std::memcmp(kind == 3 ? (const void *)first16.data() : first.data(),
                        kind == 3 ? (const void *)other16.data() : other.data(), bytes) != 0) {
            std::fprintf(stderr, "gdn_test_prefill_gemm: kind %d, route %d differs from route %d\n", kind,
                         (int)routes[r], (int)routes[0]);
            return -1;
        }
    }
    // the stores of rounded sums, as the engine launches these routes: the
    // rounding of the whole sums
    for (PRoute route : {P_WIDE, P_TILE}) {
        if (kind == 3 || (route == P_WIDE && !wide) || (route == P_TILE && kind != 0)) continue;
        GDN_HIP(hipMemset(dy, 0, out_elems * 4));
        launch_route(route, std::true_type{});
        GDN_HIP(hipGetLastError());
        GDN_HIP(hipDeviceSynchronize());
        std::vector<uint16_t> half((size_t)T * N);
        GDN_HIP(hipMemcpy(half.data(), dy, half.size() * 2, hipMemcpyDeviceToHost));
        for (size_t i = 0; i < half.size(); ++i) {
            uint32_t u;
            std::memcpy(&u, &first[i], 4);
            if (half[i] != (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16)) {
                std::fprintf(stderr, "gdn_test_prefill_gemm: kind %d, route %d: a rounded sum differs\n", kind,
                             (int)route);
                return -1;
            }
        }
    }
    // the step's kernels, one 64-token block at a time
    for (uint32_t b = 0; b < blocks; ++b) {
        const u32x4 *xb4 = x4 + (size_t)b * kMaxB * K / 8;
        BEpi ep{};
        ep.n_streams = kMaxB;
        ep.n_rows = (int)N;
        ep.y = static_cast<float *>(dr) + (size_t)b * kSplitDown * kMaxB * N;
        ep.y_rows = kMaxB;
        if (kind == 0)
            hipLaunchKernelGGL((k_bgemm<2, kKtH, 8, 1, EPI_RAW>), dim3(N / 32), dim3(8 * 64), 0, 0, w4, xb4, ep);
        if (kind == 1)
            hipLaunchKernelGGL((k_bgemm<kRtO, kKtH, 4, kSplitO, EPI_RAW>), dim3(N / 32, kSplitO), dim3(kT), 0, 0,
                               w4, xb4, ep);
        if (kind == 2)
            hipLaunchKernelGGL((k_bgemm<kRtDown, kKtI, 4, kSplitDown, EPI_RAW>), dim3(N / 32, kSplitDown),
                               dim3(kT), 0, 0, w4, xb4, ep);
        if (kind == 3)
            hipLaunchKernelGGL((k_bgu<kGuWaves>), dim3(kGuWgs), dim3(kGuWaves * 64), 0, 0, w4, xb4,
                               static_cast<uint16_t *>(dr) + (size_t)b * kMaxB * kI, kMaxB);
    }
    GDN_HIP(hipGetLastError());
    GDN_HIP(hipDeviceSynchronize());
    if (kind == 3) {
        // both outputs are X tiles of width kI: untile the first T tokens
        std::vector<uint16_t> &a = first16, r((size_t)tp * kI);
        GDN_HIP(hipMemcpy(r.data(), dr, r.size() * 2, hipMemcpyDeviceToHost));
        for (uint32_t m = 0; m < T; ++m)
            for (uint32_t k = 0; k < (uint32_t)kI; ++k) {
                const uint32_t kt = k >> 5, kk = k & 31, mm = m & 63;
                const size_t idx = (size_t)(m >> 6) * 64 * kI +
                                   (size_t)((((kt * 4 + (mm >> 4)) * 64 + ((kk >> 3) << 4) + (mm & 15)) << 3) + (kk & 7));
                const uint32_t ya = (uint32_t)a[idx] << 16, yr = (uint32_t)r[idx] << 16;
                std::memcpy(Y + (size_t)m * kI + k, &ya, 4);
                std::memcpy(Y_step + (size_t)m * kI + k, &yr, 4);
            }
    } else {
        std::vector<float> r(out_elems);
        GDN_HIP(hipMemcpy(r.data(), dr, r.size() * 4, hipMemcpyDeviceToHost));
        const int splits = kind == 0 ? 1 : kSplitDown;
        for (uint32_t m = 0; m < T; ++m)
            for (uint32_t n = 0; n < N; ++n) {
                const size_t base = (size_t)(m / kMaxB) * kSplitDown * kMaxB * N + (size_t)(m % kMaxB) * N + n;
                float v = r[base];
                for (int sp = 1; sp < splits; ++sp) v = v + r[base + (size_t)sp * kMaxB * N];
                Y[(size_t)m * N + n] = first[(size_t)m * N + n];
                Y_step[(size_t)m * N + n] = v;
            }
    }
    (void)hipFree(dw);
    (void)hipFree(dx);
    (void)hipFree(dy);
    (void)hipFree(dr);
    return 0;
}

}  // extern "C"
