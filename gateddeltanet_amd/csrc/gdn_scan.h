// gdn_scan.h -- the gated delta rule over many tokens in order, the state
// held in registers from the first token to the last: the prefill's scan
// (gdn_batch.hip) and the allocation-free recurrence (gdn_noalloc.hip).
// Not part of the ABI.
#ifndef GDN_SCAN_H
#define GDN_SCAN_H

#include "gdn_device.h"

namespace gdn {

// A chain of 256 dependent adds in the order j = 0..255 over a row of 16
// lanes, lane i holding its elements 16 i .. 16 i + 15 in p.  Every lane adds
// its own sixteen to what its left neighbour had; after pass s lanes 0..s
// hold sums of the true chain (lane s the one through element 16 s + 15), so
// lane 15 ends with the whole.  The adds take registers of their own lane:
// sixteen cross-lane moves in all, where a chain that fetched every operand
// from its lane would need one per add (an add through DPP of the chain's
// own accumulator waits two states).
__device__ __forceinline__ float chain256(const float (&p)[16]) {
    float acc = 0.0f;
#pragma unroll
    for (int s = 0; s < 16; ++s) {
        if (s) acc = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(acc), 0x111, 0xf, 0xf, true));
#pragma unroll
        for (int e = 0; e < 16; ++e) acc = acc + p[e];
    }
    return acc;
}

// From the chains' sums in lane 15 of the rows (r in rows 0 and 2, p in the
// row after it): delta in every lane of the column's two rows, and o in lane
// 15 of its p row.  (row_newbcast:15 spreads a row's lane 15 over the row,
// row_bcast:15 over the next row.)
__device__ __forceinline__ void scan_delta_o(float acc, float beta, float decay, float alpha, float v, float &delta,
                                             float &o) {
    const float d = beta * (v - decay * acc);
    const int dr = __builtin_amdgcn_update_dpp(0, __float_as_int(d), 0x15f, 0xf, 0xf, true);
    delta = __int_as_float(__builtin_amdgcn_update_dpp(dr, __float_as_int(d), 0x142, 0xa, 0xf, false));
    o = 0.0625f * (decay * acc + alpha * delta);
}

// The scan.  A workgroup is four independent waves (one per SIMD), a wave
// two state columns, and each of the wave's four 16-lane rows one 256-add
// chain of the reference's order: row 2 c + 0 sums r of column c (S^T k),
// row 2 c + 1 its p (S^T q).  Lane i of a row holds state rows 16 i .. + 15
// of its column in registers, both rows of a column the same values, so the
// products never pass through LDS.
//
// What bounds it: a wave64 FP32 add occupies its SIMD for 4 cycles, so the
// 256 adds a bit-equal chain needs are 1024 of the token's cycles whatever
// the layout; 8 heads x 256 columns x 2 chains fill the 1024 SIMDs exactly
// once at four chains per wave.  A 4096-token launch takes 3.06 ms (0.75 us a
// token); with every product written to LDS and four lanes of a wave reading
// the chains' operands back it took 4.44 ms (1.08 us).
//
// k, q, v and the per-token scalars are staged kScanTok tokens at a time in
// two LDS buffers, the next chunk's loads in flight while the current
// chunk's tokens run; one barrier per chunk.  A row's 4-value groups are
// stored so that the sixteen lanes' reads of a group are consecutive.
constexpr int kScanTok = 16;  // tokens staged per chunk (two buffers: 66 KB)
constexpr int kScanWgCols = 8;  // 4 waves x 2 columns

// Where a scan's operands are.  Per token m: k, q at + m * ldq (256 values),
// v at + m * ldv (this workgroup's columns first), o at + m * ldo, the
// scalars through `scal` (beta, decay, alpha).  NORM: k and q are raw and
// are multiplied by the token's 1/|k|, 1/|q| as they are staged (the same
// product the prefill's k_pqk stores).
struct ScanArgs {
    const float *k, *q, *v;
    float *o;
    size_t ldq, ldv, ldo;
    int n;
};

struct ScanLds {
    f32x4 kq[2][kScanTok][2][kHD / 4];  // [buffer][token][k|q][16 (g % 4) + g / 4 of 4-row group g]
    f32x4 sc[2][kScanTok];              // beta, decay, alpha
    float v[2][kScanTok][kScanWgCols];
};

// S: the workgroup's first state column of row 0, rows kHD apart (FP32, or
// BF16 bits for C == kRef, rounded after every token as the reference does).
template <int C, bool NORM, class Scal>
__device__ __forceinline__ void scan_block(const ScanArgs a, const Scal scal, void *state, ScanLds &lds) {
    static_assert(kT == 256 && kScanTok * kScanWgCols <= 128, "thread tasks below");
    constexpr int KQ = kScanTok / 2;  // staged 16-byte pieces per thread and chunk
    const int t = threadIdx.x, w = t >> 6, lane = t & 63, row = lane >> 4, i16 = lane & 15;
    const int lc = 2 * w + (row >> 1);  // this lane's column of the workgroup
    const int kind = row & 1;           // 0: r (with k), 1: p (with q)
    const int chunks = (a.n + kScanTok - 1) / kScanTok;

    // staging tasks: piece (t >> 7) + 2 j of a chunk is token, this thread's
    // k|q and 4-row group; threads 0..15 hold a token's scalars, 128..255 one
    // v each.  A token past the end re-reads the last one, unused.
    const int skind = (t >> 6) & 1, sg = t & 63;
    const float *src = (skind ? a.q : a.k) + 4 * sg;
    f32x4 kq[KQ], sc;
    float vv = 0.0f, inv[KQ];
    auto token = [&](int c, int m) { return kScanTok * c + m < a.n ? kScanTok * c + m : a.n - 1; };
    auto load_chunk = [&](int c) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < KQ; ++j) {
            const int m = token(c, (t >> 7) + 2 * j);
            kq[j] = *reinterpret_cast<const f32x4 *>(src + (size_t)m * a.ldq);
            if constexpr (NORM) inv[j] = scal.inv(m, skind);
        }
        if (t < kScanTok) sc = scal.get(token(c, t));
        if (t >= 128) {
            const int m = (t - 128) / kScanWgCols, col = (t - 128) % kScanWgCols;
            vv = a.v[(size_t)token(c, m) * a.ldv + col];
        }
    };
    auto store_chunk = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < KQ; ++j) {
            f32x4 x = kq[j];
            if constexpr (NORM) x = (f32x4){x.x * inv[j], x.y * inv[j], x.z * inv[j], x.w * inv[j]};
            lds.kq[b][(t >> 7) + 2 * j][skind][16 * (sg & 3) + (sg >> 2)] = x;
        }
        if (t < kScanTok) lds.sc[b][t] = sc;
        if (t >= 128) lds.v[b][(t - 128) / kScanWgCols][(t - 128) % kScanWgCols] = vv;
    };

    load_chunk(0);
    // rows 16 i16 .. + 15 of column lc
    float sv[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const size_t at = (size_t)(16 * i16 + i) * kHD + lc;
        if constexpr (C == kRef) sv[i] = bf16_bits_to_f32(static_cast<const uint16_t *>(state)[at]);
        else sv[i] = static_cast<const float *>(state)[at];
    }
    store_chunk(0);
    // the state waited for here: a wait inside the token loop would also wait
    // for the next chunk's loads, at each chunk's first token
#pragma unroll
    for (int i = 0; i < 16; ++i) asm volatile("" : "+v"(sv[i]));
    __syncthreads();

    f32x4 mul[4], kn[4];  // the next token's k or q; the current token's k
    auto read_mul = [&](int b, int m) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) mul[i] = lds.kq[b][m][kind][16 * i + i16];
    };
    for (int c = 0; c < chunks; ++c) {
        const int b = c & 1, n = a.n - kScanTok * c < kScanTok ? a.n - kScanTok * c : kScanTok;
        if (c + 1 < chunks) load_chunk(c + 1);
        float oacc = 0.0f;
        read_mul(b, 0);
#pragma unroll 1
        for (int m = 0; m < n; ++m) {
            float p[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) p[i] = sv[i] * mul[i >> 2][i & 3];
            // read under the chain: what the rest of this token needs, and
            // the next token's factors
            const float v = lds.v[b][m][lc];
#pragma unroll
            for (int i = 0; i < 4; ++i) kn[i] = lds.kq[b][m][0][16 * i + i16];
            const f32x4 scl = lds.sc[b][m];
            const float beta = scl.x, decay = scl.y, alpha = scl.z;
            read_mul(b, m + 1 < n ? m + 1 : m);
            __builtin_amdgcn_sched_barrier(0);
            const float acc = chain256(p);  // lane 15 of the row
            float delta, o;
            scan_delta_o(acc, beta, decay, alpha, v, delta, o);
            // lane m of a p row keeps token m's o
            const float ob = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(o), 0x15f, 0xf, 0xf, true));
            oacc = i16 == m ? ob : oacc;
            float nv[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) nv[i] = decay * sv[i] + kn[i >> 2][i & 3] * delta;
            if constexpr (C == kRef) {
                // BF16 rounding in pairs; a NaN or infinity anywhere in the
                // lane takes the integer rounding (canonical NaN)
                float mag = 0.0f;
                bool odd = false;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    odd |= nv[i] != nv[i];
                    mag = fmaxf(mag, fabsf(nv[i]));
                }
                if (odd || !(mag <= 3.402823466e38f)) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) sv[i] = rne_bf16(nv[i]);
                } else {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const uint32_t pk = cvt_pk(nv[2 * i], nv[2 * i + 1]);
                        sv[2 * i] = u2f(pk << 16);
                        sv[2 * i + 1] = u2f(pk & 0xffff0000u);
                    }
                }
            } else {
#pragma unroll
                for (int i = 0; i < 16; ++i) sv[i] = nv[i];
            }
            // used here, so that the reads stay ahead of the chain instead of
            // moving to the next token's products
#pragma unroll
            for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(mul[i]));
        }
        if (kind == 1 && i16 < n) a.o[(size_t)(kScanTok * c + i16) * a.ldo + lc] = R<C>(oacc);
        if (c + 1 < chunks) {
            // the other buffer was last read before the previous barrier
            store_chunk(b ^ 1);
            __syncthreads();
        }
    }
    if (kind == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const size_t at = (size_t)(16 * i16 + i) * kHD + lc;
            if constexpr (C == kRef) static_cast<uint16_t *>(state)[at] = bf16_hi(sv[i]);
            else static_cast<float *>(state)[at] = sv[i];
        }
    }
}

}  // namespace gdn

#endif
