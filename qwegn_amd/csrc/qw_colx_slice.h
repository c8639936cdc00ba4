// One 32-column slice of a bank row against a lane's activations, for every container: the pieces of the column-stationary
// GEMVs (gemv_colx.hip, moe_col.hip).  The arithmetic and the operand order are explained at the head of gemv_colx.hip.
#pragma once
#include "qwhip_common.h"

namespace {

// payload dwords of one 32-column slice: bits * 32 / 32 (HQ4_G32_M5 and 4-bit streams: 4)
template <int FMT>
struct qcx_fmt {
    static constexpr int BITS = FMT == QW_FMT_B8 ? 8 : (FMT == QW_FMT_B2 ? 2 : (FMT == QW_FMT_B3 ? 3 : (FMT == QW_FMT_B6 ? 6 : 4)));
    static constexpr int PW = BITS;
};

struct __attribute__((packed, aligned(4))) qcx_words4 { uint32_t q[4]; };
struct __attribute__((packed, aligned(4))) qcx_words8 { uint32_t q[8]; };

template <int FMT>
struct qcx_slice {
    uint32_t hdr;
    uint32_t q[qcx_fmt<FMT>::PW];
};

// The 16 operand pairs of one activation row for this lane's slice, in the order the masked code words come out.
// 3-bit streams: operand i pairs the elements (QCX_B3_LO[i], QCX_B3_HI[i]); operands 0..6 sit under the first mask
// (6 = codes 30, 31, cut out the plain way), 7..12 under the second, 13..15 under the third
__device__ constexpr int QCX_B3_LO[16] = {0, 3, 10, 13, 20, 23, 30, 1, 4, 11, 14, 21, 24, 2, 12, 22};
__device__ constexpr int QCX_B3_HI[16] = {5, 8, 15, 18, 25, 28, 31, 6, 9, 16, 19, 26, 29, 7, 17, 27};

// The fields of a masked 3- or 6-bit word sit at different places in its two halves: the low code of a 3-bit word reads twice the
// high one, the high code of a 6-bit word four times the low one, and the operands make up for it.  EXACT: they multiply (1x, 2x and
// 4x, 1x), which keeps every bit of an activation, subnormals too; one past 32,752 or 16,376 becomes infinite, shows in the sum
// returned, and is the caller's to see.  Not EXACT: they divide (1/2x, 1x and 1x, 1/4x); any activation passes, and those under
// 2^-13 or 2^-12 lose their last one or two bits (rows of magnitude 1e-5: 6e-3 and 1.3e-2 of the result, 1e-4: 5e-4 and 9e-4).
template <int FMT, bool EXACT>
struct qcx_scale {
    static constexpr float LO = FMT == QW_FMT_B3 ? (EXACT ? 1.0f : 0.5f) : FMT == QW_FMT_B6 ? (EXACT ? 4.0f : 1.0f) : 1.0f;
    static constexpr float HI = FMT == QW_FMT_B3 ? (EXACT ? 2.0f : 1.0f) : FMT == QW_FMT_B6 ? (EXACT ? 1.0f : 0.25f) : 1.0f;
    static constexpr float PLAIN = FMT == QW_FMT_B3 ? HI : LO;   // the operand of codes 30 and 31, cut out in step
    static constexpr float BACK = 16777216.0f / PLAIN;           // 2^24, the codes' place as f16 subnormals, over the scale
};

// 16 operand pairs of the lane's slice and the sum of its activations.
template <int FMT, bool EXACT>
__device__ __forceinline__ float qcx_operands(const h8_t* v, h2_t* xo) {
    const h2_t one = {(h1_t)1.0f, (h1_t)1.0f};
    float s0 = 0.f, s1 = 0.f;
    if constexpr (FMT == QW_FMT_B6 || FMT == QW_FMT_B3) {
        using sc = qcx_scale<FMT, EXACT>;
#pragma unroll
        for (int i = 0; i < 16; ++i) {   // 6-bit operand i: elements (e, e + 3), e = 6 (i / 3) + i % 3
            const bool plain = i == (FMT == QW_FMT_B6 ? 15 : 6);
            const int lo = FMT == QW_FMT_B3 ? QCX_B3_LO[i] : plain ? 30 : 6 * (i / 3) + i % 3;
            const int hi = FMT == QW_FMT_B3 ? QCX_B3_HI[i] : plain ? 31 : lo + 3;
            const float a = plain ? sc::PLAIN : sc::LO, b = plain ? sc::PLAIN : sc::HI;
            xo[i] = h2_t{v[lo >> 3][lo & 7] * (h1_t)a, v[hi >> 3][hi & 7] * (h1_t)b};
            if constexpr (EXACT) {
                const h2_t inv = {(h1_t)(1.0f / a), (h1_t)(1.0f / b)};
                if (i & 1) s1 = __builtin_amdgcn_fdot2(xo[i], inv, s1, false);
                else s0 = __builtin_amdgcn_fdot2(xo[i], inv, s0, false);
            }
        }
        if constexpr (!EXACT) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const h2_t nat = {v[j][2 * k], v[j][2 * k + 1]};
                    if (k & 1) s1 = __builtin_amdgcn_fdot2(nat, one, s1, false);
                    else s0 = __builtin_amdgcn_fdot2(nat, one, s0, false);
                }
            }
        }
        return s0 + s1;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            h2_t pr;
            if constexpr (FMT == QW_FMT_M5) pr = h2_t{v[j][2 * k], v[j][2 * k + 1]};
            else if constexpr (FMT == QW_FMT_B4) pr = h2_t{v[j][k], v[j][k + 4]};
            else if constexpr (FMT == QW_FMT_B2) pr = h2_t{v[2 * (j >> 1)][4 * (j & 1) + k], v[2 * (j >> 1) + 1][4 * (j & 1) + k]};
            else pr = h2_t{v[j][4 * (k >> 1) + (k & 1)], v[j][4 * (k >> 1) + (k & 1) + 2]};
            if (k & 1) s1 = __builtin_amdgcn_fdot2(pr, one, s1, false);
            else s0 = __builtin_amdgcn_fdot2(pr, one, s0, false);
            xo[4 * j + k] = pr;
        }
    }
    return s0 + s1;
}

// The slice whose header sits at byte o_hdr and whose code words at byte o_pay of `bank` (one 32-bit offset per address).
template <int FMT>
__device__ __forceinline__ void qcx_load(const uint8_t* bank, uint32_t o_hdr, uint32_t o_pay, qcx_slice<FMT>& b) {
    b.hdr = *(const uint32_t*)(bank + o_hdr);
    if constexpr (FMT == QW_FMT_B2 || FMT == QW_FMT_B3 || FMT == QW_FMT_B6) {
#pragma unroll
        for (int j = 0; j < qcx_fmt<FMT>::PW; ++j) b.q[j] = *(const uint32_t*)(bank + o_pay + 4 * j);
    } else if constexpr (FMT == QW_FMT_B8) {
        const qcx_words8 w = *(const qcx_words8*)(bank + o_pay);
#pragma unroll
        for (int j = 0; j < 8; ++j) b.q[j] = w.q[j];
    } else {
        const qcx_words4 w = *(const qcx_words4*)(bank + o_pay);
#pragma unroll
        for (int j = 0; j < 4; ++j) b.q[j] = w.q[j];
    }
}

// The slice's code words masked in place, in the order of qcx_operands.
template <int FMT>
__device__ __forceinline__ void qcx_mask(const qcx_slice<FMT>& b, uint32_t* ow) {
    if constexpr (FMT == QW_FMT_B6) {
        // window i at bit 6 e of the 192-bit slice, e = 6 (i / 3) + i % 3: code e at bits 0..5, code e + 3 at bits 18..23
        constexpr uint32_t M = 0x00FC003Fu;
#pragma unroll
        for (int i = 0; i < 15; ++i) {
            const int bit = 6 * (6 * (i / 3) + i % 3), wd = bit >> 5, sh = bit & 31;
            const uint32_t win = sh == 0 ? b.q[wd] : __builtin_amdgcn_alignbit(b.q[wd + 1], b.q[wd], sh);
            ow[i] = win & M;
        }
        ow[15] = ((b.q[5] >> 20) & 0x3Fu) | ((b.q[5] >> 10) & 0x003F0000u);   // codes 30 and 31
    } else if constexpr (FMT == QW_FMT_B3) {
        // windows of the 96-bit slice at bits -1, 8, 29, 38, 59, 68: low-half codes start at window bit 1, high-half
        // codes at bit 16 (elements: QCX_B3_LO / QCX_B3_HI)
        const uint32_t w0 = b.q[0], w1 = b.q[1], w2 = b.q[2];
        const uint32_t wa = w0 << 1;
        const uint32_t wb = __builtin_amdgcn_alignbit(w1, w0, 8);
        const uint32_t wc = __builtin_amdgcn_alignbit(w1, w0, 29);
        const uint32_t wd = __builtin_amdgcn_alignbit(w2, w1, 6);
        const uint32_t we = __builtin_amdgcn_alignbit(w2, w1, 27);
        const uint32_t wf = w2 >> 4;
        constexpr uint32_t M0 = 0x0007000Eu, M1 = 0x00380070u, M2 = 0x01C00380u;
        ow[0] = wa & M0;
        ow[1] = wb & M0;
        ow[2] = wc & M0;
        ow[3] = wd & M0;
        ow[4] = we & M0;
        ow[5] = wf & M0;
        ow[6] = ((w2 >> 26) & 7u) | ((w2 >> 13) & 0x00070000u);   // codes 30 and 31
        ow[7] = wa & M1;
        ow[8] = wb & M1;
        ow[9] = wc & M1;
        ow[10] = wd & M1;
        ow[11] = we & M1;
        ow[12] = wf & M1;
        ow[13] = wa & M2;
        ow[14] = wc & M2;
        ow[15] = we & M2;
    } else if constexpr (FMT == QW_FMT_B2) {
        // operand 8 w + j: elements (16 w + j, 16 w + j + 8), masked in place at bits 2 (j & 3) of the bytes 0 / 2 of the
        // word (j < 4) or of the word shifted down a byte (j >= 4)
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const uint32_t q = b.q[w], q8 = q >> 8;
            ow[8 * w + 0] = q & 0x00030003u;
            ow[8 * w + 1] = q & 0x000C000Cu;
            ow[8 * w + 2] = q & 0x00300030u;
            ow[8 * w + 3] = q & 0x00C000C0u;
            ow[8 * w + 4] = q8 & 0x00030003u;
            ow[8 * w + 5] = q8 & 0x000C000Cu;
            ow[8 * w + 6] = q8 & 0x00300030u;
            ow[8 * w + 7] = q8 & 0x00C000C0u;
        }
    } else if constexpr (FMT == QW_FMT_B8) {
#pragma unroll
        for (int w = 0; w < 8; ++w) {
            ow[2 * w] = b.q[w] & 0x00FF00FFu;
            ow[2 * w + 1] = (b.q[w] >> 8) & 0x00FF00FFu;
        }
    } else {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const uint32_t q = b.q[w], q8 = q >> 8;
            ow[4 * w + 0] = q & 0x000F000Fu;
            ow[4 * w + 1] = q & 0x00F000F0u;
            ow[4 * w + 2] = q8 & 0x000F000Fu;
            ow[4 * w + 3] = q8 & 0x00F000F0u;
        }
    }
}

// sum_i q_i x_i of a slice, on the operands of the same EXACT (HQ4_G32_M5: sum_i (1024 + q_i) x_i).
template <int FMT, bool EXACT>
__device__ __forceinline__ float qcx_code_dot(const uint32_t* ow, const h2_t* xo, float S) {
    float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
    if constexpr (FMT == QW_FMT_B3) {
        // a0, a1: the first mask's seven operands; a2: the second mask's six; a3: the third mask's three
#pragma unroll
        for (int i = 0; i < 7; ++i) {
            if (i & 1) a1 = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2_t, ow[i]), xo[i], a1, false);
            else a0 = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2_t, ow[i]), xo[i], a0, false);
        }
#pragma unroll
        for (int i = 7; i < 13; ++i) a2 = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2_t, ow[i]), xo[i], a2, false);
#pragma unroll
        for (int i = 13; i < 16; ++i) a3 = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2_t, ow[i]), xo[i], a3, false);
    } else {
#pragma unroll
        for (int i = 0; i < 16; i += 4) {
            a0 = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2_t, ow[i + 0]), xo[i + 0], a0, false);
            a1 = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2_t, ow[i + 1]), xo[i + 1], a1, false);
            a2 = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2_t, ow[i + 2]), xo[i + 2], a2, false);
            a3 = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2_t, ow[i + 3]), xo[i + 3], a3, false);
        }
    }
    float q;
    if constexpr (FMT == QW_FMT_B3) {
        constexpr float B = qcx_scale<FMT, EXACT>::BACK;
        q = __builtin_fmaf(a2, B * 0.125f, (a0 + a1) * B);   // fields at bits 4 / 3 of the halves: 8 q
        q = __builtin_fmaf(a3, B * 0.015625f, q);            // bits 7 / 6: 64 q
    } else if constexpr (FMT == QW_FMT_B8 || FMT == QW_FMT_B6) {
        q = ((a0 + a1) + (a2 + a3)) * qcx_scale<FMT, EXACT>::BACK;
    } else if constexpr (FMT == QW_FMT_B2) {
        q = __builtin_fmaf(a1, 4194304.0f, a0 * 16777216.0f);     // codes at bits 0..1 and 2..3 of a byte
        q = __builtin_fmaf(a2, 1048576.0f, q);                    // bits 4..5
        q = __builtin_fmaf(a3, 262144.0f, q);                     // bits 6..7
    } else {
        q = __builtin_fmaf(a0 + a2, 16777216.0f, FMT == QW_FMT_M5 ? 1024.0f * S : 0.0f);   // codes at bits 0..3
        q = __builtin_fmaf(a1 + a3, 1048576.0f, q);                                        // codes at bits 4..7
    }
    return q;
}

}  // namespace
