// A tile of 16 bank rows against fragments of 16 f16 activation rows, as the row-tile kernels take it (gemv_rows.hip has the whole,
// gemm_rows.hip and moe_rows.hip several fragments): a wave's LDS image of the slices, the codes as f16 operands, one step of 128 columns.
#pragma once
#include <type_traits>

#include "qwhip_common.h"
#include "qw_slice.h"

namespace {

template <int FMT>
constexpr uint32_t qr_code_bytes() { return 4u * (uint32_t)qg_slice_words<FMT>(); }

// The slices of a wave's 4 S slices x 16 bank rows in its part of LDS: code words [row][slice][word], headers [row][slice].  The row
// pitches put the 64 lanes of a read (16 rows x 4 words) on 64 banks, or next to it.
// The activations of one step pass through the same place: [row][16 pieces of 8 columns].
constexpr uint32_t QR_XS = 68;   // dwords between their rows
template <int FMT, int S>
struct qr_image {
    static constexpr uint32_t PW = (uint32_t)qg_slice_words<FMT>(), SL = 4u * S;
    static constexpr uint32_t RS = PW == 4u && S == 4 ? 84u : (SL * PW + 4u) | 4u, HS = SL + 4u;   // dwords; odd multiples of four
    static constexpr uint32_t DWORDS = 16u * (RS + HS) > 16u * QR_XS ? 16u * (RS + HS) : 16u * QR_XS;
};
template <int FMT, int S>
__device__ __forceinline__ void qr_park(uint32_t* img, uint32_t row, uint32_t b, const qg_slice<FMT>& s) {
    using im = qr_image<FMT, S>;
    uint32_t* w = img + row * im::RS + b * im::PW;
    if constexpr (im::PW % 4u == 0u) {
#pragma unroll
        for (uint32_t k = 0; k < im::PW; k += 4) *(u4_t*)(w + k) = u4_t{s.q[k], s.q[k + 1], s.q[k + 2], s.q[k + 3]};
    } else if constexpr (im::PW % 2u == 0u) {
#pragma unroll
        for (uint32_t k = 0; k < im::PW; k += 2) *(u2_t*)(w + k) = u2_t{s.q[k], s.q[k + 1]};
    } else {
#pragma unroll
        for (uint32_t k = 0; k < im::PW; ++k) w[k] = s.q[k];
    }
    img[16u * im::RS + row * im::HS + b] = s.hdr;
}
// Chunk c (8 codes) of slice sl of row n: one or two words, its first code at bit 0 (or where qr_codes says).
template <int FMT, int S>
__device__ __forceinline__ void qr_chunk(const uint32_t* img, uint32_t n, uint32_t sl, uint32_t c, uint32_t (&w)[2]) {
    using im = qr_image<FMT, S>;
    const uint32_t* row = img + n * im::RS + sl * im::PW;
    if constexpr (FMT == QG_FMT_B8) {
        const u2_t v = *(const u2_t*)(row + 2u * c);
        w[0] = v[0];
        w[1] = v[1];
    } else if constexpr (FMT == QG_FMT_B2) {
        w[0] = row[c >> 1] >> (16u * (c & 1u));
    } else if constexpr (FMT == QG_FMT_B3) {   // bits 24 c ..
        const uint32_t at = (24u * c) >> 5;
        w[0] = __builtin_amdgcn_alignbit(row[at + 1u], row[at], 24u * c);
    } else if constexpr (FMT == QG_FMT_B6) {   // bits 48 c ..: its low 24 bits (codes 0..3) and its high ones (4..7)
        const uint32_t at = 3u * (c >> 1) + (c & 1u), d0 = row[at], d1 = row[at + 1u], sh = 16u * (c & 1u);
        w[0] = __builtin_amdgcn_alignbit(d1, d0, sh);
        w[1] = __builtin_amdgcn_alignbit(d1 >> sh, w[0], 24);
    } else {
        w[0] = row[c];
    }
}
// The eight codes q of a chunk as f16 2^bits + q (8 bits: q), in the order of qr_x_order: the code is the top of the mantissa under that exponent
// (`base`, in a vector register), one shift and one and-or a pair.  (As f16 subnormals, code * 2^-24, the pairs cost an instruction less
// and the matrix unit drops the low bits of the products: 1e-6 of a slice's sum, and after b * sum(x), of the opposite sign, 1.6e-5 of the
// result.)  8-bit codes as they are, 1024 + q less 1024: the larger offset would cost a fifth in accuracy.
template <int FMT>
constexpr uint32_t qr_bits() { return FMT == QG_FMT_B8 ? 8u : FMT == QG_FMT_B6 ? 6u : FMT == QG_FMT_B3 ? 3u : FMT == QG_FMT_B2 ? 2u : 4u; }
template <int FMT>
constexpr uint32_t qr_base() { return FMT == QG_FMT_B8 ? 0x64006400u : (0x3C00u + (qr_bits<FMT>() << 10)) * 0x10001u; }
template <int FMT>   // w = scale * (what qr_codes gives) + (bias + QR_OFF * scale); HQ4_G32_M5: w = (1024 + q) s + b
constexpr float QR_OFF = FMT == QG_FMT_B8 ? 0.0f : (FMT == QG_FMT_M5 ? 1024.0f : 0.0f) - (float)(1u << qr_bits<FMT>());
template <int FMT, int FROM>   // the pair of codes at bits FROM and FROM + 16 of v
__device__ __forceinline__ uint32_t qr_pair(uint32_t v, uint32_t base) {
    constexpr int TO = 10 - (int)qr_bits<FMT>();
    constexpr uint32_t M = (((1u << qr_bits<FMT>()) - 1u) << TO) * 0x10001u;
    if constexpr (FROM < TO) return qw_and_or(v << (TO - FROM), M, base);
    else return qw_and_or(v >> (FROM - TO), M, base);
}
template <int FMT>
__device__ __forceinline__ h8_t qr_codes(const uint32_t (&w)[2], uint32_t base) {
    u4_t o;
    if constexpr (FMT == QG_FMT_B8) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const h2_t neg = {(h1_t)-1024.0f, (h1_t)-1024.0f};
            o[2 * h] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(w[h], w[h], 0x0C010C00u) | base) + neg);
            o[2 * h + 1] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(w[h], w[h], 0x0C030C02u) | base) + neg);
        }
    } else if constexpr (FMT == QG_FMT_B6) {
        const uint32_t a = (w[0] & 0xFFFu) | (w[1] << 16);                           // codes 0, 1 | 4, 5 (bits 28.. are not read)
        const uint32_t b = ((w[0] >> 12) & 0xFFFu) | ((w[1] << 4) & 0x0FFF0000u);   // codes 2, 3 | 6, 7
        o = u4_t{qr_pair<FMT, 0>(a, base), qr_pair<FMT, 6>(a, base), qr_pair<FMT, 0>(b, base), qr_pair<FMT, 6>(b, base)};
    } else if constexpr (FMT == QG_FMT_B3) {
        const uint32_t v = (w[0] & 0xFFFu) | ((w[0] << 4) & 0x0FFF0000u);   // codes 0..3 low, 4..7 high
        o = u4_t{qr_pair<FMT, 0>(v, base), qr_pair<FMT, 3>(v, base), qr_pair<FMT, 6>(v, base), qr_pair<FMT, 9>(v, base)};
    } else {
        // HQ4_G32_M5 and 4-bit streams: codes k and k + 4 of the word's order; 2 bits: code e + 1 sixteen bits above code e
        const uint32_t v = FMT == QG_FMT_B2 ? (w[0] & 0xFFFFu) | (w[0] << 14) : w[0];
        o = u4_t{qr_pair<FMT, 0>(v, base), qr_pair<FMT, 4>(v, base), qr_pair<FMT, 8>(v, base), qr_pair<FMT, 12>(v, base)};
    }
    return __builtin_bit_cast(h8_t, o);
}
// Eight activations in the order in which the codes come out: as they are, but for 3-, 4- and 6-bit streams, (k, k + 4).
template <int FMT>
__device__ __forceinline__ h8_t qr_x_order(h8_t v) {
    if constexpr (FMT == QG_FMT_B3 || FMT == QG_FMT_B4 || FMT == QG_FMT_B6) return h8_t{v[0], v[4], v[1], v[5], v[2], v[6], v[3], v[7]};
    else return v;
}

// A step's activation operands out of the wave's part of LDS, and (FACT) the sum of slice 4 g + c in lane (i, c).  Operand t of lane
// (i, c) is columns 8 c .. + 7 of slice 4 g + t of row i (FACT), 8 t .. + 7 of slice 4 g + c (F16W).  The sums come from the matrix unit,
// which has the time: a product of ones with the operand leaves row i's sum in every lane (i, .).
template <int FMT, bool F16W>
__device__ __forceinline__ float qr_x_step(const uint32_t* img, uint32_t i, uint32_t c, h8_t (&xo)[4]) {
    const f4_t z = {0.f, 0.f, 0.f, 0.f};
    const h8_t ones = {1, 1, 1, 1, 1, 1, 1, 1};
    float sum[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const h8_t v = *(const h8_t*)(img + i * QR_XS + 4u * (F16W ? 4u * c + t : 4u * t + c));
        xo[t] = F16W ? v : qr_x_order<FMT>(v);
        if constexpr (!F16W) sum[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, v, z, 0, 0, 0)[0];
    }
    if constexpr (F16W) return 0.f;
    return c < 2u ? (c == 0u ? sum[0] : sum[1]) : (c == 2u ? sum[2] : sum[3]);
}

template <int FMT>
constexpr bool QR_HALVES = FMT == QG_FMT_B8 || FMT == QG_FMT_B6;
// Step g of a 16-row tile out of the wave's image: acc += sum s (2^bits + q) x and accb += sum (b - 2^bits s) x (FACT), or acc, accb += w x (F16W).
template <int FMT, bool F16W, int S>
__device__ __forceinline__ void qr_step(const uint32_t* img, uint32_t g, uint32_t n, uint32_t c, const h8_t (&xo)[4], float xsum, uint32_t magic,
                                        f4_t& acc, f4_t& accb) {
    using im = qr_image<FMT, S>;
    const uint32_t* hdr = img + 16u * im::RS + n * im::HS + 4u * g;
    if constexpr (F16W) {
        qg_slice<FMT> blk;
        blk.hdr = hdr[c];
        const uint32_t* src = img + n * im::RS + (4u * g + c) * im::PW;
#pragma unroll
        for (uint32_t k = 0; k < im::PW; k += 4) {
            const u4_t v = *(const u4_t*)(src + k);
            blk.q[k] = v[0], blk.q[k + 1] = v[1], blk.q[k + 2] = v[2], blk.q[k + 3] = v[3];
        }
        const h2_t s2 = qw_splat_lo(blk.hdr), b2 = qw_splat_hi(blk.hdr);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const h8_t w = qg_dequant_chunk<FMT>(blk, j, s2, b2, magic);
            if (j & 1) accb = __builtin_amdgcn_mfma_f32_16x16x32_f16(xo[j], w, accb, 0, 0, 0);
            else acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(xo[j], w, acc, 0, 0, 0);
        }
    } else {
        const u4_t h = *(const u4_t*)hdr;
        const h2_t own = __builtin_bit_cast(h2_t, hdr[c]);
        const float bias = __builtin_fmaf(QR_OFF<FMT>, (float)own[0], (float)own[1]);
        const f4_t z = {0.f, 0.f, 0.f, 0.f};
        accb = __builtin_amdgcn_mfma_f32_16x16x4f32(xsum, bias, accb, 0, 0, 0);
#pragma unroll
        for (int t = 0; t < 4; t += 2) {
            uint32_t w[2][2];
            qr_chunk<FMT, S>(img, n, 4u * g + t, c, w[0]);
            qr_chunk<FMT, S>(img, n, 4u * g + t + 1u, c, w[1]);
            const f4_t d0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(xo[t], qr_codes<FMT>(w[0], magic), z, 0, 0, 0);
            const f4_t d1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(xo[t + 1], qr_codes<FMT>(w[1], magic), z, 0, 0, 0);
            const uint32_t h0 = h[t], h1 = h[t + 1];   // by value: the cast of a vector element takes the vector's first
            const float s0 = (float)__builtin_bit_cast(h2_t, h0)[0], s1 = (float)__builtin_bit_cast(h2_t, h1)[0];
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[r] = __builtin_fmaf(s1, d1[r], __builtin_fmaf(s0, d0[r], acc[r]));
            if constexpr (QR_HALVES<FMT>) __builtin_amdgcn_sched_barrier(0);
        }
    }
}
// Bytes of this lane's slice sl (clamped into the row) inside a bank row.
template <int FMT, class P>
__device__ __forceinline__ void qr_slice_at(const P& p, uint32_t sl, uint32_t& hdr, uint32_t& codes) {
    const uint32_t g = min(sl, p.nsl - 1u);
    if constexpr (FMT == QG_FMT_M5) {
        hdr = g * 20u;
        codes = hdr + 4u;
    } else {
        hdr = (g >> p.gshift) * p.bb;
        codes = hdr + 4u + (g & ((1u << p.gshift) - 1u)) * qr_code_bytes<FMT>();
    }
}
// One 32-bit sum an address (the bank is under 4 GiB): scalar base + 32-bit lane offset addressing.
template <int FMT, class P>
__device__ __forceinline__ void qr_load(const P& p, uint32_t hdr, uint32_t codes, qg_slice<FMT>& o) {
    if constexpr (FMT == QG_FMT_M5) {
        o.hdr = *(const uint32_t*)(p.bank + hdr);
        const qg_words4 w = *(const qg_words4*)(p.bank + codes);
#pragma unroll
        for (int j = 0; j < 4; ++j) o.q[j] = w.q[j];
    } else {
        qg_load_slice_at<FMT>(p.bank + hdr, p.bank + codes, o);
    }
}

template <int N, int I = 0, class F>
__device__ __forceinline__ void qr_for(F&& f) {   // arrays of slices stay in registers when no index is ever a variable
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        qr_for<N, I + 1>(f);
    }
}

// Step g of a 16-row tile out of the wave's image against MF fragments, the exact f16 weights: lane (n, c) has slice 4 g + c of row n.
template <int FMT, int S, int MF>
__device__ __forceinline__ void qr_weight_step(const uint32_t* img, uint32_t g, uint32_t n, uint32_t c, const h8_t (&xo)[MF][4], uint32_t magic, f4_t (&acc)[MF]) {
    using im = qr_image<FMT, S>;
    qg_slice<FMT> blk;
    blk.hdr = img[16u * im::RS + n * im::HS + 4u * g + c];
    const uint32_t* src = img + n * im::RS + (4u * g + c) * im::PW;
    if constexpr (im::PW % 4u == 0u) {
#pragma unroll
        for (uint32_t k = 0; k < im::PW; k += 4) {
            const u4_t v = *(const u4_t*)(src + k);
            blk.q[k] = v[0], blk.q[k + 1] = v[1], blk.q[k + 2] = v[2], blk.q[k + 3] = v[3];
        }
    } else if constexpr (im::PW % 2u == 0u) {
#pragma unroll
        for (uint32_t k = 0; k < im::PW; k += 2) {
            const u2_t v = *(const u2_t*)(src + k);
            blk.q[k] = v[0], blk.q[k + 1] = v[1];
        }
    } else {
#pragma unroll
        for (uint32_t k = 0; k < im::PW; ++k) blk.q[k] = src[k];
    }
    const h2_t s2 = qw_splat_lo(blk.hdr), b2 = qw_splat_hi(blk.hdr);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const h8_t w = qg_dequant_chunk<FMT>(blk, j, s2, b2, magic);
#pragma unroll
        for (int f = 0; f < MF; ++f) acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xo[f][j], w, acc[f], 0, 0, 0);
    }
}

// Four activation rows 4 q .. of bank row rr of the tile at `part`, over the waves in order.
template <int MF>
__device__ __forceinline__ f4_t qr_wave_sum(const f4_t* part, uint32_t W, uint32_t q, uint32_t rr) {
    const f4_t* src = part + (q >> 2) * 64u + (q & 3u) * 16u + rr;
    f4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (uint32_t w = 0; w < W; ++w) v += src[w * MF * 64u];
    return v;
}

}  // namespace
