// Verify GEMV (m = 2..16 activation rows already in the container's basis), every container: a workgroup takes 16 bank rows at a
// time, its waves split the row's columns, and all m rows share one v_mfma_f32_16x16x32_f16 per 32-column slice.
//
// Operand A is the activations (16 rows x 32 columns; rows past m are zero), operand B the codes of 16 bank rows, so lane
// (n = lane & 15, c = lane >> 4) ends up with outputs of bank row n for activation rows 4 c .. 4 c + 3 and needs one scale a slice.
// A step is four slices (128 columns); a wave owns S steps and keeps their activations in registers while it walks row tiles.
//  - In: a load takes 4 S consecutive slices of 16 / S bank rows (long runs: with a slice of 16 rows a quad of lanes, the contraction's
//    own layout, the address unit set the time, 34816 x 5120: 33 us), all S of a tile at once, and parks them in the wave's part of
//    LDS; the next tile's go out behind them.  No barrier: an image is private to a wave.
//  - FACT (F16W = 0): instruction t contracts slice t of the step, lane (n, c) with the eight codes of chunk c as f16; the products are
//    exact, and  s * sum(q x)  follows per slice in fp32 (qwg_aq_slice_dot, Sources/QWMetal/include/qw_dequant_multi.metalh:205-208).
//    b * sum(x) over the four slices is one v_mfma_f32_16x16x4_f32, whose operands are the headers and the slices' sums.
//  - F16W: lane (n, c) dequantizes slice c of the step to the exact f16 weights of qwhip_dequant_f16, and instruction j contracts chunk j
//    of the four slices (the arithmetic of the split-K kernel).
// The cost does not depend on m.  The partial tiles of the waves meet in LDS and are summed in wave order; rows past 6144 columns take
// several K ranges, whose sums meet in the stream's scratch and a second launch.
// OUT = 1, 2: the bank is gate|up; a unit is 16 or 32 channels' gate rows and their up rows, and the gated activation (2: and the
// FWHT-32 over its 32 channels) is formed where the tiles are summed, in fp32, rounded to f16 once: no image, no second launch.
//
// Bound: 50 to 75 vector instructions a step and wave beside the loads (4 and 6 bits), and on short launches the chain of one trip:
// loads, LDS, products, sums.  Against the kernels before, launches on cold banks back to back (us): 34816 x 5120 HQ4_G32_M5 at
// 8 / 12 / 16 rows 31.8 / 53.1 / 29.5 -> 25.3 / 26.9 / 27.4 (5.2 TB/s at 8), 3072 x 2048 6.9 / 8.7 / 10.9 -> 4.5 / 4.6 / 4.7; 24576 x 4096 in
// 36-byte blocks 17.9 / 23.6 / 17.7 -> 15.2 / 16.0 / 17.0; 22784 x 4608 at 6 bits 45 / 70 / 90 -> 24.4 / 25.4 / 25.4; 16384 x 2304 at 3 bits
// 22.4 / 37.8 / 44.9 -> 9.2 / 9.7 / 9.9; 4096 x 12288 4-bit 19.3 / 19.7 / 19.8 -> 13.1 / 13.9 / 14.4; 6144 x 24576 33.5 / 34.5 / 34.7 -> 23.0 / 24.3 /
// 25.1; 5120 x 17408 HQ8_G32 29.6 / 34.0 / 51.1 -> 25.1 / 26.2 / 26.6.  Error against 64 bits of the codes' own weights (FACT), 8 rows of
// 1536 columns: HQ4_G32_M5 6.5e-6 -> 5.2e-7, HQ8_G32 4.0e-7 -> 1.7e-7, 2 bits 1.0e-5 -> 3.9e-7.
#include <atomic>

#include "qwhip_common.h"
#include "qw_slice.h"

// gemv_sk.hip: y[m][row] = sum of the K ranges' partial sums part[range][m][n16], in range order
hipError_t qw_sk_sum(hipStream_t st, const float* part, void* y16, float* y32, uint32_t n, uint32_t m, uint32_t n16, uint32_t nkr);

namespace {

// units: row tiles (16 F rows), or blocks of 16 / 32 gated channels; flush: units between two sums of the partial tiles
#define QR_FIELDS(X)                                                                                                        \
    X(const uint8_t*, bank) X(const void*, x) X(uint32_t, K) X(uint32_t, M) X(uint32_t, nsl) X(uint32_t, row_bytes)             \
    X(uint32_t, gshift) X(uint32_t, bb) X(uint32_t, N) X(uint32_t, units) X(uint32_t, nkr) X(uint32_t, flush) X(uint32_t, inter) X(h1_t*, y16)   \
    X(float*, y32) X(float*, part) X(qw_act, act)
QW_ARG_BLOCK(qr_params, QR_FIELDS)

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
template <int FMT>
__device__ __forceinline__ void qr_slice_at(const qr_params& p, uint32_t sl, uint32_t& hdr, uint32_t& codes) {
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
template <int FMT>
__device__ __forceinline__ void qr_load(const qr_params& p, uint32_t hdr, uint32_t codes, qg_slice<FMT>& o) {
    if constexpr (FMT == QG_FMT_M5) {
        o.hdr = *(const uint32_t*)(p.bank + hdr);
        const qg_words4 w = *(const qg_words4*)(p.bank + codes);
#pragma unroll
        for (int j = 0; j < 4; ++j) o.q[j] = w.q[j];
    } else {
        qg_load_slice_at<FMT>(p.bank + hdr, p.bank + codes, o);
    }
}
// The raw activations of step g: lane takes piece lane & 15 (8 columns) of row 4 q + (lane >> 4): runs of 256 bytes (a lane
// an operand piece each, 16 runs of 64 bytes, cost the address unit three times as long).  Rows past M are zero, and so are the
// pieces past the row's end.
__device__ __forceinline__ u4_t qr_load_x(const qr_params& p, uint32_t g, uint32_t q, uint32_t lane) {
    const uint32_t col = 128u * g + 8u * (lane & 15u), row = 4u * q + (lane >> 4);
    u4_t v = {0u, 0u, 0u, 0u};
    if (row < p.M && col < p.K) v = *(const u4_t*)((const uint8_t*)p.x + (2u * row * p.K + 2u * col));
    return v;
}
template <int XDT>
__device__ __forceinline__ void qr_park_x(uint32_t* img, uint32_t q, uint32_t lane, u4_t raw) {
    *(h8_t*)(img + (4u * q + (lane >> 4)) * QR_XS + 4u * (lane & 15u)) = qg_to_f16x8<XDT>(raw);
}

// Sums the waves' partial tiles part[slot][wave][lane] of `count` row tiles, slot s being tile t0 + s * step, and stores them.
__device__ __forceinline__ void qr_store_tiles(const qr_params& p, const f4_t* part, uint32_t W, uint32_t count, uint32_t t0, uint32_t step, uint32_t kr) {
    for (uint32_t e = threadIdx.x; e < count * 16u * p.M; e += blockDim.x) {
        const uint32_t rr = e & 15u, sm = e >> 4, s = sm / p.M, m = sm - s * p.M;
        const uint32_t row = 16u * (t0 + s * step) + rr;
        const float* src = (const float*)(part + (size_t)s * W * 64u) + ((m >> 2) * 16u + rr) * 4u + (m & 3u);
        float v = 0.f;
#pragma unroll 4
        for (uint32_t w = 0; w < W; ++w) v += src[w * 256u];
        if (p.nkr > 1u) {   // rows past the bank are in the planes too
            p.part[((uint64_t)kr * p.M + m) * (16u * p.units) + row] = v;
        } else if (row < p.N) {
            const uint64_t at = (uint64_t)m * p.N + row;
            if (p.y32) p.y32[at] = v;
            if (p.y16) p.y16[at] = (h1_t)v;
        }
    }
}
// The same for one unit of 16 RT gated channels, whose RT gate tiles come first: channel c0 + j of activation row m.
template <int RT>
__device__ __forceinline__ void qr_store_gated(const qr_params& p, const f4_t* part, uint32_t W, uint32_t c0) {
    constexpr uint32_t CH = 16u * RT;
    const qw_fwht32_signs sg = qw_fwht32_lane_signs(threadIdx.x & 31u);
    for (uint32_t e = threadIdx.x; e < ((CH * p.M + 63u) & ~63u); e += blockDim.x) {   // whole waves: the rotation exchanges lanes
        const uint32_t j = e & (CH - 1u), m = min(e / CH, p.M - 1u);
        const float* src = (const float*)(part + (size_t)(j >> 4) * W * 64u) + ((m >> 2) * 16u + (j & 15u)) * 4u + (m & 3u);
        const float* up = src + (size_t)RT * W * 256u;
        float g = 0.f, u = 0.f;
#pragma unroll 4
        for (uint32_t w = 0; w < W; ++w) g += src[w * 256u], u += up[w * 256u];
        float v = qw_gated(g, u, p.act);
        if constexpr (RT == 2) {
            v = qw_fwht32_lanes(v, sg) * QW_INV_SQRT32;
            asm volatile("" : "+v"(v));   // rounded to fp32 and then to f16, as the rotation pass does (not by one mixed instruction)
        }
        if (e < CH * p.M) p.y16[(uint64_t)m * p.inter + c0 + j] = (h1_t)v;
    }
}

template <int N, int I = 0, class F>
__device__ __forceinline__ void qr_for(F&& f) {   // arrays of slices stay in registers when no index is ever a variable
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        qr_for<N, I + 1>(f);
    }
}

// S steps a wave.  blockDim.x = 64 * ceil(steps / S); dynamic LDS = the waves' images, then 2 * flush * tiles a unit * waves * 1 KiB.
template <int FMT, int XDT, bool F16W, int S, int OUT>
struct qw_gemv_rows_kernel {
static constexpr int kLaunchBound = S <= 2 ? 1024 : 768;
static __device__ __forceinline__ void run(const qr_params& p) {
    extern __shared__ __attribute__((aligned(16))) uint32_t qr_lds[];
    using im = qr_image<FMT, S>;
    constexpr uint32_t SPU = OUT == 0 ? 1u : 2u * OUT;   // row tiles of a unit
    constexpr uint32_t RPL = 16u / S;                    // bank rows of a load: 4 S slices of each
    const uint32_t tid = threadIdx.x, lane = tid & 63u, W = blockDim.x >> 6;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t G = gridDim.x / p.nkr, band = blockIdx.x / p.nkr, kr = blockIdx.x - band * p.nkr;
    const uint32_t n = lane & 15u, c = lane >> 4;             // contraction role
    const uint32_t lb = lane / RPL, lj = lane & (RPL - 1u);   // load role: slice lb of the wave's, row RPL q + lj of the tile
    uint32_t* const img = qr_lds + wave * im::DWORDS;
    f4_t* const parts = (f4_t*)(qr_lds + W * im::DWORDS);
    if (band >= p.units) return;
    const uint32_t nu = (p.units - band + G - 1u) / G;   // units of this workgroup
    const uint32_t slots = nu * SPU, per = p.flush * SPU;      // row tiles; of them between two sums
    const uint32_t magic = qw_vgpr_const(F16W ? 0x64006400u : qr_base<FMT>());

    uint32_t hdr, codes;
    qr_slice_at<FMT>(p, 4u * S * (kr * W + wave) + lb, hdr, codes);
    qg_slice<FMT> buf[S];
    auto request = [&](uint32_t slot) __attribute__((always_inline)) {
        uint32_t row;
        if constexpr (OUT == 0) {
            row = 16u * (slot * G + band);
        } else {
            const uint32_t k = slot / SPU, q = slot - k * SPU;
            row = 16u * ((k * G + band) * OUT + (q % OUT)) + (q >= OUT ? p.inter : 0u);
        }
        qr_for<S>([&](auto q) {   // rows past the bank re-read its last row (never stored)
            const uint32_t ro = min(row + RPL * q + lj, p.N - 1u) * p.row_bytes;
            qr_load<FMT>(p, ro + hdr, ro + codes, buf[q]);
        });
    };
    request(0);
    __builtin_amdgcn_sched_barrier(0);
    u4_t raw[4 * S];
    qr_for<4 * S>([&](auto i) { raw[i] = qr_load_x(p, (kr * W + wave) * S + i / 4, i % 4, lane); });
    __builtin_amdgcn_sched_barrier(0);
    h8_t xo[S][4];
    float xs[S];
    qr_for<S>([&](auto u) {
        qr_for<4>([&](auto q) { qr_park_x<XDT>(img, q, lane, raw[4 * u + q]); });
        asm volatile("" ::: "memory");   // a wave's own LDS operations complete in order
        xs[u] = qr_x_step<FMT, F16W>(img, n, c, xo[u]);
        asm volatile("" ::: "memory");
    });

    uint32_t in_flush = 0, side = 0, first = 0;   // row tiles since the last sum, the half of the partial tiles, its first slot
#pragma unroll 1
    for (uint32_t slot = 0; slot < slots; ++slot) {
        qr_for<S>([&](auto q) { qr_park<FMT, S>(img, RPL * q + lj, lb, buf[q]); });
        asm volatile("" ::: "memory");
        if (slot + 1u < slots) request(slot + 1u);
        __builtin_amdgcn_sched_barrier(0);
        f4_t acc = {0.f, 0.f, 0.f, 0.f}, accb = acc;
#pragma unroll
        for (int u = 0; u < S; ++u) {
            qr_step<FMT, F16W, S>(img, u, n, c, xo[u], xs[u], magic, acc, accb);
            __builtin_amdgcn_sched_barrier(0);
        }
        parts[(size_t)((side * per + in_flush) * W + wave) * 64u + lane] = acc + accb;
        asm volatile("" ::: "memory");
        ++in_flush;
        if (in_flush == per || slot + 1u == slots) {
            __syncthreads();   // the other half of the partial tiles is free again: its sums lie before this barrier
            const f4_t* part = parts + (size_t)side * per * W * 64u;
            if constexpr (OUT == 0) qr_store_tiles(p, part, W, in_flush, first * G + band, G, kr);
            else qr_store_gated<OUT>(p, part, W, 16u * OUT * ((slot / SPU) * G + band));
            in_flush = 0;
            side ^= 1u;
            first = slot + 1u;
        }
    }
}
};

template <typename K>
hipError_t qr_go(hipStream_t st, const qr_params& p, uint32_t wgs, uint32_t waves, size_t lds) {
    static std::atomic<bool> attr_done{false};   // per instantiation
    if (!attr_done.load(std::memory_order_acquire)) {
        const hipError_t e = hipFuncSetAttribute(qw_scalar_kernel_ptr<K>((const qr_params*)nullptr), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return e;
        attr_done.store(true, std::memory_order_release);
    }
    qw_launch_scalar<K>(dim3(wgs), dim3(64u * waves), lds, st, p);
    return hipGetLastError();
}

template <int FMT, int XDT, bool F16W>
hipError_t qr_launch(hipStream_t st, qr_params& p, size_t part_bytes, uint32_t out, uint32_t tune) {
    // as few steps a wave as 16 waves (one or two steps, 128 registers) or 12 (168) hold; longer rows in K ranges
    const uint32_t steps = qwhip_cdiv(p.nsl, 4u);
    uint32_t s = steps <= 16u ? 1u : steps <= 32u ? 2u : 4u;
    if (tune & 7u) s = max(tune & 7u, s);
    const uint32_t spu = out ? 2u * out : 1u;
    p.units = out ? p.inter / (16u * out) : qwhip_cdiv(p.N, 16u);
    p.nkr = qwhip_cdiv(steps, s * (s <= 2u ? 16u : 12u));
    if (p.nkr > 1u) {   // of the least number of ranges and the two after it, the one whose workgroups walk the fewest wave steps
        uint32_t best = ~0u, least = p.nkr;
        for (uint32_t k = least; k < least + 3u; ++k) {
            const uint32_t cost = qwhip_cdiv(p.units, 256u / k) * qwhip_cdiv(steps, s * k);
            if (cost < best) best = cost, p.nkr = k;
        }
    }
    const uint32_t waves = qwhip_cdiv(steps, s * p.nkr);
    p.nkr = qwhip_cdiv(steps, s * waves);
    if (p.nkr > 1u && (out || (uint64_t)p.nkr * p.M * p.units * 64u > part_bytes)) return hipErrorNotSupported;
    const uint32_t image = waves * 4u * (s == 1u ? qr_image<FMT, 1>::DWORDS : s == 2u ? qr_image<FMT, 2>::DWORDS : qr_image<FMT, 4>::DWORDS);
    const uint32_t part = 2u * spu * waves * 1024u, most = 160u * 1024u;   // bytes of the images, of the partial tiles of a unit
    if (image + part > most) return hipErrorNotSupported;
    const uint32_t cus = 256u * max(1u, min((s <= 2u ? 16u : 12u) / waves, most / (image + part)));
    if (out) {
        // The launch that is saved is worth 2 to 2.5 us (2 x 8192 x 3072: 9.3 us, in two launches 11.5; 2 x 7552 x 2560 8.7 / 11.1; 2 x 3840 x 1536
        // 5.8 / 7.2).  Whole units leave workgroups with a unit more than others, a row tile being 0.4 to 0.5 us per 1024 columns (2 x 8448 x
        // 2816 at 8 bits, eight tiles where five would do: 19.7 / 17.8), and up to four rows have a faster plain kernel (2 x 12544 x 5120, two
        // rows: 22.1 / 19.9, five rows: 22.6 / 22.9).
        const uint32_t tiles = qwhip_cdiv(p.units * spu, cus), longer = qwhip_cdiv(p.units, cus) * spu - tiles;
        const float plain = p.M > 4u ? 0.0f : p.M == 2u && FMT >= QG_FMT_B2 ? 0.2f : 0.1f;
        if ((longer + plain * tiles) * p.K > 5500.0f) return hipErrorNotSupported;
    }
    uint32_t per_cu = cus / 256u;
    if ((tune >> 3) & 3u) per_cu = (tune >> 3) & 3u;
    const uint32_t bands = min(p.units, 256u * per_cu / p.nkr), wgs = bands * p.nkr;
    p.flush = out ? 1u : max(1u, min(min(4u, qwhip_cdiv(p.units, bands)), (most / per_cu - image) / part));
    const size_t lds = (size_t)image + p.flush * part;
#define QR_S(SS)                                                                                                       \
    {                                                                                                                  \
        if constexpr (XDT == QWHIP_F16) {                                                                              \
            if (out == 1u) return qr_go<qw_gemv_rows_kernel<FMT, XDT, F16W, SS, 1>>(st, p, wgs, waves, lds);            \
            if (out == 2u) return qr_go<qw_gemv_rows_kernel<FMT, XDT, F16W, SS, 2>>(st, p, wgs, waves, lds);            \
        }                                                                                                              \
        return qr_go<qw_gemv_rows_kernel<FMT, XDT, F16W, SS, 0>>(st, p, wgs, waves, lds);                              \
    }
    if (s == 1u) QR_S(1) else if (s == 2u) QR_S(2) else QR_S(4)
#undef QR_S
}

}  // namespace

// Tries the row-tile kernel for a validated call with m = 1..16 rows already in the container's basis; false when the shape is outside
// its envelope.  fmt: QW_FMT_* (the codes of qw_slice.h).  f16w: contract the exact f16 weights (HQ4_G32_M5, 4- and 8-bit streams).
// inter > 0: the bank is gate|up, y16 the gated activations [m][inter], with `rotate_out` in the rotated basis.
// `tune` (0 = automatic): bits 0..2 steps a wave at least / row tiles a workgroup on long rows, bits 3.. workgroups a unit / waves / 4.
bool qw_rows_gemv(qwhip_stream_t s, const qwhip_weight_view* w, int fmt, uint32_t gshift, uint32_t bb, uint64_t row_bytes, const void* x,
                  uint32_t x_dtype, uint32_t m, bool f16w, void* y16, float* y32, uint32_t inter, bool rotate_out, uint32_t tune, hipError_t* err) {
    if (m == 0u || m > 16u || ((uintptr_t)x & 15u) != 0) return false;
    if ((uint64_t)w->n * row_bytes >= (1ull << 32)) return false;   // 32-bit offsets inside the bank
    if (f16w && fmt >= QW_FMT_B2) return false;
    const hipStream_t st = s->stream;
    const uint32_t nsl = w->k / 32u;
    if (inter && (x_dtype != QWHIP_F16 || inter % (rotate_out ? 32u : 16u) != 0)) return false;
    const size_t part_bytes = s->scratch ? s->scratch_bytes - QWHIP_STREAM_COUNTER_BYTES - QWHIP_STREAM_XROT_BYTES - s->scratch_reserved : 0u;
    qr_params p;
    p.bank = (const uint8_t*)w->blocks;
    p.x = x;
    p.K = w->k;
    p.M = m;
    p.nsl = nsl;
    p.row_bytes = (uint32_t)row_bytes;
    p.gshift = gshift;
    p.bb = bb;
    p.N = w->n;
    p.units = 0;
    p.flush = 1;
    p.inter = inter;
    p.y16 = (h1_t*)y16;
    p.y32 = y32;
    p.nkr = 1;
    p.part = (float*)(s->scratch ? s->scratch + QWHIP_STREAM_COUNTER_BYTES : nullptr);
    p.act = s->dev->act;
    const uint32_t out = inter ? (rotate_out ? 2u : 1u) : 0u;
#define QR_GO(F, W16) (x_dtype == QWHIP_F16 ? qr_launch<F, QWHIP_F16, W16>(st, p, part_bytes, out, tune) : qr_launch<F, QWHIP_BF16, W16>(st, p, part_bytes, out, tune))
    if (f16w) {
        *err = fmt == QW_FMT_M5 ? QR_GO(QG_FMT_M5, true) : fmt == QW_FMT_B4 ? QR_GO(QG_FMT_B4, true) : QR_GO(QG_FMT_B8, true);
    } else {
        switch (fmt) {
            case QW_FMT_M5: *err = QR_GO(QG_FMT_M5, false); break;
            case QW_FMT_B4: *err = QR_GO(QG_FMT_B4, false); break;
            case QW_FMT_B8: *err = QR_GO(QG_FMT_B8, false); break;
            case QW_FMT_B2: *err = QR_GO(QG_FMT_B2, false); break;
            case QW_FMT_B3: *err = QR_GO(QG_FMT_B3, false); break;
            default: *err = QR_GO(QG_FMT_B6, false); break;
        }
    }
#undef QR_GO
    if (*err == hipErrorNotSupported) return false;
    if (*err == hipSuccess && p.nkr > 1u) *err = qw_sk_sum(st, p.part, y16, y32, w->n, m, p.units * 16u, p.nkr);
    return true;
}
