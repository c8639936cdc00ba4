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
// 22.4 / 37.8 / 44.9 -> 9.2 / 9.7 / 9.9; 4096 x 12288 4-bit 20.3 / 20.5 / 20.5 -> 12.7 / 13.2 / 13.8; 6144 x 24576 34.5 / 35.6 / 35.8 -> 24.3 / 24.6 /
// 25.5; 5120 x 17408 HQ8_G32 31.1 / 35.6 / 51.6 -> 26.8 / 26.9 / 26.9.  Error against 64 bits of the codes' own weights (FACT), 8 rows of
// 1536 columns: HQ4_G32_M5 6.5e-6 -> 5.2e-7, HQ8_G32 4.0e-7 -> 1.7e-7, 2 bits 1.0e-5 -> 3.9e-7.
#include <atomic>

#include "qw_rows.h"

// gemv_sk.hip: y[m][row] = sum of the K ranges' partial sums part[range][m][n16], in range order
hipError_t qw_sk_sum(hipStream_t st, const float* part, void* y16, float* y32, uint32_t n, uint32_t m, uint32_t n16, uint32_t nkr);

namespace {

// units: row tiles (16 F rows), or blocks of 16 / 32 gated channels; flush: units between two sums of the partial tiles
#define QR_FIELDS(X)                                                                                                        \
    X(const uint8_t*, bank) X(const void*, x) X(uint32_t, K) X(uint32_t, M) X(uint32_t, nsl) X(uint32_t, row_bytes)             \
    X(uint32_t, gshift) X(uint32_t, bb) X(uint32_t, N) X(uint32_t, units) X(uint32_t, nkr) X(uint32_t, flush) X(uint32_t, inter) X(h1_t*, y16)   \
    X(float*, y32) X(float*, part) X(qw_act, act)
QW_ARG_BLOCK(qr_params, QR_FIELDS)

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

template <int FMT>
constexpr uint32_t qr_image_bytes(uint32_t s) { return 4u * (s == 1u ? qr_image<FMT, 1>::DWORDS : s == 2u ? qr_image<FMT, 2>::DWORDS : qr_image<FMT, 4>::DWORDS); }
constexpr uint32_t qr_most_waves(uint32_t s) { return s <= 2u ? 16u : 12u; }   // of 128 and of 168 registers
constexpr uint32_t QR_LDS = 160u * 1024u;

// Steps a wave (at least `least`) and K ranges of rows past 6144 columns, by the lowest price, us: the launches 5.1 and the activations; row
// tiles one after the other on a compute unit, each 0.27 for the barrier, 0.021 for every wave's part of the sums, and every step on a SIMD;
// the planes at 1.4 TB/s; and the bank's stream (8.5 TB/s, in quadrature).  Weighed by the choice it makes among 11000 measured forms of 170
// banks (n 1024 .. 20000, k 6400 .. 28672, 12 containers) at 4 to 16 rows: the form taken is 2 % slower than the best.  (Four steps a wave and
// as few ranges as hold the row, the rule before, was 13 % slower than the best: 2368 x 7936 HQ8_G32 at nine rows 15.4 us, the 4x4x4-block
// kernel 12.1, this choice 10.5.)  False where nothing fits.
template <int FMT>
bool qr_ranges(const qr_params& p, uint32_t steps, uint32_t least, size_t part_bytes, uint32_t* s_out, uint32_t* nkr_out) {
    const float unpack = FMT == QG_FMT_B8 ? 2.0f : FMT == QG_FMT_B6 ? 1.8f : FMT == QG_FMT_B3 ? 1.6f : 1.0f;
    const float bank = (float)p.N * (float)p.row_bytes / 8.5e6f;
    float best = 3e38f;
    for (uint32_t s = 1; s <= 4u; s *= 2u) {
        const uint32_t lo = max(2u, qwhip_cdiv(steps, s * qr_most_waves(s)));
        for (uint32_t k = lo; s >= least && k < lo + 7u && k <= 256u && (uint64_t)k * p.M * p.units * 64u <= part_bytes; ++k) {
            const uint32_t waves = qwhip_cdiv(steps, s * k), need = waves * (qr_image_bytes<FMT>(s) + 2048u);
            if (waves < 2u || need > QR_LDS || (k - 1u) * s * waves >= steps) continue;
            const uint32_t per_cu = max(1u, min(qr_most_waves(s) / waves, QR_LDS / need)), bands = min(p.units, 256u * per_cu / k);
            const float simd = waves * qwhip_cdiv(bands * k, 256u) * s / 4.0f;   // steps on a SIMD, side by side
            const float tile = 0.27f + 0.021f * waves + 0.076f * unpack * (s == 1u ? 0.55f : s == 2u ? 1.0f : 2.5f) * simd;
            const float t = 5.1f + 0.43f * simd + qwhip_cdiv(p.units, bands) * tile + (float)k * p.M * p.N * 8.0f / 1.43e6f, us = t * t + bank * bank;
            if (us < best) best = us, *s_out = s, *nkr_out = k;
        }
    }
    return best < 3e38f;
}

template <int FMT, int XDT, bool F16W>
hipError_t qr_launch(hipStream_t st, qr_params& p, size_t part_bytes, uint32_t out, uint32_t tune) {
    // as few steps a wave as 16 waves (one or two steps, 128 registers) or 12 (168) hold; longer rows in K ranges
    const uint32_t steps = qwhip_cdiv(p.nsl, 4u), code = (tune & 7u) == 3u ? 4u : min(tune & 7u, 4u);   // the forms there are: 1, 2 and 4
    uint32_t s = max(code, steps <= 16u ? 1u : steps <= 32u ? 2u : 4u);
    const uint32_t spu = out ? 2u * out : 1u;
    p.units = out ? p.inter / (16u * out) : qwhip_cdiv(p.N, 16u);
    p.nkr = 1;
    if (steps > s * qr_most_waves(s) && (out || !qr_ranges<FMT>(p, steps, code, part_bytes, &s, &p.nkr))) return hipErrorNotSupported;
    const uint32_t waves = qwhip_cdiv(steps, s * p.nkr);
    const uint32_t image = waves * qr_image_bytes<FMT>(s), part = 2u * spu * waves * 1024u, most = QR_LDS;   // bytes of the images, of the partial tiles of a unit
    if (image + part > most) return hipErrorNotSupported;
    const uint32_t cus = 256u * max(1u, min(qr_most_waves(s) / waves, most / (image + part)));
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
    if ((tune >> 3) & 3u) per_cu = min((tune >> 3) & 3u, most / (image + part));   // as many as LDS holds
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
// `tune` (0 = automatic): bits 0..2 steps a wave at least (3 and more: 4), bits 3..4 workgroups a unit.
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
