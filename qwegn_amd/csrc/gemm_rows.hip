// Dense GEMM of 17 to 64 activation rows on the row-tile form of gemv_rows.hip: two or four fragments of 16 rows share a tile of 16 bank
// rows, whose f16 weights a wave takes out of its LDS image once for all of them.
//
// The waves of a workgroup split the columns, so that a bank of few rows has its K loop in parallel without K ranges over workgroups, a
// tile's weights are one wave's loads ahead of its products, and nothing waits at a barrier but the tiles' sums.  The activations of a
// wave's columns stay in its registers for all its tiles: 16 registers a fragment and step, which bounds the columns of a workgroup
// (qwr_configure); more of them are K ranges into fp32 planes.
// Bound by the launch, the activations' way through LDS and then, a tile, one round of loads, unpacking, products and sums.  HQ4_G32_M5,
// cold banks, against the direct-operand kernel over K ranges (us): 32 rows on 3072 x 1536 10.2 -> 5.4, 2560 x 9728 17.8 -> 10.9,
// 7168 x 5120 17.9 -> 13.4, 34816 x 5120 44.1 -> 36.1; 64 rows on 3072 x 1536 12.3 -> 6.9, 2560 x 3584 14.9 -> 10.4.
#include <atomic>
#include <cmath>

#include "qw_gemm.h"
#include "qw_rows.h"

namespace {

#define QWR_FIELDS(X)                                                                                                       \
    X(const uint8_t*, bank) X(const void*, x) X(uint32_t, K) X(uint32_t, M) X(uint32_t, ldx) X(uint32_t, nsl) X(uint32_t, row_bytes)  \
    X(uint32_t, gshift) X(uint32_t, bb) X(uint32_t, N) X(uint32_t, units) X(uint32_t, nkr) X(uint32_t, flush) X(uint32_t, x_bf16)     \
    X(uint32_t, inter) X(uint32_t, rotate) X(void*, y) X(uint32_t, ldy) X(uint32_t, y_dtype) X(qw_act, act)
QW_ARG_BLOCK(qwr_params, QWR_FIELDS)

// Waves of a workgroup, by the registers of MF fragments over S steps: 128, 168 or 256 a lane.
constexpr uint32_t qwr_waves(uint32_t mf, uint32_t s) { return mf * s <= 4u ? 16u : mf * s <= 6u ? 12u : 8u; }

// blockDim.x = 64 * ceil(steps / (S nkr)); dynamic LDS = the waves' images, 2 * flush * waves * MF KiB of partial tiles and, GATED, the
// unit's sums, 4 tiles of 16 MF activation rows by 16 + 1.
template <int FMT, int MF, int S, bool GATED>
struct qw_gemm_rows_kernel {
static constexpr int kLaunchBound = 64 * qwr_waves(MF, S);
static __device__ __forceinline__ void run(const qwr_params& p) {
    extern __shared__ __attribute__((aligned(16))) uint32_t qwr_lds[];
    using im = qr_image<FMT, S>;
    constexpr uint32_t SPU = GATED ? 4u : 1u;    // row tiles of a unit: 32 channels' gates and ups
    constexpr uint32_t RPL = 16u / S;            // bank rows of a load: 4 S slices of each
    constexpr uint32_t ROWS = 16u * MF;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, W = blockDim.x >> 6;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t G = gridDim.x / p.nkr, band = blockIdx.x / p.nkr, kr = blockIdx.x - band * p.nkr;
    const uint32_t n = lane & 15u, c = lane >> 4;             // contraction role
    const uint32_t lb = lane / RPL, lj = lane & (RPL - 1u);   // load role: slice lb of the wave's, row RPL q + lj of the tile
    uint32_t* const img = qwr_lds + wave * im::DWORDS;
    f4_t* const parts = (f4_t*)(qwr_lds + W * im::DWORDS);
    float* const sums = (float*)(parts + (size_t)2u * p.flush * W * MF * 64u);
    if (band >= p.units) return;
    const uint32_t slots = (p.units - band + G - 1u) / G * SPU;
    const uint32_t magic = qw_vgpr_const(0x64006400u);

    uint32_t hdr, codes;
    qr_slice_at<FMT>(p, 4u * S * (kr * W + wave) + lb, hdr, codes);
    qg_slice<FMT> buf[S];
    auto request = [&](uint32_t slot) __attribute__((always_inline)) {
        uint32_t row;
        if constexpr (!GATED) {
            row = 16u * (slot * G + band);
        } else {
            const uint32_t k = slot >> 2, q = slot & 3u;
            row = 32u * (k * G + band) + 16u * (q & 1u) + (q >= 2u ? p.inter : 0u);
        }
        qr_for<S>([&](auto q) {
            const uint32_t ro = min(row + RPL * q + lj, p.N - 1u) * p.row_bytes;
            qr_load<FMT>(p, ro + hdr, ro + codes, buf[q]);
        });
    };
    request(0);
    __builtin_amdgcn_sched_barrier(0);
    u4_t raw[4 * S * MF];   // step, fragment, four rows a load: runs of 256 bytes; zero past M and past the row's end
    qr_for<4 * S * MF>([&](auto i) {
        const uint32_t col = 128u * ((kr * W + wave) * S + i / (4 * MF)) + 8u * (lane & 15u), row = 4u * (i % (4 * MF)) + (lane >> 4);
        u4_t v = {0u, 0u, 0u, 0u};
        if (row < p.M && col < p.K) v = *(const u4_t*)((const uint8_t*)p.x + (2u * row * p.ldx + 2u * col));
        raw[i] = v;
    });
    __builtin_amdgcn_sched_barrier(0);
    h8_t xo[S][MF][4];
    qr_for<S>([&](auto u) {
        qr_for<MF>([&](auto f) {
            qr_for<4>([&](auto q) {
                const u4_t v = raw[4 * MF * u + 4 * f + q];
                *(h8_t*)(img + (4u * q + c) * QR_XS + 4u * n) = p.x_bf16 ? qg_to_f16x8<QWHIP_BF16>(v) : qg_to_f16x8<QWHIP_F16>(v);
            });
            asm volatile("" ::: "memory");   // a wave's own LDS operations complete in order
            qr_for<4>([&](auto t) { xo[u][f][t] = *(const h8_t*)(img + n * QR_XS + 4u * (4u * c + t)); });
            asm volatile("" ::: "memory");
        });
    });

    uint32_t in_flush = 0, side = 0, first = 0;   // row tiles since the last sum, the half of the partial tiles, its first slot
#pragma unroll 1
    for (uint32_t slot = 0; slot < slots; ++slot) {
        qr_for<S>([&](auto q) { qr_park<FMT, S>(img, RPL * q + lj, lb, buf[q]); });
        asm volatile("" ::: "memory");
        if (slot + 1u < slots) request(slot + 1u);
        __builtin_amdgcn_sched_barrier(0);
        f4_t acc[MF];
#pragma unroll
        for (int f = 0; f < MF; ++f) acc[f] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < S; ++u) {
            qr_weight_step<FMT, S, MF>(img, u, n, c, xo[u], magic, acc);
            __builtin_amdgcn_sched_barrier(0);
        }
        f4_t* mine = parts + ((size_t)(side * p.flush + in_flush) * W + wave) * (MF * 64u) + lane;
#pragma unroll
        for (int f = 0; f < MF; ++f) mine[f * 64] = acc[f];
        asm volatile("" ::: "memory");
        ++in_flush;
        if (in_flush == p.flush || slot + 1u == slots) {
            __syncthreads();   // the other half of the partial tiles is free again: its sums lie before this barrier
            const f4_t* part = parts + (size_t)side * p.flush * W * MF * 64u;
            const uint32_t quads = 4u * ((p.M + 15u) >> 4);
            for (uint32_t e = tid; e < in_flush * 16u * quads; e += blockDim.x) {
                const uint32_t rr = e & 15u, sq = e >> 4, s = sq / quads, q = sq - s * quads;
                const f4_t v = qr_wave_sum<MF>(part + (size_t)s * W * MF * 64u, W, q, rr);
                if constexpr (GATED) {   // one tile a sum
                    float* to = sums + ((slot & 3u) * ROWS + 4u * q) * 17u + rr;
#pragma unroll
                    for (int r = 0; r < 4; ++r) to[r * 17] = (float)(h1_t)v[r];   // what the plain door stores
                } else {
                    const uint32_t row = 16u * ((first + s) * G + band) + rr;
#pragma unroll
                    for (uint32_t r = 0; r < 4; ++r) {
                        const uint32_t m = 4u * q + r;
                        if (m >= p.M || row >= p.N) continue;
                        if (p.nkr > 1u) {
                            ((float*)p.y)[((uint64_t)kr * p.M + m) * p.N + row] = v[r];
                        } else {
                            const uint64_t at = (uint64_t)m * p.ldy + row;
                            if (p.y_dtype == QWHIP_F32) qg_store<QWHIP_F32>(p.y, at, v[r]);
                            else if (p.y_dtype == QWHIP_F16) qg_store<QWHIP_F16>(p.y, at, v[r]);
                            else qg_store<QWHIP_BF16>(p.y, at, v[r]);
                        }
                    }
                }
            }
            in_flush = 0;
            side ^= 1u;
            first = slot + 1u;
            if constexpr (GATED) {
                if ((slot & 3u) == 3u) {
                    __syncthreads();
                    const uint32_t j = tid & 31u, c0 = 32u * ((slot >> 2) * G + band);
                    const qw_fwht32_signs sg = qw_fwht32_lane_signs(j);
                    for (uint32_t e = tid; e < ((32u * p.M + 63u) & ~63u); e += blockDim.x) {   // whole waves: the rotation exchanges lanes
                        const uint32_t m = min(e >> 5, p.M - 1u);
                        const float* g = sums + ((j >> 4) * ROWS + m) * 17u + (j & 15u);
                        float v = qw_gated(g[0], g[2u * ROWS * 17u], p.act);
                        if (p.rotate) {
                            v = qw_fwht32_lanes(v, sg) * QW_INV_SQRT32;
                            asm volatile("" : "+v"(v));   // rounded to fp32 and then to f16, as the rotation pass does (not by one mixed instruction)
                        }
                        if (e < 32u * p.M) ((h1_t*)p.y)[(uint64_t)m * p.ldy + c0 + j] = (h1_t)v;
                    }
                    // the next unit's sums lie behind the next tile's barrier
                }
            }
        }
    }
}
};

template <int FMT>
constexpr uint32_t qwr_image_bytes(uint32_t s) { return 4u * (s == 1u ? qr_image<FMT, 1>::DWORDS : qr_image<FMT, 2>::DWORDS); }
uint32_t qwr_image_bytes(int fmt, uint32_t s) {
    switch (fmt) {
        case QG_FMT_M5: return qwr_image_bytes<QG_FMT_M5>(s);
        case QG_FMT_B4: return qwr_image_bytes<QG_FMT_B4>(s);
        case QG_FMT_B8: return qwr_image_bytes<QG_FMT_B8>(s);
        case QG_FMT_B2: return qwr_image_bytes<QG_FMT_B2>(s);
        case QG_FMT_B3: return qwr_image_bytes<QG_FMT_B3>(s);
        default: return qwr_image_bytes<QG_FMT_B6>(s);
    }
}
uint32_t qwr_fragments(uint32_t m) { return max(2u, qwhip_cdiv(m, 16u)); }

// A launch with s steps a wave over `ranges` K ranges; waves = 0: more waves or LDS than a workgroup has, or an empty range.
struct qwr_config {
    uint32_t waves, units, per_cu, bands, flush, lds;
};
qwr_config qwr_configure(int fmt, uint32_t m, uint32_t n, uint32_t k, uint32_t s, uint32_t ranges, bool gated) {
    const uint32_t mf = qwr_fragments(m), steps = qwhip_cdiv(k, 128u), most = 160u * 1024u;
    qwr_config c = {};
    const uint32_t waves = qwhip_cdiv(steps, s * ranges), image = waves * qwr_image_bytes(fmt, s), part = 2u * waves * mf * 1024u;
    // one range fits with the gated form's sums too: both doors take one kernel, and give the same bits
    const uint32_t gated_sums = 4u * 16u * mf * 17u * 4u, sums = gated ? gated_sums : 0u;
    if (waves > qwr_waves(mf, s) || image + part + (ranges == 1u ? gated_sums : 0u) > most || (ranges - 1u) * waves * s >= steps) return c;
    c.waves = waves;
    c.units = gated ? n / 64u : n / 16u;
    c.per_cu = max(1u, min(qwr_waves(mf, s) / waves, most / (image + part + sums)));
    c.bands = min(c.units, max(1u, 256u * c.per_cu / ranges));
    c.flush = gated ? 1u : max(1u, min(min(4u, qwhip_cdiv(c.units, c.bands)), (most / c.per_cu - image) / part));
    c.lds = image + c.flush * part + sums;
    return c;
}
// A row tile on a compute unit, us, and a launch's activations: see qw_gemm_rows_choose.
double qwr_tile_us(int fmt, uint32_t m, const qwr_config& c, uint32_t s, uint32_t ranges, double* start) {
    const double unpack = fmt == QG_FMT_B8 ? 1.86 : fmt == QG_FMT_B6 ? 1.98 : fmt == QG_FMT_B3 ? 1.73 : 1.0;
    const double steps = c.waves * max(1u, qwhip_cdiv(c.bands * ranges, 256u)) * s / 4.0;   // a SIMD's
    *start = 0.184 * steps * qwr_fragments(m);
    return 0.56 + steps * (0.07 * unpack + 0.043 * qwr_fragments(m));
}

template <int FMT, int MF, int S, bool GATED>
hipError_t qwr_go(hipStream_t st, const qwr_params& p, const qwr_config& c) {
    using K = qw_gemm_rows_kernel<FMT, MF, S, GATED>;
    static std::atomic<bool> attr_done{false};   // per instantiation
    if (!attr_done.load(std::memory_order_acquire)) {
        const hipError_t e = hipFuncSetAttribute(qw_scalar_kernel_ptr<K>((const qwr_params*)nullptr), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return e;
        attr_done.store(true, std::memory_order_release);
    }
    qw_launch_scalar<K>(dim3(c.bands * p.nkr), dim3(64u * c.waves), c.lds, st, p);
    return hipGetLastError();
}
template <int FMT>
hipError_t qwr_launch(hipStream_t st, const qwr_params& p, const qwr_config& c, uint32_t s, bool gated) {
#define QWR_GO(MF, S) (gated ? qwr_go<FMT, MF, S, true>(st, p, c) : qwr_go<FMT, MF, S, false>(st, p, c))
    const uint32_t mf = qwr_fragments(p.M);
    if (s == 1u) return mf == 2u ? QWR_GO(2, 1) : mf == 3u ? QWR_GO(3, 1) : QWR_GO(4, 1);
    return mf == 2u ? QWR_GO(2, 2) : mf == 3u ? QWR_GO(3, 2) : QWR_GO(4, 2);
#undef QWR_GO
}

}  // namespace

// The steps a wave and the K ranges with the lowest price, us, if that is below `limit`; ranges (0: any): only as many.
// A launch 3.4 and the activations, a wave's registers full of them; then row tiles, one after the other on a compute unit: 0.56 for the
// barrier and the sums, and for every step on a SIMD its unpacking and its products; more ranges pay their planes, at 5 TB/s, and the
// summing launch; and no faster than the bank streams (7.4 TB/s, in quadrature).  Fitted to 4700 measured forms of 660 problems, 17 .. 64
// rows on 220 banks of 12 containers (n 1024 .. 36000, k 1024 .. 17408): 7.6 % of root mean square error.  Of the other kernels' times on
// these problems (choose_direct) the form chosen takes 0.63 up to 32 rows, 0.67 up to 48, 0.77 up to 64, none of them slower; of 836 others, half
// of them gate|up, five are slower by more than 3 %, up to 13 % (64 x 33792 x 1536 gate|up HQ4_G128 23.7 us, 26.7).  On banks of
// many rows with 64 activation rows the tiles keep the lead (64 x 34816 x 5120 HQ4_G32_M5 62 us, 53 there).
bool qw_gemm_rows_choose(int fmt, uint32_t m, uint32_t n, uint32_t k, uint64_t row_bytes, uint64_t plane_room, uint32_t ranges, double limit,
                         uint32_t* steps, uint32_t* chosen) {
    if (m > 64u || (uint64_t)n * row_bytes >= (1ull << 32)) return false;   // 32-bit offsets inside the bank
    const double bank = (double)n * (double)row_bytes / 7.4e6, planes = (double)m * n * 8.0 / 5.2e6;
    bool found = false;
    for (uint32_t s = 1; s <= 2u; ++s) {
        const uint32_t least = max(1u, qwhip_cdiv(qwhip_cdiv(k, 128u), s * qwr_waves(qwr_fragments(m), s)));
        for (uint32_t r = ranges ? ranges : least; r <= (ranges ? ranges : least + 3u); ++r) {
            if (r > 1u && r * (uint64_t)m * n * 4u > plane_room) continue;
            const qwr_config c = qwr_configure(fmt, m, n, k, s, r, false);
            if (c.waves == 0u) continue;
            double start, t = 3.4;
            t += qwhip_cdiv(c.units, c.bands) * qwr_tile_us(fmt, m, c, s, r, &start) + start;
            if (r > 1u) t += 1.6 + 0.15 * r + r * planes;
            t = std::hypot(t, bank);
            if (t < limit) limit = t, *steps = s, *chosen = r, found = true;
        }
    }
    return found;
}
// Whether gate|up of one range is faster with its activation in the launch: whole units of 32 channels leave workgroups with more tiles
// than others, the activation pass over one fp32 plane is a launch and the plane's traffic.
bool qw_gemm_rows_fuses(int fmt, uint32_t m, uint32_t n, uint32_t k, uint32_t s) {
    const qwr_config f = qwr_configure(fmt, m, n, k, s, 1u, true), c = qwr_configure(fmt, m, n, k, s, 1u, false);
    if (f.waves == 0u) return false;
    double start, start_f;
    const double fused = 4.0 * qwhip_cdiv(f.units, f.bands) * qwr_tile_us(fmt, m, f, s, 1u, &start_f);
    const double plain = qwhip_cdiv(c.units, c.bands) * qwr_tile_us(fmt, m, c, s, 1u, &start);
    return fused + start_f < plain + start + 2.0 + (double)m * n * 8.0 / 5.2e6;
}

hipError_t qw_gemm_rows(hipStream_t st, int fmt, const qw_gemm_params& g, uint32_t steps, uint32_t ranges, uint32_t xdt, uint32_t ydt, bool swiglu) {
    const qwr_config c = qwr_configure(fmt, g.M, g.N, g.K, steps, ranges, swiglu);
    if (c.waves == 0u) return hipErrorInvalidValue;
    qwr_params p;
    p.bank = g.bank;
    p.x = g.x;
    p.K = g.K;
    p.M = g.M;
    p.ldx = g.ldx;
    p.nsl = g.K / 32u;
    p.row_bytes = (uint32_t)g.row_bytes;
    p.gshift = g.gshift;
    p.bb = g.bb;
    p.N = g.N;
    p.units = c.units;
    p.nkr = ranges;
    p.flush = c.flush;
    p.x_bf16 = xdt == QWHIP_BF16 ? 1u : 0u;
    p.inter = g.inter;
    p.rotate = g.rotate_act;
    p.y = g.y;
    p.ldy = g.ldy;
    p.y_dtype = ydt;
    p.act = g.act;
    switch (fmt) {
        case QG_FMT_M5: return qwr_launch<QG_FMT_M5>(st, p, c, steps, swiglu);
        case QG_FMT_B4: return qwr_launch<QG_FMT_B4>(st, p, c, steps, swiglu);
        case QG_FMT_B8: return qwr_launch<QG_FMT_B8>(st, p, c, steps, swiglu);
        case QG_FMT_B2: return qwr_launch<QG_FMT_B2>(st, p, c, steps, swiglu);
        case QG_FMT_B3: return qwr_launch<QG_FMT_B3>(st, p, c, steps, swiglu);
        default: return qwr_launch<QG_FMT_B6>(st, p, c, steps, swiglu);
    }
}
