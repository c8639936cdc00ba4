// Grouped (MoE) GEMM of few rows an expert on the row-tile form of gemv_rows.hip: one or two fragments of an expert's sorted rows
// share a tile of 16 of its bank rows.
//
// A workgroup takes up to 32 rows of a tile-list entry and a band of the expert's row tiles; its waves split the columns and keep the
// rows' columns in registers for all the band.  The launch reads every routed expert's bank once and is bound by that stream: the
// direct-operand kernel's four waves wait for a K-step's loads and their way through LDS at a barrier each, with 1 to 32 rows to
// multiply.
#include <algorithm>
#include <atomic>
#include <cmath>

#include "qw_gemm.h"
#include "qw_rows.h"

namespace {

#define QMR_FIELDS(X)                                                                                                       \
    X(const uint8_t*, bank) X(const int32_t*, tile_count) X(const int32_t*, tile_e) X(const int32_t*, tile_r)                    \
    X(const int32_t*, expert_off) X(uint32_t, max_tiles) X(uint32_t, wgs) X(uint32_t, units) X(uint32_t, nsl) X(uint32_t, gshift) X(uint32_t, bb) X(const int32_t*, gather)  \
    X(const void*, x) X(uint64_t, expert_bytes) X(uint32_t, row_bytes) X(uint32_t, N) X(uint32_t, K) X(uint32_t, ldx)   \
    X(uint32_t, x_bf16) X(uint32_t, flush) X(uint32_t, inter) X(uint32_t, rotate) X(void*, y) X(uint32_t, ldy) X(uint32_t, y_dtype)        \
    X(qw_act, act)
QW_ARG_BLOCK(qmr_params, QMR_FIELDS)

constexpr uint32_t QMR_LISTS = 12;                  // 64 entries of the tile list each
constexpr uint32_t QMR_LDS = 160u * 1024u - 512u;   // dynamic LDS of a unit, beside the items found

// Waves of a workgroup, by the registers of MF fragments over S steps.
constexpr uint32_t qmr_waves(uint32_t mf, uint32_t s) { return mf * s <= 2u ? 16u : 12u; }

// blockDim.x = 64 * ceil(steps / S); dynamic LDS = the waves' images, 2 * flush * waves * MF KiB of partial tiles and, GATED, the unit's
// sums, 4 tiles of 16 MF rows by 16 + 1.
// Grid: every 16 MF rows of an entry are a chunk, and the chunks that there are, counted here, share the launch's workgroups, each in as many
// bands as come out even; an XCD takes a contiguous eighth of (entry, band, chunk), so that the chunks of a busy expert run side by side under
// one L2 and no XCD has more than another however the routes fall.  (With the host's bands, a grid for four chunks of every entry and eighths
// of the list, the late chunks were a round of their own behind the empty workgroups, and the XCD of the busy experts had most of them.)
// 64 rows x top-8 of 128 experts, 2048 x 768, gate|up and down, us: even routes 51 and 29 (the direct-operand kernel 70 and 42), routes
// falling as 1 / rank 50 and 28 (before 77 and 44, direct-operand 65 and 38), all tokens on the same eight 15 and 10 (35 and 19; 25 and 12).
// Finding its chunk costs a workgroup 0.4 us: 25 rows x top-2 of 16 experts, down of 2304 x 384, HQ4_G32, 6.0 -> 6.5.
template <int FMT, int S, int MF, bool GATED>
struct qw_moe_rows_kernel {
static constexpr int kLaunchBound = 64 * qmr_waves(MF, S);

static __device__ __forceinline__ void rows(const qmr_params& p, const uint8_t* bank, uint32_t m0, uint32_t M, uint32_t band, uint32_t G, uint32_t* lds) {
    using im = qr_image<FMT, S>;
    constexpr uint32_t SPU = GATED ? 4u : 1u, RPL = 16u / S, ROWS = 16u * MF;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, W = blockDim.x >> 6;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t n = lane & 15u, c = lane >> 4;             // contraction role
    const uint32_t lb = lane / RPL, lj = lane & (RPL - 1u);   // load role: slice lb of the wave's, row RPL q + lj of the tile
    uint32_t* const img = lds + wave * im::DWORDS;
    f4_t* const parts = (f4_t*)(lds + W * im::DWORDS);
    float* const sums = (float*)(parts + (size_t)2u * p.flush * W * MF * 64u);
    const uint32_t slots = (p.units - band + G - 1u) / G * SPU;
    const uint32_t magic = qw_vgpr_const(0x64006400u);

    // the rows' places first: the activations wait for them, the bank's first tile for nothing
    const uint32_t xrow = min(lane, M - 1u);
    const uint32_t src_row = p.gather ? (uint32_t)p.gather[m0 + xrow] : m0 + xrow;
    struct place { const uint8_t* bank; uint32_t nsl, gshift, bb; } at = {bank, p.nsl, p.gshift, p.bb};
    uint32_t hdr, codes;
    qr_slice_at<FMT>(at, 4u * S * wave + lb, hdr, codes);
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
            qr_load<FMT>(at, ro + hdr, ro + codes, buf[q]);
        });
    };
    request(0);
    __builtin_amdgcn_sched_barrier(0);
    u4_t raw[4 * S * MF];   // step, fragment, four rows a load: runs of 256 bytes; zero past M and past the row's end
    qr_for<4 * MF>([&](auto f) {
        const uint32_t row = 4u * f + c, from = (uint32_t)__shfl((int)src_row, (int)min(row, 63u), 64);
        qr_for<S>([&](auto u) {
            const uint32_t col = 128u * (wave * S + u) + 8u * n;
            u4_t v = {0u, 0u, 0u, 0u};
            if (row < M && col < p.K) v = *(const u4_t*)((const uint8_t*)p.x + (2u * from * p.ldx + 2u * col));
            raw[4 * MF * u + f] = v;
        });
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
            const uint32_t quads = (M + 3u) >> 2;
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
                        if (m >= M || row >= p.N) continue;
                        const uint64_t to = (uint64_t)(m0 + m) * p.ldy + row;
                        if (p.y_dtype == QWHIP_F32) qg_store<QWHIP_F32>(p.y, to, v[r]);
                        else if (p.y_dtype == QWHIP_F16) qg_store<QWHIP_F16>(p.y, to, v[r]);
                        else qg_store<QWHIP_BF16>(p.y, to, v[r]);
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
                    for (uint32_t e = tid; e < ((32u * M + 63u) & ~63u); e += blockDim.x) {   // whole waves: the rotation exchanges lanes
                        const uint32_t m = min(e >> 5, M - 1u);
                        const float* g = sums + ((j >> 4) * ROWS + m) * 17u + (j & 15u);
                        float v = qw_gated(g[0], g[2u * ROWS * 17u], p.act);
                        if (p.rotate) {
                            v = qw_fwht32_lanes(v, sg) * QW_INV_SQRT32;
                            asm volatile("" : "+v"(v));   // rounded to fp32 and then to f16, as the rotation pass does (not by one mixed instruction)
                        }
                        if (e < 32u * M) ((h1_t*)p.y)[(uint64_t)(m0 + m) * p.ldy + c0 + j] = (h1_t)v;
                    }
                    // the next unit's sums lie behind the next tile's barrier
                }
            }
        }
    }
}

// The workgroup's entry, chunk of rows and band, and the bands of this launch.  Every wave finds them: no barrier in front of the bank's loads.
struct item { uint32_t e, packed, chunk, band, bands, valid; };
static __device__ __forceinline__ item find(const qmr_params& p, uint32_t lane) {
    const uint32_t tc = min((uint32_t)max(p.tile_count[0], 0), p.max_tiles);   // the lists end there
    uint32_t te[QMR_LISTS], tr[QMR_LISTS];
#pragma unroll
    for (uint32_t j = 0; j < QMR_LISTS; ++j) {
        if (64u * j >= tc) break;
        const uint32_t t = min(64u * j + lane, tc - 1u);
        te[j] = (uint32_t)p.tile_e[t];
        tr[j] = (uint32_t)p.tile_r[t];
    }
    // chunks of an entry of 16, 32 or 64 rows: 1, 2 or 4 (MF = 1), 1, 1 or 2
    auto count = [&](uint32_t j) { return 64u * j + lane >= tc ? 0u : tr[j] >> 24 == 1u ? 1u : tr[j] >> 24 == 2u ? 2u / MF : 4u / MF; };
    uint32_t total = 0;
#pragma unroll
    for (uint32_t j = 0; j < QMR_LISTS; ++j) {
        if (64u * j >= tc) break;
        const uint32_t n = count(j);
        total += __popcll(__ballot(n > 0u)) + __popcll(__ballot(n > 1u)) + 2u * __popcll(__ballot(n > 2u));
    }
    item it = {};
    if (total == 0u) return it;
    const uint32_t bands = min(max(p.wgs / total, 1u), p.units);
    const uint32_t items = total * bands, per_xcd = (items + 7u) >> 3, at = blockIdx.x >> 3, i = (blockIdx.x & 7u) * per_xcd + at, q = i / bands;
    if (at >= per_xcd || i >= items) return it;
    uint32_t before = 0;
#pragma unroll
    for (uint32_t j = 0; j < QMR_LISTS; ++j) {
        if (64u * j >= tc) break;
        const uint32_t n = count(j);
        const unsigned long long b0 = __ballot(n > 0u), b1 = __ballot(n > 1u), b2 = __ballot(n > 2u);
        auto lower = [](unsigned long long b) { return __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u)); };
        const uint32_t mine = before + lower(b0) + lower(b1) + 2u * lower(b2);
        const unsigned long long hit = __ballot(q >= mine && q < mine + n);
        if (hit != 0ull) {
            const uint32_t l = (uint32_t)__builtin_ctzll(hit);
            const uint32_t local = i - __builtin_amdgcn_readlane(mine, l) * bands, chunks = __builtin_amdgcn_readlane(n, l);
            it.band = local >> (chunks >> 1);   // 1, 2 or 4
            it.chunk = local & (chunks - 1u);
            it.e = __builtin_amdgcn_readlane(te[j], l);
            it.packed = __builtin_amdgcn_readlane(tr[j], l);
            it.bands = bands;
            it.valid = 1u;
            return it;
        }
        before += __popcll(b0) + __popcll(b1) + 2u * __popcll(b2);
    }
    return it;
}

static __device__ __forceinline__ void run(const qmr_params& p) {
    extern __shared__ __attribute__((aligned(16))) uint32_t qmr_lds[];
    const item it = find(p, threadIdx.x & 63u);
    if (it.valid == 0u) return;
    const uint32_t e = it.e, packed = it.packed, chunk = it.chunk;
    const uint32_t code = packed >> 24, bm = code == 1u ? 16u : code == 2u ? 32u : 64u;   // rows of the entry's tile
    const uint32_t first = (packed & 0xFFFFFFu) * bm + 16u * MF * chunk;                  // row of the expert
    const uint32_t off = (uint32_t)p.expert_off[e], rows_e = (uint32_t)p.expert_off[e + 1] - off;
    if (first >= rows_e) return;
    const uint32_t M = min(min(16u * MF, bm - 16u * MF * chunk), rows_e - first);
    rows(p, p.bank + (uint64_t)e * p.expert_bytes, off + first, M, it.band, it.bands, qmr_lds);
}
};

template <int FMT, int S, int MF, bool GATED>
hipError_t qmr_go(hipStream_t st, const qmr_params& p, uint32_t wgs, uint32_t waves, size_t lds) {
    using K = qw_moe_rows_kernel<FMT, S, MF, GATED>;
    static std::atomic<bool> attr_done{false};   // per instantiation
    if (!attr_done.load(std::memory_order_acquire)) {
        const hipError_t e = hipFuncSetAttribute(qw_scalar_kernel_ptr<K>((const qmr_params*)nullptr), hipFuncAttributeMaxDynamicSharedMemorySize, (int)QMR_LDS);
        if (e != hipSuccess) return e;
        attr_done.store(true, std::memory_order_release);
    }
    qw_launch_scalar<K>(dim3(wgs), dim3(64u * waves), lds, st, p);
    return hipGetLastError();
}
template <int FMT>
constexpr uint32_t qmr_image_bytes(uint32_t s) { return 4u * (s == 1u ? qr_image<FMT, 1>::DWORDS : qr_image<FMT, 2>::DWORDS); }
uint32_t qmr_image_bytes(int fmt, uint32_t s) {
    switch (fmt) {
        case QG_FMT_M5: return qmr_image_bytes<QG_FMT_M5>(s);
        case QG_FMT_B4: return qmr_image_bytes<QG_FMT_B4>(s);
        case QG_FMT_B8: return qmr_image_bytes<QG_FMT_B8>(s);
        case QG_FMT_B2: return qmr_image_bytes<QG_FMT_B2>(s);
        case QG_FMT_B3: return qmr_image_bytes<QG_FMT_B3>(s);
        default: return qmr_image_bytes<QG_FMT_B6>(s);
    }
}

// Steps a wave: by the bank's container and columns alone, so that both doors add in one order.  Two, the waves of several workgroups to a
// unit; one where that would leave two waves, and on 8-bit banks up to 1536 columns (32 experts, 6 rows each, 1536 x 1536: 18.6 us, 19.5).
uint32_t qmr_steps(int fmt, uint32_t k) {
    const uint32_t steps = k / 128u;
    return steps <= 5u || (fmt == QG_FMT_B8 && steps <= 12u) ? 1u : 2u;
}

// What the routes make of a call: the experts that have rows and their tiles of 16, 32 and 64 rows.
struct qmr_load {
    double used, tiles[3], stream;   // stream: us of a launch that reads those experts' banks
};
// The host does not see the routes.  Prices are taken for three: even ones (rows an expert: Poisson), rows falling as 1 / rank (experts of
// neighbouring ranks together) and all rows on four experts.
void qmr_loads(const qw_gemm_params& p, uint32_t experts, qmr_load (&out)[3]) {
    const uint32_t rows = p.M;
    auto add = [](qmr_load& l, double n, double mean) {   // n experts; the tiles of Poisson rows to 5 % (up to 19 % at 0.75 of a tile)
        const double some = 1.0 - std::exp(-mean);
        l.used += n * some;
        for (int i = 0; i < 3; ++i) {
            const double b = 16 << i;
            l.tiles[i] += n * (mean < 2.2 * b ? some + std::max(0.0, mean / b - 0.55) : mean / b + 0.5);
        }
    };
    for (qmr_load& l : out) l = {};
    add(out[0], experts, rows / (double)experts);
    const double all = std::log((double)experts) + 0.577;
    for (uint32_t lo = 1, hi; lo <= experts; lo = hi + 1u) {
        hi = min(experts, max(lo, lo * 3u / 2u));
        const double n = hi - lo + 1u;
        add(out[1], n, rows * std::log((hi + 0.5) / (lo - 0.5)) / (all * n));
    }
    const uint32_t few = min(experts, 4u);
    add(out[2], few, rows / (double)few);
    for (qmr_load& l : out) l.stream = 3.9 + l.used * (double)p.N * (double)p.row_bytes / 4.75e6;
}

struct qmr_config {
    uint32_t waves, mf, units, wgs, flush, lds;   // waves = 0: none fits
    double us[3];                                 // by kind of route
};
// The launch with the lowest price, us, over the three kinds of routes (product of the even one's square, the second's and the fourth root of the
// third's): fragments of rows, and workgroups for the bands of row tiles of all chunks together (find).  A launch 3.9; then rounds of workgroups, one's activations and row tiles, a tile costing 0.36 (gate|up
// 0.42) and every step's unpacking and products on a SIMD; no faster than 4.75 TB/s of the experts that have rows.  The chunks as they are and a
// tenth more, in the mean of both: one more than the workgroups hold is another round of them.  Fitted to 19000 measured launches: up to 12
// forms of 800 calls (16 .. 256 experts, 0.1 .. 24 rows each, 12 containers) on each kind of routes, 11 % of root mean square error.
qmr_config qmr_choose(int fmt, const qw_gemm_params& p, const qmr_load (&loads)[3], bool gated) {
    const uint32_t s = qmr_steps(fmt, p.K), waves = qwhip_cdiv(p.K / 128u, s), units = gated ? p.inter / 32u : qwhip_cdiv(p.N, 16u);
    const double unpack = fmt == QG_FMT_B8 ? 1.87 : fmt == QG_FMT_B6 ? 2.04 : fmt == QG_FMT_B3 ? 1.66 : fmt == QG_FMT_B2 ? 1.42 : fmt == QG_FMT_B4 ? 1.33 : 1.0;
    qmr_config best = {};
    double lowest = 1e300;
    for (uint32_t mf = 1; mf <= 2u; ++mf) {
        const uint32_t image = waves * qmr_image_bytes(fmt, s), part = 2u * waves * mf * 1024u, sums = 4u * 16u * mf * 17u * 4u;
        if (waves > qmr_waves(mf, s) || image + part + sums > QMR_LDS) continue;
        const uint32_t per_cu = max(1u, min(qmr_waves(mf, s) / waves, QMR_LDS / (image + part + sums)));
        for (uint32_t i : {1u, 2u, 3u, 4u, 6u, 8u}) {   // workgroups a unit in all
            if (i > 2u * per_cu) break;
            double us[3];
            uint32_t run = 1;   // row tiles of a workgroup on even routes
            for (int r = 2; r >= 0; --r) {
                us[r] = 0.0;
                for (double c : {1.1 * loads[r].tiles[mf - 1u], loads[r].tiles[mf - 1u]}) {
                    const uint32_t bands = min(max(1u, (uint32_t)(256u * i / c)), units), longest = qwhip_cdiv(units, bands);
                    const double load = c * qwhip_cdiv(units, longest) / 256.0, side = std::min((double)min(per_cu, i), std::max(1.0, std::ceil(load)));
                    run = longest * (gated ? 4u : 1u);
                    const double tile = (gated ? 0.416 : 0.355) + waves * side / 4.0 * s * (0.118 * unpack + 0.054 * mf);
                    us[r] += 0.5 * std::max(loads[r].stream, 3.9 + std::max(1.0, std::ceil(load / side - 0.01)) * (0.25 * s * mf + run * tile));
                }
            }
            const double all = us[0] * us[0] * us[1] * std::sqrt(std::sqrt(us[2]));
            if (all >= lowest) continue;
            lowest = all;
            best.waves = waves, best.mf = mf, best.units = units, best.wgs = 256u * i;
            for (int r = 0; r < 3; ++r) best.us[r] = us[r];
            best.flush = gated ? 1u : max(1u, min(min(4u, run), (QMR_LDS / min(per_cu, i) - image) / part));
            best.lds = image + best.flush * part + (gated ? sums : 0u);
        }
    }
    return best;
}
// The direct-operand kernel's price, on spans of 64 rows, which it takes for this few rows an expert: 9 % of root mean square error on the
// same 2400 calls.
double qmr_direct_us(int fmt, const qw_gemm_params& p, const qmr_load& l) {
    const double load = l.tiles[2] * qwhip_cdiv(p.N, 256u) / 256.0, deep = 1.0 + 0.07 * (std::max(1.0, l.tiles[1] / l.tiles[2]) - 1.0);
    const double rounds = load <= 1.0 ? 1.0 + 0.48 * load : load <= 2.0 ? 1.41 + 0.59 * load : 0.34 + 1.32 * load;
    const double step = fmt == QG_FMT_B8 ? 1.67 : fmt == QG_FMT_B6 ? 1.54 : fmt == QG_FMT_B2 ? 1.09 : fmt == QG_FMT_B4 ? 1.17 : 1.15;
    return 4.8 + std::max(p.K / 128u * step * rounds * deep, l.used * (double)p.N * (double)p.row_bytes / 3.8e6);
}

template <int FMT>
hipError_t qmr_launch(hipStream_t st, const qmr_params& p, const qmr_config& c, uint32_t s, bool gated) {
    const uint32_t wgs = max(c.wgs, 8u * qwhip_cdiv(p.max_tiles * (4u / c.mf), 8u));   // a workgroup for every chunk there can be
#define QMR_GO(S, M) (gated ? qmr_go<FMT, S, M, true>(st, p, wgs, c.waves, c.lds) : qmr_go<FMT, S, M, false>(st, p, wgs, c.waves, c.lds))
    if (s == 1u) return c.mf == 1u ? QMR_GO(1, 1) : QMR_GO(1, 2);
    return c.mf == 1u ? QMR_GO(2, 1) : QMR_GO(2, 2);
#undef QMR_GO
}

}  // namespace

// Up to 24 rows an expert, where the price is under the direct-operand kernel's, 0.95 of it, on each kind of routes.  Over 2000 calls (16 .. 256
// experts, 0.1 .. 24 rows each, 12 containers, cold banks), of that kernel's time where this one takes them: even routes 0.68, 1 / rank 0.65, all
// tokens on the same experts 0.54; of 704 down projections 5 slower by more than 3 %, up to 1.18, of 802 gate|up calls 23, up to 1.27.  (The price
// of even routes alone, which decided before, let through calls up to 2.1 times as slow on the same experts and 1.9 times on 1 / rank, each chunk of
// 16 rows unpacking the expert again: 966 rows x top-2 of 256 experts, 1792 x 512, 20.6 us, now 11.0.  Refused with them are some even calls
// that it served better: 150 rows x top-8 of 256 experts, 1792 x 384, 45 -> 62 us.)
// Both doors take the kernel by the plain door's price: one arithmetic.
bool qw_grouped_rows(hipStream_t st, int fmt, const qw_gemm_params& g, uint32_t max_tiles, uint32_t experts, uint32_t xdt, uint32_t ydt, bool swiglu,
                     hipError_t* err) {
    if (g.M > 24u * experts || max_tiles > 64u * QMR_LISTS) return false;
    qmr_load loads[3];
    qmr_loads(g, experts, loads);
    qmr_config c = qmr_choose(fmt, g, loads, false);
    if (c.waves == 0u) return false;
    for (int r = 0; r < 3; ++r)
        if (!(c.us[r] < 0.95 * qmr_direct_us(fmt, g, loads[r]))) return false;
    if (swiglu) c = qmr_choose(fmt, g, loads, true);   // fits where the plain form does
    const uint32_t s = qmr_steps(fmt, g.K);
    qmr_params p;
    p.bank = g.bank;
    p.tile_count = g.tile_count;
    p.tile_e = g.tile_e;
    p.tile_r = g.tile_r;
    p.expert_off = g.expert_off;
    p.max_tiles = max_tiles;
    p.wgs = c.wgs;
    p.nsl = g.K / 32u;
    p.gshift = g.gshift;
    p.bb = g.bb;
    p.gather = g.gather;
    p.x = g.x;
    p.expert_bytes = (uint64_t)g.rows_per_expert * g.row_bytes;
    p.row_bytes = (uint32_t)g.row_bytes;
    p.N = g.N;
    p.units = c.units;
    p.K = g.K;
    p.ldx = g.ldx;
    p.x_bf16 = xdt == QWHIP_BF16 ? 1u : 0u;
    p.flush = c.flush;
    p.inter = g.inter;
    p.rotate = g.rotate_act;
    p.y = g.y;
    p.ldy = g.ldy;
    p.y_dtype = ydt;
    p.act = g.act;
    switch (fmt) {
        case QG_FMT_M5: *err = qmr_launch<QG_FMT_M5>(st, p, c, s, swiglu); break;
        case QG_FMT_B4: *err = qmr_launch<QG_FMT_B4>(st, p, c, s, swiglu); break;
        case QG_FMT_B8: *err = qmr_launch<QG_FMT_B8>(st, p, c, s, swiglu); break;
        case QG_FMT_B2: *err = qmr_launch<QG_FMT_B2>(st, p, c, s, swiglu); break;
        case QG_FMT_B3: *err = qmr_launch<QG_FMT_B3>(st, p, c, s, swiglu); break;
        default: *err = qmr_launch<QG_FMT_B6>(st, p, c, s, swiglu); break;
    }
    return true;
}
