// Host side of the grouped (MoE) GEMM on direct weight operands (qw_direct.h).
#include <algorithm>

#include "qw_direct_launch.h"

namespace {

// workgroups of tall spans a unit, from the mean of rows an expert (half a span of remainder where they are more than one's)
double tall_load(int fmt, const qw_gemm_params& p, uint32_t experts) {
    const double used = std::min(experts, p.M), span = fmt == QG_FMT_B8 || fmt == QG_FMT_B6 ? 96.0 : 128.0;
    return used * std::max(1.0, p.M / used / span + 0.5) * p.tiles_n / 256.0;
}
// 64-row spans, three waves a SIMD, or tall ones (128 rows, 96 on the 6- and 8-bit containers), which unpack a chunk for more products at
// two.  From 80 layers x 8 .. 10 row counts, 12 containers, 8 .. 256 experts, 64-row time over tall: under 1.5 workgroups a unit the
// taller, fewer ones leave units idle (16 experts, 128 rows each: down of 1536 x 1536 20.4 us / 33.8, gate|up of 3072 x 1536 67 / 94); past
// that 4-bit and narrower containers 0.96 .. 0.99 up to three and 1.03 .. 1.08 past, 6- and 8-bit ones 1.03 .. 1.13; on short K, whose starts
// and ends weigh more, 0.85 .. 1.0 (64 experts, 128 rows each, 2048 x 512: 37.7 / 41.6).  HQ4_G32_M5's short unpack has nothing to
// amortise on K up to 1536 (0.83 .. 1.0; past three workgroups a unit 0.99 .. 1.04 up to K = 2048, 1.05 past).  Up to 48 rows an expert both are the same spans and the three waves win (0.92 .. 1.0), but for
// three to four workgroups a unit, two rounds of either (1.04 .. 1.08).
template <int FMT>
bool few_rows(const qw_gemm_params& p, uint32_t experts) {
    const double rows = p.M / (double)std::min(experts, p.M), load = tall_load(FMT, p, experts);
    if (FMT == QG_FMT_B8 || FMT == QG_FMT_B6) return rows <= 48.0 || load < (p.K <= 512u ? 3.0 : 1.5);
    if (rows <= 48.0) return !(load > 3.0 && load <= 4.0);
    return load < 3.0 || p.K <= (FMT == QG_FMT_M5 ? 1536u : 512u);
}
template <int FMT>
hipError_t launch(hipStream_t st, const qw_gemm_params& p, uint32_t max_tiles, uint32_t experts, uint32_t xdt, uint32_t ydt, bool swiglu) {
    return qd_launch_x<FMT, false>(st, p, max_tiles, xdt, ydt, swiglu, few_rows<FMT>(p, experts));
}

}  // namespace

bool qw_grouped_direct_takes(int fmt, const qw_gemm_params& p, uint32_t experts) {
    if (p.K % 128u != 0 || p.gshift > 2u) return false;
    // 8-bit banks of short rows under a workgroup a unit: the raw image's way through LDS is a tenth of the launch (32 experts, 30 rows each,
    // 1024 x 512: 12.3 us, the 64-row kernel 11.3; from one workgroup a unit on 0.81 .. 0.97 of its time)
    return !(fmt == QG_FMT_B8 && p.K <= 640u && tall_load(fmt, p, experts) <= 1.0);
}

hipError_t qw_grouped_direct(hipStream_t st, int fmt, const qw_gemm_params& p, uint32_t max_tiles, uint32_t experts, uint32_t xdt, uint32_t ydt,
                             bool swiglu) {
    switch (fmt) {
        case QG_FMT_M5: return launch<QG_FMT_M5>(st, p, max_tiles, experts, xdt, ydt, swiglu);
        case QG_FMT_B4: return launch<QG_FMT_B4>(st, p, max_tiles, experts, xdt, ydt, swiglu);
        case QG_FMT_B8: return launch<QG_FMT_B8>(st, p, max_tiles, experts, xdt, ydt, swiglu);
        case QG_FMT_B2: return launch<QG_FMT_B2>(st, p, max_tiles, experts, xdt, ydt, swiglu);
        case QG_FMT_B3: return launch<QG_FMT_B3>(st, p, max_tiles, experts, xdt, ydt, swiglu);
        default: return launch<QG_FMT_B6>(st, p, max_tiles, experts, xdt, ydt, swiglu);
    }
}
