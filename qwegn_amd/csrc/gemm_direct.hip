// Host side of the grouped (MoE) GEMM on direct weight operands (qw_direct.h).
#include "qw_direct.h"

namespace {

template <int FMT, int YDT, bool SWIGLU, bool GACT, int XDT, int MAXF>
hipError_t launch6(hipStream_t st, const qw_gemm_params& p, uint32_t max_tiles) {
    constexpr size_t lds = 2u * MAXF * 4096u + 256u * qd_pitch<FMT>();
    auto kern = qw_gemm6_kernel<FMT, YDT, SWIGLU, GACT, XDT, MAXF>;
    static std::atomic<bool> attr_done{false};
    if (!attr_done.load(std::memory_order_acquire)) {
        const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024);
        if (e != hipSuccess) return e;
        attr_done.store(true, std::memory_order_release);
    }
    const dim3 grid(8u * qwhip_cdiv(max_tiles, 8u) * p.tiles_n);   // XCD-aware one-dimensional grid over (tile, column tile)
    hipLaunchKernelGGL(kern, grid, dim3(256), lds, st, p);
    return hipGetLastError();
}
template <int FMT, int YDT, bool SWIGLU, bool GACT, int XDT>
hipError_t launch_rows(hipStream_t st, const qw_gemm_params& p, uint32_t max_tiles, bool few) {
    if (few) return launch6<FMT, YDT, SWIGLU, GACT, XDT, 2>(st, p, max_tiles);
    return launch6<FMT, YDT, SWIGLU, GACT, XDT, qd_span<FMT>()>(st, p, max_tiles);
}
template <int FMT, int XDT>
hipError_t launch_out(hipStream_t st, const qw_gemm_params& p, uint32_t max_tiles, uint32_t ydt, bool swiglu, bool few) {
    if (swiglu) {
        if (p.act.kind) return launch_rows<FMT, QWHIP_F16, true, true, XDT>(st, p, max_tiles, few);
        return launch_rows<FMT, QWHIP_F16, true, false, XDT>(st, p, max_tiles, few);
    }
    if (ydt == QWHIP_F16) return launch_rows<FMT, QWHIP_F16, false, false, XDT>(st, p, max_tiles, few);
    if (ydt == QWHIP_BF16) return launch_rows<FMT, QWHIP_BF16, false, false, XDT>(st, p, max_tiles, few);
    return launch_rows<FMT, QWHIP_F32, false, false, XDT>(st, p, max_tiles, few);
}
template <int FMT>
hipError_t launch_x(hipStream_t st, const qw_gemm_params& p, uint32_t max_tiles, uint32_t xdt, uint32_t ydt, bool swiglu, bool few) {
    if (xdt == QWHIP_F16) return launch_out<FMT, QWHIP_F16>(st, p, max_tiles, ydt, swiglu, few);
    return launch_out<FMT, QWHIP_BF16>(st, p, max_tiles, ydt, swiglu, few);
}

}  // namespace

bool qw_grouped_direct_takes(const qw_gemm_params& p) { return p.K % 128u == 0 && p.gshift <= 2u; }

hipError_t qw_grouped_direct(hipStream_t st, int fmt, const qw_gemm_params& p, uint32_t max_tiles, uint32_t experts, uint32_t xdt, uint32_t ydt,
                             bool swiglu) {
    // 64-row spans, three waves a SIMD, against 128-row spans at two: gate|up + down of 2048 x 768, 128 experts, 8 / 32 / 64 / 128 rows
    // an expert: 114 / 126 / 178 / 256 us against 114 / 130 / 173 / 243 (HQ4_G32_M5), 118 / 131 / 182 / 270 against 120 / 133 / 174 / 253
    // (4-bit affine, group 64)
    const bool few = p.M <= 48u * experts;
    switch (fmt) {
        case QG_FMT_M5: return launch_x<QG_FMT_M5>(st, p, max_tiles, xdt, ydt, swiglu, few);
        case QG_FMT_B4: return launch_x<QG_FMT_B4>(st, p, max_tiles, xdt, ydt, swiglu, few);
        case QG_FMT_B8: return launch_x<QG_FMT_B8>(st, p, max_tiles, xdt, ydt, swiglu, few);
        case QG_FMT_B2: return launch_x<QG_FMT_B2>(st, p, max_tiles, xdt, ydt, swiglu, few);
        case QG_FMT_B3: return launch_x<QG_FMT_B3>(st, p, max_tiles, xdt, ydt, swiglu, few);
        default: return launch_x<QG_FMT_B6>(st, p, max_tiles, xdt, ydt, swiglu, few);
    }
}
