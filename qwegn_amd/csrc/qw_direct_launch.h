// Host side of the direct-operand kernel (qw_direct.h), for the translation units of its two forms.
#pragma once
#include "qw_direct.h"

namespace {

// extent: the grouped door's max_tiles; dense: K ranges
template <int FMT, int YDT, bool SWIGLU, bool GACT, int XDT, int MAXF, bool DENSE>
hipError_t qd_launch6(hipStream_t st, const qw_gemm_params& p, uint32_t extent) {
    constexpr size_t lds = 2u * MAXF * 4096u + 256u * qd_pitch<FMT>();
    auto kern = qw_gemm6_kernel<FMT, YDT, SWIGLU, GACT, XDT, MAXF, DENSE>;
    static std::atomic<bool> attr_done{false};
    if (!attr_done.load(std::memory_order_acquire)) {
        const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024);
        if (e != hipSuccess) return e;
        attr_done.store(true, std::memory_order_release);
    }
    qw_gemm_params q = p;
    if constexpr (DENSE) {
        q.tiles_m = qwhip_cdiv(p.M, 32u * MAXF);
        q.tiles_n = SWIGLU ? qwhip_cdiv(p.inter, 128u) : qwhip_cdiv(p.N, 256u);
    }
    // XCD-aware one-dimensional grid over (tile, column tile); dense: over spans and column tiles, K ranges beside it
    const dim3 grid = DENSE ? dim3(8u * qwhip_cdiv(q.tiles_m * q.tiles_n, 8u), extent) : dim3(8u * qwhip_cdiv(extent, 8u) * p.tiles_n);
    hipLaunchKernelGGL(kern, grid, dim3(256), lds, st, q);
    return hipGetLastError();
}
template <int FMT, int YDT, bool SWIGLU, bool GACT, int XDT, bool DENSE>
hipError_t qd_launch_rows(hipStream_t st, const qw_gemm_params& p, uint32_t extent, bool few) {
    if (few) return qd_launch6<FMT, YDT, SWIGLU, GACT, XDT, 2, DENSE>(st, p, extent);
    return qd_launch6<FMT, YDT, SWIGLU, GACT, XDT, qd_span<FMT>(), DENSE>(st, p, extent);
}
template <int FMT, int XDT, bool DENSE>
hipError_t qd_launch_out(hipStream_t st, const qw_gemm_params& p, uint32_t extent, uint32_t ydt, bool swiglu, bool few) {
    if constexpr (!DENSE || XDT == QWHIP_F16) {   // the dense gate|up's rows are f16: its door converts bf16 first
        if (swiglu && p.act.kind) return qd_launch_rows<FMT, QWHIP_F16, true, true, XDT, DENSE>(st, p, extent, few);
        if (swiglu) return qd_launch_rows<FMT, QWHIP_F16, true, false, XDT, DENSE>(st, p, extent, few);
    }
    if (swiglu) return hipErrorInvalidValue;
    if (ydt == QWHIP_F16) return qd_launch_rows<FMT, QWHIP_F16, false, false, XDT, DENSE>(st, p, extent, few);
    if (ydt == QWHIP_BF16) return qd_launch_rows<FMT, QWHIP_BF16, false, false, XDT, DENSE>(st, p, extent, few);
    return qd_launch_rows<FMT, QWHIP_F32, false, false, XDT, DENSE>(st, p, extent, few);
}
template <int FMT, bool DENSE>
hipError_t qd_launch_x(hipStream_t st, const qw_gemm_params& p, uint32_t extent, uint32_t xdt, uint32_t ydt, bool swiglu, bool few) {
    if (xdt == QWHIP_F16) return qd_launch_out<FMT, QWHIP_F16, DENSE>(st, p, extent, ydt, swiglu, few);
    return qd_launch_out<FMT, QWHIP_BF16, DENSE>(st, p, extent, ydt, swiglu, few);
}

}  // namespace
