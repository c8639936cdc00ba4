// Host side of the dense GEMM on direct weight operands (qw_direct.h); choose_direct in gemm.hip says which problems it takes.
#include "qw_direct.h"

namespace {

template <int FMT, int YDT, bool SWIGLU, bool GACT, int XDT, int MAXF>
hipError_t launch6(hipStream_t st, const qw_gemm_params& p, uint32_t splits) {
    constexpr size_t lds = 2u * MAXF * 4096u + 256u * qd_pitch<FMT>();
    auto kern = qw_gemm6_kernel<FMT, YDT, SWIGLU, GACT, XDT, MAXF, true>;
    static std::atomic<bool> attr_done{false};
    if (!attr_done.load(std::memory_order_acquire)) {
        const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024);
        if (e != hipSuccess) return e;
        attr_done.store(true, std::memory_order_release);
    }
    qw_gemm_params q = p;
    q.tiles_m = qwhip_cdiv(p.M, 32u * MAXF);
    q.tiles_n = SWIGLU ? qwhip_cdiv(p.inter, 128u) : qwhip_cdiv(p.N, 256u);
    const dim3 grid(8u * qwhip_cdiv(q.tiles_m * q.tiles_n, 8u), splits);
    hipLaunchKernelGGL(kern, grid, dim3(256), lds, st, q);
    return hipGetLastError();
}
template <int FMT, int YDT, bool SWIGLU, bool GACT, int XDT>
hipError_t launch_rows(hipStream_t st, const qw_gemm_params& p, uint32_t splits, bool few) {
    if (few) return launch6<FMT, YDT, SWIGLU, GACT, XDT, 2>(st, p, splits);
    return launch6<FMT, YDT, SWIGLU, GACT, XDT, qd_span<FMT>()>(st, p, splits);
}
template <int FMT, int XDT>
hipError_t launch_out(hipStream_t st, const qw_gemm_params& p, uint32_t splits, uint32_t ydt, bool few) {
    if (ydt == QWHIP_F16) return launch_rows<FMT, QWHIP_F16, false, false, XDT>(st, p, splits, few);
    if (ydt == QWHIP_BF16) return launch_rows<FMT, QWHIP_BF16, false, false, XDT>(st, p, splits, few);
    return launch_rows<FMT, QWHIP_F32, false, false, XDT>(st, p, splits, few);
}
template <int FMT>
hipError_t launch_x(hipStream_t st, const qw_gemm_params& p, uint32_t splits, uint32_t xdt, uint32_t ydt, bool swiglu, bool few) {
    if (swiglu) {   // f16 rows: the door converts bf16 first
        if (p.act.kind) return launch_rows<FMT, QWHIP_F16, true, true, QWHIP_F16>(st, p, splits, few);
        return launch_rows<FMT, QWHIP_F16, true, false, QWHIP_F16>(st, p, splits, few);
    }
    if (xdt == QWHIP_BF16) return launch_out<FMT, QWHIP_BF16>(st, p, splits, ydt, few);
    return launch_out<FMT, QWHIP_F16>(st, p, splits, ydt, few);
}

}  // namespace

hipError_t qw_dense_direct(hipStream_t st, int fmt, const qw_gemm_params& p, uint32_t splits, uint32_t xdt, uint32_t ydt, bool swiglu, bool few) {
    switch (fmt) {
        case QG_FMT_M5: return launch_x<QG_FMT_M5>(st, p, splits, xdt, ydt, swiglu, few);
        case QG_FMT_B4: return launch_x<QG_FMT_B4>(st, p, splits, xdt, ydt, swiglu, few);
        case QG_FMT_B8: return launch_x<QG_FMT_B8>(st, p, splits, xdt, ydt, swiglu, few);
        case QG_FMT_B2: return launch_x<QG_FMT_B2>(st, p, splits, xdt, ydt, swiglu, few);
        case QG_FMT_B3: return launch_x<QG_FMT_B3>(st, p, splits, xdt, ydt, swiglu, few);
        default: return launch_x<QG_FMT_B6>(st, p, splits, xdt, ydt, swiglu, few);
    }
}
