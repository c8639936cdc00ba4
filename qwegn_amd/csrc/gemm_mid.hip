// Host side of the dense GEMM on direct weight operands (qw_direct.h); choose_direct in gemm.hip says which problems it takes.
#include "qw_direct_launch.h"

hipError_t qw_dense_direct(hipStream_t st, int fmt, const qw_gemm_params& p, uint32_t splits, uint32_t xdt, uint32_t ydt, bool swiglu, bool few) {
    switch (fmt) {
        case QG_FMT_M5: return qd_launch_x<QG_FMT_M5, true>(st, p, splits, xdt, ydt, swiglu, few);
        case QG_FMT_B4: return qd_launch_x<QG_FMT_B4, true>(st, p, splits, xdt, ydt, swiglu, few);
        case QG_FMT_B8: return qd_launch_x<QG_FMT_B8, true>(st, p, splits, xdt, ydt, swiglu, few);
        case QG_FMT_B2: return qd_launch_x<QG_FMT_B2, true>(st, p, splits, xdt, ydt, swiglu, few);
        case QG_FMT_B3: return qd_launch_x<QG_FMT_B3, true>(st, p, splits, xdt, ydt, swiglu, few);
        default: return qd_launch_x<QG_FMT_B6, true>(st, p, splits, xdt, ydt, swiglu, few);
    }
}
