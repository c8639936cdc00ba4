// Argument block and output conversion of the GEMM kernels (gemm.hip, gemm_direct.hip).
#pragma once
#include "qwhip_common.h"
#include "qw_slice.h"

struct qw_gemm_params {
    const uint8_t* bank;
    const void* x;
    void* y;
    uint32_t M, N, K;
    uint32_t ldx, ldy;
    uint32_t gshift, bb;
    uint64_t row_bytes;
    uint32_t tiles_m, tiles_n;
    // grouped
    const int32_t* gather;
    const int32_t* expert_off;
    const int32_t* tile_e;
    const int32_t* tile_r;
    const int32_t* tile_count;
    uint32_t rows_per_expert;
    uint32_t inter, rotate_act;  // fused SwiGLU epilogue: gate rows [0, inter), up rows [inter, 2 inter) of an expert; FWHT-32 on the result
    qw_act act;                  // the device's gated activation (all zero: SwiGLU)
    uint32_t force_gemm2;  // tuning / tests: keep the DMA-fed kernel for the 256 x 320 shape
    uint32_t x_bf16;       // ping-pong kernel: activations are bf16, converted while the tile is staged
};

template <int YDT>
__device__ __forceinline__ void qg_store(void* y, uint64_t idx, float v) {
    if constexpr (YDT == QWHIP_F32) ((float*)y)[idx] = v;
    else if constexpr (YDT == QWHIP_F16) ((h1_t*)y)[idx] = (h1_t)v;
    else ((uint16_t*)y)[idx] = qw_f32_to_bf16(v);
}

// gemm_direct.hip: grouped GEMM on direct weight operands (K in whole pairs of 64, groups of at most 128); max_tiles as the door's,
// p.tiles_n column tiles of 256 weight rows (swiglu: of 128 outputs)
bool qw_grouped_direct_takes(int fmt, const qw_gemm_params& p, uint32_t experts);
hipError_t qw_grouped_direct(hipStream_t st, int fmt, const qw_gemm_params& p, uint32_t max_tiles, uint32_t experts, uint32_t xdt, uint32_t ydt,
                             bool swiglu);
// moe_rows.hip: grouped, few rows an expert; false where it does not take the call.
bool qw_grouped_rows(hipStream_t st, int fmt, const qw_gemm_params& p, uint32_t max_tiles, uint32_t experts, uint32_t xdt, uint32_t ydt, bool swiglu,
                     hipError_t* err);
// gemm_mid.hip: the dense form.  splits > 1: fp32 planes [splits][M][ldy] at p.y (ydt f32), no range of K pairs empty; swiglu: f16
// rows; few: spans of 64 rows.
hipError_t qw_dense_direct(hipStream_t st, int fmt, const qw_gemm_params& p, uint32_t splits, uint32_t xdt, uint32_t ydt, bool swiglu, bool few);
// gemm_rows.hip: dense, at most 64 rows, `steps` 128-column steps a wave over K ranges; the planes and swiglu as qw_dense_direct's.
hipError_t qw_gemm_rows(hipStream_t st, int fmt, const qw_gemm_params& p, uint32_t steps, uint32_t ranges, uint32_t xdt, uint32_t ydt, bool swiglu);
bool qw_gemm_rows_choose(int fmt, uint32_t m, uint32_t n, uint32_t k, uint64_t row_bytes, uint64_t plane_room, uint32_t ranges, double limit,
                         uint32_t* steps, uint32_t* chosen);
bool qw_gemm_rows_fuses(int fmt, uint32_t m, uint32_t n, uint32_t k, uint32_t steps);
