// GEMV over any container with fp32 activations and fp32 outputs, with the scalar epilogues of the reference's f32 family
// (qwg_gemv_*_f32_v4 / qwg_gemm_*_f32_bm, Sources/QWMetal/include/qw_gemm_f32_common.metalh:15-19,152-225;
// doors QWGemm.encodeHQ4F32V4 / encodeHQ4F32BM, Sources/Operators/QWGEMM/QWGemmF32.swift:178-199,311-350).
//
// Launch shape: the 16-block form of gemv_quad.hip with the fp32 matrix instruction v_mfma_f32_4x4x1_16B_f32, which multiplies
// 16 independent 4x1 by 1x4 blocks: block b (lanes 4b .. 4b + 3) is one 32-column slice, lane (b, i) converts the codes of
// bank row i, lane (b, j) keeps the 32 fp32 activations of row j, and 32 instructions contract the slice for four bank rows
// and four activation rows.  A fixed population of workgroups walks row quads; wave wv of a row set owns slice chunk
// kr * wpr + wv (16 slices) in K range kr.  One and two rows take vector FMAs
// in the same layout.  Bound by issue, not by the bank's bytes, from three rows on: the 4x4 instruction takes as long as the
// four vector FMAs it stands for, but a lane holds 32 activations instead of 128 (those spilled into the accumulator file),
// so three times the waves fit and eight rows share one pass over the bank.  Against a lane per slice with 32 activations
// of every row: 17408 x 5120, HQ4_G32_M5, 1 / 2 / 3 / 8 rows 18.6 / 21.6 / 29.9 / 57.0 -> 16.1 / 19.3 / 25.9 / 39.1 us;
// 5120 x 1024, 4-bit, 5.7 / 8.3 / 10.6 / 21.4 -> 4.6 / 5.4 / 6.2 / 10.0 us.  One and two rows of several K ranges are bound by the
// activations, which every workgroup reads (1 x 4096 x 32768, 4-bit 17.2 us in the old form, 18.6 with four lanes asking for the
// same 32 columns at the start of each range, 17.8 with a quarter each and a range ahead; 2 x 4096 x 16384, 8-bit 16.8, 18.3, 16.9).
//
// Arithmetic: all in fp32.  The reference dequantises one weight as fma(float(code [+ 1024]), scale, bias) in fp32 and
// feeds an fp32 FMA chain (qwg_unpack_hq4_word8_f32 / qwg_dot_hq4_block_f32_reg, qw_dequant_f32.metalh:10-58); here the
// affine part is applied once per slice, sum_i w_i x_i = scale * sum_i code_i x_i + bias * sum_i x_i (HQ4_G32_M5: bias stands
// for fma(1024, scale, bias), rounded once), codes converted to fp32 exactly.  Both differ from the exact sum only by
// fp32 rounding.
#include <atomic>
#include <type_traits>

#include "qwhip_common.h"

namespace {

#define QF_FIELDS(X)                                                                                                        \
    X(const uint8_t*, bank) X(const float*, x) X(float*, y) X(uint32_t, N) X(uint32_t, K) X(uint32_t, M) X(uint32_t, nsl)       \
    X(uint32_t, wpr) X(uint32_t, sets) X(uint32_t, nkr) X(uint32_t, gshift) X(uint32_t, bb) X(uint32_t, row_bytes)              \
    X(uint32_t, epi) X(float, scale)
QW_ARG_BLOCK(qf_params, QF_FIELDS)

template <int FMT>
struct qf_fmt {
    static constexpr int BITS = FMT == QW_FMT_B8 ? 8 : (FMT == QW_FMT_B2 ? 2 : (FMT == QW_FMT_B3 ? 3 : (FMT == QW_FMT_B6 ? 6 : 4)));
    static constexpr int PW = BITS;   // payload dwords of one 32-column slice
};

// Code of element e (0..31) of a slice, cut out at compile-time positions.  HQ4_G32_M5 keeps element 8w + j at bit
// 4 (j >> 1) + 16 (j & 1) of word w (unpack_hq4_word8, qw_dequant.metalh:42-62); the bit streams element e at bit e * bits.
template <int FMT>
__device__ __forceinline__ uint32_t qf_code(const uint32_t* q, int e) {
    constexpr int BITS = qf_fmt<FMT>::BITS;
    if constexpr (FMT == QW_FMT_M5) {
        const int w = e >> 3, j = e & 7;
        return (q[w] >> (4 * (j >> 1) + 16 * (j & 1))) & 15u;
    } else {
        const int off = e * BITS, wd = off >> 5, sh = off & 31;
        uint32_t c = q[wd] >> sh;
        if (sh + BITS > 32) c |= q[wd + 1] << (32 - sh);
        return c & ((1u << BITS) - 1u);
    }
}

// The four bytes of a word as floats, one conversion each (the barrier keeps the compiler from folding the shift into the
// mask in front, which would cost a second instruction a byte).
__device__ __forceinline__ f4_t qf_bytes(uint32_t v) {
    asm("" : "+v"(v));
    return f4_t{(float)(v & 255u), (float)((v >> 8) & 255u), (float)((v >> 16) & 255u), (float)(v >> 24)};
}

__device__ __forceinline__ float qf_epilogue(float v, uint32_t epi, float scale) {
    if (epi == 1u || epi == 3u) {
        const float z = v / scale;
        return z / (1.0f + expf(-z));
    }
    if (epi == 2u) return 1.0f / (1.0f + expf(-v));
    return v;
}

#define QF_DPP(v, ctrl) __builtin_amdgcn_update_dpp(0, (int)(v), ctrl, 0xF, 0xF, true)
#define QF_DPP_F32(v, ctrl) __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xF, 0xF, true))

// MG groups of four activation rows on the matrix pipe, or (MV > 0, MG = 1) one or two rows by vector FMAs: every lane of a
// block then holds the same activations and contracts its own bank row, product by product in the matrix form's order, so a
// row's bits are the same from either.  D row quads in flight per lane.  blockDim.x = 64 * wpr * sets;
// dynamic LDS = quad slots per workgroup * (4 wpr) * (4 MG) * 16 bytes.  A row's sums do not depend on M, MG or the grid.
template <int FMT, int MG, int MV, int D, int LB>
struct qw_gemv_f32_kernel {
static constexpr int kLaunchBound = LB;
static __device__ __forceinline__ void run(const qf_params& p) {
    static_assert(MV == 0 || MG == 1, "the vector form takes one or two rows");
    constexpr int PW = qf_fmt<FMT>::PW, XR = MV ? MV : MG;   // XR: activation rows a lane holds
    extern __shared__ f4_t qf_part[];   // [quad slot][wave of the set * 4 + 16-lane row][activation row] -> 4 bank rows
    const uint32_t N = p.N, wpr = p.wpr, sets = p.sets;
    const uint32_t tid = threadIdx.x;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), l64 = tid & 63u;
    const uint32_t b = l64 >> 2, j = l64 & 3u;
    const uint32_t set = wave / wpr, wv = wave - set * wpr;
    const uint32_t G = gridDim.x;
    const uint32_t NQ = (N + 3u) >> 2;
    if (blockIdx.x >= NQ) return;
    const uint32_t nq = (NQ - blockIdx.x + G - 1u) / G;    // quad slots of this workgroup
    const uint32_t nmax = (nq + sets - 1u) / sets;          // trip count, uniform over the workgroup
    const uint32_t mine = nq > set ? (nq - set + sets - 1u) / sets : 0u;
    const uint32_t W16 = wpr * 4u;
    const uint32_t step = G * sets * 4u * p.row_bytes;      // bytes between consecutive quads of one set

    // this lane's bank row inside a quad is j (the A role); rows past the bank re-read its last row (never stored)
    const uint32_t q_first = (mine ? set : 0u) * G + blockIdx.x;
    const uint32_t off_first = min(4u * q_first + j, N - 1u) * p.row_bytes;
    const uint32_t last_quad = q_first + (mine ? mine - 1u : 0u) * G * sets;
    const uint32_t off_max = min(4u * last_quad + j, N - 1u) * p.row_bytes;   // loads past the set's last quad re-read it
    // slice of this lane in K range kr (clamped into the row) and its byte offsets inside a bank row
    auto slice_of = [&](uint32_t kr, uint32_t& hdr_off, uint32_t& pay_off) {
        const uint32_t g = min((kr * wpr + wv) * 16u + b, p.nsl - 1u);
        if constexpr (FMT == QW_FMT_M5) {
            hdr_off = g * 20u;
            pay_off = hdr_off + 4u;
        } else {
            hdr_off = (g >> p.gshift) * p.bb;
            pay_off = hdr_off + 4u + (g & ((1u << p.gshift) - 1u)) * (4u * PW);
        }
        return g;
    };
    // the weight prefetch runs on across K ranges: after the last quad of a range comes the first one of the next
    uint32_t i_kr = 0, i_left = nmax, i_off = off_first, i_hdr, i_pay;
    slice_of(0, i_hdr, i_pay);
    uint32_t hdr[D], q[D][PW];
    auto issue = [&](int slot) {
        const uint32_t o_hdr = i_off + i_hdr, o_pay = i_off + i_pay;   // the bank is under 1 GiB
        hdr[slot] = *(const uint32_t*)(p.bank + o_hdr);
#pragma unroll
        for (int t = 0; t < PW; ++t) q[slot][t] = *(const uint32_t*)(p.bank + o_pay + 4 * t);
        i_off = min(i_off + step, off_max);
        if (--i_left == 0u && i_kr + 1u < p.nkr) {   // uniform over the workgroup
            ++i_kr;
            slice_of(i_kr, i_hdr, i_pay);
            i_off = off_first;
            i_left = nmax;
        }
    };
    // activations of a K range, zero for slices past the row's end; rows past M re-read row M - 1.  In the vector form the four lanes
    // of a block hold the same 32: each asks for a quarter, a range ahead, and the block exchanges them.
    f4_t xv[XR][8], xq[MV ? XR : 1][2];
    auto load_x = [&](uint32_t kr) {
        uint32_t ho, po;
        const uint32_t g = slice_of(kr, ho, po);
#pragma unroll
        for (int mg = 0; mg < XR; ++mg) {
            const float* xp = p.x + (uint64_t)min(MV ? (uint32_t)mg : 4u * mg + j, p.M - 1u) * p.K + (uint64_t)g * 32u + (MV ? 8u * j : 0u);
#pragma unroll
            for (int t = 0; t < (MV ? 2 : 8); ++t) {
                if constexpr (MV != 0) xq[mg][t] = *(const f4_t*)(xp + 4 * t);
                else xv[mg][t] = *(const f4_t*)(xp + 4 * t);
            }
        }
    };
    auto spread_x = [&]() {
        if constexpr (MV != 0) {
#pragma unroll
            for (int mg = 0; mg < XR; ++mg) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float e = xq[mg][t][i];   // (the compiler's bit cast of a vector's element takes element 0)
                        xv[mg][t][i] = QF_DPP_F32(e, 0x00);        // quad_perm [l,l,l,l]: lane l of the block holds 8 l .. 8 l + 7
                        xv[mg][2 + t][i] = QF_DPP_F32(e, 0x55);
                        xv[mg][4 + t][i] = QF_DPP_F32(e, 0xAA);
                        xv[mg][6 + t][i] = QF_DPP_F32(e, 0xFF);
                    }
                }
            }
        }
    };
    load_x(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int d = 0; d < D; ++d) issue(d);
    __builtin_amdgcn_sched_barrier(0);

    for (uint32_t kr = 0; kr < p.nkr; ++kr) {
        if constexpr (MV != 0) {
            spread_x();
            if (kr + 1u < p.nkr) load_x(kr + 1u);
        } else {
            if (kr > 0u) load_x(kr);
        }
        const bool gvalid = (kr * wpr + wv) * 16u + b < p.nsl;
        float S[XR];
#pragma unroll
        for (int mg = 0; mg < XR; ++mg) {
            if (!gvalid) {
#pragma unroll
                for (int t = 0; t < 8; ++t) xv[mg][t] = f4_t{0.f, 0.f, 0.f, 0.f};
            }
            f4_t t4 = (xv[mg][0] + xv[mg][1]) + (xv[mg][2] + xv[mg][3]);
            t4 += (xv[mg][4] + xv[mg][5]) + (xv[mg][6] + xv[mg][7]);
            S[mg] = (t4[0] + t4[1]) + (t4[2] + t4[3]);
        }
        uint32_t qslot = set;   // quad slot being consumed
        for (uint32_t ib = 0; ib < nmax; ib += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                if (ib + d >= nmax) break;
                uint32_t qq[PW];
#pragma unroll
                for (int t = 0; t < PW; ++t) qq[t] = q[d][t];
                const uint32_t hd0 = hdr[d];
                issue(d);
                using acc_t = std::conditional_t<MV != 0, float, f4_t>;
                acc_t acc[XR][4];
#pragma unroll
                for (int mg = 0; mg < XR; ++mg)
#pragma unroll
                    for (int c = 0; c < 4; ++c) acc[mg][c] = acc_t{};
                auto contract = [&](float c, int e) {
#pragma unroll
                    for (int mg = 0; mg < XR; ++mg) {
                        if constexpr (MV != 0) acc[mg][e & 3] = __builtin_fmaf(c, xv[mg][e >> 2][e & 3], acc[mg][e & 3]);
                        else acc[mg][e & 3] = __builtin_amdgcn_mfma_f32_4x4x1f32(c, xv[mg][e >> 2][e & 3], acc[mg][e & 3], 0, 0, 0);
                    }
                };
                if constexpr (FMT == QW_FMT_B8) {
#pragma unroll
                    for (int w = 0; w < 8; ++w) {
                        const f4_t c = qf_bytes(qq[w]);
#pragma unroll
                        for (int t = 0; t < 4; ++t) contract(c[t], 4 * w + t);
                    }
                } else if constexpr (FMT == QW_FMT_M5 || FMT == QW_FMT_B4) {
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        // HQ4_G32_M5: the nibble at bit 4 t + 16 u is element 2 t + u of the word; streams: nibble i is element i
                        const f4_t lo = qf_bytes(qq[w] & 0x0F0F0F0Fu), hi = qf_bytes((qq[w] >> 4) & 0x0F0F0F0Fu);
                        if constexpr (FMT == QW_FMT_M5) {
                            const float c[8] = {lo[0], lo[2], hi[0], hi[2], lo[1], lo[3], hi[1], hi[3]};
#pragma unroll
                            for (int t = 0; t < 8; ++t) contract(c[t], 8 * w + t);
                        } else {
#pragma unroll
                            for (int t = 0; t < 4; ++t) {
                                contract(lo[t], 8 * w + 2 * t);
                                contract(hi[t], 8 * w + 2 * t + 1);
                            }
                        }
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 32; ++e) contract((float)qf_code<FMT>(qq, e), e);
                }
                float* const part = (float*)(qf_part + (size_t)(qslot * W16 + wv * 4u + (l64 >> 4)) * (4u * MG));
                if constexpr (MV != 0) {
                    const h2_t hd = __builtin_bit_cast(h2_t, hd0);
                    const float sc = (float)hd[0];
                    const float bi = FMT == QW_FMT_M5 ? __builtin_fmaf(1024.0f, sc, (float)hd[1]) : (float)hd[1];
#pragma unroll
                    for (int m = 0; m < MV; ++m) {
                        const float qs = (acc[m][0] + acc[m][1]) + (acc[m][2] + acc[m][3]);
                        float r = __builtin_fmaf(sc, qs, bi * S[m]);
                        r += QF_DPP_F32(r, 0x114);
                        r += QF_DPP_F32(r, 0x118);
                        if ((l64 & 12u) == 12u && qslot < nq) {   // lane 12 + j: bank row j
                            float* dst = part + 4 * m + j;
                            if (kr == 0) *dst = r;
                            else *dst += r;
                        }
                    }
                } else {
                    // the four headers of this block's rows
                    float sc[4], bi[4];
                    const uint32_t hq[4] = {(uint32_t)QF_DPP(hd0, 0x00), (uint32_t)QF_DPP(hd0, 0x55), (uint32_t)QF_DPP(hd0, 0xAA),
                                            (uint32_t)QF_DPP(hd0, 0xFF)};   // quad_perm [i,i,i,i]
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const h2_t hd = __builtin_bit_cast(h2_t, hq[i]);
                        sc[i] = (float)hd[0];
                        // HQ4_G32_M5: weight = (1024 + code) * scale + bias = code * scale + (1024 * scale + bias); the bracket is
                        // formed with one rounding, so the large terms cancel before they meet the activations
                        bi[i] = FMT == QW_FMT_M5 ? __builtin_fmaf(1024.0f, sc[i], (float)hd[1]) : (float)hd[1];
                    }
#pragma unroll
                    for (int mg = 0; mg < MG; ++mg) {
                        f4_t v;
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float qs = (acc[mg][0][i] + acc[mg][1][i]) + (acc[mg][2][i] + acc[mg][3][i]);
                            float r = __builtin_fmaf(sc[i], qs, bi[i] * S[mg]);
                            r += QF_DPP_F32(r, 0x114);   // row_shr:4
                            r += QF_DPP_F32(r, 0x118);   // row_shr:8: lanes 12..15 of each 16-lane row hold its four blocks
                            v[i] = r;
                        }
                        if ((l64 & 12u) == 12u && qslot < nq) {
                            f4_t* dst = (f4_t*)part + 4u * mg + j;
                            if (kr == 0) *dst = v;
                            else *dst += v;
                        }
                    }
                }
                qslot += sets;
            }
        }
        // the next range's first quads are already in flight, in the slots after the last one consumed: turn the window so
        // that they sit in slots 0, 1, ... again
        if (kr + 1u < p.nkr) {
            for (uint32_t k = nmax % D; k > 0u; --k) {
                const uint32_t h0 = hdr[0];
                uint32_t q0[PW];
#pragma unroll
                for (int t = 0; t < PW; ++t) q0[t] = q[0][t];
#pragma unroll
                for (int d = 0; d + 1 < D; ++d) {
                    hdr[d] = hdr[d + 1];
#pragma unroll
                    for (int t = 0; t < PW; ++t) q[d][t] = q[d + 1][t];
                }
                hdr[D - 1] = h0;
#pragma unroll
                for (int t = 0; t < PW; ++t) q[D - 1][t] = q0[t];
            }
        }
    }
    __syncthreads();
    // fixed-order sum of the partials of each (quad slot, activation row, bank row), then the scalar epilogue
    for (uint32_t t = tid; t < nq * p.M * 4u; t += blockDim.x) {
        const uint32_t i = t & 3u, sm = t >> 2;
        const uint32_t s = sm / p.M, m = sm - s * p.M;
        const uint32_t row = 4u * (s * G + blockIdx.x) + i;
        if (row >= N) continue;
        float v = 0.f;
        const float* part = (const float*)(qf_part + (size_t)s * W16 * (4u * MG) + m) + i;
        for (uint32_t w = 0; w < W16; w += 4u) {   // W16 is a multiple of four: four partials on their way at a time
            float t4[4];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) t4[u] = part[(size_t)(w + u) * (16u * MG)];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) v += t4[u];
        }
        p.y[(uint64_t)m * N + row] = qf_epilogue(v, p.epi, p.scale);
    }
}
};

// In-place capable FWHT-32 over consecutive groups of 32 outputs of each row, butterfly order and scaling of
// qwg_fwht32_lane_f32 (Sources/QWMetal/include/qw_weight_basis.metalh:31-38); a last partial group is padded with zeros
// (the v4 kernel's epilogue 3 reads rows past N as 0, qw_gemm_f32_common.metalh:171-196).
__global__ __launch_bounds__(256) void qw_h32_f32_kernel(const float* x, float* out, uint32_t hidden, uint32_t padded) {
    const uint32_t col = blockIdx.x * 256u + threadIdx.x;
    if (col >= padded) return;   // padded is a multiple of 32: whole 32-lane groups leave together
    const uint64_t at = (uint64_t)blockIdx.y * hidden + col;
    float v = col < hidden ? x[at] : 0.0f;
    v = qw_fwht32_lanes(v, qw_fwht32_lane_signs(threadIdx.x & 31u));   // the same stages and sums, partners by DPP
    if (col < hidden) out[at] = v * 0.17677669529663689f;
}

template <int FMT, int MG, int MV>
void qf_launch1(hipStream_t st, const qf_params& p, uint32_t wgs, uint32_t threads, size_t lds) {
    using kern = qw_gemv_f32_kernel<FMT, MG, MV, FMT == QW_FMT_B8 || FMT == QW_FMT_B6 ? 2 : 3, 768>;
    static std::atomic<bool> attr_done{false};   // per instantiation
    if (!attr_done.load(std::memory_order_acquire)) {
        (void)hipFuncSetAttribute(qw_scalar_kernel_ptr<kern>((const qf_params*)nullptr), hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024);
        attr_done.store(true, std::memory_order_release);
    }
    qw_launch_scalar<kern>(dim3(wgs), dim3(threads), lds, st, p);
}

template <int FMT>
void qf_launch(hipStream_t st, const qf_params& p, uint32_t mg, uint32_t wgs, uint32_t threads, size_t lds) {
    if (p.M == 1) qf_launch1<FMT, 1, 1>(st, p, wgs, threads, lds);
    else if (p.M == 2) qf_launch1<FMT, 1, 2>(st, p, wgs, threads, lds);
    else if (mg == 1) qf_launch1<FMT, 1, 0>(st, p, wgs, threads, lds);
    else qf_launch1<FMT, 2, 0>(st, p, wgs, threads, lds);
}

}  // namespace

void qw_h32_f32_launch(hipStream_t st, const float* x, float* out, uint32_t rows, uint32_t hidden) {
    const uint32_t padded = (hidden + 31u) & ~31u;
    hipLaunchKernelGGL(qw_h32_f32_kernel, dim3((padded + 255u) / 256u, rows), dim3(256), 0, st, x, out, hidden, padded);
}

// Largest number of activation rows (8, or 0 = none) the kernel takes per launch on this bank.
uint32_t qw_f32_gemv_rows(const qwhip_weight_view* w, uint64_t row_bytes) {
    if ((uint64_t)w->n * row_bytes >= (1ull << 30)) return 0;   // 32-bit offsets inside the bank, one quad step past its end included
    return w->k <= 32768u ? 8u : 0u;
}

// One launch over m <= qw_f32_gemv_rows() activation rows already in the container's basis; epilogue 3's rotation is the
// caller's second launch.
void qw_f32_gemv(hipStream_t st, const qwhip_weight_view* w, int fmt, uint32_t gshift, uint32_t bb, uint64_t row_bytes,
                 const float* x, uint32_t m, uint32_t epi, float scale, float* y) {
    const uint32_t mr = (m + 3u) / 4u;   // groups of four activation rows
    const uint32_t nsl = w->k / 32u, nch = (nsl + 15u) / 16u;
    // at most 12 waves per row set (768 threads); longer rows take several K ranges
    const uint32_t nkr = (nch + 11u) / 12u;
    const uint32_t wpr = (nch + nkr - 1u) / nkr;
    const uint32_t nquads = (w->n + 3u) / 4u;
    // a row set fewer for every 256 quads that are missing: a workgroup of one quad beats a third of the compute units with three
    // (one row, K = 2048: 128 and 1024 rows 4.8 -> 3.1 us, 8-bit 5.6 -> 3.1; 64 x 1024, three rows 6.4 -> 3.2)
    const uint32_t sets = max(1u, min(12u / wpr, nquads / 256u));
    const uint32_t threads = 64u * wpr * sets;
    uint32_t wgs = max(1u, min(256u * max(1u, 12u / (wpr * sets)), nquads / sets));
    // the partial sums of a workgroup's rows stay in LDS: more, smaller workgroups when the bank has very many rows
    auto lds_of = [&](uint32_t g) { return (size_t)qwhip_cdiv(nquads, g) * (wpr * 4u) * (4u * mr) * 16u; };
    while (lds_of(wgs) > 96u * 1024u) wgs *= 2u;
    const size_t lds = lds_of(wgs);
    qf_params p;
    p.bank = (const uint8_t*)w->blocks;
    p.x = x;
    p.y = y;
    p.N = w->n;
    p.K = w->k;
    p.M = m;
    p.nsl = nsl;
    p.wpr = wpr;
    p.sets = sets;
    p.nkr = nkr;
    p.gshift = gshift;
    p.bb = bb;
    p.row_bytes = (uint32_t)row_bytes;
    p.epi = epi;
    p.scale = scale;
    if (fmt == QW_FMT_M5) qf_launch<QW_FMT_M5>(st, p, mr, wgs, threads, lds);
    else if (fmt == QW_FMT_B4) qf_launch<QW_FMT_B4>(st, p, mr, wgs, threads, lds);
    else if (fmt == QW_FMT_B8) qf_launch<QW_FMT_B8>(st, p, mr, wgs, threads, lds);
    else if (fmt == QW_FMT_B2) qf_launch<QW_FMT_B2>(st, p, mr, wgs, threads, lds);
    else if (fmt == QW_FMT_B3) qf_launch<QW_FMT_B3>(st, p, mr, wgs, threads, lds);
    else qf_launch<QW_FMT_B6>(st, p, mr, wgs, threads, lds);
}
