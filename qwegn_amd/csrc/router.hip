// Router logits and the dense fp32 GEMV door: out[t, e] = sum_h x[t, h] * w[e, h] on un-quantized weights, fp32 accumulate.
#include <algorithm>

#include "qwhip_common.h"

// The scalar epilogues of the dense f32 GEMV door (qwg_f32_gemv, Sources/QWMetal/gemm/qwgemm_f32.metal:120-143):
// 0 none, 1 silu(y / scale), 2 sigmoid(y), 3 2 sigmoid(y / scale).
__device__ __forceinline__ float qw_f32_gemv_epilogue(float y, uint32_t epi, float scale) {
    if (epi == 1u) {
        const float z = y / scale;
        return z / (1.0f + expf(-z));
    }
    if (epi == 2u) return 1.0f / (1.0f + expf(-y));
    if (epi == 3u) return 2.0f / (1.0f + expf(-(y / scale)));
    return y;
}


typedef __bf16 qw_bf8_t __attribute__((ext_vector_type(8)));

// Eight consecutive elements as they are stored (16 bytes, or 32 for fp32), 16-byte aligned.
template <int DT>
struct qw_raw8 {
    u4_t v[DT == QWHIP_F32 ? 2 : 1];
    __device__ __forceinline__ void load(const void* p, uint64_t i) {
        const u4_t* q = (const u4_t*)((const uint8_t*)p + i * (DT == QWHIP_F32 ? 4u : 2u));
        v[0] = q[0];
        if constexpr (DT == QWHIP_F32) v[1] = q[1];
    }
    __device__ __forceinline__ void floats(float* f) const {
        if constexpr (DT == QWHIP_F32) {
#pragma unroll
            for (int j = 0; j < 8; ++j) f[j] = __uint_as_float(v[j >> 2][j & 3]);
        } else if constexpr (DT == QWHIP_F16) {
            const h8_t h = __builtin_bit_cast(h8_t, v[0]);
#pragma unroll
            for (int j = 0; j < 8; ++j) f[j] = (float)h[j];
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                f[2 * j] = __uint_as_float(v[0][j] << 16);
                f[2 * j + 1] = __uint_as_float(v[0][j] & 0xFFFF0000u);
            }
        }
    }
};

// The upper halves of eight floats as bf16, and what they leave: taken one to three times this writes a float as a sum of
// bf16 numbers without loss (8 significant bits each: 3 for fp32, 2 for the 11 bits of f16).  An infinite value leaves NaN.
__device__ __forceinline__ qw_bf8_t qw_take_bf16(float* f) {
    u4_t w;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t a = __float_as_uint(f[2 * j]), b = __float_as_uint(f[2 * j + 1]);
        w[j] = __builtin_amdgcn_perm(b, a, 0x07060302u);
        f[2 * j] -= __uint_as_float(a & 0xFFFF0000u);
        f[2 * j + 1] -= __uint_as_float(b & 0xFFFF0000u);
    }
    return __builtin_bit_cast(qw_bf8_t, w);
}

// ------------------------------------------------------------------------------------------------
// Two token rows and more: 16 tokens x 16 NT weight rows a workgroup on the matrix cores, the hidden dimension dealt in chunks
// of 32 to its W waves (chunk c to wave c % W) and the waves' sums added in wave order, so an output does not depend on how
// many rows or experts the call has.  Operands go from memory to registers as they lie (lane (r, g): row r, columns 8 g .. 8 g + 7
// of a chunk; nothing is shared between waves, so LDS would only add a copy), four chunks in flight per wave.
// bf16 weights meet the activations as one to three bf16 products that hold every bit of them (exact products, fp32 sums: 48
// matrix-core clocks a chunk for fp32 rows, where fp32 products take 256); other weights take the fp32 matrix product.
// What bounded the kernel before (one lane per hidden column, every weight x token product one vector instruction and one LDS
// operand): 2048 x 128 x 2048 with fp32 rows took 93 us, now 17 (two passes over 16 MB of rows); 4 x 256 x 2048 with f16 rows 19 us, now 5.5.
// The last band (gate_y) is the shared-expert gate: a dot product with an fp32 row per token.
// ------------------------------------------------------------------------------------------------
template <int XDT, int WDT, int NT, int W>
__global__ __launch_bounds__(64 * W) void qw_router_mfma_kernel(const void* __restrict__ x, const void* __restrict__ wr, float* __restrict__ out,
                                                                uint32_t T, uint32_t E, uint32_t H, const float* __restrict__ sh_w,
                                                                float* __restrict__ sh_out, uint32_t gate_y, uint32_t epi, float scale) {
    constexpr uint32_t PITCH = NT * 16 + 4;   // rows 4 apart fall 16 banks apart
    __shared__ float part[W][16 * PITCH];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t t0 = blockIdx.x * 16u;
    if (blockIdx.y == gate_y) {
        for (uint32_t t = t0 + wave; t < min(t0 + 16u, T); t += W) {
            float v = 0.0f;
            for (uint32_t h = lane * 8u; h < H; h += 512u) {
                qw_raw8<XDT> a;
                qw_raw8<QWHIP_F32> b;
                a.load(x, (uint64_t)t * H + h);
                b.load(sh_w, h);
                float fa[8], fb[8];
                a.floats(fa);
                b.floats(fb);
#pragma unroll
                for (int j = 0; j < 8; ++j) v = fmaf(fb[j], fa[j], v);
            }
            v = qw_reduce64(v);
            if (lane == 0) sh_out[t] = 1.0f / (1.0f + expf(-v));
        }
        return;
    }
    const uint32_t e0 = blockIdx.y * (16u * NT), r = lane & 15u, g = lane >> 4;
    const uint64_t xi = (uint64_t)min(t0 + r, T - 1u) * H + 8u * g;   // rows past the end repeat the last one and are not stored
    uint64_t wi[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) wi[n] = (uint64_t)min(e0 + 16u * n + r, E - 1u) * H + 8u * g;
    f4_t acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[n] = f4_t{0.f, 0.f, 0.f, 0.f};
    const uint32_t chunks = H >> 5;
    constexpr int U = 4;
    for (uint32_t c = wave; c < chunks; c += W * U) {
        qw_raw8<XDT> xa[U];
        qw_raw8<WDT> wb[U][NT];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t h = 32u * (c + W * u < chunks ? c + W * u : c);
            xa[u].load(x, xi + h);
#pragma unroll
            for (int n = 0; n < NT; ++n) wb[u][n].load(wr, wi[n] + h);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u > 0 && c + W * u >= chunks) break;   // wave-uniform
            if constexpr (WDT == QWHIP_BF16) {
                constexpr int P = XDT == QWHIP_BF16 ? 1 : (XDT == QWHIP_F16 ? 2 : 3);
                qw_bf8_t a[P];
                if constexpr (XDT == QWHIP_BF16) {
                    a[0] = __builtin_bit_cast(qw_bf8_t, xa[u].v[0]);
                } else {
                    float f[8];
                    xa[u].floats(f);
#pragma unroll
                    for (int p = 0; p < P; ++p) a[p] = qw_take_bf16(f);
                }
                // the smallest terms first
#pragma unroll
                for (int p = P - 1; p >= 0; --p)
#pragma unroll
                    for (int n = 0; n < NT; ++n)
                        acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[p], __builtin_bit_cast(qw_bf8_t, wb[u][n].v[0]), acc[n], 0, 0, 0);
            } else {
                float fa[8], fb[NT][8];
                xa[u].floats(fa);
#pragma unroll
                for (int n = 0; n < NT; ++n) wb[u][n].floats(fb[n]);
#pragma unroll
                for (int j = 0; j < 8; ++j)
#pragma unroll
                    for (int n = 0; n < NT; ++n) acc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[j], fb[n][j], acc[n], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i) part[wave][(4u * g + i) * PITCH + 16u * n + r] = acc[n][i];
    __syncthreads();
    for (uint32_t o = threadIdx.x; o < 16u * 16u * NT; o += 64u * W) {
        const uint32_t row = o / (16u * NT), col = o % (16u * NT);
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < W; ++w) v += part[w][row * PITCH + col];
        if (t0 + row >= T || e0 + col >= E) continue;
        if constexpr (WDT == QWHIP_BF16 && XDT != QWHIP_BF16) {
            // the bf16 terms of an infinity, and zero terms against an infinite weight, make NaN of what may be an infinity:
            // such an output is summed again from the operands as they are
            if (v != v) {
                v = 0.0f;
                for (uint32_t h = 0; h < H; ++h)
                    v = fmaf(qw_load_f32<WDT>(wr, (uint64_t)(e0 + col) * H + h), qw_load_f32<XDT>(x, (uint64_t)(t0 + row) * H + h), v);
            }
        }
        out[(uint64_t)(t0 + row) * E + e0 + col] = qw_f32_gemv_epilogue(v, epi, scale);
    }
}

// One token row: a wavefront is a workgroup and owns one weight row (the last one the shared-expert gate), 16-byte loads, four of
// them in flight.  A row of 2048 bf16 weights is four of those loads a lane, all in flight: the launch is its own latency
// (128 x 2048: 3.2 us, with 2-byte loads and 32 workgroups 6.6).
template <int XDT, int WDT>
__global__ __launch_bounds__(64) void qw_router_row_kernel(const void* __restrict__ x, const void* __restrict__ wr, float* __restrict__ out,
                                                           uint32_t E, uint32_t H, const float* __restrict__ sh_w, float* __restrict__ sh_out,
                                                           uint32_t epi, float scale) {
    const uint32_t e = blockIdx.x, lane = threadIdx.x;
    float acc[2] = {0.0f, 0.0f};
    auto dot = [&](auto wt, const void* w, uint64_t base) {
        constexpr int WT = decltype(wt)::value;
        for (uint32_t h0 = lane * 8u; h0 < H; h0 += 2048u) {
            qw_raw8<XDT> a[4];
            qw_raw8<WT> b[4];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
                const uint32_t h = h0 + 512u * u < H ? h0 + 512u * u : h0;
                a[u].load(x, h);
                b[u].load(w, base + h);
            }
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
                float fa[8], fb[8];
                a[u].floats(fa);
                b[u].floats(fb);
                if (u == 0 || h0 + 512u * u < H) {
#pragma unroll
                    for (int j = 0; j < 8; ++j) acc[j & 1] = fmaf(fb[j], fa[j], acc[j & 1]);
                }
            }
        }
    };
    if (e == E) dot(std::integral_constant<int, QWHIP_F32>{}, sh_w, 0);
    else dot(std::integral_constant<int, WDT>{}, wr, (uint64_t)e * H);
    const float v = qw_reduce64(acc[0] + acc[1]);
    if (lane == 0) {
        if (e == E) *sh_out = 1.0f / (1.0f + expf(-v));
        else out[e] = qw_f32_gemv_epilogue(v, epi, scale);
    }
}

// ------------------------------------------------------------------------------------------------
// Any hidden size and alignment (the kernels above take whole chunks of 32 columns and 16-byte aligned rows).
// A workgroup owns TT token rows (staged as fp32 in LDS; 8 rows up to hidden = 2048, fewer on wider rows so the tile
// stays within 64 KiB, and no more than the call has) so each router row is read once per TT tokens; blockIdx.y owns a band of `eb` weight rows
// (a multiple of 4, so that few token rows still spread over the chip), a wavefront the band's rows wave, wave+4, ...;
// lanes stride the hidden dimension, so an output's summation order does not depend on the band size.  With a shared-expert gate row (fp32 [hidden]) the workgroup also writes
// sh_out[t] = sigmoid(x[t] . sh_w), the extra output column of the reference's router kernels
// (Sources/QWMetal/subsystems/qwrouter.metal:467-483,566-574,587-633).
// ------------------------------------------------------------------------------------------------
template <int XDT, int WDT, int TT>
__global__ __launch_bounds__(256) void qw_router_gemm_kernel(const void* __restrict__ x, const void* __restrict__ wr,
                                                              float* __restrict__ logits, uint32_t T, uint32_t E, uint32_t H,
                                                              const float* __restrict__ sh_w, float* __restrict__ sh_out,
                                                              uint32_t epi, float scale, uint32_t eb) {
    extern __shared__ float xs[];  // [TT][H]
    const uint32_t t0 = blockIdx.x * TT;
    const uint32_t nt = min((uint32_t)TT, T - t0);
#pragma unroll
    for (uint32_t r = 0; r < (uint32_t)TT; ++r)
        for (uint32_t h = threadIdx.x; h < H; h += 256) xs[r * H + h] = r < nt ? qw_load_f32<XDT>(x, (uint64_t)(t0 + r) * H + h) : 0.0f;
    __syncthreads();
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    const uint32_t rows = min(E + (sh_w ? 1u : 0u), (blockIdx.y + 1u) * eb);
    for (uint32_t e = blockIdx.y * eb + wave; e < rows; e += 4) {
        const bool gate_row = e == E;   // wave-uniform
        float acc[TT];
#pragma unroll
        for (int r = 0; r < TT; ++r) acc[r] = 0.0f;
        // eight weight loads in flight per lane, consumed in the order h = lane, lane + 64, ... so the sums do not depend on it
        uint32_t h = lane;
        if (!gate_row) {
            const uint64_t row = (uint64_t)e * H;
            for (; h + 7u * 64u < H; h += 8u * 64u) {
                float w[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) w[u] = qw_load_f32<WDT>(wr, row + h + (uint32_t)u * 64u);
#pragma unroll
                for (int u = 0; u < 8; ++u)
#pragma unroll
                    for (int r = 0; r < TT; ++r) acc[r] = fmaf(w[u], xs[r * H + h + (uint32_t)u * 64u], acc[r]);
            }
        }
        for (; h < H; h += 64) {
            const float w = gate_row ? sh_w[h] : qw_load_f32<WDT>(wr, (uint64_t)e * H + h);
#pragma unroll
            for (int r = 0; r < TT; ++r) acc[r] = fmaf(w, xs[r * H + h], acc[r]);
        }
#pragma unroll
        for (int r = 0; r < TT; ++r) {
            const float v = qw_reduce64(acc[r]);
            if (lane == 0 && (uint32_t)r < nt) {
                if (gate_row) sh_out[t0 + r] = 1.0f / (1.0f + expf(-v));
                else logits[(uint64_t)(t0 + r) * E + e] = qw_f32_gemv_epilogue(v, epi, scale);
            }
        }
    }
}

// Launches the matrix-core or the one-row kernel; false for a type the caller reports.
// Tile: 64 weight rows a workgroup (the activations' bf16 terms made once for four products) once that alone is a workgroup for
// every compute unit, else 16 weight rows and twice the waves: a few token rows are bound by the latency of a wave's own chunks.
template <int XDT, int WDT>
static void qw_router_launch(hipStream_t st, const void* x, const void* wr, uint32_t t, uint32_t experts, uint32_t hidden, float* out,
                             const float* sh_w, float* sh_out, uint32_t epi, float scale) {
    const uint32_t gate = sh_w ? 1u : 0u;
    if (t == 1u) {
        hipLaunchKernelGGL((qw_router_row_kernel<XDT, WDT>), dim3(experts + gate), dim3(64), 0, st, x, wr, out, experts, hidden, sh_w, sh_out, epi, scale);
        return;
    }
    const uint32_t gx = qwhip_cdiv(t, 16u);
    if ((uint64_t)gx * qwhip_cdiv(experts, 64u) >= 256u) {
        const uint32_t gy = qwhip_cdiv(experts, 64u);
        hipLaunchKernelGGL((qw_router_mfma_kernel<XDT, WDT, 4, 8>), dim3(gx, gy + gate), dim3(512), 0, st, x, wr, out, t, experts, hidden, sh_w, sh_out,
                           gate ? gy : ~0u, epi, scale);
    } else {
        const uint32_t gy = qwhip_cdiv(experts, 16u);
        hipLaunchKernelGGL((qw_router_mfma_kernel<XDT, WDT, 1, 16>), dim3(gx, gy + gate), dim3(1024), 0, st, x, wr, out, t, experts, hidden, sh_w, sh_out,
                           gate ? gy : ~0u, epi, scale);
    }
}

static bool qw_router_wide(hipStream_t st, const void* x, uint32_t x_dtype, const void* wr, uint32_t w_dtype, uint32_t t, uint32_t experts,
                           uint32_t hidden, float* out, const float* sh_w, float* sh_out, uint32_t epi, float scale) {
    if (x_dtype > QWHIP_BF16 || w_dtype > QWHIP_BF16 || qwhip_cdiv(experts, 16u) >= 65535u) return false;
#define QW_RW(XD, WD) qw_router_launch<XD, WD>(st, x, wr, t, experts, hidden, out, sh_w, sh_out, epi, scale)
#define QW_RW_W(XD)                                       \
    switch (w_dtype) {                                    \
        case QWHIP_F32: QW_RW(XD, QWHIP_F32); break;      \
        case QWHIP_F16: QW_RW(XD, QWHIP_F16); break;      \
        default: QW_RW(XD, QWHIP_BF16); break;            \
    }
    switch (x_dtype) {
        case QWHIP_F32: QW_RW_W(QWHIP_F32) break;
        case QWHIP_F16: QW_RW_W(QWHIP_F16) break;
        default: QW_RW_W(QWHIP_BF16) break;
    }
#undef QW_RW_W
#undef QW_RW
    return true;
}

static qwhip_status qw_router_gemm_impl(qwhip_stream_t s, const void* x, uint32_t x_dtype, const void* wr, uint32_t w_dtype, uint32_t t,
                                        uint32_t experts, uint32_t hidden, float* logits, const float* sh_gate_w, float* sh_gate_out,
                                        uint32_t epi, float scale) {
    QWHIP_REQUIRE(s);
    if (t == 0) return QWHIP_OK;
    QWHIP_REQUIRE(x);
    QWHIP_REQUIRE(wr);
    QWHIP_REQUIRE(logits);
    if ((sh_gate_w != nullptr) != (sh_gate_out != nullptr))
        return qwhip_fail(QWHIP_E_NULL, "router gemm: the shared-expert gate needs both its weight row and its output");
    if (experts == 0 || hidden == 0) return qwhip_fail(QWHIP_E_BAD_SHAPE, "router gemm: empty experts or hidden");
    // token rows per workgroup: the fp32 tile stays within 64 KiB
    uint32_t tt = 8;
    while (tt > 1u && ((size_t)tt * hidden * 4u > 64u * 1024u || tt >= 2u * t)) tt >>= 1;
    const size_t lds = (size_t)tt * hidden * 4u;
    if (lds > 64u * 1024u) return qwhip_fail(QWHIP_E_BAD_SHAPE, "router gemm: hidden %u exceeds the staged row (<= 16384)", hidden);
    const bool wide = hidden % 32u == 0 && (((uintptr_t)x | (uintptr_t)wr | (uintptr_t)sh_gate_w) & 15u) == 0;
    if (wide && qw_router_wide(s->stream, x, x_dtype, wr, w_dtype, t, experts, hidden, logits, sh_gate_w, sh_gate_out, epi, scale)) {
        QWHIP_TRY_HIP(hipGetLastError());
        return QWHIP_OK;
    }
    // weight rows per workgroup: about 1024 workgroups over the launch, at least one row per wavefront
    const uint32_t gx = qwhip_cdiv(t, tt), rows_total = experts + (sh_gate_w ? 1u : 0u);
    const uint32_t gy_want = std::min(qwhip_cdiv(rows_total, 4u), std::max(1u, 1024u / gx));
    const uint32_t eb = (qwhip_cdiv(rows_total, gy_want) + 3u) & ~3u;
    const dim3 grid(gx, qwhip_cdiv(rows_total, eb)), block(256);
    if (grid.y > 65535u) return qwhip_fail(QWHIP_E_BAD_SHAPE, "router gemm: %u weight rows exceed the launch grid", rows_total);
#define QW_RG(XD, WD, TT) \
    hipLaunchKernelGGL((qw_router_gemm_kernel<XD, WD, TT>), grid, block, lds, s->stream, x, wr, logits, t, experts, hidden, sh_gate_w, sh_gate_out, epi, scale, eb)
#define QW_RG_T(XD, WD)                       \
    switch (tt) {                             \
        case 8: QW_RG(XD, WD, 8); break;      \
        case 4: QW_RG(XD, WD, 4); break;      \
        case 2: QW_RG(XD, WD, 2); break;      \
        default: QW_RG(XD, WD, 1); break;     \
    }
#define QW_RG_W(XD)                                                   \
    switch (w_dtype) {                                                \
        case QWHIP_F32: QW_RG_T(XD, QWHIP_F32) break;                 \
        case QWHIP_F16: QW_RG_T(XD, QWHIP_F16) break;                 \
        case QWHIP_BF16: QW_RG_T(XD, QWHIP_BF16) break;               \
        default: return qwhip_fail(QWHIP_E_BAD_SHAPE, "router gemm: unsupported weight dtype %u", w_dtype); \
    }
    switch (x_dtype) {
        case QWHIP_F32: QW_RG_W(QWHIP_F32) break;
        case QWHIP_F16: QW_RG_W(QWHIP_F16) break;
        case QWHIP_BF16: QW_RG_W(QWHIP_BF16) break;
        default: return qwhip_fail(QWHIP_E_BAD_SHAPE, "router gemm: unsupported activation dtype %u", x_dtype);
    }
#undef QW_RG_W
#undef QW_RG_T
#undef QW_RG
    QWHIP_TRY_HIP(hipGetLastError());
    return QWHIP_OK;
}

extern "C" qwhip_status qwhip_router_gemm_shared_gate(qwhip_stream_t s, const void* x, uint32_t x_dtype, const void* wr, uint32_t w_dtype,
                                                      uint32_t t, uint32_t experts, uint32_t hidden, float* logits,
                                                      const float* sh_gate_w, float* sh_gate_out) {
    return qw_router_gemm_impl(s, x, x_dtype, wr, w_dtype, t, experts, hidden, logits, sh_gate_w, sh_gate_out, 0u, 1.0f);
}

extern "C" qwhip_status qwhip_router_gemm(qwhip_stream_t s, const void* x, uint32_t x_dtype, const void* wr, uint32_t w_dtype,
                                          uint32_t t, uint32_t experts, uint32_t hidden, float* logits) {
    return qw_router_gemm_impl(s, x, x_dtype, wr, w_dtype, t, experts, hidden, logits, nullptr, nullptr, 0u, 1.0f);
}

// Dense fp32-weight GEMV with the scalar epilogues (QWGemm.encodeF32Gemv, Sources/Operators/QWGEMM/QWGemmF32.swift:117-141 ->
// qwg_f32_gemv / qwg_f32_gemv_bm): y[t, n] = epilogue(sum_k W[n, k] x[t, k]) on the router kernel (every weight row read once
// per eight activation rows).
extern "C" qwhip_status qwhip_f32_gemv(qwhip_stream_t s, const float* w, const float* x, uint32_t rows, uint32_t n, uint32_t k,
                                       uint32_t epi, float scale, float* y) {
    if (epi > 3u) return qwhip_fail(QWHIP_E_BAD_SHAPE, "epilogue %u is not one of 0 none, 1 silu(y/scale), 2 sigmoid, 3 2 sigmoid(y/scale)", epi);
    if ((epi == 1u || epi == 3u) && !(scale != 0.0f && scale == scale))
        return qwhip_fail(QWHIP_E_BAD_SHAPE, "epilogue %u divides by its scale, which must be a non-zero number", epi);
    return qw_router_gemm_impl(s, x, QWHIP_F32, w, QWHIP_F32, rows, n, k, y, nullptr, nullptr, epi, scale);
}

