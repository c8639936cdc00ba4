// Router logits and the dense fp32 GEMV door: out[t, e] = sum_h x[t, h] * w[e, h] on un-quantized weights, fp32 accumulate.
#include <algorithm>
#include <type_traits>

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

struct __attribute__((packed, aligned(4))) qw_words4 { u4_t v; };   // 16 bytes at any 4-byte boundary

// Eight consecutive elements as they are stored: 16 bytes, 16-byte aligned, or for fp32 32 bytes, 4-byte aligned.
template <int DT>
struct qw_raw8 {
    u4_t v[DT == QWHIP_F32 ? 2 : 1];
    __device__ __forceinline__ void load(const void* p, uint64_t i) {
        const uint8_t* q = (const uint8_t*)p + i * (DT == QWHIP_F32 ? 4u : 2u);
        if constexpr (DT == QWHIP_F32) {
            v[0] = ((const qw_words4*)q)[0].v;
            v[1] = ((const qw_words4*)q)[1].v;
        } else {
            v[0] = *(const u4_t*)q;
        }
    }
    // Keeps a load from sinking into the branch behind which its value is used: all of a batch are in flight together.
    __device__ __forceinline__ void pin() {
        asm volatile("" : "+v"(v[0]));
        if constexpr (DT == QWHIP_F32) asm volatile("" : "+v"(v[1]));
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
// One summation order for every call on a weight type: a token's logits do not depend on the rows or experts beside it, so a
// token decodes, verifies and prefills to the same experts.  The hidden dimension goes in chunks of 32 columns; chunk c adds to
// partial sum c % 16, ascending, and the sixteen end as Q[i] = P[i] + P[i + 8], ((Q0 + Q1) + (Q2 + Q3)) + ((Q4 + Q5) + (Q6 + Q7)).
// bf16 weights: a chunk is one bf16 matrix product per term of the activations.  Other weights: a partial is four fp32 FMA chains
// over the columns 8 g .. 8 g + 7 of its chunks, ended as (g0 + g1) + (g2 + g3): with partial p and chain g in lane 4 p + g, a
// wavefront's own order over pieces of 512 columns (qw_router_dot), and the order of the fp32 product of four 16x1x16 blocks.
// ------------------------------------------------------------------------------------------------

// Sum over the wavefront, in that order; every lane gets it.
__device__ __forceinline__ float qw_router_fold(float v) {
    v += __shfl_xor(v, 1, 64);
    v += __shfl_xor(v, 2, 64);
    v += __shfl_xor(v, 32, 64);
    v += __shfl_xor(v, 4, 64);
    v += __shfl_xor(v, 8, 64);
    v += __shfl_xor(v, 16, 64);
    return v;
}

// R rows of x (rows past `rows` repeat the last) against one weight row by a wavefront: 16-byte loads, P pieces of 512 columns in flight.
// `w` is 4-byte aligned, `x` 16-byte.
template <int XDT, int WDT, int R, int P>
__device__ __forceinline__ void qw_router_dot(const void* x, uint32_t rows, const void* w, uint64_t wbase, uint32_t H, uint32_t lane, float* out) {
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.0f;
    for (uint32_t h0 = lane * 8u; h0 < H; h0 += 512u * P) {
        qw_raw8<XDT> a[P][R];
        qw_raw8<WDT> b[P];
#pragma unroll
        for (uint32_t u = 0; u < P; ++u) {
            const uint32_t h = h0 + 512u * u < H ? h0 + 512u * u : h0;
            b[u].load(w, wbase + h);
#pragma unroll
            for (int r = 0; r < R; ++r) a[u][r].load(x, (uint64_t)min((uint32_t)r, rows - 1u) * H + h);
        }
#pragma unroll
        for (uint32_t u = 1; u < P; ++u) {
            b[u].pin();
#pragma unroll
            for (int r = 0; r < R; ++r) a[u][r].pin();
        }
#pragma unroll
        for (uint32_t u = 0; u < P; ++u) {
            float fb[8];
            b[u].floats(fb);
            if (u > 0 && h0 + 512u * u >= H) break;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float fa[8];
                a[u][r].floats(fa);
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[r] = fmaf(fb[j], fa[j], acc[r]);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) out[r] = qw_router_fold(acc[r]);
}

// The same for bf16 weights, on the matrix cores: a piece of 512 columns is sixteen chunks, lane 16 g + p holds columns
// 8 g .. 8 g + 7 of chunk p of both rows, and the products' diagonal is what the sixteen partial sums gain.  `w` is 16-byte aligned.
template <int XDT, int R, int P>
__device__ __forceinline__ void qw_router_dot_bf16(const void* x, uint32_t rows, const void* w, uint64_t wbase, uint32_t H, uint32_t lane, float* out) {
    constexpr int TERMS = XDT == QWHIP_BF16 ? 1 : (XDT == QWHIP_F16 ? 2 : 3);
    f4_t acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = f4_t{0.f, 0.f, 0.f, 0.f};
    const uint32_t mine = 32u * (lane & 15u) + 8u * (lane >> 4);
    for (uint32_t base = 0; base < H; base += 512u * P) {          // uniform
        qw_raw8<XDT> a[P][R];
        qw_raw8<QWHIP_BF16> b[P];
#pragma unroll
        for (uint32_t u = 0; u < P; ++u) {
            const uint32_t h = base + 512u * u + mine < H ? base + 512u * u + mine : 0u;
            b[u].load(w, wbase + h);
#pragma unroll
            for (int r = 0; r < R; ++r) a[u][r].load(x, (uint64_t)min((uint32_t)r, rows - 1u) * H + h);
        }
#pragma unroll
        for (uint32_t u = 1; u < P; ++u) {
            b[u].pin();
#pragma unroll
            for (int r = 0; r < R; ++r) a[u][r].pin();
        }
#pragma unroll
        for (uint32_t u = 0; u < P; ++u) {
            if (u > 0 && base + 512u * u >= H) break;   // uniform
            const bool in = base + 512u * u + mine < H;   // a chunk past the row adds zeros
            const u4_t zero = {0u, 0u, 0u, 0u};
            const qw_bf8_t wt = __builtin_bit_cast(qw_bf8_t, in ? b[u].v[0] : zero);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                qw_bf8_t xt[TERMS];
                if constexpr (XDT == QWHIP_BF16) {
                    xt[0] = __builtin_bit_cast(qw_bf8_t, in ? a[u][r].v[0] : zero);
                } else {
                    float f[8];
                    a[u][r].floats(f);
#pragma unroll
                    for (int j = 0; j < 8; ++j) f[j] = in ? f[j] : 0.0f;
#pragma unroll
                    for (int p = 0; p < TERMS; ++p) xt[p] = qw_take_bf16(f);
                }
#pragma unroll
                for (int p = TERMS - 1; p >= 0; --p) acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xt[p], wt, acc[r], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        // partial sum p is row p of column p: register p & 3 of lane 16 (p >> 2) + p
        const uint32_t i = lane & 3u;
        float v = i == 0u ? acc[r][0] : i == 1u ? acc[r][1] : i == 2u ? acc[r][2] : acc[r][3];
        v = __shfl(v, (int)(((lane & 12u) << 2) | (lane & 15u)), 64);
        v += __shfl_xor(v, 8, 64);
        v += __shfl_xor(v, 1, 64);
        v += __shfl_xor(v, 2, 64);
        v += __shfl_xor(v, 4, 64);
        if constexpr (XDT != QWHIP_BF16) {   // what the tiles sum again (below), the wavefront does here
            if (v != v) qw_router_dot<XDT, QWHIP_BF16, 1, 4>((const uint8_t*)x + (uint64_t)min((uint32_t)r, rows - 1u) * H * (XDT == QWHIP_F32 ? 4u : 2u), 1u, w, wbase, H, lane, &v);
        }
        out[r] = v;
    }
}

// 16 tokens x 16 NT weight rows a workgroup on the matrix cores, chunk c to wave c % W.  Operands go from memory to registers as
// they lie (lane (r, g): row r, columns 8 g .. 8 g + 7 of a chunk; nothing is shared between waves, so LDS would only add a copy),
// U chunks in flight per wave.
// bf16 weights meet the activations as one to three bf16 products that hold every bit of them (exact products, fp32 sums: 48
// matrix-core clocks a chunk for fp32 rows, where fp32 products take 256); other weights take the fp32 matrix product.
// What bounded the kernel before (one lane per hidden column, every weight x token product one vector instruction and one LDS
// operand): 2048 x 128 x 2048 with fp32 rows 94 us, now 13 (two passes over 16 MB of rows); 4 x 256 x 2048 7.2 us, now 5.0;
// 2048 x 128 x 2048 all fp32 96 us, now 21, all f16 85 us, now 17.
// The last band (gate_y) is the shared-expert gate: a dot product with an fp32 row per token.
template <int XDT, int WDT, int NT, int W>
__global__ __launch_bounds__(64 * W) void qw_router_mfma_kernel(const void* __restrict__ x, const void* __restrict__ wr, float* __restrict__ out,
                                                                uint32_t T, uint32_t E, uint32_t H, const float* __restrict__ sh_w,
                                                                float* __restrict__ sh_out, uint32_t gate_y, uint32_t epi, float scale) {
    static_assert(W == 8 || W == 16, "sixteen partial sums");
    typedef float f16_t __attribute__((ext_vector_type(16)));
    constexpr uint32_t PITCH = NT * 16 + 4;   // rows 4 apart fall 16 banks apart
    __shared__ float part[W][16 * PITCH];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t t0 = blockIdx.x * 16u;
    if (blockIdx.y == gate_y) {
        for (uint32_t t = t0 + wave; t < min(t0 + 16u, T); t += W) {
            float v;
            qw_router_dot<XDT, QWHIP_F32, 1, 4>((const uint8_t*)x + (uint64_t)t * H * (XDT == QWHIP_F32 ? 4u : 2u), 1u, sh_w, 0u, H, lane, &v);
            if (lane == 0) sh_out[t] = 1.0f / (1.0f + expf(-v));
        }
        return;
    }
    const uint32_t e0 = blockIdx.y * (16u * NT), r = lane & 15u, g = lane >> 4;
    const uint64_t xi = (uint64_t)min(t0 + r, T - 1u) * H + 8u * g;   // rows past the end repeat the last one and are not stored
    uint64_t wi[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) wi[n] = (uint64_t)min(e0 + 16u * n + r, E - 1u) * H + 8u * g;
    const uint32_t chunks = H >> 5;
    constexpr int U = 4, A = 16 / W;   // the wave's partial sums: wave and, with eight waves, wave + 8
    // one product takes a register quad and the partials go side by side; four blocks take sixteen and they go one after the other
    constexpr bool SIDE = WDT == QWHIP_BF16;
    constexpr uint32_t STEP = SIDE ? W : 16;
    using acc_t = std::conditional_t<SIDE, f4_t, f16_t>;
    f4_t sum[NT];
#pragma unroll
    for (int a = 0; a < (SIDE ? 1 : A); ++a) {
        acc_t acc[SIDE ? A : 1][NT];
#pragma unroll
        for (int s = 0; s < (SIDE ? A : 1); ++s)
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[s][n] = acc_t{};
        for (uint32_t c = wave + W * a; c < chunks; c += STEP * U) {
            qw_raw8<XDT> xa[U];
            qw_raw8<WDT> wb[U][NT];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t h = 32u * (c + STEP * u < chunks ? c + STEP * u : c);
                xa[u].load(x, xi + h);
#pragma unroll
                for (int n = 0; n < NT; ++n) wb[u][n].load(wr, wi[n] + h);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (u > 0 && c + STEP * u >= chunks) break;   // wave-uniform
                if constexpr (SIDE) {
                    constexpr int M = A - 1;
                    constexpr int P = XDT == QWHIP_BF16 ? 1 : (XDT == QWHIP_F16 ? 2 : 3);
                    qw_bf8_t xt[P];
                    if constexpr (XDT == QWHIP_BF16) {
                        xt[0] = __builtin_bit_cast(qw_bf8_t, xa[u].v[0]);
                    } else {
                        float f[8];
                        xa[u].floats(f);
#pragma unroll
                        for (int p = 0; p < P; ++p) xt[p] = qw_take_bf16(f);
                    }
                    // the smallest terms first
#pragma unroll
                    for (int p = P - 1; p >= 0; --p)
#pragma unroll
                        for (int n = 0; n < NT; ++n)
                            acc[u & M][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xt[p], __builtin_bit_cast(qw_bf8_t, wb[u][n].v[0]), acc[u & M][n], 0, 0, 0);
                } else {
                    float fa[8], fb[NT][8];
                    xa[u].floats(fa);
#pragma unroll
                    for (int n = 0; n < NT; ++n) wb[u][n].floats(fb[n]);
#pragma unroll
                    for (int j = 0; j < 8; ++j)
#pragma unroll
                        for (int n = 0; n < NT; ++n) acc[0][n] = __builtin_amdgcn_mfma_f32_16x16x1f32(fa[j], fb[n][j], acc[0][n], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int n = 0; n < NT; ++n) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (SIDE) {
                    sum[n][i] = A == 1 ? acc[0][n][i] : acc[0][n][i] + acc[A - 1][n][i];
                } else {   // block g in registers 4 g .. 4 g + 3
                    const float q = (acc[0][n][i] + acc[0][n][4 + i]) + (acc[0][n][8 + i] + acc[0][n][12 + i]);
                    sum[n][i] = a == 0 ? q : sum[n][i] + q;
                }
            }
        }
    }
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i) part[wave][(4u * g + i) * PITCH + 16u * n + r] = sum[n][i];
    __syncthreads();
    for (uint32_t o = threadIdx.x; o < 16u * 16u * NT; o += 64u * W) {
        const uint32_t row = o / (16u * NT), col = o % (16u * NT);
        float q[8];
#pragma unroll
        for (int w = 0; w < 8; ++w) {
            q[w] = part[w][row * PITCH + col];
            if constexpr (W == 16) q[w] += part[w + 8][row * PITCH + col];
        }
        float v = ((q[0] + q[1]) + (q[2] + q[3])) + ((q[4] + q[5]) + (q[6] + q[7]));
        const bool live = t0 + row < T && e0 + col < E;
        if constexpr (WDT == QWHIP_BF16 && XDT != QWHIP_BF16) {
            // the bf16 terms of an infinity, and zero terms against an infinite weight, make NaN of what may be an infinity: the
            // wavefront sums such outputs again from the operands as they are, one after the other (4 x 256 x 2048 with a NaN row
            // 16 us, 5.4 without; 145 with a lane to an output)
            for (unsigned long long odd = __ballot(live && v != v); odd != 0ull; odd &= odd - 1ull) {
                const int from = __builtin_ctzll(odd);
                const uint64_t tr = t0 + __builtin_amdgcn_readlane((int)row, from), er = e0 + __builtin_amdgcn_readlane((int)col, from);
                float again;
                qw_router_dot<XDT, WDT, 1, 4>((const uint8_t*)x + tr * H * (XDT == QWHIP_F32 ? 4u : 2u), 1u, wr, er * H, H, lane, &again);
                if ((int)lane == from) v = again;
            }
        }
        if (!live) continue;
        out[(uint64_t)(t0 + row) * E + e0 + col] = qw_f32_gemv_epilogue(v, epi, scale);
    }
}

// A few token rows: a wavefront is a workgroup and owns one weight row (the last one the shared-expert gate).  A row of 2048
// weights is four loads a lane, all in flight: the launch is its own latency, where a tile of sixteen rows takes the fp32 matrix
// pipe of a compute unit 1.7 us, and repeats a row's loads and terms sixteen times.
template <int XDT, int WDT, int R>
__global__ __launch_bounds__(64) void qw_router_rows_kernel(const void* __restrict__ x, const void* __restrict__ wr, float* __restrict__ out,
                                                            uint32_t T, uint32_t E, uint32_t H, const float* __restrict__ sh_w,
                                                            float* __restrict__ sh_out, uint32_t epi, float scale) {
    constexpr int P = R <= 2 ? 4 : 2;
    const uint32_t e = blockIdx.x, lane = threadIdx.x;
    float v[R];
    if (e == E) qw_router_dot<XDT, QWHIP_F32, R, P>(x, T, sh_w, 0u, H, lane, v);
    else if constexpr (WDT == QWHIP_BF16) qw_router_dot_bf16<XDT, R, P>(x, T, wr, (uint64_t)e * H, H, lane, v);
    else qw_router_dot<XDT, WDT, R, P>(x, T, wr, (uint64_t)e * H, H, lane, v);
    if (lane != 0) return;
#pragma unroll
    for (uint32_t t = 0; t < R; ++t) {
        if (t >= T) break;
        if (e == E) sh_out[t] = 1.0f / (1.0f + expf(-v[t]));
        else out[(uint64_t)t * E + e] = qw_f32_gemv_epilogue(v[t], epi, scale);
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

// Launches the matrix-core or the few-rows kernel; false for a type the caller reports.  The choice does not show in the results.
// A wavefront per weight row up to four token rows (fp32 weights, 128 x 2048: 2 / 4 rows 2.3 / 3.1 us, tiles of sixteen rows 6.2 / 6.5),
// on bf16 weights with rows that split into terms up to two (fp32 rows, 1 / 2 / 4: 2.6 / 3.3 / 5.0 us, tiles 4.5 / 4.7 / 4.9).
// Tile: 64 weight rows a workgroup (the activations' bf16 terms made once for four products) from 160 such tiles on, else 16 weight
// rows and twice the waves: fewer tiles leave compute units idle and are bound by the latency of a wave's own chunks.  Hidden 2048,
// 64 / 128 / 192 / 256 tiles, narrow against wide: fp32 rows, bf16 weights 7.6 / 12.7 / 18.0 / 23.3 us against 12.6 / 12.6 / 12.8 / 13.2;
// f16 rows 5.8 / 9.8 / 13.6 / 17.7 against 10.9 / 11.0 / 11.0 / 11.2; all fp32 9.5 / 16.4 / 23.2 / 30.0 against 20.0 / 20.1 / 20.5 / 20.9.
template <int XDT, int WDT>
static void qw_router_launch(hipStream_t st, const void* x, const void* wr, uint32_t t, uint32_t experts, uint32_t hidden, float* out,
                             const float* sh_w, float* sh_out, uint32_t epi, float scale) {
    const uint32_t gate = sh_w ? 1u : 0u;
    constexpr bool SPLIT = WDT == QWHIP_BF16 && XDT != QWHIP_BF16;
#define QW_ROWS(R) \
    hipLaunchKernelGGL((qw_router_rows_kernel<XDT, WDT, R>), dim3(experts + gate), dim3(64), 0, st, x, wr, out, t, experts, hidden, sh_w, sh_out, epi, scale)
    if (t == 1u) {
        QW_ROWS(1);
        return;
    }
    if (t == 2u) {
        QW_ROWS(2);
        return;
    }
    if constexpr (!SPLIT) {
        if (t <= 4u) {
            QW_ROWS(4);
            return;
        }
    }
#undef QW_ROWS
    const uint32_t gx = qwhip_cdiv(t, 16u);
    if ((uint64_t)gx * qwhip_cdiv(experts, 64u) >= 160u) {
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
    const bool wide = hidden % 32u == 0 && (((uintptr_t)x | (uintptr_t)wr) & 15u) == 0;
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
// qwg_f32_gemv / qwg_f32_gemv_bm): y[t, n] = epilogue(sum_k W[n, k] x[t, k]) on the router kernels (every weight row read once
// per sixteen activation rows, per four where there are no more, per eight or fewer off the 16-byte boundaries).
extern "C" qwhip_status qwhip_f32_gemv(qwhip_stream_t s, const float* w, const float* x, uint32_t rows, uint32_t n, uint32_t k,
                                       uint32_t epi, float scale, float* y) {
    if (epi > 3u) return qwhip_fail(QWHIP_E_BAD_SHAPE, "epilogue %u is not one of 0 none, 1 silu(y/scale), 2 sigmoid, 3 2 sigmoid(y/scale)", epi);
    if ((epi == 1u || epi == 3u) && !(scale != 0.0f && scale == scale))
        return qwhip_fail(QWHIP_E_BAD_SHAPE, "epilogue %u divides by its scale, which must be a non-zero number", epi);
    return qw_router_gemm_impl(s, x, QWHIP_F32, w, QWHIP_F32, rows, n, k, y, nullptr, nullptr, epi, scale);
}

