// GEMM with the weights dequantized straight into the matrix cores' operand registers (K in whole pairs of 64, groups of at most
// 128): grouped (MoE; gemm.hip has the form for the rest), and dense where choose_direct in gemm.hip prices it below the tiles.
//
// A workgroup of four waves owns 256 weight rows of one expert and up to 32 * MAXF of its sorted rows; wave w owns tile columns
// [64 w, 64 w + 64) for all of them: NF x 2 fragments of v_mfma_f32_32x32x16_f16, NF = 1 .. MAXF (a switch in front of the K loop:
// an expert of 70 rows multiplies 96).  A weight chunk is dequantized once for up to four matrix products, where 64-row tiles
// had two: on the containers with a long unpack the vector ALU was the bound, and tails of 1 to 32 rows multiplied 64.
//  - Weights: 128 columns of the wave's 64 rows at a time, copied raw (consecutive lanes take consecutive 16-byte pieces of a
//    row: a few coalesced loads where a lane per block costs one address per lane) through a wave-private LDS image, which needs
//    no barrier; lane (j, kh) reads slice 2 s + kh of row j in K-step s and dequantizes chunk ks of it as the second operand
//    of sub-step ks.  The K order inside a K-step is permuted accordingly, the same for every form: the same bits.  Rows are an odd
//    number of whole pieces apart: aligned 16-byte stores (pieces at 88 bytes, half of them misaligned: 175 us where this
//    takes 164 on the gate|up of 2048 rows x top-8 of 128 experts, 2048 x 768).
//  - Activations: a 64-column stage per K-step through registers into LDS, XOR-swizzled, one barrier per K-step.
//  - Everything a sub-step needs is asked for one sub-step ahead: fragment a of the next one as soon as the two products that
//    read it are issued, the next weight chunk between this one's products.
// Bound, 2048 rows x top-8 of 128 experts of 2048 x 768: gate|up 153 .. 162 us by the card (HQ4_G32_M5; 6.1 vector instructions beside a
// matrix product on spans of 128, 8.8 on 64; the matrix pipe is busy 38 % of the cycles on either: at two and three waves a SIMD the
// products wait for the unpack and its operands); at 32 rows an expert and fewer the bank's stream, 252 MB in 72 us.  Layers against the
// 64-row kernel before, in turn: HQ4_G32_M5 2048 / 256 / 16 rows 286 -> 274, 134 -> 125, 100 -> 87 us; 1500 rows, top-6 of 64 experts:
// 4-bit affine g64 230 -> 186, 8-bit 330 -> 236, 6-bit 302 -> 226 us.
#pragma once
#include <atomic>

#include "qwhip_common.h"
#include "qw_gemm.h"

namespace {

template <int FMT>
__host__ __device__ constexpr int qd_chunks() {   // 16-byte pieces of one row's 128 columns: bits + 1
    return FMT == QG_FMT_B8 ? 9 : FMT == QG_FMT_B6 ? 7 : FMT == QG_FMT_B3 ? 4 : FMT == QG_FMT_B2 ? 3 : 5;
}
// 32-row fragments of a span: the wider raw pieces of the 6- and 8-bit containers leave registers for three
template <int FMT>
__host__ __device__ constexpr int qd_span() { return FMT == QG_FMT_B8 || FMT == QG_FMT_B6 ? 3 : 4; }
// bytes between the rows of a raw image: an odd number of 16-byte pieces (a block read's 32 rows meet on 16 banks at most twice)
template <int FMT>
__host__ __device__ constexpr uint32_t qd_pitch() { return 16u * (qd_chunks<FMT>() | 1); }
// wavefronts per SIMD: three where the registers of 64 rows allow it
template <int FMT, int MAXF>
__host__ __device__ constexpr int qd_waves() { return MAXF > 2 || FMT == QG_FMT_B8 || FMT == QG_FMT_B6 ? 2 : 3; }
typedef u4_t qd_piece __attribute__((aligned(4)));   // 16 bytes at 4-byte alignment

template <int N>
struct qd_int { static constexpr int value = N; };

// The workgroup's work: an expert's rows [m0, m0 + rows_valid), nf fragments of 32, and a column tile.
struct qd_item {
    uint32_t e, m0, rows_valid, nf, col;
};
// rows of n rows' span i of at most MAXF fragments
template <int MAXF>
__device__ __forceinline__ void qd_span_rows(uint32_t rows, uint32_t spans, uint32_t i, uint32_t& row0, qd_item& it) {
    const uint32_t frags = (rows + 31u) >> 5, base_f = frags / spans, more = frags - base_f * spans;
    const uint32_t f0 = i * base_f + min(i, more);
    row0 = 32u * f0;
    it.nf = base_f + (i < more ? 1u : 0u);
    it.rows_valid = min(32u * it.nf, rows - row0);
}
// rows of tile-list code `packed`'s tile
__device__ __forceinline__ uint32_t qd_tile_rows(uint32_t packed) {
    const uint32_t code = packed >> 24;
    return code == 1u ? 16u : (code == 2u ? 32u : 64u);
}
// Grid: one-dimensional and XCD-aware - workgroup L runs on XCD L % 8 (round-robin dispatch), each XCD takes one contiguous
// eighth of the expert-sorted tile list and walks (tile, column tile) column-fastest, so the spans of an expert and the column
// tiles of a span run side by side under one L2.  The list's entries are tiles of at most 64 rows.  Where all tiles of an expert
// are listed one after the other, its 32-row fragments are dealt evenly to as few spans of at most MAXF as hold them, entry i (rows
// 64 i ..) takes span i and the other entries leave; an entry of any other list (a part of one, another order) takes its own rows.
// The neighbours that this looks at are asked for together with the entry itself.
template <int MAXF>
__device__ __forceinline__ bool qd_find_item(const qw_gemm_params& p, qd_item& it) {
    const uint32_t ncol = p.tiles_n;
    const uint32_t xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3;
    const uint32_t tc = (uint32_t)max(p.tile_count[0], 0);
    const uint32_t per_xcd = (tc + 7u) >> 3;
    const uint32_t ti = slot / ncol;
    const uint32_t t = xcd * per_xcd + ti;
    if (ti >= per_xcd || t >= tc) return false;
    const uint32_t lane = threadIdx.x & 63u, near = t + lane - 31u;   // entries t - 31 .. t + 32; below 0 wraps past tc
    const uint32_t near_e = near < tc ? (uint32_t)p.tile_e[near] : ~0u, near_r = near < tc ? (uint32_t)p.tile_r[near] : 0u;
    const uint32_t e = (uint32_t)p.tile_e[t];
    const uint32_t packed = (uint32_t)p.tile_r[t];
    const uint32_t bm = qd_tile_rows(packed);
    const uint32_t first = (packed & 0xFFFFFFu) * bm;              // row of the expert
    const uint32_t off_e = (uint32_t)p.expert_off[e];
    const uint32_t rows_e = (uint32_t)p.expert_off[e + 1] - off_e;
    if (first >= rows_e) return false;
    it.e = e;
    it.col = slot - ti * ncol;

    const uint32_t tiles = (rows_e + 63u) >> 6, i = first >> 6;
    // is (le, lr) the tile of rows 64 q .. of this expert?
    const auto is_tile = [&](uint32_t le, uint32_t lr, uint32_t q) -> bool {
        const uint32_t n = qd_tile_rows(lr);
        return le == e && (lr & 0xFFFFFFu) * n == 64u * q && n >= min(64u, rows_e - 64u * q);
    };
    bool whole = t >= i && t - i + tiles <= tc;
    if (whole) {
        if (i <= 31u && tiles - i <= 33u) {
            const uint32_t q = lane + i - 31u;
            whole = __all(q >= tiles || is_tile(near_e, near_r, q));
        } else {
            for (uint32_t q = lane; q < tiles; q += 64u) whole = whole && is_tile((uint32_t)p.tile_e[t - i + q], (uint32_t)p.tile_r[t - i + q], q);
            whole = __all(whole);
        }
    }
    uint32_t row0 = first;
    if (whole) {
        const uint32_t spans = (rows_e + 32u * MAXF - 1u) / (32u * MAXF);
        if (i >= spans) return false;
        qd_span_rows<MAXF>(rows_e, spans, i, row0, it);
    } else {
        it.rows_valid = min(bm, rows_e - first);
        it.nf = (it.rows_valid + 31u) >> 5;
    }
    it.m0 = off_e + row0;
    return true;
}
// A dense problem: tiles_m spans of the M rows, the spans of a column tile side by side on one XCD, K ranges by blockIdx.y.
template <int MAXF>
__device__ __forceinline__ bool qd_find_dense(const qw_gemm_params& p, qd_item& it) {
    const uint32_t total = p.tiles_m * p.tiles_n, per_xcd = (total + 7u) >> 3;
    const uint32_t t = (blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= per_xcd || t >= total) return false;
    it.e = 0;
    it.col = t / p.tiles_m;
    qd_span_rows<MAXF>(p.M, p.tiles_m, t - it.col * p.tiles_m, it.m0, it);
    return true;
}

// Outputs of a wave, rows 32 a .. + 31 at a time through a private LDS slab, 16-byte row chunks out.  SWIGLU: the wave's two column
// fragments are (gate, up) of the same 32 outputs, rounded to f16 first (the values the two-step chain stores), then SwiGLU and
// the FWHT-32 in fp32: the arithmetic of qwhip_swiglu_fwht on the f16 gate|up matrix without writing it (the
// reference's fused form for its dense path: qmm_t_nax_swiglu_impl, Sources/QWMetal/include/qw_gemm_nax_swiglu.metalh:86-167).
template <int YDT, bool SWIGLU, bool GACT, int MAXF>
__device__ __forceinline__ void qd_epilogue(const qw_gemm_params& p, void* y, const f16_t (&acc)[MAXF][2], uint32_t nf, uint32_t m0, uint32_t rows_valid,
                                            uint32_t n0, uint32_t wave, uint32_t lane, uint8_t* lds6) {
    const uint32_t j = lane & 31u, kh = lane >> 5;
    if constexpr (SWIGLU) {
        // eight outputs a lane, four lanes a rotation group: the FWHT-32 takes three stages inside a lane and two lane exchanges
        constexpr uint32_t EP_PITCH = 2 * 64 + 16;
        uint8_t* ep = lds6 + wave * (32u * EP_PITCH);
        const uint32_t w_off = (4u * kh) * EP_PITCH + j * 2u;
        const uint32_t cc = lane & 3u, n = n0 + wave * 32u + cc * 8u;
#pragma unroll
        for (int a = 0; a < MAXF; ++a) {
            if ((uint32_t)a >= nf) break;
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int r = 0; r < 16; ++r) *(h1_t*)(ep + w_off + (8u * (r >> 2) + (r & 3)) * EP_PITCH + b * 64u) = (h1_t)acc[a][b][r];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const uint32_t row = 16u * q + (lane >> 2), grow = 32u * a + row;
                const h8_t g = *(const h8_t*)(ep + row * EP_PITCH + cc * 16u), u = *(const h8_t*)(ep + row * EP_PITCH + 64u + cc * 16u);
                float f[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) f[i] = GACT ? qw_gated((float)g[i], (float)u[i], p.act) : qw_swiglu((float)g[i], (float)u[i]);
                if (p.rotate_act) qw_fwht32_quad(f, lane);
                if (grow < rows_valid && n < p.inter) qw_store8_f16((h1_t*)y + (uint64_t)(m0 + grow) * p.ldy + n, f);
            }
        }
    } else if constexpr (YDT != QWHIP_F32) {
        constexpr uint32_t EP_PITCH = 2 * 64 + 16;
        uint8_t* ep = lds6 + wave * (32u * EP_PITCH);
        const uint32_t w_off = (4u * kh) * EP_PITCH + j * 2u;
#pragma unroll
        for (int a = 0; a < MAXF; ++a) {
            if ((uint32_t)a >= nf) break;
#pragma unroll
            for (int b = 0; b < 2; ++b) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t o = w_off + (8u * (r >> 2) + (r & 3)) * EP_PITCH + b * 64u;
                    if constexpr (YDT == QWHIP_BF16) *(uint16_t*)(ep + o) = qw_f32_to_bf16(acc[a][b][r]);
                    else *(h1_t*)(ep + o) = (h1_t)acc[a][b][r];
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t c = q * 64u + lane;
                const uint32_t row = c >> 3, cc = c & 7u;
                const u4_t v = *(const u4_t*)(ep + row * EP_PITCH + cc * 16u);
                const uint32_t grow = 32u * a + row;
                const uint32_t n = n0 + wave * 64u + cc * 8u;
                if (grow < rows_valid && n < p.N)
                    *(u4_t*)((uint16_t*)y + (uint64_t)(m0 + grow) * p.ldy + n) = v;
            }
        }
    } else {
#pragma unroll
        for (int a = 0; a < MAXF; ++a) {
            if ((uint32_t)a >= nf) break;
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const uint32_t n = n0 + wave * 64u + 32u * b + j;
                if (n < p.N) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const uint32_t row = 32u * a + 8 * (r >> 2) + 4 * kh + (r & 3);
                        if (row < rows_valid) qg_store<YDT>(y, (uint64_t)(m0 + row) * p.ldy + n, acc[a][b][r]);
                    }
                }
            }
        }
    }
}

}  // namespace

// DENSE: one bank, rows [m0, ..) of x in place, a K range per blockIdx.y into an fp32 plane of [M, ldy] each (gridDim.y = 1: into y).
template <int FMT, int YDT, bool SWIGLU, bool GACT, int XDT, int MAXF, bool DENSE = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(qd_waves<FMT, MAXF>(), qd_waves<FMT, MAXF>()))) void qw_gemm6_kernel(const qw_gemm_params p) {
    static_assert(!SWIGLU || YDT == QWHIP_F16, "fused SwiGLU stores f16");
    constexpr int C = qd_chunks<FMT>();
    constexpr uint32_t BN = 256, A_STAGE = MAXF * 4096u, RAW_OFF = 2u * A_STAGE;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds6[];
    const uint32_t tid = threadIdx.x;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63u;

    qd_item it;
    if (!(DENSE ? qd_find_dense<MAXF>(p, it) : qd_find_item<MAXF>(p, it))) return;
    const uint32_t m0 = it.m0, rows_valid = it.rows_valid, nf = it.nf;
    const uint32_t n0 = it.col * (SWIGLU ? BN / 2 : BN);
    const uint32_t pair_bytes = (4u >> p.gshift) * p.bb;             // of a row's 128 columns
    uint32_t nkp = p.K / 128u, kp0 = 0;                              // K pairs of this workgroup
    if constexpr (DENSE) {
        const uint32_t per = (nkp + gridDim.y - 1u) / gridDim.y;
        kp0 = blockIdx.y * per;
        nkp = min(per, nkp - kp0);                                   // the launcher leaves no range empty
    }
    const uint32_t bank_row0 = DENSE && !SWIGLU ? n0 : 0u;           // row offsets are 32 bits: of an expert, of a dense tile
    const uint8_t* bank = p.bank + ((uint64_t)it.e * p.rows_per_expert + bank_row0) * p.row_bytes + (uint64_t)kp0 * pair_bytes;
    const uint8_t* xbase = (const uint8_t*)p.x + (DENSE ? (uint64_t)m0 * p.ldx * 2u + (uint64_t)kp0 * 256u : 0u);

    // activation tile: chunk (row = (tid >> 3) + 32 i, 16-byte k-chunk tid & 7) -> LDS slot k-chunk ^ ((row >> 1) & 7)
    uint32_t a_voff[MAXF];
#pragma unroll
    for (int i = 0; i < MAXF; ++i) {
        const uint32_t row = (tid >> 3) + 32u * i;
        const uint32_t r = row < rows_valid ? row : rows_valid - 1u;
        const uint32_t src_row = DENSE ? r : p.gather ? (uint32_t)p.gather[m0 + r] : m0 + r;
        a_voff[i] = src_row * p.ldx * 2u + (tid & 7u) * 16u;    // activations (dense: a span's) < 4 GiB (checked by the launcher)
    }
    const uint32_t a_lds0 = (tid >> 3) * 128u + (((tid & 7u) ^ ((tid >> 4) & 7u)) << 4);   // + i * 4096 (swizzle key unchanged)

    // wave-private raw image: 16-byte piece q = lane + 64 i of the wave's 64 rows x 128 columns
    constexpr uint32_t pitch = qd_pitch<FMT>();
    uint32_t raw_goff[C], raw_loff[C];
#pragma unroll
    for (int i = 0; i < C; ++i) {
        const uint32_t q = lane + 64u * i, nl = q / (uint32_t)C, c = q - (uint32_t)C * nl;
        const uint32_t b = nl >> 5, jj = nl & 31u;
        uint32_t row;
        if constexpr (SWIGLU) row = (b ? p.inter : 0u) + min(n0 + 32u * wave + jj, p.inter - 1u);
        else row = min(n0 + 64u * wave + nl, p.N - 1u) - bank_row0;
        raw_goff[i] = row * (uint32_t)p.row_bytes + min(16u * c, pair_bytes - 16u);   // an expert's rows span < 4 GiB
        raw_loff[i] = RAW_OFF + (64u * wave + nl) * pitch + 16u * c;
    }
    // contraction role: lane (j, kh) reads slice 2 s + kh of rows 64 wave + 32 b + j in K-step s of the pair
    const uint32_t j = lane & 31u, kh = lane >> 5;
    // byte `at` of a row's pair lies at its place, or, past the whole pieces, in the last one (which ends with the row's bytes)
    const uint32_t whole = pair_bytes & ~15u;
    const auto place = [&](uint32_t at, uint32_t n) -> uint32_t { return at + n <= whole ? at : whole + at - (pair_bytes - 16u); };
    constexpr uint32_t W = qg_slice_words<FMT>(), SB = 4u * W, W0 = W > 4u ? 4u : W;
    const uint32_t rd_row = RAW_OFF + (64u * wave + j) * pitch;
    const uint32_t gm = (1u << p.gshift) - 1u;
    uint32_t rd_hdr[2], rd_q[2], rd_q1[2];
#pragma unroll
    for (uint32_t s = 0; s < 2; ++s) {
        const uint32_t si = 2u * s + kh, at = (si >> p.gshift) * p.bb, q = at + 4u + (si & gm) * SB;
        rd_hdr[s] = rd_row + at;
        rd_q[s] = rd_row + place(q, 4u * W0);
        rd_q1[s] = W > 4u ? rd_row + place(q + 16u, SB - 16u) : 0u;
    }
    const uint32_t fr_key = (j >> 1) & 7u;
    const uint32_t a_rd = j * 128u;

    f16_t acc[MAXF][2];
#pragma unroll
    for (int a = 0; a < MAXF; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.0f;
    const uint32_t magic = qw_vgpr_const(0x64006400u);
    const uint32_t last = 2u * nkp - 1u, lastp = nkp - 1u;

    auto contract = [&](auto nf_c) __attribute__((always_inline)) {
        constexpr int NF = decltype(nf_c)::value;
        u4_t a_reg[NF], raw[C];
        auto load_a = [&](uint32_t kt) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < NF; ++i) {
                asm volatile("" : "+v"(a_voff[i]));   // scalar base + 32-bit lane offset addressing (see qw_gemm3_kernel)
                a_reg[i] = *(const u4_t*)(xbase + (uint64_t)kt * 128u + a_voff[i]);
            }
        };
        auto store_a = [&](uint32_t stage) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < NF; ++i) *(h8_t*)(lds6 + stage * A_STAGE + a_lds0 + i * 4096u) = qg_to_f16x8<XDT>(a_reg[i]);
        };
        auto load_raw = [&](uint32_t kp) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < C; ++i) {
                asm volatile("" : "+v"(raw_goff[i]));
                raw[i] = *(const qd_piece*)(bank + (uint64_t)kp * pair_bytes + raw_goff[i]);
            }
        };
        auto store_raw = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < C; ++i) *(u4_t*)(lds6 + raw_loff[i]) = raw[i];
        };
        qg_slice<FMT> blk[2];
        h2_t s2[2], b2[2];
        auto read_blk = [&](uint32_t s) __attribute__((always_inline)) {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                blk[b].hdr = *(const uint32_t*)(lds6 + rd_hdr[s] + b * 32u * pitch);
                const uint32_t* q0 = (const uint32_t*)(lds6 + rd_q[s] + b * 32u * pitch);
#pragma unroll
                for (int w = 0; w < (int)W0; ++w) blk[b].q[w] = q0[w];
                if constexpr (W > 4u) {
                    const uint32_t* q1 = (const uint32_t*)(lds6 + rd_q1[s] + b * 32u * pitch);
#pragma unroll
                    for (int w = 4; w < (int)W; ++w) blk[b].q[w] = q1[w - 4];
                }
            }
        };
        auto splat = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                s2[b] = qw_splat_lo(blk[b].hdr);
                b2[b] = qw_splat_hi(blk[b].hdr);
            }
        };
        auto frag = [&](uint32_t stage, int ks, int a) __attribute__((always_inline)) -> h8_t {
            return *(const h8_t*)(lds6 + stage * A_STAGE + a_rd + (((4u * kh + (uint32_t)ks) ^ fr_key) << 4) + a * 4096u);
        };

        load_raw(0);
        load_a(0);
        store_raw();
        store_a(0);
        load_a(min(1u, last));
        load_raw(min(1u, lastp));
        __syncthreads();
        read_blk(0);
        h8_t af[NF], wc[2], wn[2];
#pragma unroll
        for (int a = 0; a < NF; ++a) af[a] = frag(0, 0, a);
        splat();
#pragma unroll
        for (int b = 0; b < 2; ++b) wc[b] = qg_dequant_chunk<FMT>(blk[b], 0, s2[b], b2[b], magic);

        for (uint32_t kp = 0; kp <= lastp; ++kp) {
#pragma unroll
            for (int s = 0; s < 2; ++s) {
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) {
                    if (ks == 3) {
                        __syncthreads();      // stage s ^ 1 holds the next K-step
                        splat();
                    }
#pragma unroll
                    for (int a = 0; a < NF; ++a) {
                        acc[a][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[a], wc[0], acc[a][0], 0, 0, 0);
                        acc[a][1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[a], wc[1], acc[a][1], 0, 0, 0);
                        af[a] = ks < 3 ? frag(s, ks + 1, a) : frag(s ^ 1, 0, a);
                        if (a == 0) wn[0] = qg_dequant_chunk<FMT>(blk[0], (ks + 1) & 3, s2[0], b2[0], magic);
                        if (a == NF / 2) wn[1] = qg_dequant_chunk<FMT>(blk[1], (ks + 1) & 3, s2[1], b2[1], magic);
                    }
                    if (ks == 0) {
                        store_a(s ^ 1);
                        load_a(min(2u * kp + s + 2u, last));
                    }
                    if (s == 1 && ks == 1) {  // the pair's last slices are in registers: its successor takes the image
                        store_raw();
                        load_raw(min(kp + 2u, lastp));
                    }
                    if (ks == 2) read_blk(s ^ 1);
                    wc[0] = wn[0];
                    wc[1] = wn[1];
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    };
    if (MAXF > 3 && nf == 4u) contract(qd_int<MAXF>{});
    else if (MAXF > 2 && nf == 3u) contract(qd_int<(MAXF < 3 ? MAXF : 3)>{});
    else if (nf == 2u) contract(qd_int<2>{});
    else contract(qd_int<1>{});
    __syncthreads();

    void* y = DENSE && YDT == QWHIP_F32 ? (void*)((float*)p.y + (uint64_t)blockIdx.y * p.M * p.ldy) : p.y;
    qd_epilogue<YDT, SWIGLU, GACT, MAXF>(p, y, acc, nf, m0, rows_valid, n0, wave, lane, lds6);
}
