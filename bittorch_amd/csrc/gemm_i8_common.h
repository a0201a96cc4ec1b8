// Shared by the tiled int8 GEMM kernels (gemm_i8.hip, gemm_i8_dma.hip): launch parameters and the output stage.
#pragma once
#include <cstddef>

#include "bt_common.h"

namespace bt {

constexpr int G_BM = 128;
constexpr int G_BN = 256;
constexpr int G_BK = 128;           // k per LDS stage (two k64 MFMA sub-steps)
constexpr int G_MB = G_BM / 16;     // 16-row blocks per tile
constexpr int G_STAGE_BYTES = G_BM * G_BK;  // 16 KiB

struct GemmParams {
    // The first 64 bytes hold what a workgroup needs to find its tile and request its first operands: the kernel
    // arguments come through the scalar cache a 64-byte line at a time.
    const int8_t* Q;      // [M, K]
    const uint8_t* W_T;   // [Kb, N]
    int64_t K, M, N;
    int tiles_m, tiles_n;
    int per_xcd;          // workgroups per XCD (grid = 8 * per_xcd)
    int wsteps, tiles16;  // WT: 16-row steps and 16-column tiles of the decode-tiled weight copy (tiles16 < 0: stored_tile16)
    int tile_n0;          // first column tile of this launch (tiles_n counts the launch's own column tiles)
    // ---- needed later
    const float* s_x;     // [M]
    void* Y;              // [M, N]
    int32_t* acc_out;     // optional [M, N]
    int64_t Kb;
    int y_dtype;
    int long_epilogue;    // A/B runs and tests (option GEMM_LONG_EPILOGUE): never the short epilogue
    int fine_from;        // gemm_i8_dma.hip: an XCD's tiles from this one on are computed in finer ones
    const int32_t* q_rowsum;  // FL kernels: sum of each row of Q over K (what the codes w + 1 of the field layout add)
    Epilogue epi;
};
static_assert(offsetof(GemmParams, s_x) == 64, "first argument line as laid out above");

// up to four consecutive outputs (left: how many the row still has) that start on any element
template <int DT>
__device__ __forceinline__ void store4_any(void* Y, const float (&v)[4], int left) {
    if constexpr (DT == BT_F32) {
        if (left >= 4) {
            u32x4_a4 o;
#pragma unroll
            for (int t = 0; t < 4; t++) o[t] = __builtin_bit_cast(uint32_t, v[t]);
            *(u32x4_a4*)Y = o;
            return;
        }
#pragma unroll
        for (int t = 0; t < 3; t++)
            if (t < left) ((float*)Y)[t] = v[t];
    } else {
        uint16_t h[4];
#pragma unroll
        for (int t = 0; t < 4; t++) h[t] = DT == BT_F16 ? f32_to_f16_bits(v[t]) : f32_to_bf16_bits(v[t]);
        if (left >= 4) {
            *(u32x2_a2*)Y = u32x2_a2{(uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16)};
            return;
        }
#pragma unroll
        for (int t = 0; t < 3; t++)
            if (t < left) ((uint16_t*)Y)[t] = h[t];
    }
}
__device__ __forceinline__ void store4(void* Y, int dt, int64_t idx, const float (&v)[4]) {
    if (dt == BT_F32) {
        st4_nt((float*)Y + idx, __builtin_bit_cast(uint32_t, v[0]), __builtin_bit_cast(uint32_t, v[1]),
               __builtin_bit_cast(uint32_t, v[2]), __builtin_bit_cast(uint32_t, v[3]));
    } else {
        uint16_t h[4];
#pragma unroll
        for (int i = 0; i < 4; i++) h[i] = (dt == BT_F16) ? f32_to_f16_bits(v[i]) : f32_to_bf16_bits(v[i]);
        st2_nt((uint16_t*)Y + idx, (uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
    }
}

// Finishes NB 16-row blocks (acc[MB0 .. MB0+NB-1]) of the tile: NB = 4 in a tile of 128 rows, 2 or 1 in the tiles of
// 64 and 32 rows a launch's remainder is cut into.
// The epilogue's operands (row scales of the wave's rows, column scales and biases as raw bits)
// are requested before the K-half exchange, whose LDS round trips cover their latency.
template <int NB>
struct EpiOperands {
    float sx[NB][4];  // [row block within the half][r]
    uint32_t ws_bits[4], bs_bits[4];
    uint2 res[NB][4]; // 16-bit residual of the lane's four columns in each of its rows (short epilogue only)
};
// The residual of a 16-bit output for the short epilogue (full tile): all 16 rows requested at once, next to the
// other epilogue operands, so that the hand-over of the K halves covers their latency.  (One load per row right
// before its use, as the long epilogue does, leaves a memory round trip per row exposed: 5 us per tile.)
template <int NB>
__device__ __forceinline__ void load_epi_residual(const GemmParams& p, int64_t m0, int mb0, int g, int64_t ncol, EpiOperands<NB>& e) {
    const uint16_t* base = (const uint16_t*)p.epi.residual + (m0 + 16 * mb0 + 4 * g) * p.N + ncol;
#pragma unroll
    for (int mbi = 0; mbi < NB; mbi++)
#pragma unroll
        for (int r = 0; r < 4; r++) e.res[mbi][r] = *(const uint2*)(base + (int64_t)(16 * mbi + r) * p.N);
}
template <int NB>
__device__ __forceinline__ void load_epi_operands(const GemmParams& p, int64_t m0, int mb0, int g, int64_t ncol,
                                                  bool col_ok, EpiOperands<NB>& e) {
#pragma unroll
    for (int mbi = 0; mbi < NB; mbi++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int64_t m = m0 + 16 * (mb0 + mbi) + 4 * g + r;
            e.sx[mbi][r] = p.s_x[m < p.M ? m : p.M - 1];
        }
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int64_t n = col_ok ? ncol + t : 0;
        e.ws_bits[t] = load_bits_rt(p.epi.scale, p.epi.scale_dtype, p.epi.scale_bcast ? 0 : n);
        e.bs_bits[t] = p.epi.bias ? load_bits_rt(p.epi.bias, p.epi.bias_dtype, n) : 0u;
    }
}

// The field layout (W_LAYOUT_TILED_FIELDS, FL = true) leaves column block t of a lane scaled by 4^t (64 for t = 3):
// float(acc) * (127 / 4^t) is the same real number as float(acc / 4^t) * 127 -- the scaled accumulator has the
// significant bits of the true one and the factor is a power of two apart from 127 -- so the epilogue takes the
// scale out in the multiplication it already has.
template <bool FL>
__device__ __forceinline__ constexpr float k127(int t) {
    return FL ? (t == 0 ? 127.0f : t == 1 ? 127.0f / 4.0f : t == 2 ? 127.0f / 16.0f : 127.0f / 64.0f) : 127.0f;
}
template <bool FL>
__device__ __forceinline__ constexpr int field_shift(int t) { return FL ? 2 * t : 0; }

template <int YDT, int MB0, int NB, bool FL = false>
__device__ __forceinline__ void gemm_epilogue(const GemmParams& p, const v4i (&acc)[2 * NB][4], int64_t m0, int g,
                                              int64_t ncol, const EpiOperands<NB>& e) {
    float ws[4], bs[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        ws[t] = bits_to_f32_rt(e.ws_bits[t], p.epi.scale_dtype);
        bs[t] = p.epi.bias ? bits_to_f32_rt(e.bs_bits[t], p.epi.bias_dtype) : 0.0f;
    }
#pragma unroll
    for (int mbi = 0; mbi < NB; mbi++) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int64_t m = m0 + 16 * (MB0 + mbi) + 4 * g + r;
            if (m >= p.M) continue;
            const float sx = e.sx[mbi][r];
            float y[4];
#pragma unroll
            for (int t = 0; t < 4; t++) {
                // float(127 a) = float(a) * 127 rounded once: |a| <= 127 K < 2^24 (checked by the host), so float(a)
                // is exact and the product rounds the same integer the reference converts (one operation less than
                // 127 a in integers first)
                const float a127f = __fmul_rn((float)acc[MB0 + mbi][t][r], k127<FL>(t));
                y[t] = epi_int8_f(a127f, sx, ws[t], bs[t]);
            }
            if (p.epi.residual) add_residual4(y, p.epi.residual, YDT, m * p.N + ncol);
            store4(p.Y, YDT, m * p.N + ncol, y);
            if (p.acc_out) {
                uint32_t a127[4];
#pragma unroll
                for (int t = 0; t < 4; t++) a127[t] = (uint32_t)times127(acc[MB0 + mbi][t][r] >> field_shift<FL>(t));
                st4_nt(p.acc_out + m * p.N + ncol, a127[0], a127[1], a127[2], a127[3]);
            }
        }
    }
}
// The same for the common case, with the bookkeeping taken out of the per-row work: every row of the tile exists,
// no residual, no accumulator output, and every row scale large enough for the two-operation division
// (all wave-uniform, checked by the caller).  A row's address is a uniform base plus a 32-bit lane offset fixed
// for the whole epilogue.  Same bits as gemm_epilogue.
template <int YDT, int MB0, int NB, bool RES = false, bool FL = false>
__device__ __forceinline__ void gemm_epilogue_fast(const GemmParams& p, const v4i (&acc)[2 * NB][4], int64_t m0, int g,
                                                   int64_t ncol, const EpiOperands<NB>& e) {
    float ws[4], bs[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        ws[t] = bits_to_f32_rt(e.ws_bits[t], p.epi.scale_dtype);
        bs[t] = p.epi.bias ? bits_to_f32_rt(e.bs_bits[t], p.epi.bias_dtype) : 0.0f;
    }
    constexpr int ES = (YDT == BT_F32) ? 4 : 2;
    const int64_t ncol0 = (int64_t)__builtin_amdgcn_readfirstlane((int)(ncol / G_BN)) * G_BN;  // the tile's first column
    const uint32_t lane_off = ((uint32_t)(4 * g) * (uint32_t)p.N + (uint32_t)(ncol - ncol0)) * ES;
    char* const base = (char*)p.Y + ((m0 + 16 * MB0) * p.N + ncol0) * ES;  // uniform
    const int64_t row_bytes = p.N * ES;
#pragma unroll
    for (int mbi = 0; mbi < NB; mbi++) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float sx = e.sx[mbi][r];
            float y[4];
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const float a127f = __fmul_rn((float)acc[MB0 + mbi][t][r], k127<FL>(t));
                const float q = div127_fast(__fmul_rn(a127f, sx));
                y[t] = __fadd_rn(__fmul_rn(q, ws[t]), bs[t]);
            }
            if constexpr (RES && YDT != BT_F32) {  // linear rounded to the output's dtype, then + residual (add_residual4)
                const uint32_t d[2] = {e.res[mbi][r].x, e.res[mbi][r].y};
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    const uint32_t h = (d[t >> 1] >> (16 * (t & 1))) & 0xffffu;
                    const float rv = (YDT == BT_F16) ? f16_bits_to_f32((uint16_t)h) : bf16_bits_to_f32((uint16_t)h);
                    y[t] = sum_in_dtype(round_to_dtype(y[t], YDT), rv, YDT);
                }
            }
            char* const dst = base + (int64_t)(16 * mbi + r) * row_bytes + lane_off;
            if constexpr (YDT == BT_F32) {
                st4_nt((float*)dst, __builtin_bit_cast(uint32_t, y[0]), __builtin_bit_cast(uint32_t, y[1]),
                       __builtin_bit_cast(uint32_t, y[2]), __builtin_bit_cast(uint32_t, y[3]));
            } else {
                uint16_t h[4];
#pragma unroll
                for (int i = 0; i < 4; i++) h[i] = (YDT == BT_F16) ? f32_to_f16_bits(y[i]) : f32_to_bf16_bits(y[i]);
                st2_nt((uint16_t*)dst, (uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
            }
        }
    }
}
template <int MB0, int NB, bool FL = false>
__device__ __forceinline__ void gemm_epilogue_dt(const GemmParams& p, const v4i (&acc)[2 * NB][4], int64_t m0, int g,
                                                 int64_t ncol, const EpiOperands<NB>& e) {
    if (p.y_dtype == BT_BF16) gemm_epilogue<BT_BF16, MB0, NB, FL>(p, acc, m0, g, ncol, e);
    else if (p.y_dtype == BT_F16) gemm_epilogue<BT_F16, MB0, NB, FL>(p, acc, m0, g, ncol, e);
    else gemm_epilogue<BT_F32, MB0, NB, FL>(p, acc, m0, g, ncol, e);
}
template <int MB0, int NB, bool FL = false>
__device__ __forceinline__ void gemm_epilogue_dt(const GemmParams& p, const v4i (&acc)[2 * NB][4], int64_t m0, int g,
                                                 int64_t ncol, const EpiOperands<NB>& e, bool fast) {
    if (fast) {  // wave-uniform
        if (p.epi.residual) {  // (16-bit outputs only: checked by the caller)
            if (p.y_dtype == BT_BF16) gemm_epilogue_fast<BT_BF16, MB0, NB, true, FL>(p, acc, m0, g, ncol, e);
            else gemm_epilogue_fast<BT_F16, MB0, NB, true, FL>(p, acc, m0, g, ncol, e);
        } else if (p.y_dtype == BT_BF16) gemm_epilogue_fast<BT_BF16, MB0, NB, false, FL>(p, acc, m0, g, ncol, e);
        else if (p.y_dtype == BT_F16) gemm_epilogue_fast<BT_F16, MB0, NB, false, FL>(p, acc, m0, g, ncol, e);
        else gemm_epilogue_fast<BT_F32, MB0, NB, false, FL>(p, acc, m0, g, ncol, e);
        return;
    }
    gemm_epilogue_dt<MB0, NB, FL>(p, acc, m0, g, ncol, e);
}

}  // namespace bt
