// fp32 activations x packed ternary weights on the bf16 matrix cores, and the two gradient products of an fp32 layer.
//
//   gemm_f32_kernel    Y = X W^T * scale + bias (the forward), and dX = (dY * scale) W (the input gradient), W ternary
//   grad_w_f32_kernel  dW = scale * dY^T X, with dBias = column sums of dY taken along
//
// Arithmetic of the forward restated from the reference's packed kernel (csrc/kernels/ternary_gemm_production.cu:158-250);
// the gradients are those of bittorch/nn/ternary_linear_cuda.py:73-111 (straight-through estimator).
//
// An fp32 value is the exact sum of three bf16 values (24 significand bits = 3 x 8), ternary weights are exact in bf16,
// and the 16-bit matrix cores sum exact products in fp32: three MFMAs do what an fp32 product does, at a sixteenth of an
// fp32 MFMA's price each.
//
// Every wave works alone: no LDS, no barrier.  An operand lane of v_mfma_f32_16x16x32_bf16 wants 8 values of one row, and
// the order of k inside an MFMA is free, so a lane loads the fp32 values themselves, splits them in registers (11 VALU
// operations per pair) and decodes the weights in the matching order.  The split of one wave's rows is hidden behind the
// MFMAs of the other wave of its SIMD: a tile of 64 x 128 needs 270 VALU operations (1080 cycles) per 96 MFMAs (1536).
#include <cfloat>
#include <cstddef>

#include "bt_common.h"

namespace bt {

typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));     // rows of any length: 4-byte alignment
typedef uint32_t u32x2_u __attribute__((ext_vector_type(2), aligned(1)));
typedef uint32_t u32_u __attribute__((aligned(1)));

__device__ __forceinline__ uint32_t f2u(float f) { return __builtin_bit_cast(uint32_t, f); }
__device__ __forceinline__ float u2f(uint32_t u) { return __builtin_bit_cast(float, u); }

// (a, b) as three dwords of two bf16 each, a in the low half: x = hi + mid + lo exactly, every term a truncation.
__device__ __forceinline__ void split_pair(float a, float b, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
    hi = perm(f2u(b), f2u(a), 0x07060302u);
    const float ra = a - u2f(f2u(a) & 0xFFFF0000u), rb = b - u2f(f2u(b) & 0xFFFF0000u);
    mid = perm(f2u(rb), f2u(ra), 0x07060302u);
    const float la = ra - u2f(f2u(ra) & 0xFFFF0000u), lb = rb - u2f(f2u(rb) & 0xFFFF0000u);
    lo = perm(f2u(lb), f2u(la), 0x07060302u);
}
// The same for any value: the smaller terms of an infinity or NaN are zero, so that it meets a weight as fp32 has it.
__device__ __forceinline__ void split_pair_any(float a, float b, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
    split_pair(fabsf(a) <= FLT_MAX ? a : 0.0f, fabsf(b) <= FLT_MAX ? b : 0.0f, hi, mid, lo);
    hi = perm(f2u(__builtin_canonicalizef(b)), f2u(__builtin_canonicalizef(a)), 0x07060302u);  // (a quiet NaN's top half is one)
}
// The same as the first with hi and mid rounded to nearest: hi leaves at most 2^-8 of x's power of two and mid at most 2^-17, and what is
// left after each has either sign (still exact: 24 bits are 8, a sign and 8, a sign and 8).  Beyond the largest bf16 value hi
// becomes an infinity and the other terms NaN.
__device__ __forceinline__ void split_pair_rn(float a, float b, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
    typedef float v2f __attribute__((ext_vector_type(2)));
    typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
    hi = __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f{a, b}), v2bf));  // v_cvt_pk_bf16_f32
    const float ra = a - u2f(hi << 16), rb = b - u2f(hi & 0xFFFF0000u);
    mid = __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f{ra, rb}), v2bf));
    const float la = ra - u2f(mid << 16), lb = rb - u2f(mid & 0xFFFF0000u);
    lo = perm(f2u(lb), f2u(la), 0x07060302u);
}

__device__ __forceinline__ v4f mfma_bf16(const u32x4& a, const u32x4& b, const v4f& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
}

// ---- forward and input gradient --------------------------------------------------------------------------------------

// where the ternary operand comes from
enum { B_ROW_MAJOR = 0,   // W_T [Kb, N], contraction over k (four codes per byte)
       B_TILED = 1,       // the decode-tiled copy, contraction over k
       B_TRANSPOSED = 2 };// W_T [Kb, N], contraction over n; output columns are k

struct GemmF32Params {
    const float* X;      // [M, C], C the contraction length
    const uint8_t* W;
    int64_t M, C, NC;    // NC: output columns
    int tiles_m, tiles_n;
    int per_xcd;         // tiles per XCD
    int fine_from;       // PARTS > 1: an XCD's tiles from this one on are shared by PARTS workgroups each
    int wsteps;          // B_TILED: 64-wide steps of the copy
    int tiles16;         // B_TILED: as in tiles16_arg
    int ldw;             // bytes of a W_T row
    int kb;              // rows of W_T
    float* Y;            // [M, NC]
    const float* a_scale;// B_TRANSPOSED: factor of X's column c (or null)
    const float* y_scale;// B_TRANSPOSED: one factor for every output (per-tensor scale), or null
    Epilogue epi;        // forward
};

// bf16 +-0.5: the weights' value here, so that the low byte is zero and a sum cannot overflow before it is doubled
constexpr uint32_t LUT_BF16_HALF = 0x00BF3F00u;

// A wave works on a tile of 16 NB rows x 64 NG columns (NB = 4, but for shared tiles), from row m_at and column c_at on (KS = 1), or tile
// (tm, tn) (KS > 1).  Parameters by value, and the place of a tile of KS > 1 formed in here: otherwise the compiler orders the output
// stage so that such launches take a microsecond longer (fp32, 600 x 768 x 3072 29.2 / 30.5, 2000 x 512 x 2048 23.1 / 24.4).
// KS > 1: all KS waves of a workgroup work on one tile, each on its run of the contraction, and add their sums through LDS
// (pairwise, always in the same order): for outputs with too few tiles to occupy the chip.
// SC: X's columns are scaled (input gradient with one scale per row of W).
// RN: forward outputs of N % 4 != 0, an instance of its own: asked at run time, every other output paid half a microsecond for
// the clamped columns and the second way to store (us, fp32, 300 x 4096 x 512 17.9 / 17.0, 4096 x 768 x 768 28.2 / 27.5).  Only
// the tile of one wave's 64 x 64 outputs gains from the question: with a branch between them the compiler sends each row's
// stores off by themselves (512 x 2048 x 1032 17.0 without, 16.0 with it; 4096 x 128 x 2048 24.1 / 23.1).
template <int SRC, int NG, int NB, int KS, bool SC, bool RN>
__device__ __forceinline__ void gemm_f32_tile(const GemmF32Params p, const int64_t m_at, const int64_t c_at, const uint32_t tm, const uint32_t tn) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 15, g = lane >> 4;
    const int64_t m0 = KS == 1 ? m_at : (int64_t)tm * 64, c0 = KS == 1 ? c_at : (int64_t)tn * (64 * NG);

    // rows and columns past the end repeat the last one: they only feed outputs that are never stored
    const uint8_t* a_base = (const uint8_t*)(p.X + m0 * p.C);
    uint32_t a_off[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int64_t left = p.M - 1 - m0;
        const uint32_t r = (uint32_t)((16 * b + i < left) ? 16 * b + i : left);
        a_off[b] = (r * (uint32_t)p.C + 8u * g) * 4u;
    }
    uint32_t b_off[NG];
    uint32_t b_shift = 0;  // RN: bits by which the last columns, loaded as the last four, stand too high
#pragma unroll
    for (int q = 0; q < NG; q++) {
        const int64_t col = c0 + 64 * q + 4 * i;
        if constexpr (SRC == B_ROW_MAJOR) {
            b_off[q] = 2u * g * (uint32_t)p.ldw + (uint32_t)(col < (RN ? p.NC - 4 : p.NC) ? col : p.NC - 4);
            if (RN && col < p.NC && col > p.NC - 4) b_shift = 8u * (uint32_t)(col - (p.NC - 4));  // (one q at most)
        } else if constexpr (SRC == B_TILED) {
            const int tt = stored_tile16((int)(col >> 4), p.tiles16);
            b_off[q] = ((uint32_t)tt * (uint32_t)p.wsteps * 64u + 16u * (g >> 1) + 4u * (i & 3)) * 4u;
        } else {
            const int kb = (int)(col >> 2);
            b_off[q] = (uint32_t)(kb < p.kb ? kb : p.kb - 1) * (uint32_t)p.ldw + 8u * g;
        }
    }
    const uint32_t sel_wt = ((uint32_t)(2 * (g & 1) + 1) << 24) | (0x0Cu << 16) | ((uint32_t)(2 * (g & 1)) << 8) | 0x0Cu;
    // this wave's steps of 32: [st0, st1) of the whole ones, and the partial one if it is the last wave
    const int nfull = (int)(p.C / 32), steps = (int)((p.C + 31) / 32);
    const int run = (KS == 1) ? nfull : (nfull + KS - 1) / KS;
    const int st0 = (KS == 1) ? 0 : min(wave * run, nfull), st1 = (KS == 1) ? nfull : min(st0 + run, nfull);
    const bool last = KS == 1 || wave == KS - 1;

    constexpr int BR = (SRC == B_TILED) ? 4 : 2;
    f32x4_u raw[NB][2];
    uint32_t braw[NG][BR];
    f32x4_u sc[2];

    auto load_a = [&](int b, int s, bool tail) {  // s uniform, tail a constant
        if (!tail) {
            const uint8_t* ab = a_base + (int64_t)s * 128;
            raw[b][0] = *(const f32x4_u*)(ab + a_off[b]);
            raw[b][1] = *(const f32x4_u*)(ab + 16 + a_off[b]);
        } else {  // the last, partial step: element by element, zero past the end
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int64_t c = (int64_t)s * 32 + 8 * g + e;
                const float v = *(const float*)(a_base + (a_off[b] - 32u * g) + 4 * (c < p.C ? c : 0));
                raw[b][e >> 2][e & 3] = c < p.C ? v : 0.0f;
            }
        }
    };
    auto load_w = [&](int s, bool tail) {
#pragma unroll
        for (int q = 0; q < NG; q++) {
            if constexpr (SRC == B_ROW_MAJOR) {
                const uint8_t* wb = p.W + (int64_t)s * 8 * p.ldw;
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    if (!tail) {
                        braw[q][r] = *(const u32_u*)(wb + (int64_t)r * p.ldw + b_off[q]);
                    } else {  // rows past the end of W_T meet zeros of X
                        const int over = 8 * s + 2 * g + r - (p.kb - 1);
                        const int row = over > 0 ? r - over : r;
                        braw[q][r] = *(const u32_u*)(wb + (int64_t)row * p.ldw + b_off[q]);
                    }
                }
            } else if constexpr (SRC == B_TILED) {
                const uint4 v = *(const uint4*)(p.W + (size_t)(s >> 1) * 256 + 128u * (s & 1) + b_off[q]);
                braw[q][0] = v.x; braw[q][1] = v.y; braw[q][2] = v.z; braw[q][BR - 1] = v.w;
            } else if (!tail) {
                const u32x2_u v = *(const u32x2_u*)(p.W + (int64_t)s * 32 + b_off[q]);
                braw[q][0] = v[0]; braw[q][1] = v[1];
            } else {
                uint32_t d[2] = {0, 0};
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int64_t n = (int64_t)s * 32 + 8 * g + e;
                    const uint32_t v = p.W[(b_off[q] - 8u * g) + (n < p.C ? n : 0)];
                    d[e >> 2] |= (n < p.C ? v : 0u) << (8 * (e & 3));
                }
                braw[q][0] = d[0]; braw[q][1] = d[1];
            }
        }
        if constexpr (SC) {
            if (!tail) {
                sc[0] = *(const f32x4_u*)(p.a_scale + (int64_t)s * 32 + 8 * g);
                sc[1] = *(const f32x4_u*)(p.a_scale + (int64_t)s * 32 + 8 * g + 4);
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int64_t c = (int64_t)s * 32 + 8 * g + e;
                    sc[e >> 2][e & 3] = p.a_scale[c < p.C ? c : 0];
                }
            }
        }
    };

    v4f acc[NB][4 * NG];
    u32x4 pl[2][3];  // the planes of two row blocks: one in the MFMAs, the next being split
    auto split = [&](int b, const f32x4_u (&scn)[2], auto any) __attribute__((always_inline)) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] = raw[b][e >> 2][e & 3];
        if constexpr (SC) {
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = __fmul_rn(x[e], scn[e >> 2][e & 3]);
        }
        // the k order of the weight decode: forward dword c = { k = c, k = 4 + c } (decode8_16bit);
        // transposed dwords = { 1, 3 }, { 0, 2 }, { 5, 7 }, { 4, 6 } of the lane's eight n
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int e0 = (SRC == B_TRANSPOSED) ? (4 * (c >> 1) + 1 - (c & 1)) : c;
            const int e1 = (SRC == B_TRANSPOSED) ? e0 + 2 : 4 + c;
            uint32_t h, m, l;
            if constexpr (decltype(any)::value) split_pair_any(x[e0], x[e1], h, m, l);
            else split_pair(x[e0], x[e1], h, m, l);
            pl[b & 1][0][c] = l; pl[b & 1][1][c] = m; pl[b & 1][2][c] = h;
        }
    };

    auto step = [&](int nx, bool more, auto any) __attribute__((always_inline)) {  // nx: the step whose operands are requested behind this one's use (uniform)
        u32x4 w[4 * NG];
        if constexpr (RN && SRC == B_ROW_MAJOR) {
#pragma unroll
            for (int q = 0; q < NG; q++)
#pragma unroll
                for (int r = 0; r < 2; r++)
                    if (c0 + 64 * q + 4 * i > p.NC - 4) braw[q][r] >>= b_shift;
        }
#pragma unroll
        for (int q = 0; q < NG; q++)
#pragma unroll
            for (int t = 0; t < 4; t++) {
                if constexpr (SRC == B_ROW_MAJOR) {
                    const uint32_t sel = ((uint32_t)(4 + t) << 24) | (0x0Cu << 16) | ((uint32_t)t << 8) | 0x0Cu;
                    w[4 * q + t] = decode8_16bit<LUT_BF16_HALF>(perm(braw[q][1], braw[q][0], sel));
                } else if constexpr (SRC == B_TILED) {
                    w[4 * q + t] = decode8_16bit<LUT_BF16_HALF>(perm(0u, braw[q][t], sel_wt));
                } else {
#pragma unroll
                    for (int d = 0; d < 2; d++) {
                        w[4 * q + t][2 * d] = perm(0u, LUT_BF16_HALF, (braw[q][d] >> (2 * t)) & 0x03000300u);
                        w[4 * q + t][2 * d + 1] = perm(0u, LUT_BF16_HALF, ((braw[q][d] << 8) >> (2 * t)) & 0x03000300u);
                    }
                }
            }
        const f32x4_u scn[2] = {sc[0], sc[1]};
        if (more) load_w(nx, false);
        split(0, scn, any);
        if (more) load_a(0, nx, false);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int b = 0; b < NB; b++) {
            if (b < NB - 1) {
                split(b + 1, scn, any);
                if (more) load_a(b + 1, nx, false);
            }
#pragma unroll
            for (int h = 0; h < 3; h++)  // smallest terms first
#pragma unroll
                for (int t = 0; t < 4 * NG; t++) acc[b][t] = mfma_bf16(pl[b & 1][h], w[t], acc[b][t]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto contract = [&](auto any) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int t = 0; t < 4 * NG; t++) acc[b][t] = v4f{0.f, 0.f, 0.f, 0.f};
        if (st0 < st1) {
            load_w(st0, false);
#pragma unroll
            for (int b = 0; b < NB; b++) load_a(b, st0, false);
            for (int s = st0; s < st1; s++) step(s + 1 < st1 ? s + 1 : s, true, any);  // (past the end: the last one again, never used)
        }
        if (last && nfull < steps) {
            load_w(nfull, true);
#pragma unroll
            for (int b = 0; b < NB; b++) load_a(b, nfull, true);
            step(0, false, any);
        }
    };
    contract(std::false_type{});
    if constexpr (SRC == B_TRANSPOSED) {
        // a non-finite value has no finite terms and left a NaN in its row: once more, with such values as they are
        bool bad = false;
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int t = 0; t < 4 * NG; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) bad |= acc[b][t][r] != acc[b][t][r];
        if (__any(bad)) contract(std::true_type{});
    }
    if constexpr (KS > 1) {
        // the upper half of the waves hands its sums to the lower half, until wave 0 has them all; NG words of 16 KiB each
        __shared__ __attribute__((aligned(16))) float xch[KS / 2 * 4096 * NG];
#pragma unroll
        for (int half = KS / 2; half >= 1; half /= 2) {
            if (wave >= half && wave < 2 * half) {
#pragma unroll
                for (int b = 0; b < NB; b++)
#pragma unroll
                    for (int t = 0; t < 4 * NG; t++)
                        *(v4f*)(xch + ((((wave - half) * NB + b) * 4 * NG + t) * 64 + lane) * 4) = acc[b][t];
            }
            __syncthreads();
            if (wave < half) {
#pragma unroll
                for (int b = 0; b < NB; b++)
#pragma unroll
                    for (int t = 0; t < 4 * NG; t++)
                        acc[b][t] += *(const v4f*)(xch + (((wave * NB + b) * 4 * NG + t) * 64 + lane) * 4);
            }
            __syncthreads();
        }
        if (wave != 0) return;
    }

#pragma unroll
    for (int q = 0; q < NG; q++) {
        const int64_t col = c0 + 64 * q + 4 * i;
        if (col >= p.NC) continue;
        float ws[4] = {1.f, 1.f, 1.f, 1.f}, bs[4] = {0.f, 0.f, 0.f, 0.f};
        if constexpr (SRC != B_TRANSPOSED) {
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const int64_t n = !RN || col + t < p.NC ? col + t : p.NC - 1;
                ws[t] = epi_scale(p.epi, n);
                bs[t] = epi_bias(p.epi, n);
            }
        }
#pragma unroll
        for (int b = 0; b < NB; b++) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int64_t m = m0 + 16 * b + 4 * g + r;
                if (m >= p.M) continue;
                float y[4];
#pragma unroll
                for (int t = 0; t < 4; t++) y[t] = acc[b][4 * q + t][r] * 2.0f;
                if constexpr (SRC == B_TRANSPOSED) {
                    if (p.y_scale) {
#pragma unroll
                        for (int t = 0; t < 4; t++) y[t] = __fmul_rn(y[t], p.y_scale[0]);
                    }
                    if (p.NC % 4 != 0) {
#pragma unroll
                        for (int t = 0; t < 4; t++)
                            if (col + t < p.NC) p.Y[m * p.NC + col + t] = y[t];
                        continue;
                    }
                } else {
#pragma unroll
                    for (int t = 0; t < 4; t++) y[t] = epi_float(y[t], ws[t], bs[t]);
                    if (KS == 8 ? p.NC % 4 != 0 : RN) {  // element by element
#pragma unroll
                        for (int t = 0; t < 4; t++) {
                            if (col + t >= p.NC) continue;
                            if (p.epi.residual) y[t] = add_residual(y[t], p.epi.residual, BT_F32, m * p.NC + col + t);
                            p.Y[m * p.NC + col + t] = y[t];
                        }
                        continue;
                    }
                    if (p.epi.residual) add_residual4(y, p.epi.residual, BT_F32, m * p.NC + col);
                }
                st4_nt(p.Y + m * p.NC + col, f2u(y[0]), f2u(y[1]), f2u(y[2]), f2u(y[3]));
            }
        }
    }
}

// KS = 1: the four waves of a workgroup are a 2 x 2 block of tiles of 64 rows.  KS > 1: see gemm_f32_tile.
// PARTS > 1 (KS = 1): a tile of the remainder, the last that would occupy a part of the compute units only, is shared by PARTS
// workgroups, whose waves take 32 or 16 rows each over the whole contraction: every output is the same chain of products as in a
// tile of its own, so that a row's bits do not depend on where it lies in the call.
template <int SRC, int NG, int KS, bool SC, bool RN, int PARTS>
__global__ __launch_bounds__(KS == 1 ? 256 : 64 * KS, 2) void gemm_f32_kernel(GemmF32Params p) {
    constexpr int TM = (KS == 1) ? 128 : 64, TN = (KS == 1) ? 128 * NG : 64 * NG;  // a workgroup's tile
    // the 8 XCDs each take a contiguous run of tiles, walked in groups of four row tiles (as in gemm_f16.hip)
    const uint32_t idx = blockIdx.x >> 3;
    const bool fine = PARTS > 1 && idx >= (uint32_t)p.fine_from;  // (uniform)
    const uint32_t f = fine ? idx - (uint32_t)p.fine_from : 0u, part = f % (uint32_t)PARTS;
    const uint32_t lin = (blockIdx.x & 7u) * (uint32_t)p.per_xcd + (fine ? (uint32_t)p.fine_from + f / (uint32_t)PARTS : idx);
    const uint32_t tiles_m = (uint32_t)p.tiles_m, tiles_n = (uint32_t)p.tiles_n;
    if (lin >= tiles_m * tiles_n) return;
    constexpr uint32_t GM = 4;
    const uint32_t group = lin / (GM * tiles_n), first_m = group * GM;
    const uint32_t gm = (tiles_m - first_m < GM) ? tiles_m - first_m : GM;
    const uint32_t in_group = lin - group * GM * tiles_n;
    const uint32_t tn = (gm == GM) ? in_group / GM : in_group / gm;
    const uint32_t tm = first_m + (in_group - tn * gm);

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t c0 = (int64_t)tn * TN + (KS == 1 ? 64 * NG * (wave & 1) : 0);
    if constexpr (PARTS > 1) {
        if (fine) {
            constexpr int NB = 4 / PARTS;
            const int64_t m0 = (int64_t)tm * TM + 16 * NB * (2 * (int)part + (wave >> 1));
            if (m0 < p.M && c0 < p.NC) gemm_f32_tile<SRC, NG, NB, KS, SC, RN>(p, m0, c0, tm, tn);
            return;
        }
    }
    const int64_t m0 = (int64_t)tm * TM + (KS == 1 ? 64 * (wave >> 1) : 0);
    if (KS == 1 && (m0 >= p.M || c0 >= p.NC)) return;  // (no barriers in a tile when KS == 1)
    gemm_f32_tile<SRC, NG, 4, KS, SC, RN>(p, m0, c0, tm, tn);
}

// Into how many workgroups a tile of the remainder is shared (KS = 1): the tiles beyond one, two ... for every compute unit of an XCD
// where they are at most half as many as compute units, so that half or three quarters of such a tile's time are saved.  (The plan is
// made without regard to it.)  us, tiles of their own / shared: 16384 x 768 x 768 forward 68.8 / 61.0, input gradient 70.9 / 65.5; 9000 x
// 2304 x 768 forward 93.5 / 86.5; four workgroups, 33792 x 256 x 1024 input gradient 71.5 / 63.6.  Less than 4 us of steps at 1.2 us each
// are not missed: 16384 x 768 x 192 23.9 / 23.8, 49000 x 256 x 160 22.0 / 22.2.
static int gemm_f32_parts(int64_t tiles, int64_t steps) {
    const int64_t cus = gemm_compute_units() / 8, per_xcd = ceil_div(tiles, 8), rem = per_xcd % cus;
    if (per_xcd < cus || rem == 0 || 2 * rem > cus) return 1;
    const int parts = 4 * rem > cus ? 2 : 4;
    return 1.2 * (double)steps * (1.0 - 1.0 / parts) > 4.0 ? parts : 1;
}
template <int SRC, int NG, int KS, bool SC, bool RN>
static int launch_gemm_f32_cfg(GemmF32Params p, const char* who, hipStream_t st) {
    p.tiles_m = (int)ceil_div(p.M, KS == 1 ? 128 : 64);
    p.tiles_n = (int)ceil_div(p.NC, KS == 1 ? 128 * NG : 64 * NG);
    const int64_t total = (int64_t)p.tiles_m * p.tiles_n;
    if (ceil_div(p.M, 64) >= (1ll << 31) || total >= (1ll << 31) - 8) {
        set_error("%s: more output tiles than one launch takes", who);
        return BT_ERR_INVALID;
    }
    p.per_xcd = (int)ceil_div(total, 8);
    const int parts = KS == 1 ? gemm_f32_parts(total, ceil_div(p.C, 32)) : 1;
    const int rem = parts > 1 ? p.per_xcd % (int)(gemm_compute_units() / 8) : 0;
    p.fine_from = p.per_xcd - rem;
    const dim3 grid((unsigned)(8 * (p.fine_from + parts * rem))), block(KS == 1 ? 256 : 64 * KS);
    if constexpr (KS == 1) {
        if (parts == 2) hipLaunchKernelGGL((gemm_f32_kernel<SRC, NG, KS, SC, RN, 2>), grid, block, 0, st, p);
        if (parts == 4) hipLaunchKernelGGL((gemm_f32_kernel<SRC, NG, KS, SC, RN, 4>), grid, block, 0, st, p);
        if (parts > 1) return check_launch(who);
    }
    hipLaunchKernelGGL((gemm_f32_kernel<SRC, NG, KS, SC, RN, 1>), grid, block, 0, st, p);
    return check_launch(who);
}
// Which split of the work?  0: tiles of 64 x 128 per wave, 1: the same with the contraction over the four waves of a
// workgroup, 2: tiles of 64 x 64 with the contraction over eight waves.  Priced with times fitted to measurements, in
// microseconds: a step of 32 costs a wave alone on its SIMD 1.2 (64 x 128) or 0.9 (64 x 64), two waves that share one 2.45
// or 2.1 together (16-bit MFMAs at 1.3 PFLOP/s; the small tile is bound by its split, 64 values per 8 MFMAs), a round of
// workgroups 5 to start and store, 8 with the sums passing through LDS.  Measured, 0 / 1 / 2: M = 16384, N = K = 768 68 / 79 /
// 131 us; M = N = K = 4096 314 / 339 / 540; M = 1000, contraction 11008, 4096 columns 433 / 243 / 387; M = 33, contraction
// 4096, 1024 columns 157 / 53 / 29; M = 64, 512 x 512 26 / 16 / 12.
static double gemm_f32_price(int64_t M, int64_t NC, int64_t C, int cfg) {
    const double simds = 4.0 * (double)gemm_compute_units();
    const int ks = cfg == 0 ? 1 : cfg == 1 ? 4 : 8;
    const double waves = (double)ceil_div(M, 64) * (double)ceil_div(NC, cfg == 2 ? 64 : 128) * ks;
    const double per_simd = (double)(int64_t)((waves + simds - 1) / simds), steps = (double)ceil_div(ceil_div(C, 32), ks);
    const double rounds = (double)(((int64_t)per_simd + 1) / 2), alone = cfg == 2 ? 0.9 : 1.2, pair = cfg == 2 ? 2.1 : 2.45;
    const bool odd = (int64_t)per_simd & 1;
    return 5.0 + steps * ((odd ? rounds - 1 : rounds) * pair + (odd ? alone : 0.0)) + rounds * (cfg == 0 ? 5.0 : 8.0);
}
static int gemm_f32_config(int64_t M, int64_t NC, int64_t C) {
    int best = 0;
    for (int c = 1; c < 3; c++)
        if (gemm_f32_price(M, NC, C, c) < gemm_f32_price(M, NC, C, best)) best = c;
    return best;
}
// microseconds of launch_gemm_f32, for the rule that chooses between it and the streaming kernel
double gemm_f32_cost(int64_t M, int64_t N, int64_t K) { return gemm_f32_price(M, N, K, gemm_f32_config(M, N, K)); }

template <int SRC, bool SC, bool RN = false>
static int launch_gemm_f32_src(const GemmF32Params& p, const char* who, hipStream_t st) {
    switch (gemm_f32_config(p.M, p.NC, p.C)) {
        case 0: return launch_gemm_f32_cfg<SRC, 2, 1, SC, RN>(p, who, st);
        case 1: return launch_gemm_f32_cfg<SRC, 2, 4, SC, RN>(p, who, st);
        default: return launch_gemm_f32_cfg<SRC, 1, 8, SC, RN>(p, who, st);
    }
}
template <int SRC>
static int launch_gemm_f32_forward(const GemmF32Params& p, const char* who, hipStream_t st) {
    return p.NC % 4 != 0 ? launch_gemm_f32_src<SRC, false, true>(p, who, st) : launch_gemm_f32_src<SRC, false>(p, who, st);
}

// the kernel's 32-bit offsets span 64 rows of X and the whole of W
bool gemm_f32_shape_ok(int64_t N, int64_t K) {
    return N >= 4 && K < (1ll << 23) && N < (1ll << 30) && ceil_div(K, 4) * N < (1ll << 32);
}
// X 4-byte, Y (and the residual) 16-byte aligned
bool gemm_f32_supported(int64_t N, int64_t K, const void* X, const void* Y) {
    return gemm_f32_shape_ok(N, K) && ((uintptr_t)X) % 4 == 0 && ((uintptr_t)Y) % 16 == 0;
}

int launch_gemm_f32(const void* X, const uint8_t* W, int w_layout, const Epilogue& epi, void* Y, int64_t M, int64_t N,
                    int64_t K, hipStream_t st) {
    GemmF32Params p = {};
    p.X = (const float*)X; p.W = W; p.M = M; p.C = K; p.NC = N; p.Y = (float*)Y; p.epi = epi;
    p.wsteps = (int)ceil_div(K, 64);
    p.tiles16 = tiles16_arg(N, w_layout);
    p.ldw = (int)N;
    p.kb = (int)ceil_div(K, 4);
    return layout_tiled(w_layout) ? launch_gemm_f32_forward<B_TILED>(p, "bt_ternary_linear_tiled_forward", st)
                                  : launch_gemm_f32_forward<B_ROW_MAJOR>(p, "bt_ternary_linear_packed_forward", st);
}

// ---- weight gradient ---------------------------------------------------------------------------------------------------

struct GradWParams {
    const float* G;       // [M, N]
    const float* X;       // [M, K]
    int64_t M, N, K;
    int tiles_n, tiles_k; // tiles of 128 x 128
    int splits;           // parts of the rows
    int per_xcd;          // workgroups per XCD (grid = 8 * per_xcd)
    int steps_per_split;  // 32-row steps of a part
    const float* scale;   // [N] or one entry
    int scale_bcast;
    float* out;           // splits == 1: dW [N, K]; otherwise partial sums [splits, N, K]
    float* bias_out;      // splits == 1: dBias [N]; otherwise partial sums [splits, 64-wide column tiles of X, N]; or null
};

// A wave owns a 64 x 64 tile of dW over its part of the rows.  Lane (i, g) loads columns 4i .. 4i+3 of rows 8g .. 8g+7 of
// both matrices: component t of those eight float4 is its operand of the MFMA whose row (column) i is matrix column 4i + t,
// so the transposition costs nothing.  Both operands are split, and of the nine products of terms six are formed: mid lo and
// lo mid are at most 2^-25 of the product each and have either sign.  Sums of up to 8 products are formed as fp32 products
// instead: an MFMA's sums are fewer but not rounded to nearest.  Relative error of 1 / 2 / 4 / 16 rows: MFMAs of all terms
// 4.3e-8 / 4.2e-8 / 4.1e-8 / 4.2e-8, the vendor's fp32 product 3.6e-8 / 4.1e-8 / 4.8e-8 / 7.8e-8.
constexpr int GRAD_W_FEW_ROWS = 8;
template <bool DIRECT>
__global__ __launch_bounds__(256, 2) void grad_w_f32_kernel(GradWParams p) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 15, g = lane >> 4;
    const uint32_t tiles = (uint32_t)(p.tiles_n * p.tiles_k);
    // each XCD takes a contiguous run of (part, tile): the tiles of one part of the rows share them in its L2
    const uint32_t lin = (blockIdx.x & 7u) * (uint32_t)p.per_xcd + (blockIdx.x >> 3);
    if (lin >= tiles * (uint32_t)p.splits) return;
    const uint32_t split = lin / tiles, tile = lin - split * tiles;
    const uint32_t tn = tile / (uint32_t)p.tiles_k, tk = tile - tn * (uint32_t)p.tiles_k;
    const int64_t n0 = (int64_t)tn * 128 + 64 * (wave >> 1), k0 = (int64_t)tk * 128 + 64 * (wave & 1);
    if (n0 >= p.N || k0 >= p.K) return;  // (no barriers below)
    // a lane's four columns; past the end the last four again (the same values are then stored twice)
    auto col_g = [&](int ii) { const int64_t c = n0 + 4 * ii; return c < p.N - 4 ? c : p.N - 4; };
    auto col_x = [&](int ii) { const int64_t c = k0 + 4 * ii; return c < p.K - 4 ? c : p.K - 4; };
    const uint32_t g_off = (8u * g * (uint32_t)p.N + (uint32_t)(col_g(i))) * 4u;
    const uint32_t x_off = (8u * g * (uint32_t)p.K + (uint32_t)(col_x(i))) * 4u;
    const int64_t s0 = (int64_t)split * p.steps_per_split;
    int64_t s1 = s0 + p.steps_per_split;
    const int64_t all = (p.M + 31) / 32, nfull = p.M / 32;
    if (s1 > all) s1 = all;

    f32x4_u gr[2][8], xr[8];
    auto load_g = [&](int64_t s, f32x4_u (&dst)[8], bool tail) {  // s uniform, tail a constant
        const uint8_t* gb = (const uint8_t*)(p.G + s * 32 * p.N);
#pragma unroll
        for (int e = 0; e < 8; e++) {
            if (!tail) {
                dst[e] = *(const f32x4_u*)(gb + (int64_t)e * p.N * 4 + g_off);
            } else {  // rows past the end: row 0 of the step again, as zeros
                const bool in = s * 32 + 8 * g + e < p.M;
                const f32x4_u a = *(const f32x4_u*)(gb + ((in ? 8u * g + e : 0u) * (uint32_t)p.N + (uint32_t)col_g(i)) * 4u);
#pragma unroll
                for (int c = 0; c < 4; c++) dst[e][c] = in ? a[c] : 0.0f;
            }
        }
    };
    auto load_x = [&](int64_t s, bool tail) {
        const uint8_t* xb = (const uint8_t*)(p.X + s * 32 * p.K);
#pragma unroll
        for (int e = 0; e < 8; e++) {
            if (!tail) {
                xr[e] = *(const f32x4_u*)(xb + (int64_t)e * p.K * 4 + x_off);
            } else {
                const bool in = s * 32 + 8 * g + e < p.M;
                const f32x4_u a = *(const f32x4_u*)(xb + ((in ? 8u * g + e : 0u) * (uint32_t)p.K + (uint32_t)col_x(i)) * 4u);
#pragma unroll
                for (int c = 0; c < 4; c++) xr[e][c] = in ? a[c] : 0.0f;
            }
        }
    };

    v4f acc[4][4];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int u = 0; u < 4; u++) acc[t][u] = v4f{0.f, 0.f, 0.f, 0.f};
    // column sums of G: every wave of a row of tiles takes the steps of its turn (all of them for tile 0 when direct)
    const int kt = (int)(k0 >> 6), nkt = (int)((p.K + 63) >> 6);
    float bsum[4] = {0.f, 0.f, 0.f, 0.f};
    int turn = DIRECT ? (kt == 0 ? 0 : -1) : (int)((kt + nkt - (int)(s0 % nkt)) % nkt);
    auto add_bias = [&](const f32x4_u (&cur)[8]) {
        if (turn == 0) {
#pragma unroll
            for (int t = 0; t < 4; t++) {
                float v = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; e++) v += cur[e][t];
                bsum[t] += v;
            }
        }
        if constexpr (!DIRECT) turn = (turn == 0) ? nkt - 1 : turn - 1;
    };

    u32x4 pg[2][3];
    auto split_g = [&](int t, const f32x4_u (&src)[8]) {
#pragma unroll
        for (int c = 0; c < 4; c++) {
            uint32_t h, m, l;
            split_pair_rn(src[2 * c][t], src[2 * c + 1][t], h, m, l);
            pg[t & 1][0][c] = h; pg[t & 1][1][c] = m; pg[t & 1][2][c] = l;
        }
    };
    auto step = [&](int64_t nx, const f32x4_u (&cur)[8], f32x4_u (&nxt)[8], bool more) {
        if (more) load_g(nx, nxt, false);
        u32x4 px[3][4];
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                uint32_t h, m, l;
                split_pair_rn(xr[2 * c][t], xr[2 * c + 1][t], h, m, l);
                px[0][t][c] = h; px[1][t][c] = m; px[2][t][c] = l;
            }
        if (more) load_x(nx, false);
        if (p.bias_out) add_bias(cur);  // uniform
        split_g(0, cur);
        __builtin_amdgcn_sched_barrier(0);
        constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};  // smallest terms first
#pragma unroll
        for (int t = 0; t < 4; t++) {
            if (t < 3) split_g(t + 1, cur);
#pragma unroll
            for (int q = 0; q < 6; q++)
#pragma unroll
                for (int u = 0; u < 4; u++) acc[t][u] = mfma_bf16(pg[t & 1][PA[q]], px[PB[q]][u], acc[t][u]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // the tile's sums over rows m .. m1 - 1 as fp32 forms the products
    auto sum_fp32 = [&](int64_t m, int64_t m1) {
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int u = 0; u < 4; u++) acc[t][u] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4  // (the loads of four rows at once; a backward of 16384 x 768 x 768 full of NaN 730 -> 590 us)
        for (; m < m1; m++) {
            const f32x4_u xv = *(const f32x4_u*)(p.X + m * p.K + col_x(i));
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const f32x4_u gv = *(const f32x4_u*)(p.G + m * p.N + col_g(4 * g + r));
#pragma unroll
                for (int t = 0; t < 4; t++)
#pragma unroll
                    for (int u = 0; u < 4; u++) acc[t][u][r] = __builtin_fmaf(gv[t], xv[u], acc[t][u][r]);
            }
        }
    };
    const int64_t sf = s1 < nfull ? s1 : nfull;  // whole steps of this part
    const bool few = p.M <= GRAD_W_FEW_ROWS;     // (a single partial step)
    if (few) {
        sum_fp32(0, p.M);
        load_g(0, gr[0], true);
        if (p.bias_out) add_bias(gr[0]);
    } else if (s0 < sf) {
        load_g(s0, gr[0], false);
        load_x(s0, false);
        int64_t s = s0;
        for (; s + 1 < sf; s += 2) {
            step(s + 1, gr[0], gr[1], true);
            step(s + 2 < sf ? s + 2 : s, gr[1], gr[0], true);  // (past the end: an earlier one again, never used)
        }
        if (s < sf) step(0, gr[0], gr[1], false);
    }
    if (!few && s1 > nfull) {  // the last part's partial step
        load_g(nfull, gr[0], true);
        load_x(nfull, true);
        step(0, gr[0], gr[1], false);
    }

    // A non-finite operand has no finite terms and left a NaN in every sum it meets, one beyond the largest bf16 value likewise,
    // and a product of rounded terms may overflow where the product does not: such a tile is summed again as fp32 forms the
    // products.
    bool bad = false;
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int r = 0; r < 4; r++) bad |= !(fabsf(acc[t][u][r]) <= FLT_MAX);
    if (bad) sum_fp32(s0 * 32, s1 * 32 < p.M ? s1 * 32 : p.M);

    float* out = p.out + (DIRECT ? 0 : (int64_t)split * p.N * p.K);
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int64_t n = col_g(4 * g + r) + t;
            const float sc = DIRECT ? p.scale[p.scale_bcast ? 0 : n] : 1.0f;
            f32x4_u v;
#pragma unroll
            for (int u = 0; u < 4; u++) v[u] = DIRECT ? __fmul_rn(acc[t][u][r], sc) : acc[t][u][r];
            *(f32x4_u*)(out + n * p.K + col_x(i)) = v;
        }
    if (p.bias_out && (!DIRECT || kt == 0)) {
        float* bo = p.bias_out + (DIRECT ? 0 : ((int64_t)split * nkt + kt) * p.N);
#pragma unroll
        for (int t = 0; t < 4; t++) {
            float v = bsum[t];
            v += __shfl_xor(v, 16, 64);
            v += __shfl_xor(v, 32, 64);
            if (g == 0) bo[col_g(i) + t] = v;
        }
    }
}

// dW = scale * sum of the partial sums, dBias = sum of its partial sums, each in a fixed order.  The first `blocks_w`
// workgroups take 1024 columns of one row of dW each, the others 16 entries of dBias (16 threads per entry: read one after
// the other, the few hundred partial sums of an entry cost 40 us of memory latency).
__global__ __launch_bounds__(256) void grad_w_reduce_kernel(const float* __restrict__ part, int splits, int64_t N, int64_t K,
                                                            const float* __restrict__ scale, int scale_bcast,
                                                            float* __restrict__ out, uint32_t blocks_w, uint32_t blocks_row,
                                                            const float* __restrict__ bias_part, int bias_parts,
                                                            float* __restrict__ bias_out) {
    const int tid = threadIdx.x;
    if (blockIdx.x < blocks_w) {
        const int64_t n = blockIdx.x / blocks_row;
        const int64_t k = 4 * ((int64_t)(blockIdx.x - n * blocks_row) * 256 + tid), at = n * K + k, total = N * K;
        const float sc = scale[scale_bcast ? 0 : n];
        if (k + 4 <= K) {
            v4f v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
            for (int s = 0; s < splits; s++) v += (v4f)*(const f32x4_u*)(part + (int64_t)s * total + at);
            f32x4_u o;
#pragma unroll
            for (int c = 0; c < 4; c++) o[c] = __fmul_rn(v[c], sc);
            *(f32x4_u*)(out + at) = o;
        } else {
            for (int64_t c = k; c < K; c++) {
                float v = 0.0f;
                for (int s = 0; s < splits; s++) v += part[(int64_t)s * total + n * K + c];
                out[n * K + c] = __fmul_rn(v, sc);
            }
        }
        return;
    }
    __shared__ float sums[256];
    const int64_t n = (int64_t)(blockIdx.x - blocks_w) * 16 + (tid & 15);
    float v = 0.0f;
    if (n < N) {
#pragma unroll 8
        for (int s = tid >> 4; s < bias_parts; s += 16) v += bias_part[(int64_t)s * N + n];
    }
    sums[tid] = v;
    __syncthreads();
    if (tid < 16 && n < N) {
        for (int s = 1; s < 16; s++) v += sums[16 * s + tid];
        bias_out[n] = v;
    }
}

// Parts of the rows: enough workgroups for two per compute unit, each part at least 8 steps of 32 rows long.
static int grad_w_splits(int64_t M, int64_t N, int64_t K) {
    const int64_t tiles = ceil_div(N, 128) * ceil_div(K, 128), steps = ceil_div(M, 32);
    return (int)std::max<int64_t>(1, std::min<int64_t>(2 * gemm_compute_units() / tiles, steps / 8));
}
static size_t align256b(size_t v) { return (v + 255) & ~(size_t)255; }

}  // namespace bt

using namespace bt;

extern "C" int bt_ternary_linear_grad_input(const float* dY, const uint8_t* W_T, const float* scale, int64_t scale_len,
                                            float* dX, int64_t M, int64_t N, int64_t K, void* stream) {
    const char* who = "bt_ternary_linear_grad_input";
    if (!dY || !W_T || !scale || !dX || M <= 0 || N <= 0 || K <= 0) {
        set_error("%s: null pointer or empty shape", who);
        return BT_ERR_INVALID;
    }
    if (scale_len != N && scale_len != 1) {
        set_error("%s: scale size doesn't match N (%lld entries, N=%lld)", who, (long long)scale_len, (long long)N);
        return BT_ERR_INVALID;
    }
    if (((uintptr_t)dY) % 4 || ((uintptr_t)dX) % 16 || N >= (1ll << 23) || K >= (1ll << 30) || ceil_div(K, 4) * N >= (1ll << 32)) {
        set_error("%s: dX must be 16-byte aligned, N below 2^23, packed weights below 4 GiB", who);
        return BT_ERR_INVALID;
    }
    GemmF32Params p = {};
    p.X = dY; p.W = W_T; p.M = M; p.C = N; p.NC = K; p.Y = dX;
    p.ldw = (int)N;
    p.kb = (int)ceil_div(K, 4);
    if (scale_len == 1 && N != 1) {
        p.y_scale = scale;
        return launch_gemm_f32_src<B_TRANSPOSED, false>(p, who, (hipStream_t)stream);
    }
    p.a_scale = scale;
    return launch_gemm_f32_src<B_TRANSPOSED, true>(p, who, (hipStream_t)stream);
}

extern "C" size_t bt_linear_grad_weight_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    const int splits = grad_w_splits(M, N, K);
    if (splits == 1) return 0;
    return align256b((size_t)splits * N * K * 4) + align256b((size_t)splits * ceil_div(K, 64) * N * 4);
}

extern "C" int bt_linear_grad_weight(const float* dY, const float* X, const float* scale, int64_t scale_len, float* dW,
                                     float* dBias, int64_t M, int64_t N, int64_t K, void* workspace, size_t workspace_bytes,
                                     void* stream) {
    const char* who = "bt_linear_grad_weight";
    if (!dY || !X || !scale || !dW || M <= 0 || N <= 0 || K <= 0) {
        set_error("%s: null pointer or empty shape", who);
        return BT_ERR_INVALID;
    }
    if (scale_len != N && scale_len != 1) {
        set_error("%s: scale size doesn't match N (%lld entries, N=%lld)", who, (long long)scale_len, (long long)N);
        return BT_ERR_INVALID;
    }
    if (N < 4 || K < 4 || N >= (1ll << 24) || K >= (1ll << 24) ||
        (((uintptr_t)dY) | ((uintptr_t)X) | ((uintptr_t)dW)) % 4) {
        set_error("%s: N and K from 4 to 2^24, 4-byte aligned buffers", who);
        return BT_ERR_INVALID;
    }
    const size_t need = bt_linear_grad_weight_workspace_bytes(M, N, K);
    if (need && (!workspace || workspace_bytes < need || ((uintptr_t)workspace) % 256)) {
        set_error("%s: workspace of %zu bytes (256-byte aligned) needed, %zu given", who, need, workspace_bytes);
        return BT_ERR_WORKSPACE;
    }
    hipStream_t st = (hipStream_t)stream;
    GradWParams p = {};
    p.G = dY; p.X = X; p.M = M; p.N = N; p.K = K;
    p.tiles_n = (int)ceil_div(N, 128); p.tiles_k = (int)ceil_div(K, 128);
    p.scale = scale; p.scale_bcast = (scale_len == 1 && N != 1) ? 1 : 0;
    const int64_t steps = ceil_div(M, 32);
    p.splits = grad_w_splits(M, N, K);
    p.steps_per_split = (int)ceil_div(steps, p.splits);
    p.splits = (int)ceil_div(steps, p.steps_per_split);  // (no empty part)
    p.per_xcd = (int)ceil_div((int64_t)p.tiles_n * p.tiles_k * p.splits, 8);
    const int64_t blocks = 8ll * p.per_xcd;
    if ((int64_t)p.tiles_n * p.tiles_k * p.splits >= (1ll << 31) - 8 || steps >= (1ll << 31)) {
        set_error("%s: more tiles than one launch takes", who);
        return BT_ERR_INVALID;
    }
    if (p.splits == 1) {
        p.out = dW;
        p.bias_out = dBias;
        hipLaunchKernelGGL(grad_w_f32_kernel<true>, dim3((unsigned)blocks), dim3(256), 0, st, p);
        return check_launch(who);
    }
    p.out = (float*)workspace;
    const int nkt = (int)ceil_div(K, 64);
    float* bias_part = (float*)((uint8_t*)workspace + align256b((size_t)grad_w_splits(M, N, K) * N * K * 4));
    p.bias_out = dBias ? bias_part : nullptr;
    hipLaunchKernelGGL(grad_w_f32_kernel<false>, dim3((unsigned)blocks), dim3(256), 0, st, p);
    int rc = check_launch(who);
    if (rc) return rc;
    const int64_t blocks_row = ceil_div(K, 1024), blocks_w = N * blocks_row, blocks_b = dBias ? ceil_div(N, 16) : 0;
    if (blocks_w + blocks_b >= (1ll << 31)) {
        set_error("%s: more tiles than one launch takes", who);
        return BT_ERR_INVALID;
    }
    hipLaunchKernelGGL(grad_w_reduce_kernel, dim3((unsigned)(blocks_w + blocks_b)), dim3(256), 0, st, (const float*)workspace,
                       p.splits, N, K, scale, p.scale_bcast, dW, (uint32_t)blocks_w, (uint32_t)blocks_row, bias_part,
                       p.splits * nkt, dBias);
    return check_launch(who);
}
