// Element arithmetic of the fused block glue (SwiGLU, RMSNorm), shared by the row kernels and by the
// streaming GEMV, which can apply either to its activation row on the way into LDS.
//   SwiGLU   h = rd( rd( g / (1 + exp(-g)) ) * u )
//   RMSNorm  y = rd( (x * r) * w ),  r = 1 / sqrt(ss / K + eps),  ss = float(sum double(x)^2)
// (rd = round to the tensor dtype; every fp32 operation rounded on its own.)
#pragma once
#include "bt_common.h"

namespace bt {

// exp(a) in fp32 by a fixed sequence of correctly rounded operations (range reduction by ln 2 in two
// parts, degree-7 polynomial, exact scaling by 2^n): a few units in the last place from exp on
// [-87, 88.7228]; +inf above (as exp overflows), exp(-87) below (callers only add it to 1).  The
// same sequence with fmaf() on a CPU gives the same bits.
__device__ __forceinline__ float exp_fixed(float a) {
    if (!(a == a)) return a;
    if (a > 88.7228f) return __builtin_inff();  // exp overflows fp32
    a = fmaxf(a, -87.0f);
    const float n = rintf(__fmul_rn(a, 1.44269504088896341f));
    float r = __builtin_fmaf(n, -0.693145751953125f, a);         // ln2 high part (exact product)
    r = __builtin_fmaf(n, -1.42860682030941723212e-6f, r);       // ln2 low part
    float p = 1.0f / 5040.0f;
    p = __builtin_fmaf(p, r, 1.0f / 720.0f);
    p = __builtin_fmaf(p, r, 1.0f / 120.0f);
    p = __builtin_fmaf(p, r, 1.0f / 24.0f);
    p = __builtin_fmaf(p, r, 1.0f / 6.0f);
    p = __builtin_fmaf(p, r, 0.5f);
    p = __builtin_fmaf(p, r, 1.0f);
    p = __builtin_fmaf(p, r, 1.0f);
    // p * 2^n, exact: the result is a normal number (n >= -126) or overflows like exp itself
    return __builtin_ldexpf(p, (int)n);
}

__device__ __forceinline__ float swiglu_value(float g, float u, int dt) {
    const float e = exp_fixed(-g);
    const float s = round_to_dtype(__fdiv_rn(g, __fadd_rn(1.0f, e)), dt);
    return round_to_dtype(__fmul_rn(s, u), dt);
}
// The same bits for eight values at once (DT is the type g and u were read from), in half the operations where DT has 16 bits:
// s is then a function of 65536 inputs, and the hardware's exp2 and reciprocal with one correction of the quotient round to
// the same s for all of them (for fp16 with the polynomial exp; tests/test_gpu_fused.py compares every input).  |g| up to
// 80 keeps every intermediate value normal; the correction loses the sign of -0.  (SwiGLU + quantization of 4096 x 6912 bf16,
// bound by its VALU work: 46.8 us with swiglu_value.)
template <int DT>
__device__ __forceinline__ void swiglu8(float (&g)[8], const float (&u)[8]) {
    if constexpr (DT != BT_F32) {
        float m = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; i++) m = fmaxf(m, fabsf(g[i]));
        if (m <= 80.0f) {  // (a NaN beside smaller values stays a NaN below)
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float e = DT == BT_BF16 ? __builtin_amdgcn_exp2f(__fmul_rn(g[i], -1.44269504088896341f)) : exp_fixed(-g[i]);
                const float d = __fadd_rn(1.0f, e), y = __builtin_amdgcn_rcpf(d), q = __fmul_rn(g[i], y);
                const float s = __builtin_fmaf(__builtin_fmaf(-d, q, g[i]), y, q);
                g[i] = round_to_dtype(__fmul_rn(round_to_dtype(copysignf(s, g[i]), DT), u[i]), DT);
            }
            return;
        }
    }
#pragma unroll
    for (int i = 0; i < 8; i++) g[i] = swiglu_value(g[i], u[i], DT);
}
// The SwiGLU output stage of the tiled GEMMs, for 16 rows of a tile: y[t][r] are a lane's projections of row 4 g + r, rounded to DT,
// t = 0, 1 those of the gate's columns c, c + 1 and t = 2, 3 the same columns of up.  It stores what the SwiGLU row kernel makes of
// stored projections, by the same element arithmetic.  Lanes 2 i and 2 i + 1 hold neighbouring columns: the even one stores two
// of the rows, the odd one the other two, in 8 bytes each.  left: rows that exist; lane_off: of row 4 g, column c.
template <int DT>
__device__ __forceinline__ void swiglu_store16(char* row, int64_t row_bytes, uint32_t lane_off, int left, int g, const float (&y)[4][4]) {
    float gate[8], up[8];
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
        for (int t = 0; t < 2; t++) {
            gate[2 * r + t] = y[t][r];
            up[2 * r + t] = y[2 + t][r];
        }
    swiglu8<DT>(gate, up);
    uint32_t d[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const uint16_t h0 = DT == BT_F16 ? f32_to_f16_bits(gate[2 * r]) : f32_to_bf16_bits(gate[2 * r]);
        const uint16_t h1 = DT == BT_F16 ? f32_to_f16_bits(gate[2 * r + 1]) : f32_to_bf16_bits(gate[2 * r + 1]);
        d[r] = (uint32_t)h0 | ((uint32_t)h1 << 16);
    }
    const bool odd = threadIdx.x & 1;
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const uint32_t keep = odd ? d[2 + r] : d[r], give = odd ? d[r] : d[2 + r];
        const uint32_t got = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)give, 0xB1, 0xf, 0xf, true);
        char* at = row + r * row_bytes + lane_off + (odd ? 2 * (uint32_t)row_bytes - 4u : 0u);
        if (4 * g + r + (odd ? 2 : 0) < left) st2_nt(at, odd ? got : keep, odd ? keep : got);
    }
}
__device__ __forceinline__ float rmsnorm_value(float x, float r, float w, int dt) {
    return round_to_dtype(__fmul_rn(__fmul_rn(x, r), w), dt);
}
__device__ __forceinline__ float rms_rstd(double ss, int K, float eps) {
    const float ms = __fdiv_rn((float)ss, (float)K);
    // sqrtf is the correctly rounded square root (__fsqrt_rn is the approximate instruction)
    return __fdiv_rn(1.0f, sqrtf(__fadd_rn(ms, eps)));
}
__device__ __forceinline__ int8_t quant_i8(float v, float inv) {
    // round_half_away, then the clamp: the conversion truncates, and truncating and clamping to integers commute
    const float x = __fmul_rn(v, inv), r = __fadd_rn(x, copysignf(0.49999997f, x));
    return (int8_t)(int)fmaxf(-127.0f, fminf(127.0f, r));
}

__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

}  // namespace bt
