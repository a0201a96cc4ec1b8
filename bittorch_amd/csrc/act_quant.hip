// Per-row int8 activation quantization for gfx950 (HBM-bound).
//
// Arithmetic restated from the reference (csrc/kernels/ternary_gemm_tensor_core.cu:343-347,
// :439, :456-457) with the row scale taken over the whole row:
//   amax = max_k |x[b,k]|;  s_x[b] = amax > 1e-6 ? amax / 127 : 1
//   q[b,k] = (int8) clamp(roundf(x[b,k] * (1 / s_x[b])), -127, 127)
// Optionally the rows' sums of q (int32), which the field-layout prefill GEMM starts its accumulators from.
#include <cstdlib>

#include "bt_common.h"

namespace bt {

// Per-row int8 activation quantizer: one wave per row, two passes over the row
// (the second pass hits in cache; a row is at most a few tens of KiB).
template <int DT>
__global__ __launch_bounds__(256) void act_quant_kernel(const void* __restrict__ X, int64_t B, int64_t K,
                                                        int8_t* __restrict__ Q, float* __restrict__ s_x,
                                                        int q_layout, int32_t* __restrict__ rowsum) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= B) return;
    const int64_t base = row * K;
    constexpr int ES = (DT == BT_F32) ? 4 : 2;
    const bool vec_ok = (K % 8 == 0) && (((uintptr_t)X) % 16 == 0) && (((uintptr_t)Q) % 8 == 0);

    auto load8 = [&](int64_t k, float (&v)[8]) {
        if (vec_ok) {
            if constexpr (DT == BT_F32) {
                const float4 a = *(const float4*)((const float*)X + base + k);
                const float4 b = *(const float4*)((const float*)X + base + k + 4);
                v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
                v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
            } else {
                const uint4 u = *(const uint4*)((const uint16_t*)X + base + k);
                const uint32_t d[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const uint16_t h = (uint16_t)(d[e >> 1] >> (16 * (e & 1)));
                    v[e] = (DT == BT_F16) ? f16_bits_to_f32(h) : bf16_bits_to_f32(h);
                }
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = (k + e < K) ? load_elem<DT>(X, base + k + e) : 0.0f;
        }
    };
    (void)ES;

    float amax = 0.0f;
    for (int64_t k = (int64_t)lane * 8; k < K; k += 512) {
        float v[8];
        load8(k, v);
#pragma unroll
        for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(v[e]));
    }
    amax = wave_max(amax);
    const float s = (amax > 1e-6f) ? __fdiv_rn(amax, 127.0f) : 1.0f;
    const float inv = __fdiv_rn(1.0f, s);
    if (lane == 0) s_x[row] = s;

    int qsum = 0;
    for (int64_t k = (int64_t)lane * 8; k < K; k += 512) {
        float v[8];
        load8(k, v);
        uint32_t lo = 0, hi = 0;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            float r = round_half_away(__fmul_rn(v[e], inv));
            r = fmaxf(-127.0f, fminf(127.0f, r));
            qsum += (int)r;  // (elements past K were loaded as zero)
            const uint32_t byte = (uint32_t)(uint8_t)(int8_t)(int)r;
            if (e < 4) lo |= byte << (8 * e);
            else hi |= byte << (8 * (e - 4));
        }
        if (vec_ok) {  // (operand order is only requested with K % 16 == 0 and aligned rows: this path)
            *(uint2*)(Q + base + k) = q_layout == Q_OPERAND_ORDER ? q_to_operand_order(lo, hi, lane & 1) : make_uint2(lo, hi);
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (k + e < K) Q[base + k + e] = (int8_t)(((e < 4 ? lo : hi) >> (8 * (e & 3))) & 0xff);
        }
    }
    if (rowsum) {  // (uniform)
        qsum = wave_sum_i32(qsum);
        if (lane == 0) rowsum[row] = qsum;
    }
}

// Eight values of the row at `base` from k on, by clamped, unconditional loads: a group past the end repeats the row's last
// one and is masked by the caller.  RAG: rows of any length that start on any element (4- or 2-byte aligned vector loads); the
// group that crosses the row's end is shifted into place and filled with zeros, and groups past it are zero.
// (Branches between the groups cost three times the kernel's time: 3847 x 8238 bf16 23 us as it is, 74 with them.)
typedef uint32_t u32x4_a16 __attribute__((ext_vector_type(4), aligned(16)));
template <int DT>
struct Group8 { uint32_t d[DT == BT_F32 ? 8 : 4]; };
template <int DT, bool RAG>
__device__ __forceinline__ void load_group8(const void* X, int64_t base, int k, int K, Group8<DT>& u) {
    typedef typename std::conditional<!RAG, u32x4_a16, typename std::conditional<DT == BT_F32, u32x4_a4, u32x4_a2>::type>::type vec;
    const uint8_t* src = (const uint8_t*)X + (base + min(k, K - 8)) * (DT == BT_F32 ? 4 : 2);
#pragma unroll
    for (int h = 0; h < (DT == BT_F32 ? 2 : 1); h++) {
        const vec v = *(const vec*)(src + 16 * h);
#pragma unroll
        for (int e = 0; e < 4; e++) u.d[4 * h + e] = v[e];
    }
}
template <int DT, bool RAG>
__device__ __forceinline__ void group8_values(Group8<DT> u, int k, int K, float (&v)[8]) {
    if constexpr (RAG) {
        const int sh = max(k + 8 - K, 0);  // values of the group past the row's end
        if constexpr (DT == BT_F32) {
            // (Chosen by value: `c ? d[i] : d[j]` chooses between two addresses, and the array then lives in LDS, 8 KiB of it
            // per workgroup: 256 rows of 1031 17.5 us that way, 3.2 this.)
            auto pick = [](bool c, uint32_t a, uint32_t b) { return c ? a : b; };
            const bool one = sh & 1, two = sh & 2, four = sh & 4;
#pragma unroll
            for (int e = 0; e < 7; e++) u.d[e] = pick(one, u.d[e + 1], u.d[e]);
#pragma unroll
            for (int e = 0; e < 6; e++) u.d[e] = pick(two, u.d[e + 2], u.d[e]);
#pragma unroll
            for (int e = 0; e < 4; e++) u.d[e] = pick(four, u.d[e + 4], u.d[e]);
#pragma unroll
            for (int e = 0; e < 8; e++) u.d[e] = pick(e + sh < 8, u.d[e], 0u);
        } else {
            const uint4 s4 = shift_group(make_uint4(u.d[0], u.d[1], u.d[2], u.d[3]), 2 * sh);
            u.d[0] = s4.x; u.d[1] = s4.y; u.d[2] = s4.z; u.d[3] = s4.w;
        }
    }
#pragma unroll
    for (int e = 0; e < 8; e++) {
        if constexpr (DT == BT_F32) {
            v[e] = __builtin_bit_cast(float, u.d[e]);
        } else {
            const uint16_t h = (uint16_t)(u.d[e >> 1] >> (16 * (e & 1)));
            v[e] = (DT == BT_F16) ? f16_bits_to_f32(h) : bf16_bits_to_f32(h);
        }
    }
}

// One workgroup per row, the row held in registers between the absmax pass and the
// quantization: X is read once and the row's latency chain is load -> reduce -> store.
// Needs K % 8 == 0, K <= 2048*ITERS and aligned pointers (16 bytes X, 8 bytes Q).  RAG: any K from 8 on and any X; Q's rows
// have Kq >= K bytes (a multiple of 16, at most 2048*ITERS), those past K zero: what the tiled GEMM reads of such rows.
template <int DT, int ITERS, bool RAG>
__global__ __launch_bounds__(256) void act_quant_row_kernel(const void* __restrict__ X, int K, int Kq,
                                                            int8_t* __restrict__ Q, float* __restrict__ s_x,
                                                            int q_layout, int32_t* __restrict__ rowsum) {
    __shared__ float part[4];
    __shared__ int part_sum[4];
    const int tid = threadIdx.x;
    const int64_t base = (int64_t)blockIdx.x * K, qbase = (int64_t)blockIdx.x * Kq;
    Group8<DT> u[ITERS];
    float v[ITERS][8];
#pragma unroll
    for (int i = 0; i < ITERS; i++) load_group8<DT, RAG>(X, base, (i * 256 + tid) * 8, K, u[i]);
#pragma unroll
    for (int i = 0; i < ITERS; i++) group8_values<DT, RAG>(u[i], (i * 256 + tid) * 8, K, v[i]);
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < ITERS; i++) {
        const bool ok = (i * 256 + tid) * 8 < K;
#pragma unroll
        for (int e = 0; e < 8; e++) amax = fmaxf(amax, ok ? fabsf(v[i][e]) : 0.0f);
    }
    amax = wave_max(amax);
    if ((tid & 63) == 0) part[tid >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
    const float s = (amax > 1e-6f) ? __fdiv_rn(amax, 127.0f) : 1.0f;
    const float inv = __fdiv_rn(1.0f, s);
    if (tid == 0) s_x[blockIdx.x] = s;
    int qsum = 0;
#pragma unroll
    for (int i = 0; i < ITERS; i++) {
        const int k = (i * 256 + tid) * 8;
        uint32_t lo = 0, hi = 0;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            float r = round_half_away(__fmul_rn(v[i][e], inv));
            r = fmaxf(-127.0f, fminf(127.0f, r));
            if (k < K) qsum += (int)r;  // (a clamped group past the end repeats the row's last one)
            const uint32_t byte = (uint32_t)(uint8_t)(int8_t)(int)r;
            if (e < 4) lo |= byte << (8 * e);
            else hi |= byte << (8 * (e - 4));
        }
        const uint2 o = q_layout == Q_OPERAND_ORDER ? q_to_operand_order(lo, hi, tid & 1) : make_uint2(lo, hi);
        if (k < Kq) st2_nt(Q + qbase + k, o.x, o.y);  // Kq % 16 == 0 in operand order: both lanes of a pair store
    }
    if (rowsum) {  // (uniform)
        qsum = wave_sum_i32(qsum);
        if ((tid & 63) == 0) part_sum[tid >> 6] = qsum;
        __syncthreads();
        if (tid == 0) rowsum[blockIdx.x] = part_sum[0] + part_sum[1] + part_sum[2] + part_sum[3];
    }
}

// Many short rows: one wave per row (four rows per workgroup), lane l holding the 8-element chunks i * 64 + l -- all
// 64 lanes busy where the workgroup kernel above leaves lanes idle, the absmax a shuffle tree, no LDS and no barrier.
// The same bits.
template <int DT, int ITERS, bool RAG>
__global__ __launch_bounds__(256) void act_quant_wave_kernel(const void* __restrict__ X, int64_t B, int K, int Kq,
                                                             int8_t* __restrict__ Q, float* __restrict__ s_x,
                                                             int q_layout, int32_t* __restrict__ rowsum) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= B) return;  // (whole waves; the kernel has no barrier)
    const int64_t base = row * K, qbase = row * Kq;
    Group8<DT> u[ITERS];
    float v[ITERS][8];
#pragma unroll
    for (int i = 0; i < ITERS; i++) load_group8<DT, RAG>(X, base, (i * 64 + lane) * 8, K, u[i]);
#pragma unroll
    for (int i = 0; i < ITERS; i++) group8_values<DT, RAG>(u[i], (i * 64 + lane) * 8, K, v[i]);
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < ITERS; i++) {
        const bool ok = (i * 64 + lane) * 8 < K;
#pragma unroll
        for (int e = 0; e < 8; e++) amax = fmaxf(amax, ok ? fabsf(v[i][e]) : 0.0f);
    }
    amax = wave_max(amax);
    const float s = (amax > 1e-6f) ? __fdiv_rn(amax, 127.0f) : 1.0f;
    const float inv = __fdiv_rn(1.0f, s);
    if (lane == 0) s_x[row] = s;
    int qsum = 0;
#pragma unroll
    for (int i = 0; i < ITERS; i++) {
        const int k = (i * 64 + lane) * 8;
        uint32_t lo = 0, hi = 0;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            float r = round_half_away(__fmul_rn(v[i][e], inv));
            r = fmaxf(-127.0f, fminf(127.0f, r));
            if (k < K) qsum += (int)r;
            const uint32_t byte = (uint32_t)(uint8_t)(int8_t)(int)r;
            if (e < 4) lo |= byte << (8 * e);
            else hi |= byte << (8 * (e - 4));
        }
        const uint2 o = q_layout == Q_OPERAND_ORDER ? q_to_operand_order(lo, hi, lane & 1) : make_uint2(lo, hi);
        if (k < Kq) st2_nt(Q + qbase + k, o.x, o.y);
    }
    if (rowsum) {  // (uniform)
        qsum = wave_sum_i32(qsum);
        if (lane == 0) rowsum[row] = qsum;
    }
}

template <int DT, bool RAG>
static bool launch_act_quant_rows(const void* X, int64_t B, int64_t K, int64_t Kq, int8_t* Q, float* s_x, int ql, int32_t* rs,
                                  hipStream_t st) {
    if (Kq > 16384 || ((uintptr_t)Q) % 8 != 0 || B > 0x7fffffff || tuning_env("BITTORCH_ACTQ_GENERIC")) return false;
    if (!RAG && (K % 8 != 0 || ((uintptr_t)X) % 16 != 0)) return false;
    const dim3 grid((unsigned)B), block(256);
    const int k = (int)K, kq = (int)Kq;
    if (B >= 2048 && K <= 3072) {  // many short rows: a wave per row (4096 x 2560 bf16 9.4 -> 7.6 us, 4096 x 1024 6.9 -> 4.5,
                                   // 4096 x 2048 7.3 -> 6.6; from K = 3584 on the workgroup kernel is as fast or faster)
        const dim3 wgrid((unsigned)((B + 3) / 4));
        switch ((kq + 511) / 512) {
            case 1: hipLaunchKernelGGL((act_quant_wave_kernel<DT, 1, RAG>), wgrid, block, 0, st, X, B, k, kq, Q, s_x, ql, rs); break;
            case 2: hipLaunchKernelGGL((act_quant_wave_kernel<DT, 2, RAG>), wgrid, block, 0, st, X, B, k, kq, Q, s_x, ql, rs); break;
            case 3: hipLaunchKernelGGL((act_quant_wave_kernel<DT, 3, RAG>), wgrid, block, 0, st, X, B, k, kq, Q, s_x, ql, rs); break;
            case 4: hipLaunchKernelGGL((act_quant_wave_kernel<DT, 4, RAG>), wgrid, block, 0, st, X, B, k, kq, Q, s_x, ql, rs); break;
            case 5: hipLaunchKernelGGL((act_quant_wave_kernel<DT, 5, RAG>), wgrid, block, 0, st, X, B, k, kq, Q, s_x, ql, rs); break;
            default: hipLaunchKernelGGL((act_quant_wave_kernel<DT, 6, RAG>), wgrid, block, 0, st, X, B, k, kq, Q, s_x, ql, rs); break;
        }
        return true;
    }
    if (Kq <= 2048) hipLaunchKernelGGL((act_quant_row_kernel<DT, 1, RAG>), grid, block, 0, st, X, k, kq, Q, s_x, ql, rs);
    else if (Kq <= 4096) hipLaunchKernelGGL((act_quant_row_kernel<DT, 2, RAG>), grid, block, 0, st, X, k, kq, Q, s_x, ql, rs);
    else if (Kq <= 8192) hipLaunchKernelGGL((act_quant_row_kernel<DT, 4, RAG>), grid, block, 0, st, X, k, kq, Q, s_x, ql, rs);
    else if (Kq <= 12288) hipLaunchKernelGGL((act_quant_row_kernel<DT, 6, RAG>), grid, block, 0, st, X, k, kq, Q, s_x, ql, rs);
    else hipLaunchKernelGGL((act_quant_row_kernel<DT, 8, RAG>), grid, block, 0, st, X, k, kq, Q, s_x, ql, rs);
    return true;
}

// q_layout = Q_OPERAND_ORDER needs K % 16 == 0, X 16-byte and Q 8-byte aligned (the callers check)
int launch_act_quant(const void* X, int x_dtype, int64_t B, int64_t K, int8_t* Q, float* s_x, int q_layout,
                     int32_t* rowsum, hipStream_t st) {
    const int ql = q_layout;
    // the operand order is written 16 bytes at a time: callers check this too, but a buffer that cannot take it
    // must never be written row-major under that name
    if (ql == Q_OPERAND_ORDER && (K % 16 != 0 || ((uintptr_t)X) % 16 != 0 || ((uintptr_t)Q) % 16 != 0)) {
        set_error("bt_act_quant_i8: the operand-order layout needs K %% 16 == 0 and 16-byte aligned X and Q");
        return BT_ERR_INVALID;
    }
    int32_t* rs = rowsum;
    const bool done = (x_dtype == BT_F32)   ? launch_act_quant_rows<BT_F32, false>(X, B, K, K, Q, s_x, ql, rs, st)
                      : (x_dtype == BT_F16) ? launch_act_quant_rows<BT_F16, false>(X, B, K, K, Q, s_x, ql, rs, st)
                                            : launch_act_quant_rows<BT_BF16, false>(X, B, K, K, Q, s_x, ql, rs, st);
    if (done) return check_launch("bt_act_quant_i8");
    const dim3 grid((unsigned)ceil_div(B, 4)), block(256);
    if (x_dtype == BT_F32) hipLaunchKernelGGL(act_quant_kernel<BT_F32>, grid, block, 0, st, X, B, K, Q, s_x, ql, rs);
    else if (x_dtype == BT_F16) hipLaunchKernelGGL(act_quant_kernel<BT_F16>, grid, block, 0, st, X, B, K, Q, s_x, ql, rs);
    else hipLaunchKernelGGL(act_quant_kernel<BT_BF16>, grid, block, 0, st, X, B, K, Q, s_x, ql, rs);
    return check_launch("bt_act_quant_i8");
}

// Rows of any length and start into operand order with rows of Kq = K rounded up to 16 (zeros behind K): the same bytes and
// scales as launch_act_quant's for the K values.
bool act_quant_padded_ok(const void* X, int x_dtype, int64_t B, int64_t K) {
    return K >= 8 && K <= 16384 && B <= 0x7fffffff && ((uintptr_t)X) % (uintptr_t)dtype_size(x_dtype) == 0;
}
int launch_act_quant_padded(const void* X, int x_dtype, int64_t B, int64_t K, int64_t Kq, int8_t* Q, float* s_x, hipStream_t st) {
    const int ql = Q_OPERAND_ORDER;
    const bool done = (x_dtype == BT_F32)   ? launch_act_quant_rows<BT_F32, true>(X, B, K, Kq, Q, s_x, ql, nullptr, st)
                      : (x_dtype == BT_F16) ? launch_act_quant_rows<BT_F16, true>(X, B, K, Kq, Q, s_x, ql, nullptr, st)
                                            : launch_act_quant_rows<BT_BF16, true>(X, B, K, Kq, Q, s_x, ql, nullptr, st);
    if (!done) {
        set_error("bt_act_quant_i8: rows of %lld values cannot be padded", (long long)K);
        return BT_ERR_INVALID;
    }
    return check_launch("bt_act_quant_i8");
}

// 16-bit rows of any length as rows of Kp = K rounded up to 8, zeros behind K: what the tiled 16-bit GEMM's 16-byte loads
// need.  Bound by its bytes; a thread copies one group of eight, the one that crosses the row's end element by element.
__global__ __launch_bounds__(256) void pad_rows_kernel(const uint16_t* __restrict__ X, int64_t groups, uint32_t row_groups, int K,
                                                       uint4* __restrict__ P) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < groups; i += (int64_t)gridDim.x * 256) {
        const int64_t row = i / row_groups;
        const int k = 8 * (int)(i - row * row_groups);
        const uint16_t* src = X + row * K + k;
        uint32_t d[4] = {0u, 0u, 0u, 0u};
        if (k + 8 <= K) {
            const u32x4_a2 v = *(const u32x4_a2*)src;
#pragma unroll
            for (int e = 0; e < 4; e++) d[e] = v[e];
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (k + e < K) d[e >> 1] |= (uint32_t)src[e] << (16 * (e & 1));
        }
        P[i] = make_uint4(d[0], d[1], d[2], d[3]);
    }
}
int launch_pad_rows(const void* X, int64_t B, int64_t K, void* P, hipStream_t st) {
    const int64_t row_groups = ceil_div(K, 8), groups = B * row_groups;
    const unsigned blocks = (unsigned)std::min<int64_t>(ceil_div(groups, 256), 1 << 20);
    hipLaunchKernelGGL(pad_rows_kernel, dim3(blocks), dim3(256), 0, st, (const uint16_t*)X, groups, (uint32_t)row_groups, (int)K, (uint4*)P);
    return check_launch("bt_ternary_linear_packed_forward(pad)");
}

// fp32 activations as three bf16 planes: x = hi + mid + lo exactly, each term the truncation to
// bf16 (upper 16 bits) of what the terms before it leave (24 significand bits = 3 x 8).  Ternary
// weights are exact in bf16, so the three products per weight are exact and the 16-bit matrix
// cores accumulate them in fp32: fp32 inputs run on the bf16 kernels without losing a bit of
// the activations.  X [B,K] fp32 -> P [B,3*Kp] bf16 bits, row b = [hi(Kp) | mid(Kp) | lo(Kp)] / 2,
// Kp = K rounded up to the kernels' 64-wide step, the padding zero (it meets padding codes or clamped
// weight rows: 0 * w = 0 exactly).
__device__ __forceinline__ void split3(float x, uint16_t& hi, uint16_t& mid, uint16_t& lo) {
    const uint32_t u0 = __builtin_bit_cast(uint32_t, x) & 0xFFFF0000u;
    const float r1 = x - __builtin_bit_cast(float, u0);
    const uint32_t u1 = __builtin_bit_cast(uint32_t, r1) & 0xFFFF0000u;
    const float r2 = r1 - __builtin_bit_cast(float, u1);
    // stored halved (exact): the bf16 kernels decode the weights as +-2.0, and x * 2 would
    // overflow for |x| above half the fp32 range
    hi = (uint16_t)(__builtin_bit_cast(uint32_t, __builtin_bit_cast(float, u0) * 0.5f) >> 16);
    mid = (uint16_t)(__builtin_bit_cast(uint32_t, __builtin_bit_cast(float, u1) * 0.5f) >> 16);
    lo = (uint16_t)(__builtin_bit_cast(uint32_t, r2 * 0.5f) >> 16);
}
// VEC: K % 4 == 0 and X 16-byte aligned (one float4 per thread and trip); otherwise element by element
template <bool VEC>
__global__ __launch_bounds__(256) void split_f32_planes_kernel(const float* __restrict__ X, int64_t B, int64_t K, int64_t Kp,
                                                               uint16_t* __restrict__ P) {
    const int64_t kq = Kp >> 2;  // groups of four per padded row
    const int64_t total = B * kq;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int64_t b = i / kq, c = i - b * kq;
        float x[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (VEC) {
            if (4 * c < K) {
                const float4 v = *(const float4*)(X + b * K + 4 * c);
                x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (4 * c + e < K) x[e] = X[b * K + 4 * c + e];
        }
        uint16_t hi[4], mid[4], lo[4];
#pragma unroll
        for (int e = 0; e < 4; e++) split3(x[e], hi[e], mid[e], lo[e]);
        uint16_t* row = P + b * 3 * Kp + 4 * c;
        *(uint2*)(row) = make_uint2((uint32_t)hi[0] | ((uint32_t)hi[1] << 16), (uint32_t)hi[2] | ((uint32_t)hi[3] << 16));
        *(uint2*)(row + Kp) = make_uint2((uint32_t)mid[0] | ((uint32_t)mid[1] << 16), (uint32_t)mid[2] | ((uint32_t)mid[3] << 16));
        *(uint2*)(row + 2 * Kp) = make_uint2((uint32_t)lo[0] | ((uint32_t)lo[1] << 16), (uint32_t)lo[2] | ((uint32_t)lo[3] << 16));
    }
}

// Kp: plane length, a multiple of 64 and >= K; P is 8-byte aligned
int launch_split_f32_planes(const void* X, int64_t B, int64_t K, int64_t Kp, void* P, hipStream_t st) {
    const int64_t total = B * (Kp >> 2);
    const unsigned blocks = (unsigned)std::min<int64_t>(std::max<int64_t>(ceil_div(total, 256), 1), 8192);
    if (K % 4 == 0 && ((uintptr_t)X) % 16 == 0)
        hipLaunchKernelGGL(split_f32_planes_kernel<true>, dim3(blocks), dim3(256), 0, st, (const float*)X, B, K, Kp, (uint16_t*)P);
    else
        hipLaunchKernelGGL(split_f32_planes_kernel<false>, dim3(blocks), dim3(256), 0, st, (const float*)X, B, K, Kp, (uint16_t*)P);
    return check_launch("bt_ternary_linear_packed_forward(split)");
}

}  // namespace bt
