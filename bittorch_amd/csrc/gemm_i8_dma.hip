// Tiled int8 x packed-ternary GEMM on activations in operand order: two independent workgroups per compute unit.
// Arithmetic as in gemm_i8.hip (csrc/kernels/ternary_gemm_tensor_core.cu:73-75, :343-347, :583-589, :652).
//
// A 256-thread workgroup (4 waves) owns a tile of 32 NB x 256 outputs; wave w works on columns 64 w .. +63 over the whole of
// K, so nothing has to be added up at the end, and two workgroups share a compute unit: while one waits, starts, drains or
// stores, the other one's MFMAs run.  Launches of at most one tile a compute unit have two such groups of waves in a workgroup
// instead, half of the stages each, which add their sums through LDS at the end (i8_splits_k).  Bound by the issue of a stage: 32 MFMAs (512 cycles) and some 60 other instructions;
// 2.2 to 2.9 POPS at K = 2560 .. 8192 (4096 x 8192 x 8192 192 us, 207 with the K halves of gemm_i8_kernel).
//   * Everything that comes from memory goes to LDS without passing through registers (global_load_lds, 16 bytes a lane):
//     the activations in the operand order the quantizer wrote them in, and each wave's packed weights (1 KiB a stage).  A
//     stage is 64 k; n = d_stages of them are in LDS, five as a rule, so a load has n - 2 stages (1500 to 4000 cycles) to arrive.
//   * A stage: 16 MFMAs of row blocks 0..3 with the decode of the next stage's weights behind them, the one barrier, 16
//     MFMAs of row blocks 4..7 under which the fragments of the next stage's row blocks 0..3 arrive.
// The loads are counted by hand (the compiler does not see them): `vmcnt` in front of the barrier of stage s leaves the
// loads of stages s + 3 .. s + n - 1 in flight, so stage s + 1 (fragments) and s + 2 (the weights decoded one stage ahead) are
// complete; that barrier also stands between the last read of stage s's buffer and the loads of stage s + n into it.
#include "gemm_i8_common.h"
#include "lds_dma.h"
#include "row_math.h"

namespace bt {

constexpr int D_BK = 64;   // k per stage
// stages in LDS: 30 to 60 KiB, two groups of waves 60 (NB = 1) and 64 KiB (what M0's 16-bit byte offset reaches)
constexpr int d_stages(int NB, int KG) { return KG == 2 && NB == 2 ? 4 : 5; }

// Output stage: row block by row block, addresses as a uniform row base plus a lane offset fixed for the whole tile.  The
// empty asm statements keep a row's address from being computed ahead of its turn (left alone, the compiler holds all 32
// row addresses and residual values at once and spills).
// RN: rows of any length, so that a lane's four columns start on any element and the last ones may be fewer.
template <bool FL, bool RN, int MB>
__device__ __forceinline__ void dma_store_acc(const GemmParams& p, const v4i (&acc)[MB][4], int64_t m0, int g, int64_t ncol,
                                              int rows_left) {
    const uint32_t lane_off = (uint32_t)(4 * g) * (uint32_t)p.N * 4u + (uint32_t)(ncol & (G_BN - 1)) * 4u;
    char* row = (char*)p.acc_out + (m0 * p.N + (int64_t)__builtin_amdgcn_readfirstlane((int)(ncol / G_BN)) * G_BN) * 4;
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
        if (16 * mb >= rows_left) return;  // (uniform)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            asm volatile("" : "+s"(row));
            if (16 * mb + 4 * g + r < rows_left) {
                uint32_t a[4];
#pragma unroll
                for (int t = 0; t < 4; t++) a[t] = (uint32_t)times127(acc[mb][t][r] >> field_shift<FL>(t));
                if constexpr (RN) {
                    for (int t = 0; t < 4; t++)
                        if (ncol + t < p.N) ((uint32_t*)(row + lane_off))[t] = a[t];
                } else {
                    st4_nt(row + lane_off, a[0], a[1], a[2], a[3]);
                }
            }
            row += p.N * 4;
        }
        row += 12 * p.N * 4;
        __builtin_amdgcn_sched_barrier(0);
    }
}
template <int YDT, bool RES, bool FL, bool RN, int MB>
__device__ __forceinline__ void dma_epilogue(const GemmParams& p, const v4i (&acc)[MB][4], int64_t m0, int g, int64_t ncol,
                                             int rows_left, const float* sx_lds, const float (&ws)[4], const float (&bs)[4]) {
    constexpr int ES = (YDT == BT_F32) ? 4 : 2;
    const uint32_t lane_off = ((uint32_t)(4 * g) * (uint32_t)p.N + (uint32_t)(ncol & (G_BN - 1))) * ES;
    const int64_t first = (m0 * p.N + (int64_t)__builtin_amdgcn_readfirstlane((int)(ncol / G_BN)) * G_BN) * ES;
    const int64_t row_bytes = p.N * ES;
    char* row = (char*)p.Y + first;
    const char* res = (const char*)p.epi.residual + first;
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
        if (16 * mb >= rows_left) return;  // (uniform)
        const float4 s4 = *(const float4*)(sx_lds + 16 * mb + 4 * g);
        const float sx[4] = {s4.x, s4.y, s4.z, s4.w};
        uint4 rv[4];
        if constexpr (RES) {  // the block's four rows at once
#pragma unroll
            for (int r = 0; r < 4; r++) {
                asm volatile("" : "+s"(res));
                const char* src = res + (16 * mb + 4 * g + r < rows_left ? lane_off : 0u);
                if constexpr (RN) {
                    uint32_t d[4];
#pragma unroll
                    for (int t = 0; t < 4; t++) d[t] = load_bits_rt(src, YDT, ncol + t < p.N ? t : 0);
                    rv[r] = YDT == BT_F32 ? make_uint4(d[0], d[1], d[2], d[3]) : make_uint4(d[0] | d[1] << 16, d[2] | d[3] << 16, 0u, 0u);
                } else if constexpr (YDT == BT_F32) rv[r] = *(const uint4*)src;
                else { const uint2 v = *(const uint2*)src; rv[r] = make_uint4(v.x, v.y, 0u, 0u); }
                res += (16 * mb + r + 1 < rows_left) ? row_bytes : 0;
            }
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            asm volatile("" : "+s"(row));
            if (16 * mb + 4 * g + r < rows_left) {
                float y[4];
#pragma unroll
                for (int t = 0; t < 4; t++) y[t] = epi_int8_f(__fmul_rn((float)acc[mb][t][r], k127<FL>(t)), sx[r], ws[t], bs[t]);
                if constexpr (RES) {
                    const uint32_t d[4] = {rv[r].x, rv[r].y, rv[r].z, rv[r].w};
#pragma unroll
                    for (int t = 0; t < 4; t++) {
                        const uint32_t bits = YDT == BT_F32 ? d[t] : (d[t >> 1] >> (16 * (t & 1))) & 0xffffu;
                        y[t] = sum_in_dtype(round_to_dtype(y[t], YDT), bits_to_f32_rt(bits, YDT), YDT);
                    }
                }
                if constexpr (RN) store4_any<YDT>(row + lane_off, y, (int)(p.N - ncol));
                else store4(row + lane_off, YDT, 0, y);
            }
            row += row_bytes;
        }
        row += 12 * row_bytes;
        if constexpr (RES) res = row - (char*)p.Y + (const char*)p.epi.residual;
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The SwiGLU output stage (SW): a lane holds two columns of the gate and the same two of up, and stores what the SwiGLU row kernel would
// make of the stored projections, bit for bit.  Bound by that arithmetic, like the 16-bit GEMM's; half of the stores and the row
// kernel's second operand are saved: 4096 x 13824 x 2560 with the quantizer 152.5 -> 144.2 us, 2048 x 5632 x 1024 27.9 -> 23.6.
template <int YDT, int MB>
__device__ __forceinline__ void dma_epilogue_swiglu(const GemmParams& p, const v4i (&acc)[MB][4], int64_t m0, int g, int64_t col,
                                                    int rows_left, const float* sx_lds, const float (&ws)[4], const float (&bs)[4]) {
    const int64_t row_bytes = p.N;  // (N / 2 outputs of two bytes)
    char* row = (char*)p.Y + m0 * row_bytes;
    const uint32_t lane_off = (uint32_t)(4 * g) * (uint32_t)row_bytes + (uint32_t)col * 2u;
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
        if (16 * mb >= rows_left) return;  // (uniform)
        const float4 s4 = *(const float4*)(sx_lds + 16 * mb + 4 * g);
        const float sx[4] = {s4.x, s4.y, s4.z, s4.w};
        float y[4][4];
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                y[t][r] = round_to_dtype(epi_int8_f(__fmul_rn((float)acc[mb][t][r], 127.0f), sx[r], ws[t], bs[t]), YDT);
        swiglu_store16<YDT>(row, row_bytes, lane_off, rows_left - 16 * mb, g, y);
        row += 16 * row_bytes;
        __builtin_amdgcn_sched_barrier(0);
    }
}

constexpr int dma_group_bytes(int NB, int KG) { return d_stages(NB, KG) * (2 * NB * 1024 + 4096); }

// One tile of 32 NB rows.  TAIL: K is not a multiple of the stage.  The activations past the end of K are some of the same
// row's and meet weights of zero: the tiled copy is padded with them, raw row-major dwords are masked.  (Where the activation
// rows are longer than the weights' K, zeros meet a repetition of the last packed row.)
// KG = 2: two groups of four waves, each on its run of the stages; they add their sums through LDS and store half the rows each.
// SW: the SwiGLU output stage on a tiled copy in natural order.  A wave's four column tiles are two of the gate and the same two of up,
// and a lane takes two columns of either, so that no sum changes lanes.
template <int SRC, int NB, int KG, bool TAIL, bool RN, bool SW>
__device__ __forceinline__ void gemm_i8_dma_tile(const GemmParams& p, const int64_t m0, const int tile_n, uint8_t* lds_all) {
    constexpr int BM = 32 * NB, D_NST = d_stages(NB, KG);
    constexpr int A_BYTES = 2 * NB * 1024, STAGE = A_BYTES + 4096;
    constexpr int A_LOADS = NB == 4 ? 2 : 1, W_LOADS = SRC == W_ROWS ? 4 : 1, LOADS = A_LOADS + W_LOADS;
    const int lane = threadIdx.x & 63;
    const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wave = wave_all & 3, group = KG == 1 ? 0 : wave_all >> 2;
    uint8_t* const lds = lds_all + group * dma_group_bytes(NB, KG);
    const int j = lane & 15, g = lane >> 4;
    const int64_t ncol = (int64_t)tile_n * G_BN + 64 * wave + 4 * j;
    const bool col_ok = ncol < p.N;
    const int nst = (int)((p.K + D_BK - 1) / D_BK);
    const int64_t k_last = (int64_t)(nst - 1) * D_BK;
    // this group's stages: st0 .. st0 + mine - 1 (every group meets `rounds` barriers in the loop; mine >= 1)
    const int rounds = KG == 1 ? nst : (nst + 1) / 2, st0 = group * rounds, mine = KG == 1 ? nst : min(rounds, nst - st0);
    const int st_tail = group == KG - 1 ? mine - 1 : nst;  // TAIL: the partial stage, if it is this group's

    // A stage's row is 64 bytes of LDS, four pieces of 16; piece q of row r lies at place q ^ (r / 4 & 2).  A 16-byte read from
    // LDS takes its lanes in groups that hold rows 0 .. 3 and 12 .. 15 of one piece with rows 4 .. 11 of the next, so it meets
    // every bank once.  (With q ^ (r / 4 % 4), and row-major weights as [row][64 columns], 7.5 M of the 15.5 M LDS cycles of
    // 2048 x 11008 x 4096 were conflicts, now none of 8.0 M; us a call, 4096 x 11008 x 4096 180.4 -> 176.4, 4096 x 13824 x 2560
    // 143.7 -> 140.9, 4096 x 2560 x 6912 91.6 -> 89.2.)  Four lanes load a row: lanes of a load that each have a row of their
    // own take the cache four times as long.  Rows past M repeat the last one (their outputs are never stored); columns past N
    // read column 0 of row-major weights and the last tile of the copy.
    const int64_t rows_left = (p.M - m0 < BM) ? p.M - m0 : BM;
    uint32_t a_off[A_LOADS], a_tail[A_LOADS];
#pragma unroll
    for (int b = 0; b < A_LOADS; b++) {
        const int row = 16 * ((A_LOADS * wave + b) % (2 * NB)) + (lane >> 2), piece = (lane & 3) ^ ((lane >> 4) & 2);
        const uint32_t r = (uint32_t)(row < rows_left ? row : rows_left - 1);
        a_off[b] = r * (uint32_t)p.K + 16u * piece;
        a_tail[b] = r * (uint32_t)p.K + (k_last + 16 * piece < p.K ? 16u * piece : 0u);
    }
    uint32_t w_off[W_LOADS], w_tail[W_LOADS];
    const bool w_in = !TAIL || SRC > W_ROWS16 || k_last + 16 * g < p.K;  // this lane's rows of the last stage exist
    if constexpr (SRC == W_ROWS) {
#pragma unroll
        for (int r = 0; r < W_LOADS; r++) {
            w_off[r] = (uint32_t)(col_ok ? ncol : 0) + (uint32_t)(4 * g + r) * (uint32_t)p.N;
            w_tail[r] = (uint32_t)(col_ok ? ncol : 0) + (uint32_t)min((int64_t)(4 * g + r), p.Kb - 1 - (k_last >> 2)) * (uint32_t)p.N;
        }
    } else if constexpr (SRC == W_ROWS16) {
        const int64_t col = (int64_t)tile_n * G_BN + 64 * wave + 16 * (lane & 3);
        w_off[0] = (uint32_t)(col < p.N ? col : 0) + (uint32_t)rows16_row(lane) * (uint32_t)p.N;
        w_tail[0] = (uint32_t)(col < p.N ? col : 0) + (uint32_t)min((int64_t)rows16_row(lane), p.Kb - 1 - (k_last >> 2)) * (uint32_t)p.N;
    } else {
        const int l = min(16 * tile_n + 4 * wave + (j >> 2), (int)(p.N >> 4) - 1);  // SW: gate and up tiles in turn
        const int tt = SW ? (l >> 1) + (l & 1 ? (int)(p.N >> 5) : 0) : stored_tile16((int)(ncol >> 4), p.tiles16);
        w_off[0] = ((uint32_t)tt * (uint32_t)p.wsteps * 64u + (uint32_t)(16 * g + 4 * (j & 3))) * 4u;
    }
    const int8_t* const a_base = p.Q + m0 * p.K;  // uniform
    const uint32_t frag_at = 64u * j + 16u * (g ^ ((j >> 2) & 2));  // lane (j, g): k = 16 g .. +15 of row j of a block
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;

    // the next stage to load: its global addresses, and the byte offset of its buffer
    const int64_t w_step = SRC <= W_ROWS16 ? 16 * p.N : 256;
    const int8_t* a_next = a_base + (int64_t)st0 * D_BK;
    const uint8_t* w_next = p.W_T + st0 * w_step;
    uint32_t into = 0;
    int st_next = 0;
    auto issue_a = [&](int b) {
        const bool last = TAIL && st_next >= st_tail;
        dma16(lds0 + into + (uint32_t)((A_LOADS * wave + b) % (2 * NB)) * 1024u, last ? a_tail[b] : a_off[b], a_next);
    };
    auto issue_w = [&](int r) {
        const bool last = TAIL && st_next >= st_tail;
        const uint32_t wd = lds0 + into + A_BYTES + (uint32_t)wave * 1024u;
        if constexpr (SRC == W_ROWS) dma4(wd + 256u * r, last ? w_tail[r] : w_off[r], w_next);
        else dma16(wd, SRC == W_ROWS16 && last ? w_tail[0] : w_off[0], w_next);
    };
    auto next_buf = [](uint32_t b) { return b + STAGE == D_NST * STAGE ? 0u : b + STAGE; };
    auto advance = [&]() {  // past the end: the last stage again, never read
        st_next++;
        a_next += st_next < mine ? D_BK : 0;
        w_next += st_next < mine ? w_step : 0;
        into = next_buf(into);
    };

    v4i acc[2 * NB][4];
#pragma unroll
    for (int mb = 0; mb < 2 * NB; mb++)
#pragma unroll
        for (int t = 0; t < 4; t++) acc[mb][t] = v4i{0, 0, 0, 0};
    if constexpr (SRC == W_FIELDS) {  // lane (j, g) holds rows 16 mb + 4 g + r of its columns
#pragma unroll
        for (int mb = 0; mb < 2 * NB; mb++) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int64_t m = m0 + 16 * mb + 4 * g + r;
                const int32_t rs = p.q_rowsum[m < p.M ? m : p.M - 1];
                acc[mb][0][r] = -rs;
                acc[mb][1][r] = -(rs << 2);
                acc[mb][2][r] = -(rs << 4);
            }
        }
    }

    uint4 a_lo[NB], a_hi[NB];
    v4i b_dec[2][4];
    uint32_t raw[4];
    auto read_raw = [&](int s, uint32_t buf) {
        const uint8_t* src = lds + buf + A_BYTES + wave * 1024;
        if constexpr (SRC <= W_ROWS16) {
#pragma unroll
            for (int r = 0; r < 4; r++) raw[r] = *(const uint32_t*)(src + 256 * r + 4 * lane);
            if (TAIL && s >= st_tail) {
#pragma unroll
                for (int r = 0; r < 4; r++) raw[r] = w_in ? raw[r] : 0u;
            }
        } else {
            if constexpr (SW) {  // lane (j, g)'s 16 bytes are those of columns 4 (j % 4) .. +3 of the wave's tile j / 4
                const uint8_t* at = src + 256 * g + 128 * (j >> 3) + 8 * (j & 7);
                const u32x2 a = *(const u32x2*)at, b = *(const u32x2*)(at + 64);
                raw[0] = a[0]; raw[1] = a[1]; raw[2] = b[0]; raw[3] = b[1];
            } else {
                const uint4 v = *(const uint4*)(src + 16 * lane);
                raw[0] = v.x; raw[1] = v.y; raw[2] = v.z; raw[3] = v.w;
            }
        }
    };
    auto read_a = [&](uint32_t buf, int mb0, uint4 (&dst)[NB]) {
        const uint8_t* src = lds + (buf + frag_at);
#pragma unroll
        for (int i = 0; i < NB; i++) {
            dst[i] = *(const uint4*)(src + (mb0 + i) * 1024);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // the decode of one stage's weights in 16 slices, one behind each MFMA of a half
    uint32_t d_t[4], d_G[4], d_H[4];
    auto decode_slice = [&](int c, v4i (&out)[4]) {
        const uint32_t lutA_lo = 0x00FF0100u, lutB_lo = 0x0000FF00u, lutB_hi = 0x00000001u;
        if constexpr (SRC == W_FIELDS) {
            out[c >> 2][c & 3] = (int)(raw[c & 3] & (0x03030303u << (2 * (c >> 2))));
            return;
        }
        if constexpr (SRC == W_TILES) {
            const int t = c >> 2;
            switch (c & 3) {
                case 0: d_G[t] = raw[t]; d_H[t] = d_G[t] >> 4; out[t][0] = (int)perm(0u, lutA_lo, d_G[t] & 0x03030303u); break;
                case 1: out[t][1] = (int)perm(lutB_hi, lutB_lo, d_G[t] & 0x0C0C0C0Cu); break;
                case 2: out[t][2] = (int)perm(0u, lutA_lo, d_H[t] & 0x03030303u); break;
                default: out[t][3] = (int)perm(lutB_hi, lutB_lo, d_H[t] & 0x0C0C0C0Cu); break;
            }
            return;
        }
        // row-major dwords: the 4x4 byte transpose in slices 2 and 3, then three slices per column
        if (c == 2) {
            d_t[0] = perm(raw[1], raw[0], 0x05010400u);
            d_t[1] = perm(raw[1], raw[0], 0x07030602u);
            d_t[2] = perm(raw[3], raw[2], 0x05010400u);
            d_t[3] = perm(raw[3], raw[2], 0x07030602u);
        } else if (c == 3) {
            d_G[0] = perm(d_t[2], d_t[0], 0x05040100u);
            d_G[1] = perm(d_t[2], d_t[0], 0x07060302u);
            d_G[2] = perm(d_t[3], d_t[1], 0x05040100u);
            d_G[3] = perm(d_t[3], d_t[1], 0x07060302u);
        } else if (c >= 4) {
            const int t = (c - 4) / 3;
            switch ((c - 4) % 3) {
                case 0: d_H[t] = d_G[t] >> 4; out[t][0] = (int)perm(0u, lutA_lo, d_G[t] & 0x03030303u); break;
                case 1:
                    out[t][1] = (int)perm(lutB_hi, lutB_lo, d_G[t] & 0x0C0C0C0Cu);
                    out[t][2] = (int)perm(0u, lutA_lo, d_H[t] & 0x03030303u);
                    break;
                default: out[t][3] = (int)perm(lutB_hi, lutB_lo, d_H[t] & 0x0C0C0C0Cu); break;
            }
        }
    };

    uint32_t buf = 0;
#pragma unroll
    for (int s = 0; s < D_NST; s++) {
#pragma unroll
        for (int b = 0; b < A_LOADS; b++) issue_a(b);
#pragma unroll
        for (int r = 0; r < W_LOADS; r++) issue_w(r);
        advance();
    }
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((D_NST - 2) * LOADS) : "memory");  // stages 0 and 1
    read_raw(0, 0);
    read_a(0, 0, a_lo);
#pragma unroll
    for (int c = 0; c < 16; c++) decode_slice(c, b_dec[0]);
    read_raw(1, STAGE);

    // Everything but the MFMAs is dealt out between them, two or three instructions behind each: an MFMA occupies the
    // matrix pipe for 16 cycles, the wave's own issue for 4, and instructions in a row of their own would leave the pipe idle.
    auto stage = [&](int s, const v4i (&b_cur)[4], v4i (&b_nxt)[4]) {
        constexpr int SL = 4 / NB;  // slots per MFMA
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int c = 0; c < 16; c++) {
            if (c % SL == 0) {
                const int i = (c / SL) >> 2, t = (c / SL) & 3;
                const v4i a = {(int)a_lo[i].x, (int)a_lo[i].y, (int)a_lo[i].z, (int)a_lo[i].w};
                acc[i][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b_cur[t], acc[i][t], 0, 0, 0);
            }
            if (c < NB) a_hi[c] = *(const uint4*)(lds + (buf + frag_at) + (NB + c) * 1024);
            decode_slice(c, b_nxt);
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((D_NST - 3) * LOADS) : "memory");
        const uint32_t nxt = next_buf(buf), nxt2 = next_buf(nxt);
#pragma unroll
        for (int c = 0; c < 16; c++) {
            if (c % SL == 0) {
                const int i = (c / SL) >> 2, t = (c / SL) & 3;
                const v4i a = {(int)a_hi[i].x, (int)a_hi[i].y, (int)a_hi[i].z, (int)a_hi[i].w};
                acc[NB + i][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b_cur[t], acc[NB + i][t], 0, 0, 0);
            }
            if (c < NB) a_lo[c] = *(const uint4*)(lds + (nxt + frag_at) + c * 1024);
            if (c == 4) read_raw(s + 2, nxt2);
            // stage s + D_NST over stage s
            if (c >= 6 && c < 6 + A_LOADS) issue_a(c - 6);
            if (c >= 8 && c < 8 + W_LOADS) issue_w(c - 8);
            if (c == 13) advance();
            __builtin_amdgcn_sched_barrier(0);
        }
        buf = nxt;
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the fragments arrived under these MFMAs (see gemm_i8_kernel)
        __builtin_amdgcn_sched_barrier(0);
    };
    int s = 0;
    for (; s + 1 < mine; s += 2) {
        stage(s, b_dec[0], b_dec[1]);
        stage(s + 1, b_dec[1], b_dec[0]);
    }
    if (s < mine) stage(s, b_dec[0], b_dec[1]);
    if (KG > 1 && mine < rounds) asm volatile("s_barrier" ::: "memory");  // (uniform; the other group has one stage more)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (no load may reach LDS that another workgroup owns by then)

    v4i sums[KG == 1 ? 1 : NB][4];
    if constexpr (KG > 1) {
        // group 0 takes the first NB row blocks, group 1 the others: each hands over the sums that it does not store
        v4i* const given = (v4i*)lds_all + wave_all * (256 * NB) + lane;
        const v4i* const taken = (const v4i*)lds_all + (wave_all ^ 4) * (256 * NB) + lane;
        __syncthreads();  // (both groups have read their last stages)
#pragma unroll
        for (int i = 0; i < NB; i++)
#pragma unroll
            for (int t = 0; t < 4; t++) {
                given[64 * (4 * i + t)] = group ? acc[i][t] : acc[NB + i][t];
                sums[i][t] = group ? acc[NB + i][t] : acc[i][t];
            }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NB; i++)
#pragma unroll
            for (int t = 0; t < 4; t++) sums[i][t] += taken[64 * (4 * i + t)];
        __syncthreads();  // (the row scales come over them)
    }

    // ---- output.  The row scales of the tile pass through the wave's own weight area in LDS (nobody else's loads reach it),
    // so that a row block's four come with one read. ----
    const int64_t half_n = p.N / 2, scol = (int64_t)tile_n * (G_BN / 2) + 32 * wave + 2 * j;  // SW: the first of this lane's outputs
    float* const sx_lds = (float*)(lds + A_BYTES + wave * 1024);
    uint32_t ws_bits[4], bs_bits[4];
#pragma unroll
    for (int q = 0; q < (NB == 4 ? 2 : 1); q++) {
        const int64_t m = m0 + 64 * q + lane;
        sx_lds[64 * q + lane] = p.s_x[m < p.M ? m : p.M - 1];
    }
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int64_t n = SW ? (scol < half_n ? scol + (t & 1) + (t >> 1) * half_n : 0) : !col_ok ? 0 : RN ? min(ncol + t, p.N - 1) : ncol + t;
        ws_bits[t] = load_bits_rt(p.epi.scale, p.epi.scale_dtype, p.epi.scale_bcast ? 0 : n);
        bs_bits[t] = p.epi.bias ? load_bits_rt(p.epi.bias, p.epi.bias_dtype, n) : 0u;
    }
    float ws[4], bs[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        ws[t] = bits_to_f32_rt(ws_bits[t], p.epi.scale_dtype);
        bs[t] = p.epi.bias ? bits_to_f32_rt(bs_bits[t], p.epi.bias_dtype) : 0.0f;
    }
    if (SW ? scol >= half_n : !col_ok) return;
    constexpr bool FL = SRC == W_FIELDS;
    auto store = [&](const auto& v, int64_t row0, int left, const float* sx) {
        if constexpr (SW) {
            if (p.y_dtype == BT_BF16) dma_epilogue_swiglu<BT_BF16>(p, v, row0, g, scol, left, sx, ws, bs);
            else dma_epilogue_swiglu<BT_F16>(p, v, row0, g, scol, left, sx, ws, bs);
            return;
        }
        if (p.acc_out) dma_store_acc<FL, RN>(p, v, row0, g, ncol, left);
        if (p.y_dtype == BT_BF16) {
            if (p.epi.residual) dma_epilogue<BT_BF16, true, FL, RN>(p, v, row0, g, ncol, left, sx, ws, bs);
            else dma_epilogue<BT_BF16, false, FL, RN>(p, v, row0, g, ncol, left, sx, ws, bs);
        } else if (p.y_dtype == BT_F16) {
            if (p.epi.residual) dma_epilogue<BT_F16, true, FL, RN>(p, v, row0, g, ncol, left, sx, ws, bs);
            else dma_epilogue<BT_F16, false, FL, RN>(p, v, row0, g, ncol, left, sx, ws, bs);
        } else {
            if (p.epi.residual) dma_epilogue<BT_F32, true, FL, RN>(p, v, row0, g, ncol, left, sx, ws, bs);
            else dma_epilogue<BT_F32, false, FL, RN>(p, v, row0, g, ncol, left, sx, ws, bs);
        }
    };
    if constexpr (KG == 1) {
        store(acc, m0, (int)rows_left, sx_lds);
    } else {
        const int first = 16 * NB * group;
        if (rows_left > first) store(sums, m0 + first, (int)rows_left - first, sx_lds + first);
    }
}

// NB: tiles of 32 NB rows.  NF > 0: the last p.fine_from .. of an XCD's tiles are computed in tiles of 32 NF rows.
template <int SRC, int NB, int NF, int KG, bool TAIL, bool RN, bool SW>
__global__ __launch_bounds__(256 * KG, KG == 2 || NB == 4 ? 2 : NB == 2 ? 3 : 4) void gemm_i8_dma_kernel(GemmParams p) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[KG * dma_group_bytes(NB, KG)];
    // XCD-aware tile order, as in gemm_i8_kernel
    const uint32_t idx = blockIdx.x >> 3;
    const bool fine = NF > 0 && idx >= (uint32_t)p.fine_from;  // (uniform)
    const uint32_t parts = NF > 0 ? NB / (NF > 0 ? NF : 1) : 1, f = fine ? idx - (uint32_t)p.fine_from : 0u;
    const uint32_t in_xcd = fine ? (uint32_t)p.fine_from + f / parts : idx;
    const uint32_t lin = (blockIdx.x & 7u) * (uint32_t)p.per_xcd + in_xcd;
    const uint32_t tiles_m = (uint32_t)p.tiles_m, tiles_n = (uint32_t)p.tiles_n;
    if (lin >= tiles_m * tiles_n) return;
    constexpr uint32_t GM = 4;
    const uint32_t group = lin / (GM * tiles_n);
    const uint32_t first_m = group * GM;
    const uint32_t gm = (tiles_m - first_m < GM) ? tiles_m - first_m : GM;
    const uint32_t in_group = lin - group * GM * tiles_n;
    const uint32_t tn = (gm == GM) ? in_group / GM : in_group / gm;
    const int64_t m0 = (int64_t)(first_m + (in_group - tn * gm)) * (32 * NB);
    if constexpr (NF > 0) {
        if (fine) {
            const int64_t mf = m0 + (int64_t)(f % parts) * (32 * NF);
            if (mf < p.M) gemm_i8_dma_tile<SRC, NF, 1, TAIL, RN, SW>(p, mf, (int)tn, lds);
            return;
        }
    }
    gemm_i8_dma_tile<SRC, NB, KG, TAIL, RN, SW>(p, m0, (int)tn, lds);
}

// A launch of one tile of 64 or 32 rows for each compute unit at most: two groups of waves, half of the stages each, so that a
// SIMD has two waves where one's chain of LDS reads, decode and MFMAs left it idle half of the time.  One / two groups, us a
// call with the quantizer, row-major weights: tiles of 32 rows, 256 x 7680 x 2560 18.7 / 17.1, 512 x 4096 x 11008 50.0 / 42.2;
// of 64 rows, 256 x 11008 x 4096 28.2 / 24.0, 1000 x 2560 x 6912 42.5 / 34.9, 1000 x 4096 x 11008 62.8 / 51.8.  The gain grows
// with K; below 24 stages it is lost in the exchange of the sums.  The field layout keeps one group (its sums start at minus
// the row sums).
static bool i8_splits_k(int64_t stages) { return stages >= 24; }

// Rows of the tiles in units of 32 (4, 2 or 1), or 0 where gemm_i8_kernel is the better one: tiled weights in whole stages with
// at most one tile of 128 x 256 for each compute unit, but not with two groups of waves on finer tiles.  Measured, decode-tiled
// weights, gemm_i8_kernel / tiles of 32 / 64 / 128 rows here, us: one tile of 32 rows for each compute unit at most, 256 x 4096 x
// 4096 16.2 / 14.6 / 17.2 / 18.1, 512 x 2560 x 6912 24.3 / 21.8 / 25.2 / 27.1; of 64 rows, 256 x 11008 x 4096 20.5 / 21.9 / 18.6 /
// 21.9, 1000 x 2560 x 6912 30.1 / 32.7 / 25.9 / 31.5; of 128 rows, 512 x 11008 x 4096 26.4 / 30.9 / 29.1 / 29.4, 2048 x 4096 x 4096
// 30.1 / 40.2 / 32.7 / 32.8, 2048 x 4096 x 11008 67.6 / 105 / 78.0 / 77.1; 16 stages (one group), 128 x 16384 x 1024 8.3 / 8.5 /
// 10.1 / 8.6.  The field layout has one group here, so it stays there.  With more tiles (tiled / row-major weights, us, that kernel
// first): 4096 x 13824 x 2560 133 -> 122 / 148 -> 134; 2048 x 11008 x 4096 93 -> 82 / 104 -> 88; 4096 x 2560 x 6912 (64-row tiles)
// 67 -> 65 / 85 -> 73; 4096 x 8192 x 8192 207 -> 192 / 250 -> 208; 3000 x 1008 x 1040, K not in whole stages, 38 -> 13 / 16 -> 14.
// The prices are microseconds of a compute unit's run of tiles, fitted to the same runs.
static int gemm_i8_dma_plan(int64_t M, int64_t N, int64_t K, bool tiled, bool fields, double* us) {
    const int64_t C = gemm_compute_units(), tn = ceil_div(N, G_BN);
    const int64_t t4 = ceil_div(M, 128) * tn, t2 = ceil_div(M, 64) * tn, t1 = ceil_div(M, 32) * tn;
    const bool whole = gemm_whole_tiles();
    const bool split = i8_splits_k(ceil_div(K, D_BK)) && !fields;
    if (tiled && K % 128 == 0 && N % 4 == 0 && t4 <= C && (t2 > C || !split || whole)) return 0;
    if (t1 <= C && !whole) { *us = split ? 5.7 + 0.0027 * (double)K : 5.2 + 0.0035 * (double)K; return 1; }
    if (t2 <= C && !whole) { *us = split ? 5.5 + 0.0034 * (double)K : 5.2 + 0.0045 * (double)K; return 2; }
    const int parts = gemm_dma_parts(t4);
    const double n4 = parts == 1 ? (double)ceil_div(t4, C) : (double)(2 * (t4 / (2 * C))) + (parts == 2 ? 1.2 : 0.6);
    const double p4 = n4 * (3.5 + 0.0055 * (double)K), p2 = (double)ceil_div(t2, C) * (2.2 + 0.0029 * (double)K);
    const bool half = p2 < p4 && !whole;
    *us = 2.0 + (half ? p2 : p4);
    return half ? 2 : 4;
}
int gemm_i8_dma_rows(int64_t M, int64_t N, int64_t K, bool tiled, bool fields) {
    double us;
    return gemm_i8_dma_plan(M, N, K, tiled, fields, &us);
}
// microseconds of launch_gemm_i8: this file's plan, or gemm_i8_kernel's rounds of whole tiles (of finer ones at their price)
double gemm_i8_cost(int64_t M, int64_t N, int64_t K, bool tiled, bool operand_order) {
    double us;
    if (operand_order && gemm_i8_dma_plan(M, N, K, tiled, false, &us)) return us;
    return gemm_split(M, N, tiled && K % 128 == 0).rounds * (8.6 + 0.0044 * (double)K);
}

template <int SRC, int NB, bool TAIL, bool RN = false, bool SW = false>
static int launch_gemm_i8_dma_src(GemmParams p, hipStream_t st) {
    p.tile_n0 = 0;
    p.tiles_n = (int)ceil_div(p.N, G_BN);
    p.tiles_m = (int)ceil_div(p.M, 32 * NB);
    const int64_t total = (int64_t)p.tiles_m * p.tiles_n;
    if (total >= (1ll << 29)) {
        set_error("bt_ternary_gemm_i8: %lld tiles of %d x 256 outputs are more than one launch takes", (long long)total, 32 * NB);
        return BT_ERR_INVALID;
    }
    p.per_xcd = (int)ceil_div(total, 8);
    p.fine_from = p.per_xcd;
    const dim3 block(256);
    if constexpr (NB == 4) {
        const int parts = gemm_dma_parts(total);
        if (parts > 1) {
            const int rem = p.per_xcd % (int)(2 * gemm_compute_units() / 8);
            p.fine_from = p.per_xcd - rem;
            const dim3 grid((unsigned)(8 * (p.fine_from + parts * rem)));
            if (parts == 2) hipLaunchKernelGGL((gemm_i8_dma_kernel<SRC, 4, 2, 1, TAIL, RN, SW>), grid, block, 0, st, p);
            else hipLaunchKernelGGL((gemm_i8_dma_kernel<SRC, 4, 1, 1, TAIL, RN, SW>), grid, block, 0, st, p);
            return check_launch("bt_ternary_gemm_i8");
        }
    }
    if constexpr (NB != 4 && SRC != W_FIELDS) {
        if (total <= gemm_compute_units() && i8_splits_k(ceil_div(p.K, D_BK))) {
            hipLaunchKernelGGL((gemm_i8_dma_kernel<SRC, NB, 0, 2, TAIL, RN, SW>), dim3((unsigned)(8 * p.per_xcd)), dim3(512), 0, st, p);
            return check_launch("bt_ternary_gemm_i8");
        }
    }
    hipLaunchKernelGGL((gemm_i8_dma_kernel<SRC, NB, 0, 1, TAIL, RN, SW>), dim3((unsigned)(8 * p.per_xcd)), block, 0, st, p);
    return check_launch("bt_ternary_gemm_i8");
}
template <int NB>
static int launch_gemm_i8_dma_rows(const GemmParams& p, int src, bool swiglu, hipStream_t st) {
    const bool tail = p.K % D_BK != 0;
    if (swiglu) return tail ? launch_gemm_i8_dma_src<W_TILES, NB, true, false, true>(p, st) : launch_gemm_i8_dma_src<W_TILES, NB, false, false, true>(p, st);
    if (src == W_TILES && p.N % 4 != 0) return launch_gemm_i8_dma_src<W_TILES, NB, true, true>(p, st);
    if (src == W_FIELDS) return launch_gemm_i8_dma_src<W_FIELDS, NB, false>(p, st);
    if (src == W_TILES) return tail ? launch_gemm_i8_dma_src<W_TILES, NB, true>(p, st) : launch_gemm_i8_dma_src<W_TILES, NB, false>(p, st);
    if (src == W_ROWS16) return tail ? launch_gemm_i8_dma_src<W_ROWS16, NB, true>(p, st) : launch_gemm_i8_dma_src<W_ROWS16, NB, false>(p, st);
    return tail ? launch_gemm_i8_dma_src<W_ROWS, NB, true>(p, st) : launch_gemm_i8_dma_src<W_ROWS, NB, false>(p, st);
}
// swiglu: the SwiGLU output stage (a natural-order tiled copy of [gate | up], N % 32 == 0, a 16-bit output [M, N / 2], neither residual nor acc_out)
int launch_gemm_i8_dma(const GemmParams& p, int rows, bool tiled, bool fields, bool swiglu, hipStream_t st) {
    const int src = w_source(tiled, fields, p.W_T, p.N);
    return rows == 4 ? launch_gemm_i8_dma_rows<4>(p, src, swiglu, st)
         : rows == 2 ? launch_gemm_i8_dma_rows<2>(p, src, swiglu, st) : launch_gemm_i8_dma_rows<1>(p, src, swiglu, st);
}

}  // namespace bt
