// Ternary weights times a few tens of rows: short prompts, batched decode steps.  16-bit rows, and int8 rows in operand order.
//
// Arithmetic as in gemm_f16.hip and gemm_i8.hip.  Between the streaming kernel, which decodes the weights again for every 16 rows, and
// the tiled GEMMs, whose tiles of 256 columns are too few to occupy the chip: a workgroup owns 16 RB rows x 16 NACC columns, so that
// a weight is decoded once for all of the rows, and its eight waves split K.  Every wave works alone on its run of steps of 128 bytes
// of a row (64 or 128 values): the rows come eight lanes to a row (whole cache lines; a lane a row would take the cache four times
// as long), D steps ahead, and pass through the wave's own LDS into matrix fragments, without a barrier.  The waves' sums meet in
// LDS, in wave order.
#include <cstdio>

#include "row_math.h"

namespace bt {

struct RowsParams {
    const uint8_t* X;     // [M, K] fp16 or bf16 bits, or int8
    const uint8_t* W;     // the decode-tiled copy, or W_T [Kb, N]
    int64_t row_bytes;    // of X (a multiple of 16)
    int64_t M, N, Kb;
    int wsteps;           // 64-wide steps of the copy
    int tiles16;          // as in tiles16_arg
    int tiles;            // column tiles
    int per_xcd;          // column tiles per XCD (grid.x = 8 * per_xcd); 0: tiles in launch order
    void* Y;              // [M, N], SW: [M, N / 2]
    int y_dtype;
    const float* s_x;     // MODE_I8: [M]
    int32_t* acc_out;     // MODE_I8: optional [M, N]
    Epilogue epi;
};

constexpr int ROWS_WAVES = 8;
// Row blocks whose sums a wave hands over at once, and the LDS of a wave: a step's rows, then those sums.
constexpr int rows_pass(int RB, int NACC) { return RB > 4 && NACC == 4 ? (RB + 1) / 2 : RB; }
constexpr int rows_wave_bytes(int RB, int NACC) {
    return std::max(RB * 2048, rows_pass(RB, NACC) * NACC * 1024);
}
constexpr int rows_depth(int RB) { return RB <= 3 ? 3 : 2; }  // steps whose rows are on their way (two: 256 x 2560 x 6912 20.9 us, three: 18.0)
typedef uint32_t u32_any __attribute__((aligned(4)));

// ROWS: row-major weights (NACC = 4, N % 4 == 0): lane (j, g) takes columns 4 j .. +3; otherwise the decode-tiled copy, column j of
// every 16-column tile.
// SW: the SwiGLU output stage on a copy in gate/up pair order (NACC even: tiles 2 i and 2 i + 1 are the gate's and up's)
// TAIL: a partial step, or rows of X longer than the weights'
template <int MODE, bool ROWS, int RB, int NACC, bool SW, bool TAIL>
__global__ __launch_bounds__(64 * ROWS_WAVES, 2) void few_rows_kernel(RowsParams p) {
    constexpr bool I8 = MODE == MODE_I8;
    constexpr int D = rows_depth(RB), AL = 2 * RB, YDT = MODE == MODE_F16 ? BT_F16 : BT_BF16;
    constexpr int WR = I8 ? 2 * NACC : NACC;  // raw dwords of a lane and step
    typedef typename std::conditional<I8, v4i, v4f>::type acc_t;
    __shared__ __attribute__((aligned(16))) uint8_t lds_all[ROWS_WAVES * rows_wave_bytes(RB, NACC)];
    // consecutive tiles on one XCD
    const int tile = p.per_xcd ? (int)(blockIdx.x & 7) * p.per_xcd + (int)(blockIdx.x >> 3) : (int)blockIdx.x;
    if (tile >= p.tiles) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 15, g = lane >> 4;
    uint8_t* const lds = lds_all + wave * rows_wave_bytes(RB, NACC);
    const int64_t m0 = (int64_t)blockIdx.y * (16 * RB);
    const int rows_left = (int)((p.M - m0 < 16 * RB) ? p.M - m0 : 16 * RB);
    const int nst = (int)((p.row_bytes + 127) >> 7), run = (nst + ROWS_WAVES - 1) / ROWS_WAVES;
    const int st0 = min(wave * run, nst), st1 = min(nst, st0 + run);

    // Load b brings rows 8 b .. +7 of the step, piece lane % 8 of 16 bytes; rows past the end repeat the last one (never stored).
    const uint8_t* const x0 = p.X + m0 * p.row_bytes;
    const uint32_t piece = lane & 7;
    uint32_t a_off[AL];
#pragma unroll
    for (int b = 0; b < AL; b++) {
        const int row = 8 * b + (lane >> 3);
        a_off[b] = (uint32_t)(row < rows_left ? row : rows_left - 1) * (uint32_t)p.row_bytes + 16u * piece;
    }
    // Lane (j, g) takes pieces 2 g and 2 g + 1 of a row, one after the other (sub-steps 0 and 1): eight values each, kb rows
    // 4 g + 2 sub, + 1 of the step's 16, or sixteen values, kb rows 8 g + 4 sub .. + 3 of its 32.
    uint32_t w_off[ROWS ? 1 : NACC], w_col = 0;
    if constexpr (ROWS) {
        const int64_t col = (int64_t)tile * 64 + 4 * j;
        w_col = (uint32_t)(col < p.N ? col : 0);
        w_off[0] = w_col + (I8 ? 8u : 4u) * (uint32_t)g * (uint32_t)p.N;
    } else {
#pragma unroll
        for (int t = 0; t < NACC; t++)
            w_off[t] = ((uint32_t)stored_tile16(tile * NACC + t, p.tiles16) * (uint32_t)p.wsteps * 64u + (I8 ? 32u * g + j : (uint32_t)lane)) * 4u;
    }
    // a row of a step is 128 bytes of LDS, piece q of row r at place q ^ f(r): no bank twice (fd_place of gemm_f16.hip)
    const uint32_t put = (uint32_t)(lane >> 3) * 128u, put_at[2] = {put + 16u * (piece ^ ((lane >> 4) & 1u)), put + 16u * (piece ^ (((lane >> 4) & 1u) | 6u))};
    const uint32_t at_j = ((j >> 1) & 1u) | ((j >> 3) & 1u) * 6u;
    const uint32_t frag_at[2] = {128u * j + 16u * ((2u * g) ^ at_j), 128u * j + 16u * ((2u * g + 1u) ^ at_j)};

    u32x4 xa[D][AL];
    uint32_t raw[D][WR];
    const bool past = TAIL && 128 * (nst - 1) + 16 * (int)piece >= (int)p.row_bytes;  // this lane's pieces of the partial step lie past the end
    const uint32_t kept = past ? 0u : 0xFFFFFFFFu;
    const u32x4 keep = {kept, kept, kept, kept};
    // In the partial step such a lane loads the row's first piece of the step instead, and where the copy ends in the middle of a step
    // of 128 values, the lanes of its second half load the first.
    const uint32_t x_back = past ? 16u * piece : 0u, w_back = 2 * (nst - 1) + 1 >= p.wsteps && g >= 2 ? 256u : 0u;
    auto load = [&](int f, int s) __attribute__((always_inline)) {  // s uniform
        const uint8_t* xb = x0 + (int64_t)s * 128;
        const bool last = TAIL && s == nst - 1;  // (uniform)
        if constexpr (ROWS) {
            constexpr int SR = I8 ? 32 : 16;  // rows of W_T a step
            const uint8_t* wb = p.W + (int64_t)s * SR * p.N;
            const uint32_t end = (uint32_t)(p.Kb - 1 - (int64_t)s * SR) * (uint32_t)p.N + w_col;  // TAIL: rows past the last one meet zeros
#pragma unroll
            for (int r = 0; r < WR; r++) {
                if constexpr (TAIL) raw[f][r] = *(const u32_any*)(wb + min(w_off[0] + (uint32_t)r * (uint32_t)p.N, end));
                else raw[f][r] = *(const u32_any*)(wb + (int64_t)r * p.N + w_off[0]);
            }
        } else if constexpr (I8) {
            const uint8_t* wb = p.W + (int64_t)s * 512;
            const uint32_t back = last ? w_back : 0u;
#pragma unroll
            for (int x = 0; x < WR; x++) raw[f][x] = ldw_nt(wb + (w_off[x % NACC] + 64u * (x / NACC) - back));
        } else {
            const uint8_t* wb = p.W + (int64_t)s * 256;
#pragma unroll
            for (int t = 0; t < NACC; t++) raw[f][t] = ldw_nt(wb + w_off[t]);
        }
        const uint32_t back = last ? x_back : 0u;
#pragma unroll
        for (int b = 0; b < AL; b++) xa[f][b] = *(const u32x4*)(xb + (TAIL ? a_off[b] - back : a_off[b]));
    };
    acc_t acc[RB][NACC];
#pragma unroll
    for (int b = 0; b < RB; b++)
#pragma unroll
        for (int t = 0; t < NACC; t++) acc[b][t] = acc_t{0, 0, 0, 0};
    auto step = [&](int f, int s) __attribute__((always_inline)) {
        if (TAIL && s == nst - 1) {  // (uniform)
#pragma unroll
            for (int b = 0; b < AL; b++) xa[f][b] &= keep;
        }
#pragma unroll
        for (int b = 0; b < AL; b++) *(u32x4*)(lds + 1024 * b + put_at[b & 1]) = xa[f][b];
        u32x4 w[2][NACC];
        if constexpr (I8) {
#pragma unroll
            for (int sub = 0; sub < 2; sub++) {
                uint32_t G[4];
                if constexpr (ROWS) {
                    transpose4x4_bytes(raw[f][4 * sub], raw[f][4 * sub + 1], raw[f][4 * sub + 2], raw[f][4 * sub + 3], G);
                } else {
#pragma unroll
                    for (int t = 0; t < NACC; t++) G[t] = raw[f][sub * NACC + t];
                }
#pragma unroll
                for (int t = 0; t < NACC; t++) w[sub][t] = __builtin_bit_cast(u32x4, decode16_i8(G[t]));
            }
        } else {  // decode: see gemm_f16.hip
            constexpr uint32_t LUT = (MODE == MODE_F16) ? LUT_F16_ONE : LUT_BF16_TWO;
            uint32_t hi[NACC][4];
#pragma unroll
            for (int t = 0; t < NACC; t++)
#pragma unroll
                for (int e = 0; e < 4; e++) hi[t][e] = perm(0u, LUT, (raw[f][t] >> (2 * e)) & 0x03030303u);
#pragma unroll
            for (int t = 0; t < NACC; t++)
#pragma unroll
                for (int x = 0; x < 8; x++) {
                    const int r = x >> 1, e = 2 * (x & 1), q = ROWS ? r : t, byte = ROWS ? t : r;
                    w[x >> 2][t][x & 3] = perm(hi[q][e + 1], hi[q][e], ((uint32_t)(4 + byte) << 24) | (0x0Cu << 16) | ((uint32_t)byte << 8) | 0x0Cu);
                }
        }
        load(f, s + D < st1 ? s + D : st1 - 1);  // (past the end: the last one again, never used)
#pragma unroll
        for (int b = 0; b < RB; b++)
#pragma unroll
            for (int sub = 0; sub < 2; sub++) {
                const u32x4 a = *(const u32x4*)(lds + 2048 * b + frag_at[sub]);
#pragma unroll
                for (int t = 0; t < NACC; t++) {
                    if constexpr (I8)
                        acc[b][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i, a), __builtin_bit_cast(v4i, w[sub][t]), acc[b][t], 0, 0, 0);
                    else if constexpr (MODE == MODE_F16)
                        acc[b][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, w[sub][t]), acc[b][t], 0, 0, 0);
                    else
                        acc[b][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, w[sub][t]), acc[b][t], 0, 0, 0);
                }
            }
    };
    if (st0 < st1) {
#pragma unroll
        for (int f = 0; f < D; f++) load(f, min(st0 + f, st1 - 1));
        int s = st0;
        for (; s + D <= st1; s += D) {
#pragma unroll
            for (int f = 0; f < D; f++) step(f, s + f);
        }
#pragma unroll
        for (int f = 0; f < D - 1; f++) {
            if (s + f < st1) step(f, s + f);  // (uniform)
        }
    }

    auto total = [&](int at) {
        acc_t v = *(const acc_t*)(lds_all + at * 16);
#pragma unroll
        for (int w = 1; w < ROWS_WAVES; w++) v += *(const acc_t*)(lds_all + w * rows_wave_bytes(RB, NACC) + at * 16);
        return v;
    };
    // a thread finishes rows 4 g .. +3 of a column (SW: of a column of the gate and the same of up)
    constexpr int PASS = rows_pass(RB, NACC), COLS = SW ? NACC / 2 : NACC;
    const int64_t Ny = SW ? p.N / 2 : p.N;
#pragma unroll
    for (int b0 = 0; b0 < RB; b0 += PASS) {
        if (b0) __syncthreads();
#pragma unroll
        for (int b = b0; b < RB && b < b0 + PASS; b++)
#pragma unroll
            for (int t = 0; t < NACC; t++) *(acc_t*)(lds + (((b - b0) * NACC + t) * 64 + lane) * 16) = acc[b][t];
        __syncthreads();
        const int sets = std::min(PASS, RB - b0) * COLS;
        for (int set = wave; set < sets; set += ROWS_WAVES) {  // (uniform)
            const int b = set / COLS, t = set - b * COLS, row0 = 16 * (b0 + b) + 4 * g;
            const int64_t col = ROWS ? (int64_t)tile * 64 + 4 * j + t : ((int64_t)tile * COLS + t) * 16 + j;
            if (col >= Ny || row0 >= rows_left) continue;
            if constexpr (I8) {
                const v4i v = total((b * NACC + t) * 64 + lane);
                const float ws = epi_scale(p.epi, col), bs = epi_bias(p.epi, col);
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    if (row0 + r >= rows_left) continue;
                    const int64_t row = m0 + row0 + r, at = row * p.N + col;
                    const int32_t sum = v[r];
                    if (p.acc_out) p.acc_out[at] = times127(sum);
                    float y = epi_int8_f(__fmul_rn((float)sum, 127.0f), p.s_x[row], ws, bs);
                    if (p.epi.residual) y = add_residual(y, p.epi.residual, p.y_dtype, at);
                    if (p.y_dtype == BT_F32) store_elem<BT_F32>(p.Y, at, y);
                    else if (p.y_dtype == BT_F16) store_elem<BT_F16>(p.Y, at, y);
                    else store_elem<BT_BF16>(p.Y, at, y);
                }
            } else {
                float y[SW ? 2 : 1][4];
#pragma unroll
                for (int u = 0; u < (SW ? 2 : 1); u++) {
                    const v4f v = total((b * NACC + (SW ? 2 * t + u : t)) * 64 + lane);
                    const int64_t n = col + u * Ny;
                    const float ws = epi_scale(p.epi, n), bs = epi_bias(p.epi, n);
#pragma unroll
                    for (int r = 0; r < 4; r++) y[u][r] = epi_float(MODE == MODE_BF16 ? v[r] * 0.5f : v[r], ws, bs);  // (bf16 weights were decoded as +-2.0)
                }
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    if (row0 + r >= rows_left) continue;
                    const int64_t at = (m0 + row0 + r) * Ny + col;
                    float v = y[0][r];
                    if constexpr (SW) v = swiglu_value(round_to_dtype(y[0][r], YDT), round_to_dtype(y[SW ? 1 : 0][r], YDT), YDT);
                    else if (p.epi.residual) v = add_residual(v, p.epi.residual, YDT, at);
                    store_elem<YDT>(p.Y, at, v);
                }
            }
        }
    }
}

// Which tile, and what the launch takes in microseconds.  A workgroup reads its rows' whole length from L2, at 66 KB a microsecond
// and compute unit whatever the tile (25 bytes a cycle), so wide tiles of few rows are the cheapest that occupy the chip in one
// round; a second round costs more than the first.  Tiles of 32 x 64 / 48 x 64 / 64 x 64 / 80 x 64 / 32 x 32, us, bf16: 64 x 7680 x 2560
// 7.3 / 9.0 / 10.4 / 12.2 / 8.2; 77 x 7680 x 2560 11.7 / 8.9 / 10.6 / 12.4 / 10.1; 128 x 7680 x 2560 12.0 / 14.9 / 10.6 / 12.5 / 12.3;
// 77 x 11008 x 4096 23.4 / 22.6 / 25.6 / 18.5 / 20.5; 64 x 4096 x 4096 8.6 / 10.7 / 12.2 / 15.0 / 7.3.  int8 rows are half the bytes and
// bound by the decode and the chain of a step, 0.5 us and 0.2 a row block; 16 x 64 / 32 x 64 / 48 x 64 / 64 x 64 / 80 x 64, us, tiled:
// 64 x 7680 x 2560 7.8 / 6.9 / 8.5 / 9.3 / 10.8, 128 x 4096 x 11008 19.3 / 14.9 / 18.4 / 20.1 / 24.7, 16 x 11008 x 4096 6.6 / 7.4 / 8.5 / 9.5 / 11.3.
// On tiled int8 weights, from memory, such a launch takes 2 to 14 % longer than that, the more the fuller the chip is.
struct RowsPlan {
    int rb, nacc;
    double us;
};
// Column tiles of an XCD where consecutive ones lie on one XCD, or 0: in launch order
static int rows_per_xcd(int64_t tiles, int64_t blocks) { return blocks > 1 && tiles % 8 != 0 && tiles < 64 ? 0 : (int)ceil_div(tiles, 8); }
static RowsPlan few_rows_plan(bool i8, bool rows, int64_t M, int64_t N, int64_t row_bytes) {
    const int64_t C = gemm_compute_units();
    const double steps = (double)ceil_div(ceil_div(row_bytes, 128), ROWS_WAVES);
    auto price = [&](int rb, int nacc) {
        const int64_t blocks = ceil_div(M, 16 * rb), tiles = ceil_div(N, 16 * nacc), per_xcd = rows_per_xcd(tiles, blocks);
        const double rounds = (double)ceil_div(blocks * tiles, C);
        // Rows that no L2 holds come from behind it, once for each XCD that has a tile of them, at 6 TB/s: 2048 x 512 x 11008 bf16 58 us for
        // 360 MB, 1000 x 256 x 11008 in tiles of 32 columns 29 us for 176 MB.
        const double bytes = (double)M * (double)row_bytes, fetch = bytes > ROWS_L2_BYTES ? 2.0 + (double)std::min<int64_t>(tiles, 8) * bytes / 6.5e6 : 0.0;
        if (i8) {
            // (an XCD's workgroups are on its own compute units: of 5 x 100 some have 65 for 32, three rounds; 224 x 6400 x 11008 47 us)
            const double turns = per_xcd ? (double)ceil_div(per_xcd * blocks, C / 8) : rounds, full = (double)(blocks * tiles) / ((double)C * turns);
            return std::max(fetch, (0.2 + 0.8 * turns) * (2.7 + 0.65 * rb + steps * (0.5 + 0.2 * rb)) * (rows ? 1.0 : 1.02 + 0.12 * full));
        }
        return std::max(fetch, 2.6 + rounds * (rounds > 1 ? 1.45 : 1.0) * (0.7 + steps * ROWS_WAVES * (2048.0 * rb + 256.0 * nacc) / 66000.0));
    };
    static const int cfg[6][2] = {{2, 2}, {1, 4}, {2, 4}, {3, 4}, {4, 4}, {5, 4}};
    auto has = [&](const int* c) { return c[1] == 2 ? !rows && !i8 : c[0] > 1 || i8; };
    RowsPlan best = {0, 0, 0.0};
    for (const auto& c : cfg) {
        const double us = price(c[0], c[1]);
        if (has(c) && (!best.rb || us < best.us)) best = {c[0], c[1], us};
    }
    if (const char* env = option(OPT_ROWS_CFG)) {
        int rb = 0, nacc = 0;
        if (sscanf(env, "%d,%d", &rb, &nacc) == 2)
            for (const auto& c : cfg)
                if (has(c) && c[0] == rb && c[1] == nacc) best = {rb, nacc, 0.0};
    }
    return best;
}
// i8: K int8 values a row, otherwise K 16-bit ones; rows: row-major weights
double few_rows_cost(bool i8, bool rows, int64_t M, int64_t N, int64_t K) { return few_rows_plan(i8, rows, M, N, i8 ? K : 2 * K).us; }

template <int MODE, bool ROWS, int RB, int NACC, bool SW>
static int launch_rows_cfg(RowsParams p, hipStream_t st) {
    const int64_t blocks = ceil_div(p.M, 16 * RB);
    p.tiles = (int)ceil_div(p.N, 16 * NACC);
    p.per_xcd = rows_per_xcd(p.tiles, blocks);
    const dim3 grid((unsigned)(p.per_xcd ? 8 * p.per_xcd : p.tiles), (unsigned)blocks), block(64 * ROWS_WAVES);
    const bool tail = p.row_bytes % 128 != 0 || 4 * p.Kb * (MODE == MODE_I8 ? 1 : 2) < p.row_bytes;
    if (tail) hipLaunchKernelGGL((few_rows_kernel<MODE, ROWS, RB, NACC, SW, true>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((few_rows_kernel<MODE, ROWS, RB, NACC, SW, false>), grid, block, 0, st, p);
    return check_launch("few_rows");
}
template <int MODE, bool ROWS, int RB, int NACC>
static int launch_rows_epi(const RowsParams& p, bool sw, hipStream_t st) {
    if constexpr (MODE != MODE_I8 && !ROWS) {
        if (sw) return launch_rows_cfg<MODE, ROWS, RB, NACC, true>(p, st);
    }
    return launch_rows_cfg<MODE, ROWS, RB, NACC, false>(p, st);
}
template <int MODE, bool ROWS>
static int launch_rows_mode(const RowsParams& p, bool sw, hipStream_t st) {
    const RowsPlan pl = few_rows_plan(MODE == MODE_I8, ROWS, p.M, p.N, p.row_bytes);
    if constexpr (!ROWS && MODE != MODE_I8) {
        if (pl.nacc == 2) return launch_rows_epi<MODE, ROWS, 2, 2>(p, sw, st);
    }
    if constexpr (MODE == MODE_I8) {
        if (pl.rb == 1) return launch_rows_epi<MODE, ROWS, 1, 4>(p, sw, st);
    }
    return pl.rb == 2 ? launch_rows_epi<MODE, ROWS, 2, 4>(p, sw, st) : pl.rb == 3 ? launch_rows_epi<MODE, ROWS, 3, 4>(p, sw, st)
         : pl.rb == 4 ? launch_rows_epi<MODE, ROWS, 4, 4>(p, sw, st) : launch_rows_epi<MODE, ROWS, 5, 4>(p, sw, st);
}

// Rows of whole groups of 16 bytes, 16-byte aligned; row-major weights (tiled = false) 4-byte aligned with N % 4 == 0.  32-bit offsets
// span 80 rows of X, and 32 rows of W_T or the whole copy (below 4 GiB: checked by the caller).
bool few_rows_supported(int64_t N, int64_t row_bytes, const void* X, const void* W, bool tiled) {
    return row_bytes % 16 == 0 && row_bytes >= 16 && row_bytes < (1ll << 24) && N < (1ll << 26) && ((uintptr_t)X) % 16 == 0 &&
           (tiled || (N % 4 == 0 && ((uintptr_t)W) % 4 == 0));
}

// X: M rows of K values (Kw: the weights' K where the rows are longer, zeros behind it; 0: K); int8 ones in operand order, with s_x.
// epi_op: 0, or EPI_SWIGLU_PAIRS (16-bit rows, W_LAYOUT_TILED in pair order, N % 32 == 0, no residual; Y is [M, N / 2])
int launch_few_rows(int mode, const void* X, const float* s_x, const uint8_t* W, int w_layout, const Epilogue& epi, void* Y, int y_dtype,
                    int32_t* acc_out, int64_t M, int64_t N, int64_t K, int epi_op, hipStream_t st, int64_t Kw) {
    RowsParams p = {};
    p.X = (const uint8_t*)X; p.W = W; p.Y = Y; p.epi = epi; p.y_dtype = y_dtype; p.s_x = s_x; p.acc_out = acc_out;
    p.row_bytes = mode == MODE_I8 ? K : 2 * K;
    p.M = M; p.N = N; p.Kb = ceil_div(Kw ? Kw : K, 4);
    p.wsteps = (int)ceil_div(K, 64);
    p.tiles16 = tiles16_arg(N, w_layout);
    const bool sw = epi_op == EPI_SWIGLU_PAIRS;
    if (layout_tiled(w_layout))
        return mode == MODE_I8 ? launch_rows_mode<MODE_I8, false>(p, sw, st) : mode == MODE_F16 ? launch_rows_mode<MODE_F16, false>(p, sw, st)
                                                                                              : launch_rows_mode<MODE_BF16, false>(p, sw, st);
    return mode == MODE_I8 ? launch_rows_mode<MODE_I8, true>(p, sw, st) : mode == MODE_F16 ? launch_rows_mode<MODE_F16, true>(p, sw, st)
                                                                                         : launch_rows_mode<MODE_BF16, true>(p, sw, st);
}

}  // namespace bt
