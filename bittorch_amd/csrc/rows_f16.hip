// fp16 / bf16 x decode-tiled ternary weights for a few tens of rows: short prompts, batched decode steps.
//
// Arithmetic as in gemm_f16.hip.  Between the streaming kernel, which decodes the weights again for every 16 rows, and the tiled GEMM,
// whose tiles of 256 columns are too few to occupy the chip: a workgroup owns 16 RB rows x 16 NACC columns, so that a weight is
// decoded once for all of the rows, and its eight waves split K.  Every wave works alone on its run of 64-wide steps: the rows come
// eight lanes to a row (whole cache lines; a lane a row would take the cache four times as long), D steps ahead, and pass
// through the wave's own LDS into matrix fragments, without a barrier.  The waves' sums meet in LDS, in wave order.
#include <cstdio>

#include "row_math.h"

namespace bt {

struct RowsParams {
    const uint16_t* X;    // [M, K] fp16 or bf16 bits
    const uint8_t* W;     // the decode-tiled copy
    int64_t K, M, N;      // K: length of an activation row (a multiple of 8)
    int wsteps;           // 64-wide steps of the copy
    int tiles16;          // as in tiles16_arg
    int tiles;            // column tiles
    int per_xcd;          // column tiles per XCD (grid.x = 8 * per_xcd); 0: tiles in launch order
    void* Y;              // [M, N], SW: [M, N / 2]
    Epilogue epi;
};

constexpr int ROWS_WAVES = 8;
// Row blocks whose sums a wave hands over at once, and the LDS of a wave: a step's rows, then those sums.
constexpr int rows_pass(int RB, int NACC) { return RB > 4 && NACC == 4 ? (RB + 1) / 2 : RB; }
constexpr int rows_wave_bytes(int RB, int NACC) {
    return std::max(RB * 2048, rows_pass(RB, NACC) * NACC * 1024);
}
constexpr int rows_depth(int RB) { return RB <= 3 ? 3 : 2; }  // steps whose rows are on their way (two: 256 x 2560 x 6912 20.9 us, three: 18.0)

// SW: the SwiGLU output stage on a copy in gate/up pair order (NACC even: tiles 2 i and 2 i + 1 are the gate's and up's)
// TAIL: K % 64 != 0
template <int MODE, int RB, int NACC, bool SW, bool TAIL>
__global__ __launch_bounds__(64 * ROWS_WAVES, 2) void rows_f16_kernel(RowsParams p) {
    constexpr int D = rows_depth(RB), AL = 2 * RB, YDT = MODE == MODE_F16 ? BT_F16 : BT_BF16;
    __shared__ __attribute__((aligned(16))) uint8_t lds_all[ROWS_WAVES * rows_wave_bytes(RB, NACC)];
    // consecutive tiles on one XCD
    const int tile = p.per_xcd ? (int)(blockIdx.x & 7) * p.per_xcd + (int)(blockIdx.x >> 3) : (int)blockIdx.x;
    if (tile >= p.tiles) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 15, g = lane >> 4;
    uint8_t* const lds = lds_all + wave * rows_wave_bytes(RB, NACC);
    const int64_t m0 = (int64_t)blockIdx.y * (16 * RB);
    const int rows_left = (int)((p.M - m0 < 16 * RB) ? p.M - m0 : 16 * RB);
    const int nst = (int)((p.K + 63) >> 6), run = (nst + ROWS_WAVES - 1) / ROWS_WAVES;
    const int st0 = min(wave * run, nst), st1 = min(nst, st0 + run);

    // Load b brings rows 8 b .. +7 of the step, piece lane % 8 of 16 bytes; rows past the end repeat the last one (never stored).
    const uint8_t* const x0 = (const uint8_t*)(p.X + m0 * p.K);
    const uint32_t piece = lane & 7;
    uint32_t a_off[AL];
#pragma unroll
    for (int b = 0; b < AL; b++) {
        const int row = 8 * b + (lane >> 3);
        a_off[b] = (uint32_t)(row < rows_left ? row : rows_left - 1) * (uint32_t)p.K * 2u + 16u * piece;
    }
    uint32_t w_off[NACC];
#pragma unroll
    for (int t = 0; t < NACC; t++) w_off[t] = ((uint32_t)stored_tile16(tile * NACC + t, p.tiles16) * (uint32_t)p.wsteps * 64u + (uint32_t)lane) * 4u;
    // a row of a step is 128 bytes of LDS, piece q of row r at place q ^ f(r): no bank twice (fd_place of gemm_f16.hip)
    const uint32_t put = (uint32_t)(lane >> 3) * 128u, put_at[2] = {put + 16u * (piece ^ ((lane >> 4) & 1u)), put + 16u * (piece ^ (((lane >> 4) & 1u) | 6u))};
    const uint32_t at_j = ((j >> 1) & 1u) | ((j >> 3) & 1u) * 6u;
    const uint32_t frag_at[2] = {128u * j + 16u * ((2u * g) ^ at_j), 128u * j + 16u * ((2u * g + 1u) ^ at_j)};

    u32x4 xa[D][AL];
    uint32_t raw[D][NACC];
    const bool past = TAIL && 64 * (nst - 1) + 8 * (int)piece >= (int)p.K;  // this lane's pieces of the partial step lie past the end
    const uint32_t kept = past ? 0u : 0xFFFFFFFFu;
    const u32x4 keep = {kept, kept, kept, kept};
    auto load = [&](int f, int s) __attribute__((always_inline)) {  // s uniform
        const uint8_t *wb = p.W + (int64_t)s * 256, *xb = x0 + (int64_t)s * 128;
#pragma unroll
        for (int t = 0; t < NACC; t++) raw[f][t] = ldw_nt(wb + w_off[t]);
        if (TAIL && s == nst - 1) {  // (uniform)
#pragma unroll
            for (int b = 0; b < AL; b++) xa[f][b] = *(const u32x4*)(past ? x0 + (a_off[b] - 16u * piece) : xb + a_off[b]);
        } else {
#pragma unroll
            for (int b = 0; b < AL; b++) xa[f][b] = *(const u32x4*)(xb + a_off[b]);
        }
    };
    v4f acc[RB][NACC];
#pragma unroll
    for (int b = 0; b < RB; b++)
#pragma unroll
        for (int t = 0; t < NACC; t++) acc[b][t] = v4f{0.f, 0.f, 0.f, 0.f};
    constexpr uint32_t LUT = (MODE == MODE_F16) ? LUT_F16_ONE : LUT_BF16_TWO;
    auto step = [&](int f, int s) __attribute__((always_inline)) {
        if (TAIL && s == nst - 1) {  // (uniform)
#pragma unroll
            for (int b = 0; b < AL; b++) xa[f][b] &= keep;
        }
#pragma unroll
        for (int b = 0; b < AL; b++) *(u32x4*)(lds + 1024 * b + put_at[b & 1]) = xa[f][b];
        // decode: see gemm_f16.hip
        u32x4 w[2][NACC];
#pragma unroll
        for (int t = 0; t < NACC; t++) {
            uint32_t hi[4];
#pragma unroll
            for (int e = 0; e < 4; e++) hi[e] = perm(0u, LUT, (raw[f][t] >> (2 * e)) & 0x03030303u);
#pragma unroll
            for (int x = 0; x < 8; x++) {
                const int r = x >> 1, e = 2 * (x & 1);
                w[x >> 2][t][x & 3] = perm(hi[e + 1], hi[e], ((uint32_t)(4 + r) << 24) | (0x0Cu << 16) | ((uint32_t)r << 8) | 0x0Cu);
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
                    if constexpr (MODE == MODE_F16)
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
        v4f v = *(const v4f*)(lds_all + at * 16);
#pragma unroll
        for (int w = 1; w < ROWS_WAVES; w++) v += *(const v4f*)(lds_all + w * rows_wave_bytes(RB, NACC) + at * 16);
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
            for (int t = 0; t < NACC; t++) *(v4f*)(lds + (((b - b0) * NACC + t) * 64 + lane) * 16) = acc[b][t];
        __syncthreads();
        const int sets = std::min(PASS, RB - b0) * COLS;
        for (int set = wave; set < sets; set += ROWS_WAVES) {  // (uniform)
            const int b = set / COLS, t = set - b * COLS, row0 = 16 * (b0 + b) + 4 * g;
            const int64_t col = ((int64_t)tile * COLS + t) * 16 + j;
            if (col >= Ny || row0 >= rows_left) continue;
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

// Which tile, and what the launch takes in microseconds.  A workgroup reads its rows' whole length from L2, at 66 KB a microsecond
// and compute unit whatever the tile (25 bytes a cycle), so wide tiles of few rows are the cheapest that occupy the chip in one
// round; a second round costs more than the first.  Tiles of 32 x 64 / 48 x 64 / 64 x 64 / 80 x 64 / 32 x 32, us, bf16: 64 x 7680 x 2560
// 7.3 / 9.0 / 10.4 / 12.2 / 8.2; 77 x 7680 x 2560 11.7 / 8.9 / 10.6 / 12.4 / 10.1; 128 x 7680 x 2560 12.0 / 14.9 / 10.6 / 12.5 / 12.3;
// 77 x 11008 x 4096 23.4 / 22.6 / 25.6 / 18.5 / 20.5; 64 x 4096 x 4096 8.6 / 10.7 / 12.2 / 15.0 / 7.3.
struct RowsPlan {
    int rb, nacc;
    double us;
};
static RowsPlan rows_f16_plan(int64_t M, int64_t N, int64_t K) {
    const int64_t C = gemm_compute_units();
    const double steps = (double)ceil_div(ceil_div(K, 64), ROWS_WAVES);
    auto price = [&](int rb, int nacc) {
        const double rounds = (double)ceil_div(ceil_div(M, 16 * rb) * ceil_div(N, 16 * nacc), C);
        return 2.6 + rounds * (rounds > 1 ? 1.35 : 1.0) * (0.7 + steps * ROWS_WAVES * (2048.0 * rb + 256.0 * nacc) / 66000.0);
    };
    static const int cfg[5][2] = {{2, 2}, {2, 4}, {3, 4}, {4, 4}, {5, 4}};
    RowsPlan best = {0, 0, 0.0};
    for (const auto& c : cfg) {
        const double us = price(c[0], c[1]);
        if (!best.rb || us < best.us) best = {c[0], c[1], us};
    }
    if (const char* env = option(OPT_ROWS_CFG)) {
        int rb = 0, nacc = 0;
        if (sscanf(env, "%d,%d", &rb, &nacc) == 2)
            for (const auto& c : cfg)
                if (c[0] == rb && c[1] == nacc) best = {rb, nacc, 0.0};
    }
    return best;
}
double rows_f16_cost(int64_t M, int64_t N, int64_t K) { return rows_f16_plan(M, N, K).us; }

template <int MODE, int RB, int NACC, bool SW>
static int launch_rows_cfg(RowsParams p, hipStream_t st) {
    const int64_t blocks = ceil_div(p.M, 16 * RB);
    p.tiles = (int)ceil_div(p.N, 16 * NACC);
    p.per_xcd = blocks > 1 && p.tiles % 8 != 0 && p.tiles < 64 ? 0 : (int)ceil_div(p.tiles, 8);
    const dim3 grid((unsigned)(p.per_xcd ? 8 * p.per_xcd : p.tiles), (unsigned)blocks), block(64 * ROWS_WAVES);
    if (p.K % 64 != 0) hipLaunchKernelGGL((rows_f16_kernel<MODE, RB, NACC, SW, true>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((rows_f16_kernel<MODE, RB, NACC, SW, false>), grid, block, 0, st, p);
    return check_launch("rows_f16");
}
template <int MODE, int RB, int NACC>
static int launch_rows_epi(const RowsParams& p, bool sw, hipStream_t st) {
    return sw ? launch_rows_cfg<MODE, RB, NACC, true>(p, st) : launch_rows_cfg<MODE, RB, NACC, false>(p, st);
}
template <int MODE>
static int launch_rows_mode(const RowsParams& p, RowsPlan pl, bool sw, hipStream_t st) {
    if (pl.nacc == 2) return launch_rows_epi<MODE, 2, 2>(p, sw, st);
    return pl.rb == 2 ? launch_rows_epi<MODE, 2, 4>(p, sw, st) : pl.rb == 3 ? launch_rows_epi<MODE, 3, 4>(p, sw, st)
         : pl.rb == 4 ? launch_rows_epi<MODE, 4, 4>(p, sw, st) : launch_rows_epi<MODE, 5, 4>(p, sw, st);
}

bool rows_f16_supported(int64_t N, int64_t K, const void* X) {
    return K % 8 == 0 && K >= 8 && K < (1ll << 23) && N < (1ll << 30) && ((uintptr_t)X) % 16 == 0;
}

// epi_op: 0, or EPI_SWIGLU_PAIRS (W_LAYOUT_TILED in pair order, N % 32 == 0, no residual; Y is [M, N / 2])
int launch_rows_f16(int mode, const void* X, const uint8_t* W, int w_layout, const Epilogue& epi, void* Y, int64_t M, int64_t N,
                    int64_t K, int epi_op, hipStream_t st) {
    RowsParams p = {};
    p.X = (const uint16_t*)X; p.W = W; p.Y = Y; p.epi = epi;
    p.M = M; p.N = N; p.K = K;
    p.wsteps = (int)ceil_div(K, 64);
    p.tiles16 = tiles16_arg(N, w_layout);
    const RowsPlan pl = rows_f16_plan(M, N, K);
    const bool sw = epi_op == EPI_SWIGLU_PAIRS;
    return mode == MODE_F16 ? launch_rows_mode<MODE_F16>(p, pl, sw, st) : launch_rows_mode<MODE_BF16>(p, pl, sw, st);
}

}  // namespace bt
