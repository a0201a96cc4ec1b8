// Weight gradient of 16-bit layers on gfx950: dW[n, k] = scale[n] * sum_m dY[m, n] X[m, k], dY [M, N] and X [M, K] fp16 or
// bf16 (the straight-through estimator of bittorch/nn/ternary_linear_cuda.py:73-111), fp32 sums, the scale and the masters'
// dtype in the epilogue.
//
// The contraction runs over the rows of both operands, so an MFMA fragment, 8 consecutive m of one column, is a column of a
// row-major matrix.  Lane (i, g) of a wave loads columns 8 i .. +7 of rows 8 g .. +7, eight 16-byte loads; 32 byte permutes
// turn them into the fragments of eight 16-column blocks, block t holding the columns 8 i + t, and go to LDS in fragment
// order: no address of a wave's LDS access meets another's bank, and a lane's outputs are eight consecutive k of a row.
//
// A 256-thread workgroup owns 256 x 256 outputs, a wave 128 x 128 of them (256 accumulators a lane, one wave a SIMD): a stage
// of 32 m is 64 MFMAs a wave (1024 cycles) for 64 KiB read from and 32 KiB written to LDS per workgroup, and an XCD's 32
// workgroups read 12 strips of 256 columns.  The matrix cores are busy for 62 % of the time (69 % in
// one long round), and the rest goes to the issue of a lone wave's other instructions.  4096 x 11008 x 4096 (rows, dY's columns,
// X's), fp16 to fp32, 345 us = 1.07 PFLOP/s, the last of three rounds of tiles two thirds full; the vendor's product (393 us in a
// profile) and the pass that scaled and widened its result 449.  The same stages make tiles of 128 x 128 for outputs that would
// leave compute units idle: a stage is 64 m, half of them for each wave of an operand, and a wave 64 x 64 outputs (768 x 768 of 300
// rows 10.2 us, 17.5 in tiles of 256).
#include "bt_common.h"

namespace bt {

struct GradW16Params {
    const uint16_t* G;    // [M, N]
    const uint16_t* X;    // [M, K]
    int64_t M, N, K;
    int tiles_n, tiles_k; // tiles of 32 T x 32 T
    int whole;            // tiles per XCD that sum over all rows
    int tail_from;        // tiles from this one on are summed in parts of the rows,
    int splits;           // so many (1: there are none),
    int per_xcd_tail;     // so many (tile, part) per XCD (grid = 8 * (whole + per_xcd_tail)),
    int64_t part_rows;    // of so many rows, a multiple of 128 (the last part: what is left),
    int long_first;       // 1: two parts of unequal length, an XCD's long ones in front of its short ones,
    float* part;          // into [part][tile][accumulator][thread]
    int scale_bcast, scale_dtype;
    const void* scale;    // [N] or one entry
    void* out;            // [N, K]
};

// first row and column of a tile of 32 T x 32 T outputs
template <int T>
__device__ __forceinline__ void grad_w16_tile(uint32_t lin, uint32_t tiles_n, uint32_t tiles_k, int64_t& n0, int64_t& k0) {
    constexpr uint32_t GM = 4;
    const uint32_t group = lin / (GM * tiles_k), first_n = group * GM;
    const uint32_t gm = (tiles_n - first_n < GM) ? tiles_n - first_n : GM;
    const uint32_t in_group = lin - group * GM * tiles_k, tk = in_group / gm;
    n0 = (int64_t)(first_n + (in_group - tk * gm)) * (32 * T);
    k0 = (int64_t)tk * (32 * T);
}

// One row's sums of `count` consecutive columns: each is rounded as the 16-bit product of two matrices would be, scaled and
// rounded again, what the unfused operations give.
template <int DT, bool OUT32, int COUNT>
__device__ __forceinline__ void grad_w16_store(void* out, int64_t at, const float (&sum)[COUNT], float scale) {
    const float s16 = round_to_dtype(scale, DT);
    float v[COUNT];
#pragma unroll
    for (int b = 0; b < COUNT; b++) v[b] = round_to_dtype(__fmul_rn(round_to_dtype(sum[b], DT), s16), DT);
    if constexpr (OUT32) {
#pragma unroll
        for (int b = 0; b < COUNT; b += 4) *(v4f*)((float*)out + at + b) = v4f{v[b], v[b + 1], v[b + 2], v[b + 3]};
    } else {
        uint32_t d[COUNT / 2];
#pragma unroll
        for (int b = 0; b < COUNT / 2; b++) {
            const uint16_t l16 = DT == BT_F16 ? f32_to_f16_bits(v[2 * b]) : f32_to_bf16_bits(v[2 * b]);
            const uint16_t h16 = DT == BT_F16 ? f32_to_f16_bits(v[2 * b + 1]) : f32_to_bf16_bits(v[2 * b + 1]);
            d[b] = (uint32_t)l16 | (uint32_t)h16 << 16;
        }
        if constexpr (COUNT == 8) *(u32x4*)((uint16_t*)out + at) = u32x4{d[0], d[1], d[2], d[3]};
        else *(u32x2*)((uint16_t*)out + at) = u32x2{d[0], d[1]};
    }
}

template <int MODE, bool OUT32, int T>
__global__ __launch_bounds__(256, 1) void grad_w16_kernel(GradW16Params p) {
    constexpr int DT = MODE == MODE_F16 ? BT_F16 : BT_BF16;
    constexpr int SROWS = T == 8 ? 32 : 64;  // rows of a stage
    constexpr uint32_t BUF = 32768;  // a stage in LDS: [G, X][half][block t][lane] x 16 bytes
    __shared__ __attribute__((aligned(16))) uint8_t lds[2 * BUF];
    // each XCD takes a contiguous run of tiles, walked in groups of four row tiles, so that its L2 holds what it shares
    const uint32_t tiles_n = (uint32_t)p.tiles_n, tiles_k = (uint32_t)p.tiles_k, idx = blockIdx.x >> 3;
    const bool tail = idx >= (uint32_t)p.whole;  // (uniform)
    uint32_t lin, item = 0, part = 0;
    if (tail) {
        const uint32_t tiles = tiles_n * tiles_k - (uint32_t)p.tail_from;
        const uint32_t j = idx - (uint32_t)p.whole, per_xcd = (uint32_t)p.per_xcd_tail;
        if (p.long_first) {  // (uniform)
            const uint32_t half = per_xcd / 2, tile = (blockIdx.x & 7u) * half + (j < half ? j : j - half);
            if (tile >= tiles) return;
            part = j < half ? 0u : 1u;
            item = part * tiles + tile;
        } else {
            item = (blockIdx.x & 7u) * per_xcd + j;
            if (item >= tiles * (uint32_t)p.splits) return;
            part = item / tiles;
        }
        lin = (uint32_t)p.tail_from + (item - part * tiles);
    } else {
        lin = (blockIdx.x & 7u) * (uint32_t)p.whole + idx;
        if (lin >= (uint32_t)p.tail_from) return;
    }
    const int64_t m_first = part * p.part_rows, rows = tail ? min(p.part_rows, p.M - m_first) : p.M;
    int64_t n0, k0;
    grad_w16_tile<T>(lin, tiles_n, tiles_k, n0, k0);

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 15, g = lane >> 4;
    const int hi = wave >> 1, lo = wave & 1;

    // Loads: waves 0 and 1 the halves of G's stage, 2 and 3 of X's (T == 8: of its 256 columns, else of its 64 rows).  The
    // buffer ends with the matrix, so rows past M are zeros; columns past the end read the next row and only reach outputs
    // that are not stored.
    const int64_t ld = hi ? p.K : p.N;
    const uint8_t* src = (const uint8_t*)((hi ? p.X : p.G) + m_first * ld);
    const int64_t step_bytes = 2 * SROWS * ld;
    int64_t left = rows * ld * 2;
    uint32_t voff[8];
    const uint32_t col = (uint32_t)(hi ? k0 : n0) + (T == 8 ? 128u * lo : 0u) + 8u * i, row = 8u * g + (T == 8 ? 0u : 32u * lo);
#pragma unroll
    for (int e = 0; e < 8; e++) voff[e] = ((row + e) * (uint32_t)ld + col) * 2u;
    u32x4 r[4][8];
    auto load = [&](int set, int e) {
        const uint32_t bytes = left > 0x7fffffff ? 0x7fffffffu : left > 0 ? (uint32_t)left : 0u;
        r[set][e] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
            __builtin_amdgcn_make_buffer_rsrc((void*)src, 0, bytes, 0x00027000), voff[e], 0, 0));
    };
    auto advance = [&]() { src += step_bytes; left -= step_bytes; };
    uint8_t* const w_at = lds + 16384 * hi + 8192 * lo + 16 * lane;
    u32x4 frag;
    auto permute = [&](int set, int t, int q) {  // dword q of block t
        frag[q] = perm(r[set][2 * q + 1][t >> 1], r[set][2 * q][t >> 1], (t & 1) ? 0x07060302u : 0x05040100u);
    };
    auto write = [&](int buf, int t) { *(u32x4*)(w_at + buf * BUF + 1024 * t) = frag; };

    v4f acc[T][T];
#pragma unroll
    for (int a = 0; a < T; a++)
#pragma unroll
        for (int b = 0; b < T; b++) acc[a][b] = v4f{0.f, 0.f, 0.f, 0.f};
    u32x4 fa[8], fb[8];
    // T == 8: fragment t is block t of the wave's 128 columns; else block t % 4 of its four, of the stage's half t / 4
    const uint8_t* const a_at = lds + (T == 8 ? 8192 : 4096) * hi + 16 * lane;
    const uint8_t* const b_at = lds + 16384 + (T == 8 ? 8192 : 4096) * lo + 16 * lane;
    auto at = [](int buf, int t) { return buf * BUF + (T == 8 ? 1024 * t : 8192 * (t >> 2) + 1024 * (t & 3)); };
    auto read_a = [&](int buf, int t) { fa[t] = *(const u32x4*)(a_at + at(buf, t)); };
    auto read_b = [&](int buf, int t) { fb[t] = *(const u32x4*)(b_at + at(buf, t)); };
    auto mfma = [&](int a, int b) {
        v4f& c = acc[a % T][b % T];
        if constexpr (MODE == MODE_F16) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(fa[a]), "v"(fb[b]));
        else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(fa[a]), "v"(fb[b]));
    };

#pragma unroll
    for (int s = 0; s < 4; s++) {
#pragma unroll
        for (int e = 0; e < 8; e++) load(s, e);
        advance();
    }
    auto put = [&](int set, int buf, int t) {
#pragma unroll
        for (int q = 0; q < 4; q++) permute(set, t, q);
        write(buf, t);
    };
#pragma unroll
    for (int t = 0; t < 8; t++) put(0, 0, t);
#pragma unroll
    for (int e = 0; e < 4; e++) load(0, e);
#pragma unroll
    for (int t = 0; t < 4; t++) put(1, 1, t);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int t = 0; t < 4; t++) { read_a(0, t); read_b(0, t); }

    // Stage s (set and buffer constants of its place in the loop).  Four runs of 16 MFMAs go round the quarters of the wave's
    // tile, the next stage the other way round, so that one set of fragments serves: each quarter of them is read behind the
    // last run that used it, one run ahead of its own first.  A stage's blocks 0 to 3 are written behind the barrier of the
    // stage before the last, blocks 4 to 7 in front of the last one's; its loads are issued three stages before that.
    auto stage = [&](auto SC) {
        constexpr int S = decltype(SC)::value, B = S & 1, F = B ? 4 : 0, O = 4 - F;  // first and other half of X's blocks
        constexpr int S1 = (S + 1) & 3, S2 = (S + 2) & 3;
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (T == 4) {  // two runs of 16, a half of the rows each; the same order of writes and loads
#pragma unroll
            for (int c = 0; c < 16; c++) {
                mfma(c >> 2, c & 3);
                if (c % 4 == 1) read_b(B, 4 + c / 4);
                if (c % 4 == 3) read_a(B, 4 + c / 4);
                if (c % 4 == 2) load(S, 4 + c / 4);
                permute(S1, 4 + (c >> 2), c & 3);
                if (c % 4 == 3) write(1 - B, 4 + (c >> 2));
                __builtin_amdgcn_sched_barrier(0);
            }
            advance();
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int c = 0; c < 16; c++) {
                mfma(4 + (c >> 2), 4 + (c & 3));
                if (c % 4 == 1) read_b(1 - B, c / 4);
                if (c % 4 == 3) read_a(1 - B, c / 4);
                if (c % 4 == 2) load(S1, c / 4);
                permute(S2, c >> 2, c & 3);
                if (c % 4 == 3) write(B, c >> 2);
                __builtin_amdgcn_sched_barrier(0);
            }
            return;
        }
#pragma unroll
        for (int c = 0; c < 16; c++) {
            mfma(c >> 2, F + (c & 3));
            if (c < 8 && c % 2 == 0) read_b(B, O + c / 2);
            if (c == 5 || c == 13) load(S, 4 + c / 8);
            permute(S1, 4 + (c >> 3), (c >> 1) & 3);  // (the second of a pair repeats the first: no instruction)
            if ((c & 7) == 7) write(1 - B, 4 + (c >> 3));
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int c = 0; c < 16; c++) {
            mfma(c >> 2, O + (c & 3));
            if (c < 8 && c % 2 == 0) read_a(B, 4 + c / 2);
            if (c == 5 || c == 11) load(S, 6 + c / 8);
            if (c == 12) advance();
            if (c < 8) {
                permute(S1, 6 + (c >> 2), c & 3);
                if ((c & 3) == 3) write(1 - B, 6 + (c >> 2));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 16; c++) {
            mfma(4 + (c >> 2), O + (c & 3));
            if (c < 8 && c % 2 == 0) read_a(1 - B, c / 2);
            if (c == 5 || c == 13) load(S1, c / 8);
            if (c >= 8) {
                permute(S2, (c - 8) >> 2, c & 3);
                if ((c & 3) == 3) write(B, (c - 8) >> 2);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int c = 0; c < 16; c++) {
            mfma(4 + (c >> 2), F + (c & 3));
            if (c < 8 && c % 2 == 0) read_b(1 - B, O + c / 2);
            if (c == 5 || c == 13) load(S1, 2 + c / 8);
            if (c < 8) {
                permute(S2, 2 + (c >> 2), c & 3);
                if ((c & 3) == 3) write(B, 2 + (c >> 2));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    asm volatile("s_nop 7" ::: "memory");  // (nor that they read the accumulators cleared above)
    __builtin_amdgcn_sched_barrier(0);
    for (int64_t m = 0; m < rows; m += 4 * SROWS) {  // (stages past the last row are zeros)
        stage(std::integral_constant<int, 0>{});
        stage(std::integral_constant<int, 1>{});
        stage(std::integral_constant<int, 2>{});
        stage(std::integral_constant<int, 3>{});
    }
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // (the compiler does not see the matrix instructions' latency)
    __builtin_amdgcn_sched_barrier(0);

    if (tail) {  // (uniform)
        v4f* o = (v4f*)p.part + (int64_t)item * (256 * T * T) + threadIdx.x;
#pragma unroll
        for (int a = 0; a < T; a++)
#pragma unroll
            for (int b = 0; b < T; b++) o[256 * (T * a + b)] = acc[a][b];
        return;
    }
    // lane (i, g): T == 8: rows 8 (4 g + c) + a of the wave's 128, columns 8 i .. +7; T == 4: rows 8 (4 g + c) + 4 hi + a of the
    // tile's 128, columns 8 i + 4 lo .. +3
    const int64_t k = k0 + (T == 8 ? 128 : 4) * lo + 8 * i;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const int64_t n = n0 + (T == 8 ? 128 : 4) * hi + 8 * (4 * g + c);
        if (n >= p.N || k >= p.K) continue;
        float sc[T];
#pragma unroll
        for (int a = 0; a < T; a++) sc[a] = load_elem_rt(p.scale, p.scale_dtype, p.scale_bcast ? 0 : n + a);
#pragma unroll
        for (int a = 0; a < T; a++) {
            float v[T];
#pragma unroll
            for (int b = 0; b < T; b++) v[b] = acc[a][b][c];
            grad_w16_store<DT, OUT32>(p.out, (n + a) * p.K + k, v, sc[a]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// The tiles summed in parts: a thread adds the parts of four of an accumulator row's column blocks, in order, and finishes
// their 4 x 4 outputs.  Bound by reading the parts.
template <int MODE, bool OUT32, int T>
__global__ __launch_bounds__(256) void grad_w16_reduce_kernel(GradW16Params p) {
    constexpr int DT = MODE == MODE_F16 ? BT_F16 : BT_BF16;
    constexpr uint32_t H = T / 4;
    const uint32_t tiles = (uint32_t)(p.tiles_n * p.tiles_k - p.tail_from);
    const uint32_t tile = blockIdx.x / (T * H), a = (blockIdx.x / H) % T, h = blockIdx.x % H, tid = threadIdx.x;
    int64_t n0, k0;
    grad_w16_tile<T>((uint32_t)p.tail_from + tile, (uint32_t)p.tiles_n, (uint32_t)p.tiles_k, n0, k0);
    const uint32_t i = tid & 15, g = (tid >> 4) & 3, lo = (tid >> 6) & 1, hi = tid >> 7;
    const v4f* src = (const v4f*)p.part + (int64_t)tile * (256 * T * T) + 256 * (T * a + 4 * h) + tid;
    v4f sum[4];
#pragma unroll
    for (int b = 0; b < 4; b++) sum[b] = src[256 * b];
#pragma unroll 4
    for (int s = 1; s < p.splits; s++) {
        src += (int64_t)tiles * (256 * T * T);
#pragma unroll
        for (int b = 0; b < 4; b++) sum[b] += src[256 * b];
    }
    const int64_t k = k0 + (T == 8 ? 128 : 4) * lo + 8 * i + 4 * h;
    if (k >= p.K) return;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const int64_t n = n0 + (T == 8 ? 128 : 4) * hi + 8 * (4 * g + c) + a;
        if (n >= p.N) continue;
        const float v[4] = {sum[0][c], sum[1][c], sum[2][c], sum[3][c]};
        grad_w16_store<DT, OUT32>(p.out, n * p.K + k, v, load_elem_rt(p.scale, p.scale_dtype, p.scale_bcast ? 0 : n));
    }
}

// Tiles of 256 or of 128 (T = 8, 4): whole rounds of a tile for each compute unit, and what remains as one round more, or in
// parts of the rows where that takes less.  Parts of equal length fill what would be idle when at most half of the compute units
// have a tile.  With some more tiles than that, each is cut in two parts of unequal length: an XCD starts its long parts, the
// compute units left over take its short ones, two in turn at most, and the lengths are chosen for both to end together (three
// and more in turn are no better: their rows are no longer those that the long parts read, 16384 x 3584 x 3584 390 / 435 us).  Priced in microseconds, f
// the share of compute units that a round fills (one wave a SIMD leaves clock and memory to the others), by the measurements of
// 112 sizes, most of them within 5 %:
//   a round   5.4 + 10 f + (0.0183 + 0.0055 f) rows for tiles of 256, 1.2 + 4.5 f + (0.0073 + 0.0018 f) rows for tiles of 128
//   parts     5 + 0.11 or 2.5 + 0.04 a part in place of the constant: writing the sums and adding them up
// Measured, bf16 to fp32, tiles of 256 whole / in parts / tiles of 128 / the vendor's product with scale_widen_kernel behind it
// (the vendor's takes up to 1.6 times as long at neighbouring sizes): 300 x 768 x 768 17.9 / 16.4 / 10.3 / 13.1; 2048 x 2048 x 2048
// 53.2 / 45.6 / 29.3 / 37.0; 4096 x 2560 x 2560 96.8 / 78.5 / 83.2 / 81.8; 4096 x 3584 x 3584 111 / - / 143 / 141;
// 4096 x 2048 x 4096 97.2 / 89.2 / 88.4 / 84.0; in two unequal parts, 8192 x 3072 x 3072 188 / 162 / 191 / 176 and
// 16384 x 3072 x 3072 348 / 291 / 373 / 327.
struct GradW16Plan { int T; int64_t tiles, tail, splits, part_rows; bool long_first; double us; };
static GradW16Plan grad_w16_plan(int64_t M, int64_t N, int64_t K) {
    GradW16Plan best = {};
    const int64_t C = gemm_compute_units();
    for (int T = 8; T >= 4; T -= 4) {
        const int64_t side = 32 * T, unit = T == 8 ? 128 : 256;  // rows of four stages
        auto rows_us = [&](int64_t wgs, int64_t rows) {
            const double fill = (double)wgs / (double)C;
            return (T == 8 ? 0.0183 + 0.0055 * fill : 0.0073 + 0.0018 * fill) * (double)(ceil_div(rows, unit) * unit);
        };
        auto round_us = [&](int64_t wgs) {
            const double fill = (double)wgs / (double)C;
            return (T == 8 ? 5.4 + 10.0 * fill : 1.2 + 4.5 * fill) + rows_us(wgs, M);
        };
        auto parts_us = [&](int64_t parts) { return T == 8 ? 5.0 + 0.11 * (double)parts : 2.5 + 0.04 * (double)parts; };
        GradW16Plan r = {T, ceil_div(N, side) * ceil_div(K, side), 0, 1, M, false, 0.0};
        const int64_t rounds = r.tiles / C, rem = r.tiles % C;
        const double whole = 5.0 + (double)rounds * round_us(C);
        r.us = whole + (rem ? round_us(rem) : 0.0);
        auto consider = [&](int64_t rows, bool long_first, double us) {
            const int64_t splits = ceil_div(M, rows);
            if (splits > 1 && us < r.us) { r.us = us; r.tail = rem; r.splits = splits; r.part_rows = rows; r.long_first = long_first; }
        };
        for (int64_t want = 2; rem && want <= std::min<int64_t>(C / rem, ceil_div(M, unit)); want++) {
            const int64_t rows = ceil_div(ceil_div(M, want), unit) * unit, parts = rem * ceil_div(M, rows);
            consider(rows, false, whole + parts_us(parts) + rows_us(parts, rows));
        }
        // an XCD's C / 8 compute units: `held` with a long part, `left` for as many short ones, `turns` each at most
        const int64_t held = ceil_div(rem, 8), left = C / 8 - held;
        if (T == 8 && 2 * rem > C && 2 * left >= held) {
            const int64_t turns = ceil_div(held, left), rows = ceil_div(ceil_div(M * turns, turns + 1), unit) * unit;
            consider(rows, true, whole + parts_us(2 * rem) + rows_us(C, rows));
        }
        if (!best.T || r.us < best.us) best = r;
    }
    return best;
}

template <int MODE, bool OUT32, int T>
static void launch_grad_w16_tiles(const GradW16Params& p, int64_t tail, hipStream_t st) {
    hipLaunchKernelGGL((grad_w16_kernel<MODE, OUT32, T>), dim3((unsigned)(8 * (p.whole + p.per_xcd_tail))), dim3(256), 0, st, p);
    if (tail) hipLaunchKernelGGL((grad_w16_reduce_kernel<MODE, OUT32, T>), dim3((unsigned)(T * T / 4 * tail)), dim3(256), 0, st, p);
}
template <int MODE, bool OUT32>
static void launch_grad_w16(const GradW16Params& p, const GradW16Plan& plan, hipStream_t st) {
    if (plan.T == 8) launch_grad_w16_tiles<MODE, OUT32, 8>(p, plan.tail, st);
    else launch_grad_w16_tiles<MODE, OUT32, 4>(p, plan.tail, st);
}

}  // namespace bt

using namespace bt;

extern "C" size_t bt_linear_grad_weight_16_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    const GradW16Plan plan = grad_w16_plan(M, N, K);
    return (size_t)(plan.tail * plan.splits * plan.T * plan.T) << 12;
}

extern "C" int bt_linear_grad_weight_16(const void* dY, const void* X, int dtype, const void* scale, int scale_dtype,
                                        int64_t scale_len, void* dW, int out_dtype, int64_t M, int64_t N, int64_t K,
                                        void* workspace, size_t workspace_bytes, void* stream) {
    const char* who = "bt_linear_grad_weight_16";
    if (!dY || !X || !scale || !dW || M <= 0 || N <= 0 || K <= 0) {
        set_error("%s: null pointer or empty shape", who);
        return BT_ERR_INVALID;
    }
    if (scale_len != N && scale_len != 1) {
        set_error("%s: scale size doesn't match N (%lld entries, N=%lld)", who, (long long)scale_len, (long long)N);
        return BT_ERR_INVALID;
    }
    if ((dtype != BT_F16 && dtype != BT_BF16) || (scale_dtype != BT_F32 && scale_dtype != BT_F16 && scale_dtype != BT_BF16) || (out_dtype != dtype && out_dtype != BT_F32)) {
        set_error("%s: unsupported dtype %d -> %d", who, dtype, out_dtype);
        return BT_ERR_INVALID;
    }
    // (32-bit byte offsets span a stage's 32 rows and the columns of a last tile)
    if (N % 8 || K % 8 || N >= (1ll << 24) || K >= (1ll << 24) || (((uintptr_t)dY) | ((uintptr_t)X) | ((uintptr_t)dW)) % 16 ||
        ((uintptr_t)scale) % dtype_size(scale_dtype) || ceil_div(N, 128) * ceil_div(K, 128) >= (1ll << 28) || M >= (1ll << 40) / std::max(N, K)) {
        set_error("%s: N and K must be multiples of 8 below 2^24, buffers 16-byte aligned", who);
        return BT_ERR_INVALID;
    }
    const size_t need = bt_linear_grad_weight_16_workspace_bytes(M, N, K);
    if (need && (!workspace || workspace_bytes < need || ((uintptr_t)workspace) % 256)) {
        set_error("%s: workspace of %zu bytes (256-byte aligned) needed, %zu given", who, need, workspace_bytes);
        return BT_ERR_WORKSPACE;
    }
    const GradW16Plan plan = grad_w16_plan(M, N, K);
    GradW16Params p = {};
    p.G = (const uint16_t*)dY; p.X = (const uint16_t*)X; p.M = M; p.N = N; p.K = K; p.out = dW;
    p.scale = scale; p.scale_dtype = scale_dtype; p.scale_bcast = scale_len == 1 ? 1 : 0;
    p.tiles_n = (int)ceil_div(N, 32 * plan.T); p.tiles_k = (int)ceil_div(K, 32 * plan.T);
    p.whole = (int)ceil_div(plan.tiles - plan.tail, 8);
    p.tail_from = (int)(plan.tiles - plan.tail);
    p.splits = (int)plan.splits; p.part_rows = plan.part_rows; p.part = (float*)workspace;
    p.long_first = plan.long_first ? 1 : 0;
    p.per_xcd_tail = (int)(plan.long_first ? 2 * ceil_div(plan.tail, 8) : ceil_div(plan.tail * plan.splits, 8));
    hipStream_t st = (hipStream_t)stream;
    if (dtype == BT_F16) {
        if (out_dtype == BT_F32) launch_grad_w16<MODE_F16, true>(p, plan, st);
        else launch_grad_w16<MODE_F16, false>(p, plan, st);
    } else {
        if (out_dtype == BT_F32) launch_grad_w16<MODE_BF16, true>(p, plan, st);
        else launch_grad_w16<MODE_BF16, false>(p, plan, st);
    }
    return check_launch(who);
}
