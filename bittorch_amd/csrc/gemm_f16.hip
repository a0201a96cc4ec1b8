// Large-batch fp16 / bf16 x packed-ternary GEMM for gfx950 on the 16-bit matrix cores: the float path of the packed
// forward for batches too tall for the streaming kernel.
//
// Arithmetic restated from the reference's large-batch packed kernel
// (csrc/kernels/ternary_gemm_production.cu:158-250, accumulate :226-235, epilogue :244-247):
//   acc_f32[m,n] = sum_k x[m,k] * w[k,n];   y[m,n] = acc * scale[n] + bias[n]
// (fp32 accumulation of exact products; the summation order differs from the reference's
// sequential loop, which the 16-bit output tolerance covers).
//
// A 256-thread workgroup (4 waves) owns a tile of 16 NR x 256 outputs, wave w columns 64 w .. +63 over the whole of K; two
// workgroups share a compute unit, so that one's MFMAs run while the other waits, starts, drains or stores (a 512-thread
// workgroup that split K over the two waves of a SIMD: 6.9 us a round of tiles with nothing beside it, fp16 / bf16 row-major
// weights, 4096 x 11008 x 4096 338 -> 260 us, tiled 300 -> 257; 16384 x 768 x 768 30 -> 21.5; 512 x 4096 x 4096 49 -> 31).
// A launch of at most one tile a compute unit has two such groups of waves in a workgroup, half of the stages each, which add
// their sums through LDS at the end (f16_splits_k).  Bound by the issue of a stage, 64 MFMAs (1024 cycles) and some 150 other
// instructions, 80 of them vector ones: 1.46 PFLOP/s at that size (252 us).
// Activations and packed weights go to LDS by global_load_lds, n = fd_stages of 64 k, three for tiles of 128 rows.  The order
// of k inside an MFMA is free: lane (j, g) of the stage's first sub-step takes k = 16 g .. +7 and of the second 16 g + 8 .. +15,
// so the 16 weight bytes a lane loads are all its own, and the weights are decoded in natural order, so the activations are fed
// as they lie in memory.
// A stage is four runs of 16 MFMAs (two halves of the rows for each sub-step).  The decode of the second sub-step's weights is
// dealt out behind the MFMAs of the first, that of the next stage's first sub-step behind the second's.
// Loads are counted by hand: in front of a stage's third run vmcnt leaves the loads of stages s + 2 .. s + n - 1 in flight, so
// stage s + 1 is complete (its weights are read there, its activations behind the barrier in front of the fourth run); the loads
// of stage s + n go out behind that barrier, into the buffer whose last fragments were read before it.
#include <cstddef>

#include "lds_dma.h"
#include "row_math.h"

namespace bt {

constexpr int F_BN = 256;
constexpr int F_BK = 64;            // k per stage (two k32 MFMA sub-steps)

struct GemmFParams {
    // The first 64 bytes hold what a workgroup needs to find its tile and request its first operands: the kernel
    // arguments come through the scalar cache a 64-byte line at a time.
    const uint16_t* X;    // [M, K] fp16 or bf16 bits
    const uint8_t* W_T;   // [Kb, N]
    int64_t K, M, N;      // K: length of an activation row
    int tiles_m, tiles_n;
    int per_xcd;          // tiles per XCD
    int wstages;          // 64-wide stages of W_T
    int tiles16;          // W_TILES: 16-column tiles of the copy (its 16-row steps are the stages; < 0: stored_tile16)
    int fine_from;        // an XCD's tiles from this one on are computed in finer ones
    // ---- needed later
    void* Y;              // [M, N]
    int64_t Kb;           // packed weight rows
    Epilogue epi;
};
static_assert(offsetof(GemmFParams, Y) == 64, "first argument line as laid out above");

// Stages of activations in LDS; of weights one fewer, since a wave has its own in registers half a stage before it needs them.
// NB: 32 rows of them.  One group of four waves: 56, 44, 36 KiB; two groups: 64 (NB = 2), 56 (NB = 1).
constexpr int fd_stages(int NB, int KG) { return NB == 4 || (NB == 2 && KG == 2) ? 3 : NB == 2 || KG == 2 ? 4 : 5; }
constexpr int fd_group_bytes(int NB, int KG) { return fd_stages(NB, KG) * NB * 4096 + (fd_stages(NB, KG) - 1) * 4096; }

// Piece q of row r of a stage lies at place q ^ fd_place(r / 2).  A 16-byte read from LDS takes its lanes in groups that hold
// rows 0 .. 3 and 12 .. 15 of one pair of pieces with rows 4 .. 11 of the next pair: those must differ.  (With r / 2 itself every
// fragment read met half of the banks twice: 2.2 M of the 4.9 M LDS cycles of 1000 x 2560 x 6912 were conflicts, now none of
// 2.7 M; 49.6 -> 44.1 us there with the decode below.)
__device__ __forceinline__ uint32_t fd_place(uint32_t half_row) { return (half_row & 1u) | ((half_row >> 2) & 1u) * 6u; }

// y = sum * scale + bias, row block by row block (the empty asm keeps a row's address from being computed ahead of its turn)
// RN: rows of any length, so that a lane's four columns start on any element and the last ones may be fewer.
template <int MODE, bool RES, bool RN, int MB>
__device__ __forceinline__ void fd_epilogue(const GemmFParams& p, const v4f (&acc)[MB][4], int64_t m0, int g, int64_t ncol,
                                            int rows_left, const float (&ws)[4], const float (&bs)[4]) {
    constexpr int YDT = MODE == MODE_F16 ? BT_F16 : BT_BF16;
    const uint32_t lane_off = ((uint32_t)(4 * g) * (uint32_t)p.N + (uint32_t)(ncol & (F_BN - 1))) * 2u;
    const int64_t first = (m0 * p.N + (int64_t)__builtin_amdgcn_readfirstlane((int)(ncol / F_BN)) * F_BN) * 2;
    const int64_t row_bytes = p.N * 2;
    char* row = (char*)p.Y + first;
    const char* res = (const char*)p.epi.residual + first;
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
        if (16 * mb >= rows_left) return;  // (uniform)
        uint2 rv[4];
        if constexpr (RES) {  // the block's four rows at once; lanes past the last row read a row that exists
#pragma unroll
            for (int r = 0; r < 4; r++) {
                asm volatile("" : "+s"(res));
                const char* src = res + (16 * mb + 4 * g + r < rows_left ? lane_off : 0u);
                if constexpr (RN) {
                    uint32_t d[4];
#pragma unroll
                    for (int t = 0; t < 4; t++) d[t] = ((const uint16_t*)src)[ncol + t < p.N ? t : 0];
                    rv[r] = make_uint2(d[0] | d[1] << 16, d[2] | d[3] << 16);
                } else {
                    rv[r] = *(const uint2*)src;
                }
                res += (16 * mb + r + 1 < rows_left) ? row_bytes : 0;
            }
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            asm volatile("" : "+s"(row));
            if (16 * mb + 4 * g + r < rows_left) {
                uint16_t h[4];
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    float a = acc[mb][t][r];
                    if constexpr (MODE == MODE_BF16) a *= 0.5f;  // weights were decoded as +-2.0
                    float y = epi_float(a, ws[t], bs[t]);
                    if constexpr (RES) {
                        const uint32_t bits = ((t < 2 ? rv[r].x : rv[r].y) >> (16 * (t & 1))) & 0xffffu;
                        y = sum_in_dtype(round_to_dtype(y, YDT), bits_to_f32_rt(bits, YDT), YDT);
                    }
                    h[t] = YDT == BT_F16 ? f32_to_f16_bits(y) : f32_to_bf16_bits(y);
                }
                if (RN && ncol + 4 > p.N) {
                    for (int t = 0; t < 3; t++)
                        if (ncol + t < p.N) ((uint16_t*)(row + lane_off))[t] = h[t];
                } else if constexpr (RN) {
                    *(u32x2_a2*)(row + lane_off) = u32x2_a2{(uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16)};
                } else {
                    st2_nt(row + lane_off, (uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
                }
            }
            row += row_bytes;
        }
        row += 12 * row_bytes;
        if constexpr (RES) res = row - (char*)p.Y + (const char*)p.epi.residual;
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The SwiGLU output stage (EPI_SWIGLU_PAIRS): a lane holds columns c, c + 1 of the gate in t = 0, 1 and the same of up in t = 2, 3,
// and stores what the SwiGLU row kernel would make of the rounded outputs: the same element arithmetic, hence the same bits.  Bound by
// that arithmetic, 64 values a lane behind the last stage of a tile (3 us where all tiles end together); it saves the projections'
// way to memory and back and a launch.  GEMM and row kernel / this, us, bf16: 1000 x 13824 x 2560 73.4 / 65.4, 4096 x 13824 x 2560
// 238 / 217, 300 x 8192 x 2048 23.8 / 19.5.  (4-byte stores of each row 67.2 and 222 on the first two.)
template <int MODE, int MB>
__device__ __forceinline__ void fd_epilogue_swiglu(const GemmFParams& p, const v4f (&acc)[MB][4], int64_t m0, int g, int64_t col,
                                                   int rows_left, const float (&ws)[4], const float (&bs)[4]) {
    constexpr int YDT = MODE == MODE_F16 ? BT_F16 : BT_BF16;
    const int64_t row_bytes = p.N;  // (N / 2 outputs of two bytes)
    char* row = (char*)p.Y + m0 * row_bytes;
    const uint32_t lane_off = (uint32_t)(4 * g) * (uint32_t)row_bytes + (uint32_t)col * 2u;
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
        if (16 * mb >= rows_left) return;  // (uniform)
        float y[4][4];
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float a = acc[mb][t][r];
                if constexpr (MODE == MODE_BF16) a *= 0.5f;  // weights were decoded as +-2.0
                y[t][r] = round_to_dtype(epi_float(a, ws[t], bs[t]), YDT);
            }
        swiglu_store16<YDT>(row, row_bytes, lane_off, rows_left - 16 * mb, g, y);
        row += 16 * row_bytes;
        __builtin_amdgcn_sched_barrier(0);
    }
}

// One tile of 16 NR rows (48: a wave stages 64, the last ones repeated).  TAIL: K is not a multiple of 64 (of 8 it is): the lanes whose k lies past
// the end load something of their own row or column instead and their activations are zeroed on the way to the MFMAs.
// KG = 2: two groups of four waves, each on its run of the stages; they add their sums through LDS and store half the rows each
// (of 48: 32 and 16).
// SW: the SwiGLU output stage on a copy in gate/up pair order (stored tiles 2 i, 2 i + 1 are 16 columns of the gate and the same of up):
// a lane takes two columns of either, so that no sum changes lanes.
template <int MODE, int SRC, int NR, int KG, bool TAIL, bool RN, bool SW>
__device__ __forceinline__ void gemm_f16_tile(const GemmFParams& p, const int64_t m0, const int tile_n, uint8_t* lds_all) {
    constexpr int NB = (NR + 1) / 2, BM = 16 * NR, A_BYTES = NB * 4096, NST = fd_stages(NB, KG), W_AT = NST * A_BYTES;
    constexpr int A_LOADS = NB, W_LOADS = SRC == W_ROWS ? 4 : 1, LOADS = A_LOADS + W_LOADS;
    const int lane = threadIdx.x & 63;
    const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wave = wave_all & 3, group = KG == 1 ? 0 : wave_all >> 2;
    uint8_t* const lds = lds_all + group * fd_group_bytes(NB, KG);
    const int j = lane & 15, g = lane >> 4;
    const int64_t ncol = (int64_t)tile_n * F_BN + 64 * wave + 4 * j;
    const bool col_ok = ncol < p.N;
    const int nst = (int)((p.K + F_BK - 1) / F_BK);
    const int64_t k_last = (int64_t)(nst - 1) * F_BK;
    // this group's stages: st0 .. st0 + mine - 1 (every group meets `rounds` barriers in the loop; mine >= 1)
    const int rounds = KG == 1 ? nst : (nst + 1) / 2, st0 = group * rounds, mine = KG == 1 ? nst : min(rounds, nst - st0);
    const int st_tail = group == KG - 1 ? mine - 1 : rounds;  // TAIL: the partial stage, if it is this group's

    // A stage's row is 128 bytes of LDS, eight pieces of 16 at the places fd_place gives them.  A wave loads whole rows, eight
    // lanes each: lanes of a load that each have a row of their own take the cache four times as long.  Wave w loads rows
    // 8 NB w .. +8 NB-1, eight at a time.  Rows past M repeat the last one, columns past N column 0 or the copy's last tile
    // (never stored).
    const int64_t rows_left = (p.M - m0 < BM) ? p.M - m0 : BM;
    uint32_t a_off[A_LOADS], a_tail[A_LOADS];
#pragma unroll
    for (int b = 0; b < A_LOADS; b++) {
        const int row = 8 * (NB * wave + b) + (lane >> 3), piece = (lane & 7) ^ fd_place(row >> 1);
        const uint32_t r = (uint32_t)(row < rows_left ? row : rows_left - 1);
        a_off[b] = (r * (uint32_t)p.K + 8u * piece) * 2u;
        a_tail[b] = k_last + 8 * piece < p.K ? a_off[b] : r * (uint32_t)p.K * 2u;
    }
    uint32_t w_off[W_LOADS], w_tail[W_LOADS];
    if constexpr (SRC == W_ROWS16) {
        const int64_t col = (int64_t)tile_n * F_BN + 64 * wave + 16 * (lane & 3);
        w_off[0] = (uint32_t)(col < p.N ? col : 0) + (uint32_t)rows16_row(lane) * (uint32_t)p.N;
        w_tail[0] = (k_last >> 2) + rows16_row(lane) < p.Kb ? w_off[0] : (uint32_t)(col < p.N ? col : 0);
    } else if constexpr (SRC == W_TILES) {
        const int tt = stored_tile16((int)(ncol >> 4), p.tiles16);
        w_off[0] = ((uint32_t)tt * (uint32_t)p.wstages * 64u + (uint32_t)(16 * g + 4 * (j & 3))) * 4u;
    } else {
#pragma unroll
        for (int r = 0; r < W_LOADS; r++) {
            w_off[r] = (uint32_t)(col_ok ? ncol : 0) + (uint32_t)(4 * g + r) * (uint32_t)p.N;
            w_tail[r] = (k_last >> 2) + 4 * g + r < p.Kb ? w_off[r] : (uint32_t)(col_ok ? ncol : 0);
        }
    }
    u32x4 keep[2] = {};  // TAIL: which values of a lane's fragment lie inside K in the last stage
    if constexpr (TAIL) {
#pragma unroll
        for (int sub = 0; sub < 2; sub++) {
            const uint32_t m = k_last + 16 * g + 8 * sub < p.K ? 0xFFFFFFFFu : 0u;
            keep[sub] = u32x4{m, m, m, m};
        }
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;

    const int64_t w_step = SRC == W_TILES ? 256 : 16 * p.N;
    const uint8_t* a_next = (const uint8_t*)(p.X + m0 * p.K + (int64_t)st0 * F_BK);
    const uint8_t* w_next = p.W_T + st0 * w_step;
    uint32_t into = 0, w_into = W_AT;
    int st_next = 0;
    auto issue_a = [&](int b) {
        const bool last = TAIL && st_next >= st_tail;
        dma16(lds0 + into + (uint32_t)(NB * wave + b) * 1024u, last ? a_tail[b] : a_off[b], a_next);
    };
    auto issue_w = [&](int r) {
        const bool last = TAIL && st_next >= st_tail;
        const uint32_t wd = lds0 + w_into + (uint32_t)wave * 1024u;
        if constexpr (SRC == W_TILES) dma16(wd, w_off[0], w_next);
        else if constexpr (SRC == W_ROWS16) dma16(wd, last ? w_tail[0] : w_off[0], w_next);
        else dma4(wd + 256u * r, last ? w_tail[r] : w_off[r], w_next);
    };
    auto next_buf = [](uint32_t b) { return b + A_BYTES == W_AT ? 0u : b + A_BYTES; };
    auto next_wbuf = [](uint32_t b) { return b + 4096 == fd_group_bytes(NB, KG) ? (uint32_t)W_AT : b + 4096; };
    auto advance = [&]() {  // past the end: the last stage again, never read
        st_next++;
        a_next += st_next < mine ? 2 * F_BK : 0;
        w_next += st_next < mine ? w_step : 0;
        into = next_buf(into);
        w_into = next_wbuf(w_into);
    };

    v4f acc[NR][4];
#pragma unroll
    for (int mb = 0; mb < NR; mb++)
#pragma unroll
        for (int t = 0; t < 4; t++) acc[mb][t] = v4f{0.f, 0.f, 0.f, 0.f};

    // two sets of fragments: the halves of a sub-step (NB = 4) or whole sub-steps
    constexpr int RB = NB == 4 ? 4 : NR;
    u32x4 a_x[RB], a_y[RB], b0[4], b1[4];
    uint32_t raw[4];
    // lane (j, g): k = 16 g + 8 sub .. +7 of row 16 mb + j
    const uint32_t at_j = fd_place(j >> 1), frag_at[2] = {128u * j + 16u * ((2u * g) ^ at_j), 128u * j + 16u * ((2u * g + 1) ^ at_j)};
    auto frag = [&](uint32_t buf, int sub, int mb) { return *(const u32x4*)(lds + (buf + frag_at[sub]) + 2048 * mb); };
    auto read_raw = [&](uint32_t wbuf) {
        const uint8_t* src = lds + wbuf + wave * 1024;
        if constexpr (SRC == W_TILES) {
            if constexpr (SW) {  // lane (j, g)'s 16 bytes are those of columns 4 (j % 4) .. +3 of stored tile j / 4
                const uint8_t* at = src + 256 * g + 128 * (j >> 3) + 8 * (j & 7);
                const u32x2 a = *(const u32x2*)at, b = *(const u32x2*)(at + 64);
                raw[0] = a[0]; raw[1] = a[1]; raw[2] = b[0]; raw[3] = b[1];
            } else {
                const u32x4 v = *(const u32x4*)(src + 16 * lane);
#pragma unroll
                for (int t = 0; t < 4; t++) raw[t] = v[t];
            }
        } else {
#pragma unroll
            for (int r = 0; r < 4; r++) raw[r] = *(const uint32_t*)(src + 256 * r + 4 * lane);
        }
    };
    // Decode of a raw dword's 16 codes: code c of its four bytes becomes the high bytes of four operand values by one table
    // lookup (the low bytes of +-1 in fp16 and of +-2 in bf16 are zero), and an operand dword is the high bytes of codes 2 h and
    // 2 h + 1 of one byte: 19 operations for eight dwords.  Byte by byte it took 28.
    // Column t's codes of its byte r (k = 4 r .. +3) are in byte r of raw[t] (the copy) or byte t of raw[r] (rows); sub-step s
    // takes bytes 2 s and 2 s + 1.
    constexpr uint32_t LUT = (MODE == MODE_F16) ? LUT_F16_ONE : LUT_BF16_TWO;
    uint32_t hi[4][4];
    auto table = [&](int e) { hi[e >> 2][e & 3] = perm(0u, LUT, (raw[e >> 2] >> (2 * (e & 3))) & 0x03030303u); };
    auto emit = [&](int e, int sub, u32x4 (&out)[4]) {  // dword e % 4 of column e / 4
        const int t = e >> 2, d = e & 3, r = 2 * sub + (d >> 1), h = d & 1;
        const int q = SRC == W_TILES ? t : r, byte = SRC == W_TILES ? r : t;
        out[t][d] = perm(hi[q][2 * h + 1], hi[q][2 * h], ((uint32_t)(4 + byte) << 24) | (0x0Cu << 16) | ((uint32_t)byte << 8) | 0x0Cu);
    };
    // The first sub-step's tables are all of them (the copy) or those of raw[0] and raw[1] (rows).
    constexpr int T0 = SRC == W_TILES ? 16 : 8;
    auto mfma = [&](const u32x4& a, const u32x4& b, v4f& c) {
        if constexpr (MODE == MODE_F16)
            c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
        else
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
    };

    uint32_t buf = 0, wbuf = W_AT;
#pragma unroll
    for (int s = 0; s < NST; s++) {
#pragma unroll
        for (int b = 0; b < A_LOADS; b++) issue_a(b);
        if (s == NST - 1) break;
#pragma unroll
        for (int r = 0; r < W_LOADS; r++) issue_w(r);
        advance();
    }
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NST - 1) * LOADS - W_LOADS) : "memory");  // stage 0
    read_raw(wbuf);
#pragma unroll
    for (int i = 0; i < RB; i++) a_x[i] = frag(0, 0, i);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the first weights' place is free again
#pragma unroll
    for (int r = 0; r < W_LOADS; r++) issue_w(r);
    advance();
#pragma unroll
    for (int e = 0; e < T0; e++) table(e);
#pragma unroll
    for (int e = 0; e < 16; e++) emit(e, 0, b0);

    // Everything but the MFMAs is dealt out between them (16 slots a run), two or three instructions behind each:
    // instructions in a row of their own would leave the matrix pipe idle.
    constexpr int SL = NB == 1 ? 2 : 1;  // slots per MFMA
    for (int s = 0; s < mine; s++) {
        const uint32_t nxt = next_buf(buf);
        auto run_mfma = [&](int c, const u32x4 (&a)[RB], const u32x4 (&b)[4], int mb0) {
            if (c % SL != 0 || c >= 4 * SL * RB) return;
            const int i = (c / SL) >> 2, t = (c / SL) & 3;
            mfma(a[i], b[t], acc[mb0 + i][t]);
        };
        auto mask = [&](u32x4 (&a)[RB], int sub) {
            if constexpr (TAIL) {
                if (s == st_tail) {  // (uniform)
#pragma unroll
                    for (int i = 0; i < RB; i++) a[i] &= keep[sub];
                }
            }
        };
        auto load_next = [&](int c) {  // stage s + NST over stage s
            if (c >= 5 && c < 5 + A_LOADS) issue_a(c - 5);
            if (c >= 10 && c < 10 + W_LOADS) issue_w(c - 10);
            if (c == 15) advance();
        };
        mask(a_x, 0);
        if constexpr (NB == 4) {
#pragma unroll
            for (int c = 0; c < 16; c++) {
                run_mfma(c, a_x, b0, 0);
                if (c < 4) a_y[c] = frag(buf, 0, 4 + c);
                if (c % 2 == 0) {
                    if (SRC == W_TILES) emit(c / 2, 1, b1);
                    else table(8 + c / 2);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            mask(a_y, 0);
#pragma unroll
            for (int c = 0; c < 16; c++) {
                run_mfma(c, a_y, b0, 4);
                if (c < 4) a_x[c] = frag(buf, 1, c);
                if (SRC != W_TILES) emit(c, 1, b1);
                else if (c % 2 == 0) emit(8 + c / 2, 1, b1);
                __builtin_amdgcn_sched_barrier(0);
            }
            mask(a_x, 1);
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 2) * LOADS) : "memory");  // stage s + 1
#pragma unroll
            for (int c = 0; c < 16; c++) {
                run_mfma(c, a_x, b1, 0);
                if (c == 0) read_raw(next_wbuf(wbuf));
                if (c < 4) a_y[c] = frag(buf, 1, 4 + c);
                if (c >= 8) {  // (the weights have arrived)
                    table(c - 8);
                    if (T0 == 16) table(c);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            mask(a_y, 1);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
            for (int c = 0; c < 16; c++) {
                run_mfma(c, a_y, b1, 4);
                if (c < 4) a_x[c] = frag(nxt, 0, c);
                emit(c, 0, b0);
                load_next(c);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            // fewer rows: a run is a whole sub-step, so that the fragments of the next one have a run to arrive in
#pragma unroll
            for (int c = 0; c < 16; c++) {
                run_mfma(c, a_x, b0, 0);
                if (c < RB) a_y[c] = frag(buf, 1, c);
                if (SRC == W_TILES) {
                    if (c < 12) emit(c, 1, b1);
                    else if (c < 14) { emit(2 * c - 12, 1, b1); emit(2 * c - 11, 1, b1); }
                } else {
                    if (c < 4) { table(8 + 2 * c); table(9 + 2 * c); }
                    else if (c < 12) { emit(2 * (c - 4), 1, b1); emit(2 * (c - 4) + 1, 1, b1); }
                }
                if (c == 15) {
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 2) * LOADS) : "memory");  // stage s + 1
                    read_raw(next_wbuf(wbuf));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            mask(a_y, 1);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
            for (int c = 0; c < 16; c++) {
                run_mfma(c, a_y, b1, 0);
                if (c < RB) a_x[c] = frag(nxt, 0, c);
                if (T0 == 16) {
                    if (c >= 4 && c < 12) { table(2 * (c - 4)); table(2 * (c - 4) + 1); }
                    else if (c >= 12) {
#pragma unroll
                        for (int e = 0; e < 4; e++) emit(4 * (c - 12) + e, 0, b0);
                    }
                } else {
                    if (c >= 4 && c < 8) { table(2 * (c - 4)); table(2 * (c - 4) + 1); }
                    else if (c >= 8) { emit(2 * (c - 8), 0, b0); emit(2 * (c - 8) + 1, 0, b0); }
                }
                load_next(c);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        buf = nxt;
        wbuf = next_wbuf(wbuf);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the fragments arrived under these MFMAs
        __builtin_amdgcn_sched_barrier(0);
    }
    if (KG > 1 && mine < rounds) asm volatile("s_barrier" ::: "memory");  // (uniform; the other group has one stage more)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (no load may reach LDS that another workgroup owns by then)

    const int64_t half_n = p.N / 2, scol = (int64_t)tile_n * (F_BN / 2) + 32 * wave + 2 * j;  // SW: the first of this lane's outputs
    float ws[4], bs[4];
    uint32_t ws_bits[4], bs_bits[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int64_t n = SW ? (scol < half_n ? scol + (t & 1) + (t >> 1) * half_n : 0) : !col_ok ? 0 : RN ? min(ncol + t, p.N - 1) : ncol + t;
        ws_bits[t] = load_bits_rt(p.epi.scale, p.epi.scale_dtype, p.epi.scale_bcast ? 0 : n);
        bs_bits[t] = p.epi.bias ? load_bits_rt(p.epi.bias, p.epi.bias_dtype, n) : 0u;
    }
#pragma unroll
    for (int t = 0; t < 4; t++) {
        ws[t] = bits_to_f32_rt(ws_bits[t], p.epi.scale_dtype);
        bs[t] = p.epi.bias ? bits_to_f32_rt(bs_bits[t], p.epi.bias_dtype) : 0.0f;
    }
    const bool stores = SW ? scol < half_n : col_ok;
    auto store = [&](const auto& sums, int64_t row0, int left) {
        if constexpr (SW) fd_epilogue_swiglu<MODE>(p, sums, row0, g, scol, left, ws, bs);
        else if (p.epi.residual) fd_epilogue<MODE, true, RN>(p, sums, row0, g, ncol, left, ws, bs);
        else fd_epilogue<MODE, false, RN>(p, sums, row0, g, ncol, left, ws, bs);
    };
    if constexpr (KG == 1) {
        if (stores) store(acc, m0, (int)rows_left);
    } else {
        // group 0 takes the first NB row blocks, group 1 the others: each hands over the sums that it does not store
        v4f* const mine_at = (v4f*)lds_all + wave_all * (256 * NB) + lane;
        const v4f* const theirs_at = (const v4f*)lds_all + (wave_all ^ 4) * (256 * NB) + lane;
        v4f sums[NB][4];
        __syncthreads();  // (both groups have read their last stages)
#pragma unroll
        for (int i = 0; i < NB; i++)
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const int other = NB + i < NR ? NB + i : NR - 1;  // (48 rows: the last block twice, stored once)
                mine_at[64 * (4 * i + t)] = group ? acc[i][t] : acc[other][t];
                sums[i][t] = group ? acc[other][t] : acc[i][t];
            }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NB; i++)
#pragma unroll
            for (int t = 0; t < 4; t++) sums[i][t] += theirs_at[64 * (4 * i + t)];
        const int left = (int)rows_left - 16 * NB * group;
        if (stores && left > 0) store(sums, m0 + 16 * NB * group, left);
    }
}

// NR: tiles of 16 NR rows.  NF > 0: an XCD's tiles from p.fine_from on are computed in tiles of 16 NF rows.
template <int MODE, int SRC, int NR, int NF, int KG, bool TAIL, bool RN, bool SW>
__global__ __launch_bounds__(256 * KG, KG == 2 || NR == 8 ? 2 : NR == 4 ? 3 : 4) void gemm_f16_kernel(GemmFParams p) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[KG * fd_group_bytes((NR + 1) / 2, KG)];
    // XCD-aware tile order: the 8 XCDs each take a contiguous run of tiles, walked in groups of four row tiles, so that one
    // XCD's L2 holds a compact block of rows and columns
    const uint32_t idx = blockIdx.x >> 3;
    const bool fine = NF > 0 && idx >= (uint32_t)p.fine_from;  // (uniform)
    const uint32_t parts = NF > 0 ? NR / (NF > 0 ? NF : 1) : 1, f = fine ? idx - (uint32_t)p.fine_from : 0u;
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
    const int64_t m0 = (int64_t)(first_m + (in_group - tn * gm)) * (16 * NR);
    if constexpr (NF > 0) {
        if (fine) {
            const int64_t mf = m0 + (int64_t)(f % parts) * (16 * NF);
            if (mf < p.M) gemm_f16_tile<MODE, SRC, NF, 1, TAIL, RN, SW>(p, mf, (int)tn, lds);
            return;
        }
    }
    gemm_f16_tile<MODE, SRC, NR, KG, TAIL, RN, SW>(p, m0, (int)tn, lds);
}

// X and Y are read and written in 16- and 8-byte pieces; 32-bit byte offsets span a tile's rows of X, 16 rows of Y and, for
// row-major weights, 16 rows of W_T.  W_T 4-byte aligned and N % 4 == 0, or the decode-tiled copy (256-byte aligned, below
// 4 GiB: checked by the caller), with which Y's rows have any length.
bool gemm_f16_supported(int64_t N, int64_t K, const void* X, const void* W_T, const void* Y, bool tiled) {
    return (tiled || N % 4 == 0) && N < (1ll << 27) && K % 8 == 0 && K >= 8 && K < (1ll << 23) && ((uintptr_t)W_T) % 4 == 0 &&
           ((uintptr_t)X) % 16 == 0 && ((uintptr_t)Y) % 16 == 0;
}

// A launch of one tile of 64 or 32 rows for each compute unit at most: two groups of waves, half of the stages each.  With one
// group a SIMD has a single wave, whose chain of LDS reads, decode and MFMAs leaves it idle half of the time.  One / two groups,
// us, decode-tiled bf16: tiles of 32 rows, 512 x 2560 x 6912 43.2 / 34.1, 128 x 4096 x 11008 62.3 / 49.2, 256 x 7680 x 2560
// 19.3 / 17.1, 128 x 6000 x 1536 13.0 / 12.0; of 64 rows, 1000 x 2560 x 6912 49.6 / 44.1, 256 x 11008 x 4096 32.7 / 29.7,
// 512 x 6000 x 1536 15.8 / 15.7.  Fewer stages than 24 would not pay for the exchange of the sums; deeper launches have
// the other tiles' waves for company (1000 x 13824 x 2560 66.9 / 81.2).
static bool f16_splits_k(int64_t stages) { return stages >= 24; }

// Rows of the tiles in units of 16, and what the launch takes in microseconds.  Up to one tile of 32, then of 48 (where two groups of
// waves share it), then of 64 rows for each compute unit the launch is one tile deep; beyond that a compute unit's run of tiles is priced.  Measured (tiles of 128 / 64 /
// 32 rows, us, row-major weights): M = 512, 1024, 1536, 2048, 3072, 4096 with N = K = 4096 30 / 30 / 25, 33 / 31 / 40,
// 49 / 49 / 53, 52 / 54 / 75, 89 / 81 / 107, 95 / 106 / 139; 1000 x 13824 x 2560 60 / 66 / 81; 1000 x 2560 x 6912 66 / 45 / 62;
// 16384 x 768 x 768 21 / 20 / 26; 4096 x 11008 x 4096 (the last round in halves) 251 / 264 / 333.
// Tiles of 48 rows, us, decode-tiled / row-major bf16, those of 64 / 48 rows: 1000 x 2560 x 6912 45.1 / 43.7, 42.3 / 41.0; 1200 x 2560 x
// 6912 43.1 / 40.5, 42.4 / 39.7; 832 x 2560 x 2560 19.8 / 18.3; 768 x 4096 x 4096 29.0 / 26.7; 384 x 8192 x 8192 50.0 / 47.3; 350 x 8192 x
// 1536 14.5 / 13.5 (a stage has a quarter fewer MFMAs, its loads and decode are the same).
static int gemm_f16_plan(int64_t M, int64_t N, int64_t K, double* us) {
    const int64_t C = gemm_compute_units(), tn = ceil_div(N, F_BN);
    const int64_t t4 = ceil_div(M, 128) * tn, t2 = ceil_div(M, 64) * tn, t1 = ceil_div(M, 32) * tn;
    const bool whole = gemm_whole_tiles(), split = f16_splits_k(ceil_div(K, F_BK));
    if (t1 <= C && !whole) { *us = split ? 5.7 + 0.0042 * (double)K : 4.0 + 0.0055 * (double)K; return 2; }
    if (split && ceil_div(M, 48) * tn <= C && !whole) { *us = 5.9 + 0.0049 * (double)K; return 3; }
    if (t2 <= C && !whole) { *us = split ? 6.0 + 0.0056 * (double)K : 5.0 + 0.0065 * (double)K; return 4; }
    const int parts = gemm_dma_parts(t4);
    const double n4 = parts == 1 ? (double)ceil_div(t4, C) : (double)(2 * (t4 / (2 * C))) + (parts == 2 ? 1.2 : 0.6);
    const double p4 = n4 * (2.0 + 0.0113 * (double)K), p2 = (double)ceil_div(t2, C) * (1.3 + 0.0062 * (double)K);
    const bool half = p2 < p4 && !whole;
    *us = 4.0 + (half ? p2 : p4);
    return half ? 4 : 8;
}
double gemm_f16_cost(int64_t M, int64_t N, int64_t K) {
    double us;
    gemm_f16_plan(M, N, K, &us);
    return us;
}

template <int MODE, int SRC, int NR, bool TAIL, bool RN = false, bool SW = false>
static int launch_gemm_f16_cfg(GemmFParams p, hipStream_t st) {
    const char* who = SRC == W_TILES ? "bt_ternary_linear_tiled_forward" : "bt_ternary_linear_packed_forward";
    p.tiles_n = (int)ceil_div(p.N, F_BN);
    p.tiles_m = (int)ceil_div(p.M, 16 * NR);
    const int64_t total = (int64_t)p.tiles_m * p.tiles_n;
    if (total >= (1ll << 29)) {
        set_error("%s: %lld tiles of %d x 256 outputs are more than one launch takes", who, (long long)total, 16 * NR);
        return BT_ERR_INVALID;
    }
    p.per_xcd = (int)ceil_div(total, 8);
    p.fine_from = p.per_xcd;
    const dim3 block(256);
    if constexpr (NR == 8) {
        const int parts = gemm_dma_parts(total);
        if (parts > 1) {
            const int rem = p.per_xcd % (int)(2 * gemm_compute_units() / 8);
            p.fine_from = p.per_xcd - rem;
            const dim3 grid((unsigned)(8 * (p.fine_from + parts * rem)));
            if (parts == 2) hipLaunchKernelGGL((gemm_f16_kernel<MODE, SRC, 8, 4, 1, TAIL, RN, SW>), grid, block, 0, st, p);
            else hipLaunchKernelGGL((gemm_f16_kernel<MODE, SRC, 8, 2, 1, TAIL, RN, SW>), grid, block, 0, st, p);
            return check_launch(who);
        }
    }
    if constexpr (NR != 8) {
        if (NR == 3 || (total <= gemm_compute_units() && f16_splits_k(p.wstages))) {
            hipLaunchKernelGGL((gemm_f16_kernel<MODE, SRC, NR, 0, 2, TAIL, RN, SW>), dim3((unsigned)(8 * p.per_xcd)), dim3(512), 0, st, p);
            return check_launch(who);
        }
    }
    if constexpr (NR != 3) hipLaunchKernelGGL((gemm_f16_kernel<MODE, SRC, NR, 0, 1, TAIL, RN, SW>), dim3((unsigned)(8 * p.per_xcd)), block, 0, st, p);
    return check_launch(who);
}
template <int MODE, int SRC, int NR>
static int launch_gemm_f16_src(const GemmFParams& p, int epi_op, hipStream_t st) {
    if constexpr (SRC == W_TILES) {
        if (epi_op == EPI_SWIGLU_PAIRS)
            return p.K % F_BK != 0 ? launch_gemm_f16_cfg<MODE, SRC, NR, true, false, true>(p, st)
                                   : launch_gemm_f16_cfg<MODE, SRC, NR, false, false, true>(p, st);
        // (rows of any length come with K of any length: one instance)
        if (p.N % 4 != 0) return launch_gemm_f16_cfg<MODE, SRC, NR, true, true>(p, st);
    }
    return p.K % F_BK != 0 ? launch_gemm_f16_cfg<MODE, SRC, NR, true>(p, st) : launch_gemm_f16_cfg<MODE, SRC, NR, false>(p, st);
}
template <int MODE, int NR>
static int launch_gemm_f16_mode(const GemmFParams& p, int src, int epi_op, hipStream_t st) {
    return src == W_TILES ? launch_gemm_f16_src<MODE, W_TILES, NR>(p, epi_op, st)
         : src == W_ROWS16 ? launch_gemm_f16_src<MODE, W_ROWS16, NR>(p, 0, st) : launch_gemm_f16_src<MODE, W_ROWS, NR>(p, 0, st);
}
template <int MODE>
static int launch_gemm_f16_rows(const GemmFParams& p, int rows, int src, int epi_op, hipStream_t st) {
    return rows == 8 ? launch_gemm_f16_mode<MODE, 8>(p, src, epi_op, st) : rows == 4 ? launch_gemm_f16_mode<MODE, 4>(p, src, epi_op, st)
         : rows == 3 ? launch_gemm_f16_mode<MODE, 3>(p, src, epi_op, st) : launch_gemm_f16_mode<MODE, 2>(p, src, epi_op, st);
}
// epi_op: 0, or EPI_SWIGLU_PAIRS (w_layout W_LAYOUT_TILED in pair order, N % 32 == 0, no residual; Y is [M, N / 2])
// Kw: the weights' K where the rows of X are longer (zeros behind it; 0: K)
int launch_gemm_f16(int mode, const void* X, const uint8_t* W_T, int w_layout, const Epilogue& epi, void* Y, int64_t M,
                    int64_t N, int64_t K, hipStream_t st, int64_t Kw, int epi_op) {
    GemmFParams p = {};
    p.X = (const uint16_t*)X; p.W_T = W_T; p.Y = Y; p.epi = epi;
    p.M = M; p.N = N; p.K = K; p.Kb = ceil_div(Kw ? Kw : K, 4);
    p.wstages = (int)ceil_div(K, F_BK);
    p.tiles16 = tiles16_arg(N, w_layout);
    double us;
    const int rows = gemm_f16_plan(M, N, K, &us), src = w_source(layout_tiled(w_layout), false, W_T, N);
    return mode == MODE_F16 ? launch_gemm_f16_rows<MODE_F16>(p, rows, src, epi_op, st) : launch_gemm_f16_rows<MODE_BF16>(p, rows, src, epi_op, st);
}

}  // namespace bt
