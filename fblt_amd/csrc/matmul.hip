/*
 * fp32 matrix product out[M,N] = a[M,K] * b[K,N] (row-major), the projection
 * GEMMs either side of the attention core (reference contract:
 * csrc/ops/matmul.h, CPU loop csrc/ops/linalg_cpu.c:8-18, device twin
 * csrc/ops/linalg.cu:48-134).
 *
 * Three kernels:
 *
 *  - "skinny" (M <= 32: the n new rows of a decode / verify step): one thread
 *    per output column, the column of b read coalesced across the wave, the
 *    rows of a through the scalar cache; every output is the reference's own
 *    sum -- k ascending, product and sum rounded separately -- so this path
 *    is bit-identical to blt_matmul_cpu.
 *
 *  - "mfma" (everything else; from three terms a sum on): 64x64 or 128x128 output tiles per workgroup of eight
 *    wavefronts, K in steps of 32 or 64 through double-buffered LDS tiles, on the f16 or bf16
 *    matrix instructions with both operands taken apart on the way to LDS
 *    (split_f16.h, split_bf16.h).  The product is accumulated
 *    TRANSPOSED (MFMA A operand = b tile, B operand = a tile), which puts one
 *    output ROW in each lane with four consecutive columns per register
 *    group: rows are stored with 16-byte stores, and an optional epilogue can
 *    rotate (column 2i, column 2i+1) pairs lane-locally -- the rotary position
 *    embedding of the Q and K blocks of a packed QKV projection
 *    (csrc/models/attention.c:76-90) -- without a second pass over the
 *    result.  Summation order differs from the reference's (fp32 tolerance).
 *    On fp32 instructions -> on bf16 parts -> on f16 parts: 2048 x 512 . 512 x 2048 41.0 -> 30.4 -> 20.6 us, 2048 x 2048 .
 *    2048 x 512 45.3 -> 37.0 -> 28.6, 8192 x 512 . 512 x 1536 84.2 as bf16 -> 65.2.
 *
 *  - "splitk" (outputs too small to give every compute unit a 64x64 tile,
 *    e.g. 512x128 * 128x384; sums of one or two terms; more than 2^25 columns): one 32x32 output tile per workgroup, its four
 *    wavefronts take the 32-wide K chunks round-robin straight from global
 *    memory (no LDS staging, no barrier in the loop) and add their partial
 *    tiles through LDS at the end.  Same accumulator layout and epilogue as
 *    the mfma kernel; the serial MFMA chain per wave is a quarter as long and
 *    there are four times as many workgroups.
 */
#include "blt_hip.h"
#include "blt_fatal.h"
#include "hip_check.h"
#include "lane_ops.h"
#include "launch.h"
#include "matmul.h"
#include "split_bf16.h"
#include "split_f16.h"
#include "cross_rows_device.h"

#include <stdint.h>
#include <stdlib.h>

#include <algorithm>
#include <map>

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int TM = 64, TN = 64; /* smallest workgroup tile of the mfma kernel */

/* One (64*WT)x(64*WT) output tile per workgroup of eight wavefronts: four quadrants of WT x WT MFMA tiles, and for each
 * quadrant two waves that take half of every K step (16 of 32); their sums meet in LDS at the end.  The
 * operands are taken apart into two f16 parts (split_f16.h) or three bf16 parts (split_bf16.h) once per workgroup, on the
 * way from registers to the double-buffered LDS tiles: rows of a as [row][k], columns of b as [column][k], so that a fragment is one
 * 16-byte read.  WT = 2 halves the split and the LDS reads per output.
 * f16 first, if K is long enough; a workgroup that meets operands out of its range, before the first product as a rule, or
 * finds its results too small for it (half_lost()) starts again as bf16.  Half the matrix instructions, four fifths of the vector ones, half the error (K = 2048: 2.2e-7
 * against 4.9e-7), and a clock that gives way less (8192 x 2048 . 2048 x 1536, random operands against ones: 268 and 210 us
 * as bf16, 196 and 160 as f16, 189 random ones as the loop is now).  Bound: no one unit.  A step of the large tile takes some 2000
 * cycles, and in it a SIMD's matrix unit 770, its vector unit 320 instructions, the compute unit's LDS 800 and 150 of bank conflicts; by the
 * counters vector instructions issue in 0.4 ... 0.5 of a launch's cycles and the matrix unit is busy in a quarter.  What is between them
 * is eight waves that meet at a barrier a step; requests and fragments further ahead, three buffers and another order of issue changed
 * nothing.
 * VEC: a 16-byte aligned with lda and K multiples of 4.  ROPE: rotate pairs of the first g.rope_cols columns in
 * the epilogue.
 * NORM: the row statistic comes from the values on their way to LDS, the norm weight is multiplied in there, the row's
 * scale after the product: two vector instructions per value of a against a pass over a of its own (2048 rows of
 * 512: 14 us with sums in the reference's order).
 * GATED: the left quadrants are columns of a*b, the right ones the same columns of a*b2; they meet in LDS
 * (2048 x 512 . 512 x (2 x 2048): two products and the activation 71 us, this way 63, with eight waves finishing 52).
 * The end is shared by all eight waves and stores rows: a layer of 2048 rows and width 512 took 132.5 us with four waves
 * storing from registers, of which the rotation alone 5.6, and takes 124.0. */
template <int WT, bool NORM, bool F16>
struct MfmaShape {
    static constexpr int BT = 64 * WT;          /* rows and columns of the tile */
    static constexpr int STEP = F16 && WT == 1 && !NORM ? 64 : 32; /* of K: the small tile's work in 32 is short against a barrier */
    static constexpr int EPT = BT * STEP / 512; /* values of each operand a thread carries per step */
    static constexpr int LP = STEP + 8;         /* LDS row: 16-byte reads of eight consecutive rows hit different banks */
    static constexpr int PART = BT * LP, PARTS = F16 ? 2 : 3;
    struct Tiles {
        __bf16 a[PARTS][PART], b[PARTS][PART]; /* of either type */
    };
    static constexpr size_t LDS_BYTES = 2 * sizeof(Tiles);
};
/* Most columns of b that the tiles take: a tested limit, not a reach.  A lane's 32-bit offset is its column's alone, but the lines
 * have been drawn and tested where a whole step's rows would still fit such offsets. */
template <int WT>
constexpr uint32_t widest_b() {
    constexpr int steps[] = {MfmaShape<WT, false, false>::STEP, MfmaShape<WT, false, true>::STEP, MfmaShape<WT, true, false>::STEP,
                             MfmaShape<WT, true, true>::STEP};
    int most = 0;
    for (int step : steps) most = std::max(most, step);
    return 0xFFFFFFFFu / 4u / (uint32_t)most;
}
static_assert(widest_b<1>() <= widest_b<2>(), "what is too wide for the small tile goes to the large one");
template <int WT, bool NORM>
constexpr size_t MFMA_LDS_BYTES = std::max(MfmaShape<WT, NORM, true>::LDS_BYTES, MfmaShape<WT, NORM, false>::LDS_BYTES);

/* Operands of the f16 form are taken times these: up to 4094 of a and 1023 of b, and in the first step the largest value of each
 * thread's run from 2^-15 and 2^-17 on, so that operands whose results would be found too small are seen before they are
 * multiplied (8192 x 512 . 512 x 1536 with b of deviation 4e-6: 89 us, found at the end 149). */
constexpr float HALF_A = 16.0f, HALF_B = 64.0f, HALF_FIRST = 0x1p-11f;

/* K from which the f16 form is taken, by WT: the error of its parts is that of the longer chain of roundings of the bf16 form
 * at K = 100 and less from there on; 64x64 tiles lose their first two steps of 64 to filling and draining (2048 x 128 . 128 x 1024
 * 7.8 us as bf16, 9.1 as f16; K = 256 10.9 and 11.4; K = 512 19.2 and 16.8), 128x128 ones gain from the start (8192 x 128 .
 * 128 x 1536 36.4 -> 33.0). */
constexpr uint32_t HALF_K[2] = {384, 128};

/* The f16 form holds what it takes apart to 2^-36 absolutely (split_f16.h), so a result may be off by K (A + B) 2^-36, A and B the
 * largest values of its row of a and its column of b as taken apart.  Where no result of a row or of a column within 32
 * rows reaches 2^20 times that -- its values lie far below others, or meet only what is far below others: [1, x] . [x, 1] with x
 * small --, the workgroup starts again as bf16.  (The terms' errors have either sign: of K = 512 a fortieth of the bound, typically.)
 * Zeros are exact: a row or column of nothing else does not count.  Looking at the results, and no longer at each run of values:
 * a layer of 2048 rows and width 512 126.5 -> 122.9 us, 1024 x 512 . 512 x 1024 10.6 -> 10.5; with a run of values out of range in
 * the last step, or a row that ends in such, 8192 x 512 . 512 x 1536 80.0 -> 66.7, the same as without.  Starting again costs
 * the first form's time: 2048 x 512 . 512 x 2048 23.5 us, with such a row 26.8, with a value of 1e5 in the last step 37.5, with
 * all of an operand tiny 29.8. */
__device__ __forceinline__ float half_trusted(uint32_t k, float most) { return (float)k * 0x1p-16f * most; }

/* The largest magnitudes that a workgroup's threads took apart, noted before a barrier */
template <int BT>
struct HalfTops {
    static constexpr uint32_t SHARE = 512u / BT; /* threads of a row of a, neighbours; of a column of b, BT apart */
    float a[BT], b[512];
    float2 wave[8];
    uint32_t lost[8]; /* by wave */
    __device__ __forceinline__ void note(float most_a, float most_b) {
        const uint32_t tid = threadIdx.x;
        static_assert(SHARE == 4u || SHARE == 8u, "a quad or two");
        most_a = fmaxf(most_a, dpp_mov<DPP_XOR1>(most_a)), most_a = fmaxf(most_a, dpp_mov<DPP_XOR2>(most_a));
        if (SHARE == 8u) most_a = fmaxf(most_a, dpp_mov<DPP_HALF_MIRROR>(most_a));
        a[tid / SHARE] = most_a, b[tid] = most_b;
        most_a = across_keys<1>(most_a, OpMax()), most_b = across_keys<1>(most_b, OpMax());
        wave[tid >> 6] = make_float2(most_a, most_b);
    }
    __device__ __forceinline__ float column(uint32_t at) const {
        float t = 0.f;
#pragma unroll
        for (uint32_t s = 0; s < SHARE; s++) t = fmaxf(t, b[s * BT + at]);
        return t;
    }
};

/* Is a row or a column of this wave's 32 rows lost?  sum: as accumulated; lane (h, c) holds of row `row` the columns
 * col0 + 32 j + 8 (r / 4) + 4 h + r % 4.  First with one bound for all, the tile's: two instructions a result, a bit for each
 * that does not reach it.  With bounds of their own where that finds something.
 * rows, cols: how many there are of the output, the last one repeats. */
template <int WT, int BT>
__device__ __forceinline__ bool half_lost(const floatx16 (&sum)[WT], const HalfTops<BT> &tops, uint32_t k, uint32_t row, uint32_t col0,
                                          int rows, int cols) {
    if (rows <= 0 || cols <= 0) return false;
    float2 most = tops.wave[0];
#pragma unroll
    for (int w = 1; w < 8; w++) most = make_float2(fmaxf(most.x, tops.wave[w].x), fmaxf(most.y, tops.wave[w].y));
    const float bound = half_trusted(k, most.x + most.y);
    constexpr uint32_t ALL = WT == 2 ? ~0u : 0xFFFFu;
    uint32_t below = 0u;
#pragma unroll
    for (int j = 0; j < WT; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) below = __builtin_amdgcn_alignbit(below, __float_as_uint(fabsf(sum[j][r]) - bound), 31);
    float column = __uint_as_float(below);
    column = swap16(row0_all(column, OpAnd()), OpAnd());
    const bool none = __float_as_uint(swap32(__uint_as_float(below), OpAnd())) == ALL && tops.a[row] > 0.f;
    if (!__any(none || __float_as_uint(column) != 0u)) return false;

    const uint32_t h = threadIdx.x >> 5 & 1u;
    float row_most = tops.a[row], col_most = 0.f, out = 0.f;
#pragma unroll
    for (int j = 0; j < WT; j++)
#pragma unroll
        for (int r = 0; r < 16; r++)
            col_most = fmaxf(col_most, tops.column(col0 + 32 * j + 8 * (r / 4) + 4 * h + r % 4)), out = fmaxf(out, fabsf(sum[j][r]));
    col_most = swap32(col_most, OpMax()), out = swap32(out, OpMax());
    bool lost = out < half_trusted(k, row_most + col_most) && row_most > 0.f && col_most > 0.f;
    row_most = across_keys<1>(row_most, OpMax());
#pragma unroll
    for (int j = 0; j < WT; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const float t = tops.column(col0 + 32 * j + 8 * (r / 4) + 4 * h + r % 4);
            const uint64_t in = __ballot(!(fabsf(sum[j][r]) < half_trusted(k, row_most + t)) || t == 0.f);
            lost |= row_most > 0.f && ((uint32_t)in == 0u || (uint32_t)(in >> 32) == 0u);
        }
    return lost;
}

/* The sums of a wave over its half of K, scaled (by HALF_A HALF_B, or 2^32), and a thread's share of its row's sum of squares.
 * F16: as f16 parts; most_a, most_b: the largest magnitudes this thread took apart.  Returns true, the same for all threads and with
 * nothing of use in acc, if a run of values of the first step is out of their range.  (One above it later is infinite as f16, and
 * so are its row's or column's results.) */
template <bool VEC, int WT, bool NORM, bool GATED, bool F16>
__device__ __forceinline__ bool mfma_sums(const MatmulArgs &g, unsigned char *lds, floatx16 (&acc)[WT][WT], float &ss, float &most_a,
                                          float &most_b) {
    using Shape = MfmaShape<WT, NORM, F16>;
    constexpr int BT = Shape::BT, EPT = Shape::EPT, LP = Shape::LP, PARTS = Shape::PARTS, TK = Shape::STEP;
    auto *tiles = reinterpret_cast<typename Shape::Tiles *>(lds);
    typedef __bf16 piece __attribute__((ext_vector_type(EPT))); /* of either type */

    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t h = lane >> 5, c = lane & 31u;
    const uint32_t wr = (wave & 3u) >> 1, wc = wave & 1u; /* wave's quadrant of the tile */
    const uint32_t kg = wave >> 2;                         /* its half of a K step */
    constexpr uint32_t COLS = GATED ? BT / 2 : BT; /* columns of a product */
    const uint32_t row0 = blockIdx.y * BT, col0 = blockIdx.x * COLS;

    /* this thread's values of a step: EPT consecutive k of one row of a, of one column of b; rows and columns past the end
     * repeat the last one (their results are not stored), k past the end is zeroed on the way to LDS */
    const uint32_t a_row = tid / (TK / EPT), a_k = (tid % (TK / EPT)) * EPT;
    const uint32_t b_col = tid % BT, b_k = (tid / BT) * EPT;
    const float *const arow = g.a + (size_t)min(row0 + a_row, g.m - 1u) * g.lda;
    /* b or b2: one of them per wave, for the small tile per half of a wave */
    const bool gates = GATED && (WT == 2 ? (wave & 1u) != 0u : b_col >= COLS);
    const uint32_t b_at = min(col0 + b_col % COLS, g.n - 1u);
    /* A wave takes whole rows of b: a row's address is the wave's, and the lane adds its column, one register for all of them.
     * (Not where the lanes of a wave take from both matrices.) */
    constexpr bool ONE = !GATED || WT == 2;
    const float *const bmat = gates ? g.b2 : g.b;
    const uint32_t b_first = ONE ? wave * 64u / BT * EPT : b_k;
    struct Values {
        float a[EPT], b[EPT], w[NORM ? EPT : 1];
    };
    auto request = [&](Values &v, uint32_t k0) __attribute__((always_inline)) {
        const float *b_row = bmat + (size_t)(k0 + b_first) * g.ldb;
        uint32_t column = 4u * b_at;
        asm volatile("" : "+v"(column)); /* row and column kept apart: joined they are a 64-bit sum of the lane for each row */
#pragma unroll
        for (int i = 0; i < EPT; i++, b_row += g.ldb) {
            if constexpr (ONE) {
                auto row = (const __attribute__((address_space(1))) char *)b_row;
                asm("" : "+s"(row));
                v.b[i] = *(const __attribute__((address_space(1))) float *)(row + column);
            } else {
                v.b[i] = b_row[b_at];
            }
        }
#pragma unroll
        for (int i = 0; i < EPT; i += 4) {
            if (VEC) {
                const float4 t = *reinterpret_cast<const float4 *>(arow + k0 + a_k + i);
                v.a[i] = t.x, v.a[i + 1] = t.y, v.a[i + 2] = t.z, v.a[i + 3] = t.w;
            } else {
                v.a[i] = arow[k0 + a_k + i], v.a[i + 1] = arow[k0 + a_k + i + 1];
                v.a[i + 2] = arow[k0 + a_k + i + 2], v.a[i + 3] = arow[k0 + a_k + i + 3];
            }
            if constexpr (NORM) {
                const float *w = g.norm_w + k0 + a_k + i;
                if (VEC) {
                    const float4 t = *reinterpret_cast<const float4 *>(w);
                    v.w[i] = t.x, v.w[i + 1] = t.y, v.w[i + 2] = t.z, v.w[i + 3] = t.w;
                } else {
                    v.w[i] = w[0], v.w[i + 1] = w[1], v.w[i + 2] = w[2], v.w[i + 3] = w[3];
                }
            }
        }
    };
    ss = most_a = most_b = 0.f;
    constexpr float UP_A = F16 ? HALF_A : SPLIT_UP, UP_B = F16 ? HALF_B : SPLIT_UP;
    auto park = [&](const Values &v, uint32_t buf, bool counts) __attribute__((always_inline)) {
        float pa[EPT], pb[EPT], squares = 0.f;
#pragma unroll
        for (int i = 0; i < EPT; i++) {
            if constexpr (NORM) squares = fmaf(v.a[i], v.a[i], squares), pa[i] = v.a[i] * v.w[i] * UP_A;
            else pa[i] = v.a[i] * UP_A;
            pb[i] = v.b[i] * UP_B;
        }
        if constexpr (NORM) ss += counts ? squares : 0.f;
        piece parts[3];
        if constexpr (F16) most_a = fmaxf(most_a, half_top(pa)), most_b = fmaxf(most_b, half_top(pb)), split_f16<EPT>(pa, parts[0], parts[1]);
        else split_bf16<EPT>(pa, parts[0], parts[1], parts[2]);
#pragma unroll
        for (int t = 0; t < PARTS; t++) *reinterpret_cast<piece *>(&tiles[buf].a[t][a_row * LP + a_k]) = parts[t];
        if constexpr (F16) split_f16<EPT>(pb, parts[0], parts[1]);
        else split_bf16<EPT>(pb, parts[0], parts[1], parts[2]);
#pragma unroll
        for (int t = 0; t < PARTS; t++) *reinterpret_cast<piece *>(&tiles[buf].b[t][b_col * LP + b_k]) = parts[t];
    };

    floatx16 small[WT][WT]; /* F16: the products with a low part, times HALF_UP */
#pragma unroll
    for (int i = 0; i < WT; i++)
#pragma unroll
        for (int j = 0; j < WT; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = small[i][j][r] = 0.f;

    struct Fragments {
        bf16x8 a[WT][PARTS][TK / 32], b[WT][PARTS][TK / 32];
    };
    auto read = [&](uint32_t buf, Fragments &f) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < PARTS; t++)
#pragma unroll
            for (int i = 0; i < WT; i++)
#pragma unroll
                for (int k = 0; k < TK / 32; k++) {
                    const uint32_t at = TK / 2u * kg + 16u * k + 8u * h;
                    f.a[i][t][k] = *reinterpret_cast<const bf16x8 *>(&tiles[buf].a[t][(wr * (32u * WT) + 32u * i + c) * LP + at]);
                    f.b[i][t][k] = *reinterpret_cast<const bf16x8 *>(&tiles[buf].b[t][(wc * (32u * WT) + 32u * i + c) * LP + at]);
                }
    };
    auto multiply = [&](const Fragments &f) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < WT; i++)
#pragma unroll
            for (int j = 0; j < WT; j++)
#pragma unroll
                for (int k = 0; k < TK / 32; k++) {
                    if constexpr (F16) {
                        small[i][j] = mfma_f16(f.b[j][1][k], f.a[i][0][k], small[i][j]);
                        acc[i][j] = mfma_f16(f.b[j][0][k], f.a[i][0][k], acc[i][j]);
                        small[i][j] = mfma_f16(f.b[j][0][k], f.a[i][1][k], small[i][j]);
                    } else {
                        const bf16x8 a[3] = {f.a[i][0][k], f.a[i][1][k], f.a[i][2][k]}, b[3] = {f.b[j][0][k], f.b[j][1][k], f.b[j][2][k]};
                        acc[i][j] = mfma_split(b, a, acc[i][j]);
                    }
                }
    };
    /* Whole steps: two register sets take turns, the values of step s+1 and s+2 are on their way while step s
     * runs, so a request has two steps of matrix work to arrive in.  Past the last one it is requested and
     * parked again, into the buffer nobody reads: no branch between the matrix instructions and the split. */
    const uint32_t steps = g.k / TK;
    if (steps != 0u) {
        Values v0, v1;
        auto of_step = [&](uint32_t s) { return min(s, steps - 1u) * TK; };
        request(v0, 0);
        __builtin_amdgcn_sched_barrier(0);
        request(v1, of_step(1u));
        __builtin_amdgcn_sched_barrier(0);
        park(v0, 0, true);
        request(v0, of_step(2u));
        __builtin_amdgcn_sched_barrier(0);
        if (F16) { /* an operand that is out of range is so everywhere, as a rule */
            if (__syncthreads_or(!half_range(most_a, HALF_FIRST) || !half_range(most_b, HALF_FIRST))) return true;
        } else {
            __syncthreads();
        }
        auto step = [&](uint32_t s, Values &v) __attribute__((always_inline)) {
            /* v holds the values of step s+1 */
            Fragments f;
            read(s & 1u, f);
            multiply(f);
            park(v, (s & 1u) ^ 1u, s + 1u < steps);
            if (F16) __builtin_amdgcn_sched_group_barrier(0x100, 4 * WT * TK / 32, 0); /* fragments first */
            /* behind each matrix instruction its share of the step's vector instructions (75 of the large tile as f16, 90 with the
             * norm): eight each, and the last ones had none beside them (8192 x 2048 . 2048 x 1536 193.1 -> 188.9 us) */
            constexpr int SHARE = !F16 ? (WT == 2 ? 4 : 8) : WT == 2 ? (NORM ? 7 : 6) : (NORM ? 16 : 12);
#pragma unroll
            for (int n = 0; n < (F16 ? 3 : 6) * WT * WT * TK / 32; n++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, SHARE, 0);
            }
            request(v, of_step(s + 3u));
            __syncthreads();
        };
        /* In pairs, an odd step behind the loop: with a branch around the second one the compiler made the first wait for all that was
         * on its way, the values of the step after it included, and requests out of order before the loop do the same (2048 rows of a
         * layer of 512 columns 121.4 -> 117.2 us with this and whole rows of b (above), 1500 119.4 -> 113.1, 640 95.5 -> 85.3). */
        uint32_t s = 0;
        for (; s + 1u < steps; s += 2u) {
            step(s, v1);
            step(s + 1u, v0);
        }
        if (s < steps) step(s, v1);
    }
    if (g.k % TK != 0u) { /* what is left of K, zeros behind it */
        const uint32_t k0 = steps * TK;
        Values v;
#pragma unroll
        for (int i = 0; i < EPT; i++) {
            const uint32_t ka = min(k0 + a_k + i, g.k - 1u), kb = min(k0 + b_k + i, g.k - 1u);
            const float x = arow[ka], y = bmat[(size_t)kb * g.ldb + b_at];
            v.a[i] = k0 + a_k + i < g.k ? x : 0.f, v.b[i] = k0 + b_k + i < g.k ? y : 0.f;
            if constexpr (NORM) v.w[i] = g.norm_w[ka];
        }
        park(v, 0, true); /* the loop ended on a barrier */
        __syncthreads();
        Fragments f;
        read(0, f);
        multiply(f);
        __syncthreads();
    }
    if (F16) {
#pragma unroll
        for (int i = 0; i < WT; i++)
#pragma unroll
            for (int j = 0; j < WT; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] = fmaf(small[i][j][r], HALF_DOWN, acc[i][j][r]);
    }
    return false;
}

/* of K, for each of `slices`: whole steps of either form */
__host__ __device__ __forceinline__ uint32_t tile_slice(uint32_t k, uint32_t slices) { return ((k + slices - 1u) / slices + 63u) / 64u * 64u; }

/* Products in slices of K; ALL_BITS: on parts that hold every bit of the operands, bf16 ones from the start */
enum : int { WHOLE, SLICES, SLICES_ALL_BITS };
/* SLICED (small tile): gridDim.z workgroups a tile, each with its run of K as a product of its own; the one that comes last adds
 * up what all of them left, in their order. */
template <bool VEC, bool ROPE, int WT, bool NORM, bool GATED, int SLICED = WHOLE>
__global__ __launch_bounds__(512, WT == 1 ? 4 : 2) void matmul_mfma_kernel(MatmulArgs g) {
    static_assert(SLICED == WHOLE || (WT == 1 && !ROPE && !NORM && !GATED), "plain products");
    if constexpr (SLICED != WHOLE) {
        const uint32_t per = tile_slice(g.k, g.slices), k0 = blockIdx.z * per;
        g.a += k0, g.b += (size_t)k0 * g.ldb;
        g.k = min(per, g.k - k0); /* the launcher leaves no slice empty */
    }
    constexpr int BT = MfmaShape<WT, NORM, true>::BT;
    extern __shared__ __attribute__((aligned(16))) unsigned char mm_lds[];
    __shared__ float row_ss[NORM ? BT : 1];
    __shared__ HalfTops<BT> tops;

    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t h = lane >> 5, c = lane & 31u;
    const uint32_t wr = (wave & 3u) >> 1, wc = wave & 1u; /* wave's quadrant of the tile */
    const uint32_t kg = wave >> 2;                         /* its half of a K step */
    constexpr uint32_t COLS = GATED ? BT / 2 : BT; /* columns of a product */
    const uint32_t row0 = blockIdx.y * BT, col0 = blockIdx.x * COLS;

    /* The two waves of a quadrant add their sums through one area, row by row, once the tile buffers are free: of the large tile each
     * the half that it finishes (row tile `mine`), of the small one all to the first.  The finished quadrant goes back there,
     * and all waves store rows of it: a lane holds a column's worth of rows, so from registers a store (and a load of the
     * rotation or of the residual) would touch 32 rows with 32 bytes each. */
    constexpr uint32_t SIDE = 32u * WT, PITCH = SIDE + 4u, SHARE = 512u / BT; /* SHARE: threads of a row of a, neighbours */
    static_assert(4 * SIDE * PITCH * sizeof(float) <= MFMA_LDS_BYTES<WT, NORM>, "the results pass through the tile buffers");
    const auto area = [&](uint32_t quadrant) { return reinterpret_cast<float *>(mm_lds) + quadrant * (SIDE * PITCH); };
    const auto place = [&](uint32_t tile, int j, int q) {
        return reinterpret_cast<float4 *>(area(wave & 3u) + (32u * tile + c) * PITCH + 32u * j + 8u * q + 4u * h);
    };
    const uint32_t mine = WT == 2 ? kg : 0u;
    const bool finishes = WT == 2 || kg == 0u;
    floatx16 sum[WT];
    auto meet = [&](const floatx16 (&acc)[WT][WT], float ss) __attribute__((always_inline)) {
        if constexpr (NORM) {
#pragma unroll
            for (uint32_t d = 1u; d < SHARE; d *= 2u) ss += __shfl_xor(ss, (int)d, 64);
            if (tid % SHARE == 0u) row_ss[tid / SHARE] = ss;
        }
#pragma unroll
        for (int j = 0; j < WT; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                float4 give;
                float *const g4 = &give.x;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    g4[e] = WT == 2 && kg != 0u ? acc[0][j][4 * q + e] : acc[WT - 1][j][4 * q + e];
                    sum[j][4 * q + e] = WT == 2 && kg != 0u ? acc[WT - 1][j][4 * q + e] : acc[0][j][4 * q + e];
                }
                if (WT == 2 || kg == 1u) *place(WT == 2 ? 1u - kg : 0u, j, q) = give;
            }
        __syncthreads();
        if (!finishes) return;
#pragma unroll
        for (int j = 0; j < WT; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float4 got = *place(mine, j, q);
                sum[j][4 * q + 0] += got.x, sum[j][4 * q + 1] += got.y, sum[j][4 * q + 2] += got.z, sum[j][4 * q + 3] += got.w;
            }
    };

    const bool gate_wave = GATED && wc == 1u;
    const uint32_t wave_col = col0 + (GATED ? 0u : wc * SIDE), my_row = SIDE * wr + 32u * mine + c;
    MatmulArgs to = g;
    const bool joined = GATED && g.out2 == nullptr; /* four waves a pair of quadrants then, two a quadrant else */
    if (gate_wave && !joined) to.out = g.out2, to.residual = nullptr;
    const bool vst = VEC && g.n % 4u == 0u && (g.ldo % 4u == 0u) && ((reinterpret_cast<uintptr_t>(to.out) & 15u) == 0u) &&
                     ((reinterpret_cast<uintptr_t>(to.residual) & 15u) == 0u);
    constexpr uint32_t PER = SIDE / 4u, ROWS = 64u / PER; /* lanes a row, rows at once */
    const uint32_t share = joined ? SIDE / 4u : SIDE / 2u, first = (joined ? 2u * wc + kg : kg) * share;
    const float *const from = area(joined ? 2u * wr : wave & 3u), *const gates = area(2u * wr + 1u);

    /* What the end needs from memory, the rotation or the residual of this thread's pieces, asked for while the waves of a quadrant meet:
     * asked for where it is used, piece after piece, each waits behind the store
     * and the branch of the one before (2048 rows of a layer of 512 columns 116.3 -> 113.6 us, 1500 113.0 -> 110.5, 301 62.5 -> 61.6). */
    constexpr int PIECES = SIDE / 2u / ROWS;
    float4 extra[PIECES]; /* cosines and sines, or the residual */
    const bool rotates = ROPE && !g.stage_k && wave_col < g.rope_cols;
    const bool prompt = !GATED && vst && (ROPE ? rotates && !to.residual : to.residual != nullptr);
    auto ask = [&]() __attribute__((always_inline)) {
        if (!prompt) return;
        const uint32_t col = lane % PER * 4u;
#pragma unroll
        for (int i = 0; i < PIECES; i++) { /* past the end: the last row or column again */
            const uint32_t row = min(row0 + SIDE * wr + first + min(ROWS * i, share - 1u) + lane / PER, g.m - 1u);
            if constexpr (ROPE) {
                const size_t at = (size_t)row * (g.head_dim / 2u) + ((wave_col + col) % g.head_dim) / 2u;
                const float2 c2 = *reinterpret_cast<const float2 *>(g.rope_cos + at), s2 = *reinterpret_cast<const float2 *>(g.rope_sin + at);
                extra[i] = make_float4(c2.x, c2.y, s2.x, s2.y);
            } else {
                extra[i] = *reinterpret_cast<const float4 *>(to.residual + (size_t)row * g.ldo + min(wave_col + col, g.n - 4u));
            }
        }
    };

    /* the finished rows, back to the area */
    auto put = [&]() __attribute__((always_inline)) {
        const float scale = NORM ? 1.0f / sqrtf(row_ss[my_row] / (float)g.k + 1e-6f) : 1.0f; /* reductions_cpu.c:345-346 */
#pragma unroll
        for (int j = 0; j < WT; j++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                *place(mine, j, q) = make_float4(sum[j][4 * q + 0] * scale, sum[j][4 * q + 1] * scale, sum[j][4 * q + 2] * scale,
                                                 sum[j][4 * q + 3] * scale);
    };

    /* One result in some thousand does not reach half_lost()'s bound because its terms happen to cancel.  Where one to three rows
     * or columns are by themselves at an edge, such a one would be all of a column, and some tile of nearly every launch start again
     * (200 x 512 . 512 x 2048 10.9 -> 18.9 us): bf16 from the start. */
    const auto few = [](uint32_t left, uint32_t whole, uint32_t block) { return left < whole && left % block - 1u < 3u; };
    bool half = SLICED != SLICES_ALL_BITS && g.k >= HALF_K[WT - 1] && !few(g.m - row0, BT, 32u) && !few(g.n - col0, COLS, SIDE);
    if (half) {
        floatx16 acc[WT][WT];
        float ss, most_a, most_b;
        half = !mfma_sums<VEC, WT, NORM, GATED, true>(g, mm_lds, acc, ss, most_a, most_b);
        if (half) {
            tops.note(most_a, most_b);
            ask();
            meet(acc, ss);
            bool lost = false;
            if (finishes) {
                lost = half_lost<WT, BT>(sum, tops, g.k, my_row, wc * SIDE, (int)(g.m - row0) - (int)(my_row - c), (int)(g.n - wave_col));
#pragma unroll
                for (int j = 0; j < WT; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) lost |= !isfinite(sum[j][r]), sum[j][r] *= 1.0f / (HALF_A * HALF_B);
                put();
            }
            lost = __any(lost);
            if (lane == 0u) tops.lost[wave] = lost;
            __syncthreads();
            uint32_t any = 0u;
#pragma unroll
            for (int w = 0; w < 8; w++) any |= tops.lost[w];
            half = any == 0u;
        }
    }
    if (!half) {
        floatx16 acc[WT][WT];
        float ss, none;
        mfma_sums<VEC, WT, NORM, GATED, false>(g, mm_lds, acc, ss, none, none);
        ask();
        meet(acc, ss);
        if (finishes) {
            bool bad = false;
#pragma unroll
            for (int j = 0; j < WT; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    bad |= !isfinite(sum[j][r]);
                    sum[j][r] *= SPLIT_DOWN;
                }
            if (__any(bad)) {
                /* something is not finite, or too large for the scaled sums: these rows again on the fp32 instructions, which
                 * tell infinities from NaN */
                const float *ar = g.a + (size_t)min(row0 + my_row, g.m - 1u) * g.lda;
#pragma unroll
                for (int j = 0; j < WT; j++) {
                    const float *bc = (gate_wave ? g.b2 : g.b) + min(wave_col + 32u * j + c, g.n - 1u);
#pragma unroll
                    for (int r = 0; r < 16; r++) sum[j][r] = 0.f;
                    /* sums of 64, then their sum: closer than one chain (K = 512: 1.5e-7 against 4.1e-7) */
                    for (uint32_t k0 = 0; k0 < g.k; k0 += 64u) {
                        floatx16 part;
#pragma unroll
                        for (int r = 0; r < 16; r++) part[r] = 0.f;
                        for (uint32_t k = k0 + h; k < min(k0 + 64u, g.k) + h; k += 2u) { /* an odd K ends with a product of zeros */
                            float x = k < g.k ? ar[k] : 0.f;
                            const float y = k < g.k ? bc[(size_t)k * g.ldb] : 0.f;
                            if (NORM && k < g.k) x *= g.norm_w[k];
                            part = __builtin_amdgcn_mfma_f32_32x32x2f32(y, x, part, 0, 0, 0);
                        }
                        sum[j] += part;
                    }
                }
            }
            put();
        }
        __syncthreads();
    }

    float4 total[SLICED != WHOLE ? PIECES : 1];
    if constexpr (SLICED != WHOLE) {
        /* device-scope stores and loads, and an explicit wait for the stores' completion before the barrier that precedes this
         * workgroup's ticket, as for the split states of the KV step (kv_step.h) */
        __shared__ uint32_t ticket;
        constexpr uint32_t WORDS = BT * BT / 2; /* a slice's sums, two a word */
        const uint32_t tile = blockIdx.y * gridDim.x + blockIdx.x;
        uint64_t *const words = reinterpret_cast<uint64_t *>(g.slice_sums) + (size_t)tile * g.slices * WORDS + tid;
        uint64_t *const own = words + (size_t)blockIdx.z * WORDS;
#pragma unroll
        for (int i = 0; i < PIECES; i++) {
            const float4 v = *reinterpret_cast<const float4 *>(from + (first + ROWS * i + lane / PER) * PITCH + lane % PER * 4u);
            __hip_atomic_store(own + (2 * i) * 512, (uint64_t)__float_as_uint(v.y) << 32 | __float_as_uint(v.x), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(own + (2 * i + 1) * 512, (uint64_t)__float_as_uint(v.w) << 32 | __float_as_uint(v.z), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
        blt_vector_memory_done(); /* every wave's sums are out before thread 0 draws the ticket */
        __syncthreads();
        if (tid == 0u) ticket = __hip_atomic_fetch_add(&g.slice_tickets[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (ticket != g.slices - 1u) return;
        if (tid == 0u) g.slice_tickets[tile] = 0u; /* re-armed for the next launch */
        static_assert(4 * PIECES * 512 == BT * BT, "a thread's pieces are all of a slice's sums");
#pragma unroll
        for (int i = 0; i < PIECES; i++) total[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        for (uint32_t z = 0; z < g.slices; z += 2u) { /* slice order, whoever comes last; two on their way */
            uint64_t t[2][2 * PIECES];
#pragma unroll
            for (uint32_t u = 0; u < 2u; u++)
#pragma unroll
                for (int i = 0; i < 2 * PIECES; i++)
                    t[u][i] = __hip_atomic_load(words + (size_t)min(z + u, g.slices - 1u) * WORDS + i * 512, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (uint32_t u = 0; u < 2u; u++) {
                if (z + u >= g.slices) break;
#pragma unroll
                for (int i = 0; i < PIECES; i++) {
                    total[i].x += __uint_as_float((uint32_t)t[u][2 * i]), total[i].y += __uint_as_float((uint32_t)(t[u][2 * i] >> 32));
                    total[i].z += __uint_as_float((uint32_t)t[u][2 * i + 1]), total[i].w += __uint_as_float((uint32_t)(t[u][2 * i + 1] >> 32));
                }
            }
        }
    }
#pragma unroll
    for (uint32_t r = 0; r < SIDE / 2u; r += ROWS) {
        if (r >= share) break;
        const uint32_t at = first + r + lane / PER, col = lane % PER * 4u;
        const uint32_t row = row0 + SIDE * wr + at;
        float4 v = SLICED != WHOLE ? total[SLICED != WHOLE ? r / ROWS : 0] : *reinterpret_cast<const float4 *>(from + at * PITCH + col);
        if (joined) {
            const float4 gate = *reinterpret_cast<const float4 *>(gates + at * PITCH + col);
            v.x = silu_times(gate.x, v.x), v.y = silu_times(gate.y, v.y), v.z = silu_times(gate.z, v.z), v.w = silu_times(gate.w, v.w);
        }
        if (row >= g.m) continue;
        if (!prompt) {
            matmul_store4<ROPE>(to, row, wave_col + col, v, vst);
            continue;
        }
        const float4 e = extra[r / ROWS];
        if constexpr (ROPE) {
            if (wave_col + col < g.rope_cols) v = rope_rotate4(v, make_float2(e.x, e.y), make_float2(e.z, e.w));
        } else {
            v.x = e.x + v.x, v.y = e.y + v.y, v.z = e.z + v.z, v.w = e.w + v.w;
        }
        if (wave_col + col < g.n) *reinterpret_cast<float4 *>(to.out + (size_t)row * g.ldo + wave_col + col) = v;
    }
}

/* 32x32 output tile (bx, by) per workgroup, K split over the NW waves (4, or 8 for long K:
 * the serial chain of chunk loads per wave halves); the first four waves finish the tile. */
template <bool VEC, bool ROPE, bool GATED, int NW = 4, bool CROSS = false>
__device__ __forceinline__ void splitk_tile(const MatmulArgs &g, const uint32_t bx, const uint32_t by,
                                            float (*part)[16][64], float (*part_ss)[32], float *qt = nullptr) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t h = lane >> 5, c = lane & 31u;
    const uint32_t row = by * 32u + c, col = bx * 32u + c;
    const float *arow = g.a + (size_t)min(row, g.m - 1u) * g.lda;
    const float *bcol = g.b + min(col, g.n - 1u);
    const float *b2col = GATED ? g.b2 + min(col, g.n - 1u) : nullptr;

    float ss = 0.f; /* this lane's share of sum_k a[row][k]^2 (norm_w only) */
    /* fragments of one 32-wide K chunk: lane (h, c) holds a[row][k0 + 16h + t] and b[k0 + 16h + t][col] */
    /* Every load of a chunk is issued before anything waits: addresses past K are clamped to the
     * last valid element and the value replaced by zero afterwards, so no load sits behind a
     * branch, and the norm arithmetic (which needs the a values) comes after the b requests. */
    auto fetch = [&](uint32_t k0, float (&fa)[16], float (&fb)[16], float (&fg)[16]) __attribute__((always_inline)) {
        const uint32_t kb = k0 + 16u * h;
        if (VEC) { /* K is a multiple of 4 here: a 16-byte piece is inside or outside as a whole */
#pragma unroll
            for (int t = 0; t < 16; t += 4) {
                const float4 v = *reinterpret_cast<const float4 *>(arow + min(kb + t, g.k - 4u));
                const bool in = kb + t < g.k;
                fa[t + 0] = in ? v.x : 0.f, fa[t + 1] = in ? v.y : 0.f;
                fa[t + 2] = in ? v.z : 0.f, fa[t + 3] = in ? v.w : 0.f;
            }
        } else {
#pragma unroll
            for (int t = 0; t < 16; t++) {
                const float v = arow[min(kb + t, g.k - 1u)];
                fa[t] = kb + t < g.k ? v : 0.f;
            }
        }
#pragma unroll
        for (int t = 0; t < 16; t++) {
            const float v = bcol[(size_t)min(kb + t, g.k - 1u) * g.ldb];
            fb[t] = kb + t < g.k ? v : 0.f;
        }
        if (GATED) {
#pragma unroll
            for (int t = 0; t < 16; t++) {
                const float v = b2col[(size_t)min(kb + t, g.k - 1u) * g.ldb];
                fg[t] = kb + t < g.k ? v : 0.f;
            }
        }
        if (g.norm_w) { /* uniform: sum of squares of the raw row, then the norm weight folded into a */
            float nw[16];
#pragma unroll
            for (int t = 0; t < 16; t++) nw[t] = g.norm_w[min(kb + t, g.k - 1u)];
#pragma unroll
            for (int t = 0; t < 16; t++) {
                ss += fa[t] * fa[t];
                fa[t] *= nw[t]; /* fa is already zero past K */
            }
        }
    };

    floatx16 acc, acc2;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.f, acc2[r] = 0.f;
    uint32_t chunks = (g.k + 31u) / 32u, first = 0u;
    if (g.slices > 1u) { /* this workgroup's share of the chunks */
        const uint32_t per = (chunks + g.slices - 1u) / g.slices;
        first = min(blockIdx.z * per, chunks);
        chunks = min(first + per, chunks);
    }
    float fa[16], fb[16], fg[GATED ? 16 : 1];
    float dummy[GATED ? 1 : 16]; /* stands in for the gate fragment when there is none */
    (void)dummy;
    uint32_t ch = first + wave;
    if (ch < chunks) {
        if constexpr (GATED) fetch(ch * 32u, fa, fb, fg);
        else fetch(ch * 32u, fa, fb, dummy);
    }
    while (ch < chunks) {
        const uint32_t nx = ch + (uint32_t)NW;
        float na[16], nb[16], ng[GATED ? 16 : 1];
        if (nx < chunks) {
            if constexpr (GATED) fetch(nx * 32u, na, nb, ng);
            else fetch(nx * 32u, na, nb, dummy);
        }
#pragma unroll
        for (int t = 0; t < 16; t++) {
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[t], fa[t], acc, 0, 0, 0);
            if (GATED) acc2 = __builtin_amdgcn_mfma_f32_32x32x2f32(fg[t], fa[t], acc2, 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < 16; t++) {
            fa[t] = na[t], fb[t] = nb[t];
            if (GATED) fg[t] = ng[t];
        }
        ch = nx;
    }

#pragma unroll
    for (int r = 0; r < 16; r++) {
        part[wave][r][lane] = acc[r];
        if (GATED) part[NW + wave][r][lane] = acc2[r];
    }
    if (g.norm_w) {
        ss += __shfl_xor(ss, 32, 64);
        if (h == 0) part_ss[wave][c] = ss;
    }
    __syncthreads();
    if (NW > 4 && wave >= 4u) return; /* no barrier follows */
    float row_scale = 1.0f;
    if (g.norm_w) {
        float tot = (part_ss[0][c] + part_ss[1][c]) + (part_ss[2][c] + part_ss[3][c]);
        if (NW > 4) tot += (part_ss[4][c] + part_ss[5][c]) + (part_ss[6][c] + part_ss[7][c]);
        row_scale = 1.0f / sqrtf(tot / (float)g.k + 1e-6f); /* reductions_cpu.c:345-346 */
    }
    /* wave w < 4 finishes register group w: out[row][col0 + 8w + 4h + 0..3] */
    auto total = [&](uint32_t first, uint32_t reg) __attribute__((always_inline)) {
        float t = (part[first + 0][reg][lane] + part[first + 1][reg][lane]) +
                  (part[first + 2][reg][lane] + part[first + 3][reg][lane]);
        if (NW > 4)
            t += (part[first + 4][reg][lane] + part[first + 5][reg][lane]) +
                 (part[first + 6][reg][lane] + part[first + 7][reg][lane]);
        return t;
    };
    float v4[4], second[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        v4[i] = total(0u, 4u * wave + i) * row_scale;
        if (GATED) {
            const float gate = total((uint32_t)NW, 4u * wave + i) * row_scale;
            if (g.out2) second[i] = gate; /* two products, two outputs */
            else v4[i] = silu_times(gate, v4[i]);
        }
    }
    if (!GATED && !CROSS && g.slices > 1u) {
        /* Device-scope stores and loads, and an explicit wait for the stores' completion before the
         * barrier that precedes this workgroup's ticket, as for the split softmax states of the
         * KV step (kv_step.h).  The waves past the fourth have left. */
        __shared__ uint32_t ticket;
        const uint32_t tile = by * gridDim.x + bx;
        float *sums = g.slice_sums + (size_t)tile * g.slices * 1024u + 4u * threadIdx.x;
#pragma unroll
        for (int i = 0; i < 4; i++)
            __hip_atomic_store(sums + (size_t)blockIdx.z * 1024u + i, v4[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        blt_vector_memory_done(); /* every wave's sums are out before thread 0 draws the ticket */
        __syncthreads();
        if (threadIdx.x == 0)
            ticket = __hip_atomic_fetch_add(&g.slice_tickets[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (ticket != g.slices - 1u) return;
        if (threadIdx.x == 0) g.slice_tickets[tile] = 0u; /* re-armed for the next launch */
#pragma unroll
        for (int i = 0; i < 4; i++) v4[i] = __hip_atomic_load(sums + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        for (uint32_t z = 1; z < g.slices; z++) /* slice order, whoever comes last */
#pragma unroll
            for (int i = 0; i < 4; i++)
                v4[i] += __hip_atomic_load(sums + (size_t)z * 1024u + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (CROSS) {
        /* The tile is the projected query of 32 rows for head bx: park it, then wave w takes rows
         * 8w .. 8w+7 with eight lanes per row (four columns each).  Softmax as
         * blt_softmax_masked_row_inplace: maximum over finite scores, non-finite scores weigh
         * nothing, an empty or all-dead row gives zeros (same statements as kv_cross_rows_kernel). */
#pragma unroll
        for (int i = 0; i < 4; i++) qt[c * 33u + 8u * wave + 4u * h + i] = v4[i];
        __syncthreads(); /* the waves past the fourth have left */
        const uint32_t rr = 8u * wave + (lane >> 3), s8 = lane & 7u;
        const uint32_t R = by * 32u + rr;
        if (R >= g.m) return;
        const float4 q4 = make_float4(qt[rr * 33u + 4u * s8], qt[rr * 33u + 4u * s8 + 1u], qt[rr * 33u + 4u * s8 + 2u],
                                      qt[rr * 33u + 4u * s8 + 3u]);
        const uint32_t lo = g.cross_lo[R], hi = g.cross_hi[R];
        const size_t base = (size_t)(R / g.cross_rows_per_seq) * g.cross_slab_rows * g.n + bx * 32u + 4u * s8;
        auto score = [&](uint32_t j) {
            const float4 k4 = *reinterpret_cast<const float4 *>(g.cross_k + base + (size_t)j * g.n);
            float p = q4.x * k4.x + q4.y * k4.y + q4.z * k4.z + q4.w * k4.w;
            p += __shfl_xor(p, 1, 64);
            p += __shfl_xor(p, 2, 64);
            p += __shfl_xor(p, 4, 64);
            return p * g.cross_scale;
        };
        float mx = -__builtin_huge_valf();
        for (uint32_t j = lo; j < hi; j++) {
            const float sc = score(j);
            if (isfinite(sc)) mx = fmaxf(mx, sc);
        }
        float sum = 0.f;
        float4 o4 = make_float4(0.f, 0.f, 0.f, 0.f);
        for (uint32_t j = lo; j < hi; j++) {
            const float sc = score(j);
            const float e = isfinite(sc) ? expf(sc - mx) : 0.f;
            if (e == 0.f) continue;
            sum += e;
            const float4 vv = *reinterpret_cast<const float4 *>(g.cross_v + base + (size_t)j * g.n);
            o4.x += e * vv.x, o4.y += e * vv.y, o4.z += e * vv.z, o4.w += e * vv.w;
        }
        const float inv = sum > 0.f ? 1.0f / sum : 0.f;
        *reinterpret_cast<float4 *>(g.cross_out + (size_t)R * g.n + bx * 32u + 4u * s8) =
            make_float4(o4.x * inv, o4.y * inv, o4.z * inv, o4.w * inv);
        return;
    }
    if (row >= g.m) return;
    const bool vst = VEC && (g.ldo % 4u == 0u) && ((reinterpret_cast<uintptr_t>(g.out) & 15u) == 0u) &&
                     ((reinterpret_cast<uintptr_t>(g.residual) & 15u) == 0u) &&
                     ((reinterpret_cast<uintptr_t>(g.out2) & 15u) == 0u);
    const uint32_t oc = bx * 32u + 8u * wave + 4u * h;
    matmul_store4<ROPE>(g, row, oc, make_float4(v4[0], v4[1], v4[2], v4[3]), vst);
    if (GATED && g.out2) {
        MatmulArgs g2 = g;
        g2.out = g.out2;
        g2.residual = nullptr;
        matmul_store4<false>(g2, row, oc, make_float4(second[0], second[1], second[2], second[3]), vst);
    }
}

/* WAVES: registers for as many on a SIMD.  Left alone the compiler takes three registers more than four allow, and then a compute unit
 * holds one workgroup of eight waves: a product of 384 tiles (512 x 256 x 768) took 7.5 us, 6.5 with two at a time.  Where each
 * has a compute unit to itself the limit costs a little (512 x 1024 x 256 in two slices 8.55 / 8.76). */
template <bool VEC, bool ROPE, bool GATED, int NW = 4, bool CROSS = false, int WAVES = 2>
__global__ __launch_bounds__(64 * NW, WAVES) void matmul_splitk_kernel(MatmulArgs g) {
    __shared__ float part[(GATED ? 2 : 1) * NW][16][64];
    __shared__ float part_ss[NW][32];
    __shared__ float qt[CROSS ? 32 * 33 : 1];
    splitk_tile<VEC, ROPE, GATED, NW, CROSS>(g, blockIdx.x, blockIdx.y, part, part_ss, qt);
}

/* Two independent products in one launch: the tile rows of the second are
 * stacked under those of the first (rows0 tile rows); the second carries a
 * second weight matrix, the first too if BOTH, or the first is rotated if ROPE.  For pairs of small products whose launches would
 * otherwise each pay the fixed launch cost. */
template <bool VEC, bool BOTH, bool ROPE = false>
__global__ __launch_bounds__(256, 2) void matmul_splitk_pair_kernel(MatmulArgs g0, MatmulArgs g1, uint32_t rows0) {
    __shared__ float part[8][16][64];
    __shared__ float part_ss[4][32];
    if (blockIdx.y < rows0) { /* uniform per workgroup */
        if (blockIdx.x * 32u >= g0.n) return;
        splitk_tile<VEC, ROPE, BOTH>(g0, blockIdx.x, blockIdx.y, part, part_ss);
    } else {
        if (blockIdx.x * 32u >= g1.n) return;
        splitk_tile<VEC, false, true>(g1, blockIdx.x, blockIdx.y - rows0, part, part_ss);
    }
}

constexpr uint32_t SKINNY_KC = 512; /* k values of the a rows staged in LDS at a time */

/* One output column per thread, R rows of a per workgroup (grid.y walks the row groups).  Every
 * output is the reference's own sum: k ascending, product and sum rounded separately.  What the
 * kernel is built around is the latency of that serial chain: the rows of a sit in LDS (one
 * broadcast 16-byte read per four k), the column of b is fetched sixteen k ahead of the chain --
 * the requests of block t+1 are in flight while block t is summed -- and every row gets a thread
 * per column of its own (R = 1 at launch) rather than a share of a thread. */
template <int R, bool GATED, bool CROSS = false>
__global__ __launch_bounds__(256) void matmul_skinny_kernel(MatmulArgs g) {
#pragma clang fp contract(off) /* product and sum rounded separately, as the reference's loop */
    constexpr uint32_t KC = SKINNY_KC, UN = 16;
    __shared__ __attribute__((aligned(16))) float sa[R][KC];
    __shared__ float inv_rms[R];
    __shared__ float sq[CROSS ? R : 1][CROSS ? 256 : 1]; /* the projected rows, for the cross-attention epilogue */
    const uint32_t jj = blockIdx.x * 256u + threadIdx.x;
    const uint32_t j = min(jj, g.n - 1u);
    const uint32_t r0 = blockIdx.y * R;
    float acc[R], acc2[R];
#pragma unroll
    for (int r = 0; r < R; r++) acc[r] = 0.0f, acc2[r] = 0.0f;
    const float *bcol = g.b + j;
    const float *gcol = GATED ? g.b2 + j : nullptr;
    for (uint32_t kc = 0; kc < g.k; kc += KC) {
        const uint32_t klen = min(KC, g.k - kc);
        __syncthreads(); /* the previous chunk has been consumed */
        for (uint32_t t = threadIdx.x; t < R * KC; t += 256u) {
            const uint32_t r = t / KC, kk = t % KC;
            const uint32_t row = min(r0 + r, g.m - 1u);
            sa[r][kk] = g.a[(size_t)row * g.lda + kc + min(kk, klen - 1u)];
        }
        __syncthreads();
        if (g.norm_w) { /* uniform; the host sends such a product here only when k <= KC (one chunk) */
            /* the reference's row norm (csrc/ops/reductions_cpu.c:325-352) on the staged rows: sum of
             * squares in element order by one lane per row, then x * inv_rms * w element by element */
            if ((threadIdx.x & 63u) == 0 && (threadIdx.x >> 6) < (uint32_t)R) {
                const uint32_t r = threadIdx.x >> 6;
                float sumsq = 0.0f;
                uint32_t q = 0;
                for (; q + 4u <= klen; q += 4u) {
                    const float4 t = *reinterpret_cast<const float4 *>(&sa[r][q]);
                    sumsq = sumsq + t.x * t.x;
                    sumsq = sumsq + t.y * t.y;
                    sumsq = sumsq + t.z * t.z;
                    sumsq = sumsq + t.w * t.w;
                }
                for (; q < klen; q++) sumsq = sumsq + sa[r][q] * sa[r][q];
                inv_rms[r] = 1.0f / sqrtf(sumsq / (float)klen + 1e-6f);
            }
            __syncthreads();
            for (uint32_t t = threadIdx.x; t < R * KC; t += 256u) {
                const uint32_t r = t / KC, kk = t % KC;
                if (kk < klen) sa[r][kk] = sa[r][kk] * inv_rms[r] * g.norm_w[kk];
            }
            __syncthreads();
        }
        const uint32_t full = klen / UN * UN;
        if (full) {
            float bv[UN], gv[UN];
#pragma unroll
            for (uint32_t u = 0; u < UN; u++) {
                bv[u] = bcol[(size_t)(kc + u) * g.ldb];
                gv[u] = GATED ? gcol[(size_t)(kc + u) * g.ldb] : 0.0f;
            }
            for (uint32_t k0 = 0; k0 < full; k0 += UN) {
                /* the next block's column values (the last round fetches its own block again) */
                const uint32_t kn = kc + min(k0 + UN, full - UN);
                float nb[UN], ng[UN];
#pragma unroll
                for (uint32_t u = 0; u < UN; u++) {
                    nb[u] = bcol[(size_t)(kn + u) * g.ldb];
                    ng[u] = GATED ? gcol[(size_t)(kn + u) * g.ldb] : 0.0f;
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (uint32_t u4 = 0; u4 < UN; u4 += 4) {
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        const float4 a4 = *reinterpret_cast<const float4 *>(&sa[r][k0 + u4]);
                        const float av[4] = {a4.x, a4.y, a4.z, a4.w};
#pragma unroll
                        for (int t = 0; t < 4; t++) {
                            acc[r] = acc[r] + av[t] * bv[u4 + t];
                            if (GATED) acc2[r] = acc2[r] + av[t] * gv[u4 + t];
                        }
                    }
                }
#pragma unroll
                for (uint32_t u = 0; u < UN; u++) bv[u] = nb[u], gv[u] = ng[u];
            }
        }
        for (uint32_t k = full; k < klen; k++) {
            const float bj = bcol[(size_t)(kc + k) * g.ldb];
            const float gj = GATED ? gcol[(size_t)(kc + k) * g.ldb] : 0.0f;
#pragma unroll
            for (int r = 0; r < R; r++) {
                acc[r] = acc[r] + sa[r][k] * bj;
                if (GATED) acc2[r] = acc2[r] + sa[r][k] * gj;
            }
        }
    }
    if (CROSS) { /* one workgroup holds whole rows (n <= 256): a wave per (row, head) */
#pragma unroll
        for (int r = 0; r < R; r++) sq[r][threadIdx.x] = acc[r];
        __syncthreads();
        const uint32_t xhd = g.cross_head_dim, heads = g.n / xhd;
        for (uint32_t p = threadIdx.x >> 6; p < (uint32_t)R * heads; p += 4u) {
            const uint32_t r = p / heads, hh = p % heads, row = r0 + r;
            if (row >= g.m) continue;
            const size_t slab = (size_t)(row / g.cross_rows_per_seq) * g.cross_slab_rows * g.n + hh * xhd;
            cross_row_head(&sq[r][hh * xhd], g.cross_k + slab, g.cross_v + slab, g.cross_lo[row], g.cross_hi[row], g.n,
                           xhd, g.cross_scale, g.cross_out + (size_t)row * g.n + hh * xhd, threadIdx.x & 63u);
        }
        return;
    }
    if (jj >= g.n) return;
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (r0 + r >= g.m) continue;
        float v = (GATED && !g.out2) ? silu_times(acc2[r], acc[r]) : acc[r];
        if (g.residual) v = g.residual[(size_t)(r0 + r) * g.ldo + j] + v;
        g.out[(size_t)(r0 + r) * g.ldo + j] = v;
        if (GATED && g.out2) g.out2[(size_t)(r0 + r) * g.ldo + j] = acc2[r];
    }
}

template <int R>
void launch_skinny(const MatmulArgs &g, hipStream_t s) {
    const dim3 grid((g.n + 255u) / 256u, (g.m + R - 1u) / R);
    if (g.cross_k) blt_launch("matmul_skinny_cross", matmul_skinny_kernel<R, false, true>, grid, dim3(256), 0, s, g);
    else if (g.b2) blt_launch("matmul_skinny", matmul_skinny_kernel<R, true>, grid, dim3(256), 0, s, g);
    else blt_launch("matmul_skinny", matmul_skinny_kernel<R, false>, grid, dim3(256), 0, s, g);
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

} // namespace

namespace {

enum Path { PATH_SKINNY, PATH_SPLITK, PATH_MFMA };

Path choose_path(const MatmulArgs &g) {
    const bool rope = g.rope_cos != nullptr && g.rope_cols > 0;
    /* up to this many rows the thread-per-column kernel, whose sums run in the reference's order
     * (bit-identical results) */
    constexpr uint32_t exact_rows = 32u;
    if (g.m <= exact_rows && !rope && !g.tolerant) return PATH_SKINNY;
    /* up to 111 64x64 tiles (a bit under half the compute units), 79 of a pair of products: quarter tiles, K split
     * over the waves.  Measured in whole blocks: 108 tiles of K = 128 a tenth of a product faster than on the tile kernel,
     * 128 ... 132 tiles of K = 256 ... 1024 a tenth slower; pairs of 72 tiles of K = 128 faster, of 80 and 128
     * tiles of K = 256 and 512 slower (block of 200 rows of 512: 54.8 -> 49.7 us on the tile kernel). */
    const uint64_t splitk_below = g.b2 ? 80u : 112u;
    /* wider than the tile kernel has been tested (widest_b); this one computes every address in 64 bits */
    if (g.ldb > widest_b<2>()) return PATH_SPLITK;
    /* one or two products an element: three parts drop the bits that fp32 rounds them to (error against float64 3.5e-8
     * and 3.4e-8, on the fp32 instructions 2.5e-8 and 3.1e-8; from three on the parts are closer, 3.3e-8 against 3.6e-8) */
    if (g.k < 3u) return PATH_SPLITK;
    if ((uint64_t)((g.n + TN - 1) / TN) * ((g.m + TM - 1) / TM) < splitk_below) return PATH_SPLITK;
    return PATH_MFMA;
}

struct SliceScratch {
    float *sums = nullptr;
    size_t sum_floats = 0;
    uint32_t *tickets = nullptr;
    size_t ticket_count = 0;
};
__global__ void clear_words_kernel(uint32_t *w, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256u + threadIdx.x;
    if (i < n) w[i] = 0u;
}

} // namespace

bool matmul_slice_scratch(size_t floats, size_t count, hipStream_t s, float **sums, uint32_t **tickets) {
    if (blt_stream_captured_by_caller(s)) return false;
    static thread_local std::map<hipStream_t, SliceScratch> by_stream;
    SliceScratch &sc = by_stream[blt_stream_key()];
    if (blt_stream_capturing() && (floats > sc.sum_floats || count > sc.ticket_count)) return false;
    /* outgrown buffers are left to the process: a launch still in flight may be using them */
    if (floats > sc.sum_floats) {
        sc.sum_floats = std::max(floats, 2 * sc.sum_floats);
        HIP_CHECK(hipMalloc((void **)&sc.sums, sc.sum_floats * sizeof(float)));
    }
    if (count > sc.ticket_count) {
        sc.ticket_count = std::max<size_t>(2 * count, 1024);
        HIP_CHECK(hipMalloc((void **)&sc.tickets, sc.ticket_count * sizeof(uint32_t)));
        /* a fill kernel, not a memset, on the stream the launches follow */
        blt_launch("matmul_clear_words", clear_words_kernel, dim3((unsigned)((sc.ticket_count + 255) / 256)), dim3(256), 0,
                   s ? s : blt_stream(), sc.tickets, sc.ticket_count);
    }
    *sums = sc.sums;
    *tickets = sc.tickets;
    return true;
}

namespace {

/* Slices of K per output tile: long K over few tiles leaves most of the chip idle and every wave
 * with a serial chain of chunk loads (2048 x 512 weights under 118 rows: 64 tiles, eight chunks per
 * wave).  As many slices as keep one chunk per wave and give one workgroup per compute unit: measured
 * over 12 ... 256 tiles and K = 1024 ... 4096, the best count was the one that brought the launch
 * to about 256 workgroups, and more made it slower again. */
uint32_t slices_for(const MatmulArgs &g, dim3 grid, bool eight) {
    if (g.b2 || g.cross_k || g.norm_w) return 1u;
    const uint32_t chunks = (g.k + 31u) / 32u;
    const uint64_t tiles = (uint64_t)grid.x * grid.y;
    const uint32_t room = chunks / (eight ? 8u : 4u);
    if (chunks < 32u || tiles > 128u) return 1u;
    return std::max(1u, std::min(room, 256u / (uint32_t)tiles));
}

template <bool VEC, bool ROPE>
void launch_splitk(const MatmulArgs &g_in, dim3 grid, hipStream_t s) {
    /* eight waves once every wave still gets a chunk (K >= 256) and the launch leaves the chip room for them */
    const bool eight = g_in.k >= 256u && (uint64_t)grid.x * grid.y <= 512u;
    MatmulArgs g = g_in;
    g.slices = slices_for(g, grid, eight);
    const size_t tiles = (size_t)grid.x * grid.y;
    if (g.slices > 1u && matmul_slice_scratch(tiles * g.slices * 1024u, tiles, s, &g.slice_sums, &g.slice_tickets)) grid.z = g.slices;
    else g.slices = 1u;
    if (g.cross_k) {
        if constexpr (VEC && !ROPE)
            blt_launch("matmul_splitk_cross", matmul_splitk_kernel<true, false, false, 4, true>, grid, dim3(256), 0, s, g);
        return;
    }
    if (g.b2) blt_launch("matmul_splitk", matmul_splitk_kernel<VEC, ROPE, true>, grid, dim3(256), 0, s, g);
    else if (eight && VEC && (uint64_t)grid.x * grid.y * grid.z > 256u)
        blt_launch("matmul_splitk", matmul_splitk_kernel<VEC, ROPE, false, 8, false, VEC ? 4 : 2>, grid, dim3(512), 0, s, g);
    else if (eight) blt_launch("matmul_splitk", matmul_splitk_kernel<VEC, ROPE, false, 8>, grid, dim3(512), 0, s, g);
    else blt_launch("matmul_splitk", matmul_splitk_kernel<VEC, ROPE, false>, grid, dim3(256), 0, s, g);
}

} // namespace

bool matmul_takes_cross(const MatmulArgs &g) {
    if (g.b2 || g.residual || (g.rope_cos != nullptr && g.rope_cols > 0) || g.cross_head_dim == 0u ||
        g.n % g.cross_head_dim != 0u)
        return false;
    const Path path = choose_path(g);
    if (path == PATH_SKINNY) return g.n <= 256u && g.cross_head_dim <= 256u;
    return path == PATH_SPLITK && g.cross_head_dim == 32u && g.n % 32u == 0u && g.k % 4u == 0u;
}
bool matmul_takes_norm(const MatmulArgs &g) { return choose_path(g) != PATH_SKINNY || g.k <= SKINNY_KC; }

namespace {
bool vec_ok(const MatmulArgs &g) {
    return aligned16(g.a) && aligned16(g.b) && aligned16(g.norm_w) && g.lda % 4u == 0 && g.ldb % 4u == 0 && g.k % 4u == 0 && g.n % 4u == 0;
}
} // namespace

bool matmul_pair_ok(const MatmulArgs &g0, const MatmulArgs &g1) {
    const auto rotated = [](const MatmulArgs &g) { return g.rope_cos != nullptr && g.rope_cols > 0; };
    const auto plain = [](const MatmulArgs &g) {
        return g.m != 0 && g.n != 0 && g.k != 0 && (g.m > 32u || g.tolerant) && choose_path(g) == PATH_SPLITK && !g.residual;
    };
    /* the first product may normalise its rows on the way (four waves: the tile code's own sums) */
    return plain(g0) && plain(g1) && !rotated(g1) && !(rotated(g0) && g0.b2 != nullptr) && (g0.b2 == nullptr || g0.out2 != nullptr) && g1.b2 != nullptr && g1.out2 != nullptr && !g1.norm_w;
}

void matmul_f32_launch_pair(const MatmulArgs &g0, const MatmulArgs &g1, hipStream_t s) {
    BLT_REQUIRE(matmul_pair_ok(g0, g1), "matmul: this pair of products cannot share a launch");
    const uint32_t rows0 = (g0.m + 31u) / 32u, rows1 = (g1.m + 31u) / 32u;
    const uint32_t cols = (std::max(g0.n, g1.n) + 31u) / 32u;
    const dim3 grid(cols, rows0 + rows1);
    const auto launch = [&](auto kernel) { blt_launch("matmul_splitk", kernel, grid, dim3(256), 0, s, g0, g1, rows0); };
    const bool vec = vec_ok(g0) && vec_ok(g1);
    if (g0.rope_cos != nullptr && g0.rope_cols > 0) launch(vec ? matmul_splitk_pair_kernel<true, false, true> : matmul_splitk_pair_kernel<false, false, true>);
    else if (g0.b2) launch(vec ? matmul_splitk_pair_kernel<true, true> : matmul_splitk_pair_kernel<false, true>);
    else launch(vec ? matmul_splitk_pair_kernel<true, false> : matmul_splitk_pair_kernel<false, false>);
}

namespace {
template <bool VEC, bool ROPE, int WT, bool NORM, bool GATED, int SLICED = WHOLE>
void launch_mfma_as(const MatmulArgs &g, dim3 grid, hipStream_t s) {
    constexpr size_t lds = MFMA_LDS_BYTES<WT, NORM>;
    const auto kernel = matmul_mfma_kernel<VEC, ROPE, WT, NORM, GATED, SLICED>;
    if constexpr (lds > 64u * 1024u - 512u) { /* from 64 KB on a kernel has to ask for its LDS first */
        static const hipError_t asked =
            hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        HIP_CHECK(asked);
    }
    blt_launch(SLICED != WHOLE ? "matmul_mfma_slices" : "matmul_mfma", kernel, grid, dim3(512), lds, s, g);
}
/* Slices of K per 64x64 tile; 1: not taken for it.  Up to 128 tiles with a long K leave half of the chip empty.  As many slices as
 * keep to one workgroup a compute unit (two on one take turns with its LDS and vector units: 192 tiles of K = 2048 24.5 us, as
 * 384 27.0; 256 28.8 and 30.4), of at least HALF_K each.  The 64x64 tile whole against this, 1000 rows of 2048 to 512 columns 23.7 /
 * 18.8 us, 900 of 1024 14.0 / 12.3, error against float64 2.2e-7 / 1.4e-7 (K = 2048).
 * Fewer than 112 tiles are products on the fp32 instructions otherwise, and hold every bit of their operands: so they do here, on
 * bf16 parts.  As f16 parts a result that comes from a row's smallest values only was as far off as those parts are, another
 * of the row being large (values of 1e-9 beside ones near 1: 2.3e-5 of their products).  bf16 parts round six times for 16 terms, so only short slices are as close as the 32x32 tiles are, eight waves
 * to a K: error, this / 32x32 tiles, in six slices 0.70 ... 0.72, five 0.76 ... 0.80, four 0.83 ... 0.88, three of K up to 2560
 * 0.96 ... 1.00 but of 4096 1.01, two 1.2; none up to 128 of the 32x32 tiles, which take slices of their own.  That many slices where
 * it takes two workgroups on some compute units too.  us, 32x32 tiles / this, 301 rows of 2048 to 512 columns 17.2 / 13.5, 420
 * 18.0 / 14.3, 640 31.5 / 17.3, 700 31.6 / 24.5, 832 31.7 / 25.1, 832 of 1280 21.8 / 18.6, 420 of 1536 14.3 / 12.9, 301 of 4096 32.5 / 18.1,
 * 832 57.8 / 37.5. */
uint32_t tile_slices(const MatmulArgs &g, bool rope, bool all_bits) {
    if (g.b2 || rope || g.norm_w || g.cross_k || g.k < 1024u || g.m <= (uint32_t)TM || g.ldb > widest_b<1>()) return 1u;
    const uint64_t tiles = (uint64_t)((g.n + TN - 1u) / TN) * ((g.m + TM - 1u) / TM);
    if (tiles < 16u || tiles > 128u || tiles * g.k < 80u * 1024u) return 1u; /* 16: the last workgroup adds its slices one after the other */
    if (all_bits && (uint64_t)((g.n + 31u) / 32u) * ((g.m + 31u) / 32u) <= 128u) return 1u;
    const uint32_t least = !all_bits ? 2u : g.k <= 2560u ? 3u : 4u, room = 256u / (uint32_t)tiles;
    for (uint32_t n = std::min(all_bits ? std::max(room, least) : room, g.k / HALF_K[0]); n >= least; n--) {
        const uint32_t before = (n - 1u) * tile_slice(g.k, n);
        if (before < g.k && g.k - before >= HALF_K[0]) return n; /* the last one is not empty, nor bf16 for being short */
    }
    return 1u;
}
/* false: not taken, or no place for the sums in a capture */
template <bool VEC>
bool launch_sliced(const MatmulArgs &g_in, bool rope, bool all_bits, hipStream_t s) {
    MatmulArgs g = g_in;
    g.slices = tile_slices(g, rope, all_bits);
    const dim3 grid((g.n + TN - 1u) / TN, (g.m + TM - 1u) / TM, g.slices);
    const size_t tiles = (size_t)grid.x * grid.y;
    if (g.slices < 2u || !matmul_slice_scratch(tiles * g.slices * (TM * TN), tiles, s, &g.slice_sums, &g.slice_tickets)) return false;
    if (all_bits) launch_mfma_as<VEC, false, 1, false, false, SLICES_ALL_BITS>(g, grid, s);
    else launch_mfma_as<VEC, false, 1, false, false, SLICES>(g, grid, s);
    return true;
}
template <bool VEC, int WT>
void launch_mfma(const MatmulArgs &g, bool rope, hipStream_t s) {
    constexpr uint32_t BT = MfmaShape<WT, false, true>::BT;
    const uint32_t cols = g.b2 ? BT / 2u : BT;
    const dim3 grid((g.n + cols - 1u) / cols, (g.m + BT - 1u) / BT);
    if (g.b2) {
        if (g.norm_w) launch_mfma_as<VEC, false, WT, true, true>(g, grid, s);
        else launch_mfma_as<VEC, false, WT, false, true>(g, grid, s);
    } else if (rope) {
        if (g.norm_w) launch_mfma_as<VEC, true, WT, true, false>(g, grid, s);
        else launch_mfma_as<VEC, true, WT, false, false>(g, grid, s);
    } else {
        if (g.norm_w) launch_mfma_as<VEC, false, WT, true, false>(g, grid, s);
        else launch_mfma_as<VEC, false, WT, false, false>(g, grid, s);
    }
}
} // namespace

void matmul_f32_launch(const MatmulArgs &g, hipStream_t s) {
    if (g.m == 0 || g.n == 0) return;
    const bool rope = g.rope_cos != nullptr && g.rope_cols > 0;
    const Path path = choose_path(g);
    BLT_REQUIRE(g.b2 == nullptr || !rope, "matmul: a gated product is not rotated");
    BLT_REQUIRE(g.norm_w == nullptr || matmul_takes_norm(g), "matmul: the fused row norm is not available for this shape");
    if (path == PATH_SKINNY) {
        BLT_REQUIRE(g.cross_k == nullptr || (matmul_takes_cross(g) && g.cross_v && g.cross_out && g.cross_lo &&
                                             g.cross_hi && g.cross_rows_per_seq >= 1u),
                    "matmul: the cross-attention epilogue is not available for this shape");
        /* one row per workgroup (measured against 2 and 4 at every shape of the decoder: the extra
         * chains of a lane cost more than the re-reads of b from L2) */
        launch_skinny<1>(g, s);
        return;
    }
    const bool vec = vec_ok(g);
    if (g.cross_k) {
        BLT_REQUIRE(matmul_takes_cross(g) && vec && g.cross_v && g.cross_out && g.cross_lo && g.cross_hi &&
                        g.cross_rows_per_seq >= 1u && aligned16(g.cross_k) && aligned16(g.cross_v) &&
                        aligned16(g.cross_out),
                    "matmul: the cross-attention epilogue is not available for this shape");
    }
    const bool all_bits = path == PATH_SPLITK;
    if (vec ? launch_sliced<true>(g, rope, all_bits, s) : launch_sliced<false>(g, rope, all_bits, s)) return;
    if (path == PATH_SPLITK) {
        const dim3 sgrid((g.n + 31u) / 32u, (g.m + 31u) / 32u);
        if (rope) {
            if (vec) launch_splitk<true, true>(g, sgrid, s);
            else launch_splitk<false, true>(g, sgrid, s);
        } else {
            if (vec) launch_splitk<true, false>(g, sgrid, s);
            else launch_splitk<false, false>(g, sgrid, s);
        }
        return;
    }
    /* One 128x128 workgroup lives on a compute unit, 256 at a time; of the 64x64 ones, which split and read twice as much per
     * output, two, 512 at a time: the large tile once its rounds are at least nine sixteenths full, four and a half rounds
     * of the small one for two (K = 512, small against large: 128 large tiles 16.8 us against 19.4, 144 23.0 against
     * 20.0, 176 23.0 against 20.4, 256 26.9 against 20.6, 288 37.5 against 38.6, 352 43.1 against 39.4). */
    const uint32_t big_cols = g.b2 ? 64u : 128u;
    const uint64_t big_tiles = (uint64_t)((g.n + big_cols - 1u) / big_cols) * ((g.m + 127u) / 128u);
    const bool big = big_tiles >= (big_tiles + 255u) / 256u * 144u || g.ldb > widest_b<1>();
    if (big) {
        if (vec) launch_mfma<true, 2>(g, rope, s);
        else launch_mfma<false, 2>(g, rope, s);
    } else {
        if (vec) launch_mfma<true, 1>(g, rope, s);
        else launch_mfma<false, 1>(g, rope, s);
    }
}

uint32_t matmul_tolerant() {
    static const uint32_t on = [] {
        const char *e = getenv("BLT_HIP_EXACT_STEP");
        return (e && atoi(e) == 1) ? 0u : 1u;
    }();
    return on;
}

void matmul_later_launch(CrossLater &later, hipStream_t s) {
    if (later.kv_waits) matmul_f32_launch(later.kv, s);
    later.kv_waits = false;
}

extern "C" void blt_matmul_hip(const blt_tensor *a, const blt_tensor *b, blt_tensor *out) {
    BLT_REQUIRE(a != NULL && b != NULL && out != NULL, "matmul: inputs must not be NULL");
    BLT_REQUIRE(a->ndim == 2 && b->ndim == 2 && out->ndim == 2, "matmul: all tensors must be 2D");
    BLT_REQUIRE(a->backend == BLT_BACKEND_HIP && b->backend == BLT_BACKEND_HIP && out->backend == BLT_BACKEND_HIP,
                "matmul: HIP implementation called with a non-HIP tensor");
    BLT_REQUIRE(a->dtype == BLT_DTYPE_FP32 && b->dtype == BLT_DTYPE_FP32,
                "matmul: the HIP backend takes FP32 operands only (BF16 weights are not supported)");
    BLT_REQUIRE(out->dtype == BLT_DTYPE_FP32, "matmul: output must be FP32");
    BLT_REQUIRE(a->shape[1] == b->shape[0], "matmul inner dimensions do not match");
    BLT_REQUIRE(out->shape[0] == a->shape[0] && out->shape[1] == b->shape[1], "matmul output shape is incorrect");
    const size_t m = a->shape[0], k = a->shape[1], n = b->shape[1];
    if (m == 0 || n == 0) return;
    if (k == 0) { /* an empty sum: the product is all zeros (csrc/ops/linalg_cpu.c:8-18 stores sum = 0) */
        blt_hip_memset(out->data, 0, m * n * sizeof(float));
        return;
    }
    BLT_REQUIRE(m <= 0x7FFFFFFFu && k <= 0x7FFFFFFFu && n <= 0x7FFFFFFFu, "matmul: dimensions exceed 2^31-1");
    MatmulArgs g;
    __builtin_memset(&g, 0, sizeof(g));
    g.k = (uint32_t)k;
    g.lda = (uint32_t)k, g.ldb = (uint32_t)n, g.ldo = (uint32_t)n;
    /* a grid holds fewer than 2^32 threads in x, up to sixteen of them a column, and 65535 workgroups in y, of 32 rows and more */
    constexpr size_t most_cols = 1u << 27, most_rows = 1u << 20;
    for (size_t row = 0; row < m; row += most_rows)
        for (size_t col = 0; col < n; col += most_cols) {
            g.a = (const float *)a->data + row * k, g.b = (const float *)b->data + col;
            g.out = (float *)out->data + row * n + col;
            g.m = (uint32_t)std::min(m - row, most_rows), g.n = (uint32_t)std::min(n - col, most_cols);
            matmul_f32_launch(g, 0);
        }
    HIP_CHECK_LAUNCH("blt_matmul");
}
