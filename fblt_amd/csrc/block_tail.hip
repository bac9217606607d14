/*
 * Everything of a transformer block behind its attention in ONE launch (csrc/models/transformer.c:112-128,
 * csrc/infer/kv_cache.c:384-414):
 *
 *   resid = x + comb * proj
 *   act   = silu(RMSNorm(resid) * gate) .* (RMSNorm(resid) * up)
 *   out   = resid + act * down
 *
 * As launches these are three products of 4 to 7 us each whatever their size, because each waits for the one before
 * and for a trip of its own to memory.  All three are row-local, so here a workgroup takes 16 rows from the
 * attention's output to the block's, and the hidden layer is dealt to several workgroups (grid x): each computes
 * all of resid -- again, 2 * 16 * E * E operations that would otherwise be a launch --, its own HS hidden columns,
 * and its share of the last product's sum.  The shares go to a per-stream buffer, the workgroup that draws the last
 * ticket of its row tile adds them in the order of the slices.  Nobody waits for another workgroup.
 *
 * Weights are on their way to registers from the first instruction on, the ones used first first: each is used by one
 * wave only, so LDS would add a trip and save nothing.  fp32 matrix instructions: under 16 rows, taking a weight apart into
 * bf16 parts costs more than the matrix time it saves.
 *
 * Bound: latency.  E = 128, hidden 512, 512 rows: 10.9 us in the kernel trace, of which (parts left out, one after the other)
 * an empty launch with all requests 3, the barriers and the partial sums through LDS 2.5, fp32 matrix time of the compute
 * unit 2.2, the ticket 1.9.  Whole blocks, three launches -> this: 128 rows
 * 25.0 -> 17.3 us, 512 rows 29.5 -> 21.6; E = 64 22.7 -> 13.9 and 26.1 -> 17.2; E = 256, 128 rows 31.5 -> 28.4.
 * Relative error of the block against float64: 1.57e-7 -> 1.45e-7 (E = 128, 128 rows), 1.64e-7 -> 1.47e-7 (256 of 256).
 */
#include "blt_hip.h"
#include "blt_fatal.h"
#include "hip_check.h"
#include "lane_ops.h"
#include "launch.h"
#include "matmul.h"

#include <cstring>

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

/* Columns go in groups of 64, a wave per (group, share of the terms): lane (g, c) loads four consecutive columns
 * 4 c .. 4 c + 3 of row 4 g + t of every block of 16 terms, 16 bytes, and column j of the four is the tile of every fourth
 * column from j on.  A load instruction costs a compute unit's vector memory path about the same whatever it
 * brings: with a tile of 16 consecutive columns a wave and 4 bytes a lane, four times the loads, a block of 512 rows took
 * 23.3 us instead of 21.6. */
template <int E_, int NW_, bool PROJ_>
struct TailShape {
    static constexpr int E = E_, HS = 64, NW = NW_, THREADS = 64 * NW;
    static constexpr bool PROJ = PROJ_;
    static constexpr int ROW = E + 4, ACT = HS + 4; /* LDS rows, four banks apart */
    template <int COLS, int TERMS>
    struct Product {
        static constexpr int GROUPS = COLS / 64, SHARES = NW / GROUPS, BLOCKS = TERMS / 16 / SHARES, PITCH = COLS + 4;
        static constexpr int PART = SHARES * 16 * PITCH; /* floats of the partial tiles */
        static_assert(GROUPS * SHARES == NW && BLOCKS * SHARES * 16 == TERMS, "waves over groups and shares");
    };
    using Proj = Product<E, E>;
    using Gated = Product<2 * HS, E>; /* the up columns, then the gate columns */
    using Down = Product<E, HS>;
    static constexpr int EPT = 16 * E / THREADS; /* of the 16 rows of E, and of HS, a thread finishes */
    static constexpr int APT = 16 * HS / THREADS;
    static constexpr int AREA = Proj::PART > Gated::PART ? Proj::PART : Gated::PART;
};

/* the weights of a wave's product: from `w`, row-major with `ld` columns, rows from term0 on */
template <int BLOCKS>
__device__ __forceinline__ void request(floatx4 (&v)[4 * BLOCKS], const float *w, size_t ld, uint32_t term0) {
    const uint32_t lane = threadIdx.x & 63u;
    const float *p = w + (size_t)(term0 + 4u * (lane >> 4)) * ld + 4u * (lane & 15u);
#pragma unroll
    for (int i = 0; i < 4 * BLOCKS; i++) v[i] = *reinterpret_cast<const floatx4 *>(p + (size_t)(16 * (i / 4) + i % 4) * ld);
}
/* the wave's sums over its share of the terms, to rows of PITCH of its part */
template <int BLOCKS, int PITCH>
__device__ __forceinline__ void multiply(const float *rows, uint32_t row_pitch, uint32_t term0, const floatx4 (&v)[4 * BLOCKS], float *part) {
    const uint32_t lane = threadIdx.x & 63u, g = lane >> 4, c = lane & 15u;
    const float *mine = rows + c * row_pitch + term0 + 4u * g;
    floatx4 acc[4];
#pragma unroll
    for (int j = 0; j < 4; j++) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < BLOCKS; b++) {
        const floatx4 a = *reinterpret_cast<const floatx4 *>(mine + 16 * b);
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int j = 0; j < 4; j++) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], v[4 * b + t][j], acc[j], 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; r++)
        *reinterpret_cast<floatx4 *>(part + (4u * g + r) * PITCH + 4u * c) = floatx4{acc[0][r], acc[1][r], acc[2][r], acc[3][r]};
}
/* N consecutive values, the shares' sums added */
template <int SHARES, int PITCH, int N>
__device__ __forceinline__ void gather(const float *part, float (&out)[N]) {
    typedef float values __attribute__((ext_vector_type(N)));
    values v = *reinterpret_cast<const values *>(part);
#pragma unroll
    for (int s = 1; s < SHARES; s++) v += *reinterpret_cast<const values *>(part + s * 16 * PITCH);
#pragma unroll
    for (int i = 0; i < N; i++) out[i] = v[i];
}

template <typename Shape>
struct TailLds {
    __attribute__((aligned(16))) float rows[16 * Shape::ROW], part[Shape::AREA], act[16 * Shape::ACT];
    uint32_t ticket;
};

/* slice `slice` of row tile `tile` */
template <typename Shape>
__device__ __forceinline__ void tail_tile(const BlockTailArgs &a, uint32_t slices, uint32_t slice, uint32_t tile, TailLds<Shape> &lds) {
    using Proj = typename Shape::Proj;
    using Gated = typename Shape::Gated;
    using Down = typename Shape::Down;
    constexpr int E = Shape::E, HS = Shape::HS, ROW = Shape::ROW, ACT = Shape::ACT, EPT = Shape::EPT, APT = Shape::APT;
    typedef float rowpart __attribute__((ext_vector_type(EPT)));
    float *const rows = lds.rows, *const part = lds.part, *const act = lds.act;
    const uint32_t tid = threadIdx.x;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t row0 = 16u * tile;
    /* what this thread finishes of the 16 rows */
    constexpr uint32_t TPR = E / EPT; /* threads of a row: neighbours in one wave */
    static_assert(TPR <= 64, "a row's threads are in one wave");
    const uint32_t f_row = tid / TPR, f_col = EPT * (tid % TPR);
    const size_t f_at = (size_t)min(row0 + f_row, a.rows - 1u) * E + f_col;

    floatx4 wp[Shape::PROJ ? 4 * Proj::BLOCKS : 1], wg[4 * Gated::BLOCKS], wd[4 * Down::BLOCKS];
    const uint32_t p_group = wave % Proj::GROUPS, p_term = wave / Proj::GROUPS * (16 * Proj::BLOCKS);
    const uint32_t g_group = wave % Gated::GROUPS, g_term = wave / Gated::GROUPS * (16 * Gated::BLOCKS);
    const uint32_t d_group = wave % Down::GROUPS, d_term = wave / Down::GROUPS * (16 * Down::BLOCKS);
    rowpart in;
    if constexpr (Shape::PROJ) in = *reinterpret_cast<const rowpart *>(a.comb + f_at);
    const rowpart x = *reinterpret_cast<const rowpart *>(a.x + f_at);
    const rowpart norm_w = *reinterpret_cast<const rowpart *>(a.norm_w + f_col);
    if constexpr (Shape::PROJ) request<Proj::BLOCKS>(wp, a.proj + 64u * p_group, E, p_term);
    __builtin_amdgcn_sched_barrier(0); /* requests in the order in which they are used, all before the first wait */
    const bool is_gate = g_group >= (uint32_t)Gated::GROUPS / 2u;
    request<Gated::BLOCKS>(wg, (is_gate ? a.gate : a.up) + slice * HS + 64u * (g_group % (Gated::GROUPS / 2)), a.hidden, g_term);
    request<Down::BLOCKS>(wd, a.down + (size_t)slice * HS * E + 64u * d_group, E, d_term);
    __builtin_amdgcn_sched_barrier(0);

    float resid[EPT];
    if constexpr (Shape::PROJ) {
        *reinterpret_cast<rowpart *>(rows + f_row * ROW + f_col) = in;
        __syncthreads();
        multiply<Proj::BLOCKS, Proj::PITCH>(rows, ROW, p_term, wp, part + wave / Proj::GROUPS * (16 * Proj::PITCH) + 64u * p_group);
        __syncthreads();
        gather<Proj::SHARES, Proj::PITCH, EPT>(part + f_row * Proj::PITCH + f_col, resid);
#pragma unroll
        for (int i = 0; i < EPT; i++) resid[i] = x[i] + resid[i];
    } else {
#pragma unroll
        for (int i = 0; i < EPT; i++) resid[i] = x[i];
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < EPT; i++) ss += resid[i] * resid[i];
    ss = key_sum<TPR < 32 ? TPR : 32>(ss);
    if (TPR == 64) ss = swap32(ss, OpSum());
    const float scale = 1.0f / sqrtf(ss / (float)E + 1e-6f); /* reductions_cpu.c:345-346 */
    rowpart n;
#pragma unroll
    for (int i = 0; i < EPT; i++) n[i] = resid[i] * scale * norm_w[i];
    *reinterpret_cast<rowpart *>(rows + f_row * ROW + f_col) = n;
    __syncthreads();
    multiply<Gated::BLOCKS, Gated::PITCH>(rows, ROW, g_term, wg, part + wave / Gated::GROUPS * (16 * Gated::PITCH) + 64u * g_group);
    __syncthreads();
    {
        typedef float values __attribute__((ext_vector_type(APT)));
        const uint32_t h_row = tid / (HS / APT), h_col = APT * (tid % (HS / APT));
        float up[APT], gate[APT];
        gather<Gated::SHARES, Gated::PITCH, APT>(part + h_row * Gated::PITCH + h_col, up);
        gather<Gated::SHARES, Gated::PITCH, APT>(part + h_row * Gated::PITCH + HS + h_col, gate);
        values v;
#pragma unroll
        for (int i = 0; i < APT; i++) v[i] = silu_times(gate[i], up[i]);
        *reinterpret_cast<values *>(act + h_row * ACT + h_col) = v;
    }
    __syncthreads();
    multiply<Down::BLOCKS, Down::PITCH>(act, ACT, d_term, wd, part + wave / Down::GROUPS * (16 * Down::PITCH) + 64u * d_group);
    __syncthreads();
    float sum[EPT];
    gather<Down::SHARES, Down::PITCH, EPT>(part + f_row * Down::PITCH + f_col, sum);

    if (slices > 1u) {
        /* device-scope stores and loads, and an explicit wait for the stores' completion before the barrier that
         * precedes the workgroup's ticket */
        constexpr uint32_t WORDS = 16 * E / 2; /* a slice's sums, two a word */
        uint64_t *mine = a.sums + (size_t)tile * slices * WORDS + tid;
#pragma unroll
        for (int i = 0; i < EPT / 2; i++)
            __hip_atomic_store(mine + (size_t)slice * WORDS + i * Shape::THREADS,
                               (uint64_t)__float_as_uint(sum[2 * i + 1]) << 32 | __float_as_uint(sum[2 * i]), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        blt_vector_memory_done();
        __syncthreads();
        if (tid == 0u)
            lds.ticket = __hip_atomic_fetch_add(&a.tickets[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (lds.ticket != slices - 1u) return;
        if (tid == 0u) a.tickets[tile] = 0u; /* re-armed for the next launch */
#pragma unroll
        for (int i = 0; i < EPT; i++) sum[i] = 0.f;
        for (uint32_t z = 0; z < slices; z += 8u) { /* slice order, whoever comes last */
            uint64_t t[8][EPT / 2];
#pragma unroll
            for (uint32_t u = 0; u < 8u; u++)
#pragma unroll
                for (int i = 0; i < EPT / 2; i++)
                    t[u][i] = __hip_atomic_load(mine + (size_t)min(z + u, slices - 1u) * WORDS + i * Shape::THREADS, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (uint32_t u = 0; u < 8u; u++)
#pragma unroll
                for (int i = 0; i < EPT; i++)
                    sum[i] += z + u < slices ? __uint_as_float((uint32_t)(t[u][i / 2] >> (32 * (i % 2)))) : 0.f;
        }
    }
    rowpart out;
#pragma unroll
    for (int i = 0; i < EPT; i++) out[i] = resid[i] + sum[i];
    if (row0 + f_row < a.rows) *reinterpret_cast<rowpart *>(a.out + f_at) = out;
}

template <typename Shape>
__global__ __launch_bounds__(Shape::THREADS) void block_tail_kernel(BlockTailArgs a) {
    __shared__ TailLds<Shape> lds;
    tail_tile<Shape>(a, gridDim.x, blockIdx.x, blockIdx.y, lds);
}

/* A cross block of 16 rows a workgroup: norm, query projection, the rows' attention, output projection, residual
 * (csrc/models/cross_attention.c:101-157, csrc/infer/kv_cache.c:303-324).  A row sees few keys, a handful of bytes or the
 * patches of its own window, so the rows of K and V come straight from memory, eight keys in flight, the first before there
 * is a query, to the threads that hold the query: EPT columns each, a head's threads neighbours.  Running maximum over
 * finite scores; a score that is not finite weighs nothing, a row without keys gives zeros.
 *
 * Bound: latency: weights and keys on their way, two products with their partial sums through LDS; 7.2 us in the kernel trace
 * for 512 rows of 128 that see a patch each, 9.4 for 128 rows of up to 16 bytes (a further trip to memory for every eight
 * keys past the first), against 5.6 + 4.3 and 6.1 + 4.2 with a gap as two launches. */
/* Rows that it is taken for.  No crossover lies there: prompts of two layers as launches / this, us, 8192 rows 245 / 221, 16384 362 /
 * 333, 32768 619 / 566, 65536 1189 / 1085 (64 columns 32768 rows 387 / 330). */
constexpr uint32_t CROSS_ROWS = 16384;
constexpr uint32_t CROSS_KEYS = 4;

/* Where rows find their key ranges: in memory ... */
struct RangesThere {};
__device__ __forceinline__ void find_range(const CrossBlockArgs &a, RangesThere, uint32_t row, uint32_t &lo, uint32_t &hi) {
    lo = a.lo[row], hi = a.hi[row];
}
__device__ __forceinline__ void leave_ranges(RangesThere, uint32_t, uint32_t) {}
/* ... or in the kernel arguments, and then the first of a row tile's workgroups leaves them there.  With a launch that only brings them a
 * prompt of 512 bytes takes 66.2 us, so 64.6. */
__device__ __forceinline__ uint32_t range_start(const CrossWords &w, uint32_t row) {
    return (w.words[w.batch + (row >> 1)] >> (16u * (row & 1u))) & 0xFFFFu;
}
__device__ __forceinline__ void find_range(const CrossBlockArgs &, const CrossWords &w, uint32_t row, uint32_t &lo, uint32_t &hi) {
    lo = range_start(w, row), hi = w.span ? lo + w.span : range_start(w, row + 1u);
}
__device__ __forceinline__ void leave_ranges(const CrossWords &w, uint32_t tile, uint32_t threads) {
    const uint32_t tid = threadIdx.x, row = 16u * tile + tid;
    if (tid < 16u && row < w.rows) {
        const uint32_t lo = range_start(w, row);
        w.lo[row] = lo, w.hi[row] = w.span ? lo + w.span : range_start(w, row + 1u);
    }
    if (tile == 0u)
        for (uint32_t b = tid; b < w.batch; b += threads) w.lens[b] = w.words[b];
}

/* then(): further requests, behind the first keys'.  Returns the thread's columns of its row; rows and part are free for the taking
 * behind a barrier. */
template <typename Shape, uint32_t KEYS, typename Range, typename Then>
__device__ __forceinline__ floatx4 cross_rows(const CrossBlockArgs &a, uint32_t tile, float *rows, float *part, Range range, Then then) {
    using Proj = typename Shape::Proj;
    constexpr int E = Shape::E, ROW = Shape::ROW, EPT = Shape::EPT;
    static_assert(EPT == 4, "a thread holds 16 bytes of a row");
    const uint32_t tid = threadIdx.x;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr uint32_t TPR = E / EPT;
    const uint32_t row0 = 16u * tile, f_row = tid / TPR, f_col = EPT * (tid % TPR);
    const uint32_t row = min(row0 + f_row, a.rows - 1u);
    const size_t f_at = (size_t)row * E + f_col;
    const uint32_t group = wave % Proj::GROUPS, term = wave / Proj::GROUPS * (16 * Proj::BLOCKS);
    float *const mine = part + wave / Proj::GROUPS * (16 * Proj::PITCH) + 64u * group;

    floatx4 wq[4 * Proj::BLOCKS], wp[4 * Proj::BLOCKS];
    floatx4 x = *reinterpret_cast<const floatx4 *>(a.x + f_at), norm_w = {1.f, 1.f, 1.f, 1.f}, resid = {0.f, 0.f, 0.f, 0.f};
    if (a.norm_w) norm_w = *reinterpret_cast<const floatx4 *>(a.norm_w + f_col);
    request<Proj::BLOCKS>(wq, a.wq + 64u * group, E, term);
    __builtin_amdgcn_sched_barrier(0);
    uint32_t lo, hi;
    range(row, lo, hi);
    const uint32_t lanes = a.head_dim / EPT; /* of a head: a power of two up to TPR */
    const size_t slab = (size_t)(row / a.rows_per_seq) * a.slab_rows * E + f_col;
    struct Keys {
        floatx4 k[KEYS], v[KEYS];
    } even, odd; /* taking turns */
    const auto fetch = [&](Keys &to, uint32_t j) __attribute__((always_inline)) { /* past the last key: that one again */
        if (j >= hi) return;
#pragma unroll
        for (uint32_t u = 0; u < KEYS; u++) to.k[u] = *reinterpret_cast<const floatx4 *>(a.k + slab + (size_t)min(j + u, hi - 1u) * E);
#pragma unroll
        for (uint32_t u = 0; u < KEYS; u++) to.v[u] = *reinterpret_cast<const floatx4 *>(a.v + slab + (size_t)min(j + u, hi - 1u) * E);
    };
    if (a.residual) resid = *reinterpret_cast<const floatx4 *>(a.residual + f_at);
    request<Proj::BLOCKS>(wp, a.proj + 64u * group, E, term);
    __builtin_amdgcn_sched_barrier(0);
    fetch(even, lo); /* the keys do not wait for the query */
    fetch(odd, lo + KEYS);
    then();
    __builtin_amdgcn_sched_barrier(0);

    if (a.norm_w) {
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < EPT; i++) ss += x[i] * x[i];
        ss = key_sum<TPR>(ss);
        x *= 1.0f / sqrtf(ss / (float)E + 1e-6f) * norm_w; /* reductions_cpu.c:345-346 */
    }
    *reinterpret_cast<floatx4 *>(rows + f_row * ROW + f_col) = x;
    __syncthreads();
    multiply<Proj::BLOCKS, Proj::PITCH>(rows, ROW, term, wq, mine);
    __syncthreads();
    float q[EPT];
    gather<Proj::SHARES, Proj::PITCH, EPT>(part + f_row * Proj::PITCH + f_col, q);

    float m = -__builtin_huge_valf(), l = 0.f;
    floatx4 o = {0.f, 0.f, 0.f, 0.f};
    const auto attend = [&](const Keys &from, uint32_t j) __attribute__((always_inline)) {
        float s[KEYS], top = m;
#pragma unroll
        for (uint32_t u = 0; u < KEYS; u++) s[u] = q[0] * from.k[u][0] + q[1] * from.k[u][1] + q[2] * from.k[u][2] + q[3] * from.k[u][3];
        for (uint32_t d = 1u; d < lanes; d *= 2u)
#pragma unroll
            for (uint32_t u = 0; u < KEYS; u++) s[u] += __shfl_xor(s[u], (int)d, 64);
#pragma unroll
        for (uint32_t u = 0; u < KEYS; u++) {
            s[u] *= a.scale;
            if (j + u >= hi || !isfinite(s[u])) s[u] = -__builtin_huge_valf();
            top = fmaxf(top, s[u]);
        }
        if (top == -__builtin_huge_valf()) return; /* nothing of weight yet */
        const float fade = expf(m - top);
        m = top, l *= fade, o *= fade;
#pragma unroll
        for (uint32_t u = 0; u < KEYS; u++) {
            const float e = expf(s[u] - top);
            if (e == 0.f) continue; /* its value row may be anything */
            l += e, o += e * from.v[u];
        }
    };
    for (uint32_t j = lo; j < hi; j += 2u * KEYS) { /* the same for a row's threads */
        attend(even, j);
        fetch(even, j + 2u * KEYS);
        if (j + KEYS < hi) attend(odd, j + KEYS);
        fetch(odd, j + 3u * KEYS);
    }
    /* A key seen early whose weight has faded to zero since: its infinite value row times zero is in the sums.  Then the row once
     * more with the maximum known, so that such a key never enters. */
    const uint64_t lost = __ballot(!(isfinite(o[0]) && isfinite(o[1]) && isfinite(o[2]) && isfinite(o[3])));
    if ((lost >> (tid & 63u & ~(TPR - 1u)) & (~0ull >> (64u - TPR))) != 0u) {
        l = 0.f, o = floatx4{0.f, 0.f, 0.f, 0.f};
        for (uint32_t j = lo; j < hi; j++) {
            const floatx4 k = *reinterpret_cast<const floatx4 *>(a.k + slab + (size_t)j * E);
            float s = q[0] * k[0] + q[1] * k[1] + q[2] * k[2] + q[3] * k[3];
            for (uint32_t d = 1u; d < lanes; d *= 2u) s += __shfl_xor(s, (int)d, 64);
            s *= a.scale;
            const float e = isfinite(s) ? expf(s - m) : 0.f;
            if (e != 0.f) l += e, o += e * *reinterpret_cast<const floatx4 *>(a.v + slab + (size_t)j * E);
        }
    }
    o *= l > 0.f ? 1.0f / l : 0.f;
    *reinterpret_cast<floatx4 *>(rows + f_row * ROW + f_col) = o;
    __syncthreads();
    multiply<Proj::BLOCKS, Proj::PITCH>(rows, ROW, term, wp, mine);
    __syncthreads();
    float sum[EPT];
    gather<Proj::SHARES, Proj::PITCH, EPT>(part + f_row * Proj::PITCH + f_col, sum);
#pragma unroll
    for (int i = 0; i < EPT; i++) resid[i] += sum[i];
    return resid;
}

template <typename Shape, uint32_t KEYS, typename Ranges>
__device__ __forceinline__ void cross_tile(const CrossBlockArgs &a, const Ranges &w, uint32_t tile, float *rows, float *part) {
    leave_ranges(w, tile, Shape::THREADS);
    const floatx4 out = cross_rows<Shape, KEYS>(
        a, tile, rows, part, [&](uint32_t row, uint32_t &lo, uint32_t &hi) __attribute__((always_inline)) { find_range(a, w, row, lo, hi); }, [] {});
    const uint32_t row = 16u * tile + threadIdx.x / (Shape::E / 4);
    if (row < a.rows) *reinterpret_cast<floatx4 *>(a.out + (size_t)row * Shape::E + 4u * (threadIdx.x % (Shape::E / 4))) = out;
}

/* A cross block and the QKV product of its rows: workgroup x of a row tile takes the columns of Q, K or V, each with the cross block
 * of its own -- again, as in the tail --, and the first stores that block's rows.
 * Bound: latency, a chain of two products behind each other and the norm between; for 512 rows of 128 that see a patch each 9.9 us in
 * the kernel trace, against 6.9 and 5.6 and the gap as two launches (a prompt of 512 bytes, two layers: 70.2 / 66.6 us). */
template <typename Shape, typename Ranges>
__global__ __launch_bounds__(Shape::THREADS) void cross_qkv_kernel(CrossBlockArgs a, MatmulArgs g, Ranges w_in) {
    using Proj = typename Shape::Proj;
    constexpr int E = Shape::E, ROW = Shape::ROW;
    constexpr uint32_t TPR = E / 4;
    __shared__ __attribute__((aligned(16))) float rows[16 * ROW], part[Proj::PART];
    const uint32_t tid = threadIdx.x, third = blockIdx.x, tile = blockIdx.y;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t group = wave % Proj::GROUPS, share = wave / Proj::GROUPS, term = share * (16 * Proj::BLOCKS);
    const uint32_t f_row = tid / TPR, f_col = 4u * (tid % TPR), row = 16u * tile + f_row;
    floatx4 w[4 * Proj::BLOCKS], norm_w;
    if (third == 0u) leave_ranges(w_in, tile, Shape::THREADS);
    const auto range = [&](uint32_t r, uint32_t &lo, uint32_t &hi) __attribute__((always_inline)) { find_range(a, w_in, r, lo, hi); };
    floatx4 x = cross_rows<Shape, CROSS_KEYS>(a, tile, rows, part, range, [&]() __attribute__((always_inline)) {
        norm_w = *reinterpret_cast<const floatx4 *>(g.norm_w + f_col);
        request<Proj::BLOCKS>(w, g.b + third * E + 64u * group, g.ldb, term);
    });
    if (third == 0u && row < a.rows) *reinterpret_cast<floatx4 *>(a.out + (size_t)row * E + f_col) = x;
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) ss += x[i] * x[i];
    ss = key_sum<TPR>(ss);
    x *= 1.0f / sqrtf(ss / (float)E + 1e-6f) * norm_w; /* reductions_cpu.c:345-346 */
    *reinterpret_cast<floatx4 *>(rows + f_row * ROW + f_col) = x;
    __syncthreads();
    multiply<Proj::BLOCKS, Proj::PITCH>(rows, ROW, term, w, part + share * (16 * Proj::PITCH) + 64u * group);
    __syncthreads();
    float v[4];
    gather<Proj::SHARES, Proj::PITCH, 4>(part + f_row * Proj::PITCH + f_col, v);
    if (row >= a.rows) return;
    const float4 result = make_float4(v[0], v[1], v[2], v[3]);
    if constexpr (std::is_same<Ranges, CrossWords>::value) {
        if (g.stage_k) { /* the lengths are on their way too */
            const uint32_t b = row / g.stage_n;
            matmul_stage4(g, row, b, w_in.words[b] + row % g.stage_n, third * E + f_col, result);
            return;
        }
    }
    matmul_store4<true>(g, row, third * E + f_col, result, true);
}

template <typename Shape, typename Ranges>
__global__ __launch_bounds__(Shape::THREADS) void cross_block_kernel(CrossBlockArgs a, Ranges w) {
    __shared__ __attribute__((aligned(16))) float rows[16 * Shape::ROW], part[Shape::Proj::PART];
    cross_tile<Shape, CROSS_KEYS>(a, w, blockIdx.x, rows, part);
}

/* A block's tail and a cross block that neither reads nor writes anything of it, in the first `first` rows of workgroups: the
 * encoder's, whose patches take up a layer's bytes while the next layer goes on with them.  Its few workgroups fit beside the tail's: 128
 * patches of 512 bytes, 128 columns, take 9.6 us as a launch and make this one 16.2 us where the tail alone is 11.4 ... 12.2 (64 columns,
 * 757 bytes: 7.1, and 8.9 for 6.6).  Half the keys in flight: more registers than the tail has would halve the workgroups of a compute
 * unit. */
template <typename Shape, typename Ranges>
__global__ __launch_bounds__(Shape::THREADS, 4) void block_tail_beside_kernel(BlockTailArgs a, CrossBlockArgs c, uint32_t first, Ranges w) {
    __shared__ TailLds<Shape> lds;
    if (blockIdx.y < first) {
        const uint32_t tile = blockIdx.y * gridDim.x + blockIdx.x;
        if (tile < (c.rows + 15u) / 16u) cross_tile<Shape, CROSS_KEYS / 2>(c, w, tile, lds.rows, lds.part);
    } else {
        tail_tile<Shape>(a, gridDim.x, blockIdx.x, blockIdx.y - first, lds);
    }
}

template <typename Shape>
void launch_tail(const BlockTailArgs &a, dim3 grid, hipStream_t s, const CrossBlockArgs *beside = nullptr) {
    if constexpr (Shape::PROJ) {
        if (beside) {
            const uint32_t first = ((beside->rows + 15u) / 16u + grid.x - 1u) / grid.x;
            const dim3 both(grid.x, grid.y + first);
            if (beside->words)
                blt_launch("block_tail", block_tail_beside_kernel<Shape, CrossWords>, both, dim3(Shape::THREADS), 0, s, a, *beside, first,
                           *beside->words);
            else
                blt_launch("block_tail", block_tail_beside_kernel<Shape, RangesThere>, both, dim3(Shape::THREADS), 0, s, a, *beside, first,
                           RangesThere());
            return;
        }
    }
    blt_launch("block_tail", block_tail_kernel<Shape>, grid, dim3(Shape::THREADS), 0, s, a);
}

} // namespace

bool block_tail_launch(BlockTailArgs a, uint32_t embed_dim, hipStream_t s, CrossLater *later) {
    if (a.rows == 0u || a.hidden == 0u || (embed_dim != 64u && embed_dim != 128u && embed_dim != 256u) || a.hidden % 64u != 0u)
        return false;
    for (const void *p : {(const void *)a.comb, (const void *)a.x, (const void *)a.proj, (const void *)a.norm_w, (const void *)a.up,
                          (const void *)a.gate, (const void *)a.down, (const void *)a.out, (const void *)a.resid})
        if ((reinterpret_cast<uintptr_t>(p) & 15u) != 0u) return false;
    /* A workgroup's time hardly depends on its load, so the launch takes as many times that as the chip needs rounds, and the
     * products as launches fill it better.  Whole blocks (projection to output, attention included), launches / this:
     *   E = 64 (four workgroups of four waves a compute unit): 256 x 4 = 1024 workgroups 68.7 / 61.6 us
     *   E = 128 (two of eight waves): 512 workgroups 35.2 / 30.1 (1024 rows) and 31.4 / 28.4 (hidden layer of 1024), 768
     *   workgroups 49.2 / 49.2, 1024 53.8 / 57.3
     *   E = 256 (one of sixteen waves, the projection a launch of its own): 256 workgroups 34.2 / 33.2; 512 as 256 of twice
     *   the hidden columns 41.3 / 41.3 */
    const uint64_t workgroups = (uint64_t)((a.rows + 15u) / 16u) * (a.hidden / 64u);
    /* Who comes last adds up all slices, eight at a time, which counts from 33 slices on (from 17 at 256 columns):
     *   E = 64: 48 slices, 624 workgroups 31.7 / 28.7; 64, 512 29.9 / 26.7 and 832 33.6 / 35.7; 128, 512 34.0 / 32.6 and 896 37.7 / 46.3
     *   E = 128: 64 slices, 256 workgroups 29.9 / 26.4 and 448 32.4 / 33.2; 96, 288 32.9 / 35.7; 128, 384 36.2 / 42.9
     *   E = 256: 32 slices, 128 workgroups 32.6 / 32.3 and 224 33.3 / 34.2; 48, 144 33.5 / 36.1 */
    const bool many = a.hidden / 64u > (embed_dim == 256u ? 16u : 32u);
    const uint32_t most = embed_dim == 64u ? (many ? 640u : 1024u) : embed_dim == 128u ? (many ? 256u : 512u) : many ? 128u : 256u;
    if (workgroups > most) return false;
    const uint32_t slices = a.hidden / 64u, tiles = (a.rows + 15u) / 16u;
    if (slices > 1u && !matmul_slice_scratch((size_t)tiles * slices * 16u * embed_dim, tiles, s, (float **)&a.sums, &a.tickets))
        return false;
    const dim3 grid(slices, tiles);
    /* with a cross block that waits, as long as all workgroups have a place at once */
    const CrossBlockArgs *beside = nullptr;
    if (later != nullptr && later->cross_waits && embed_dim != 256u && workgroups + (later->cross.rows + 15u) / 16u <= most) {
        matmul_later_launch(*later, s); /* its keys */
        beside = &later->cross, later->cross_waits = false;
    }
    if (embed_dim == 64u) {
        launch_tail<TailShape<64, 4, true>>(a, grid, s, beside);
    } else if (embed_dim == 128u) {
        launch_tail<TailShape<128, 8, true>>(a, grid, s, beside);
    } else { /* 1024 threads leave a wave 128 registers, and its share of proj is 64 of them */
        MatmulArgs g;
        std::memset(&g, 0, sizeof(g));
        g.a = a.comb, g.b = a.proj, g.residual = a.x, g.out = a.resid;
        g.m = a.rows, g.k = g.n = g.lda = g.ldb = g.ldo = embed_dim;
        g.tolerant = 1u;
        matmul_f32_launch(g, s);
        a.x = a.resid;
        launch_tail<TailShape<256, 16, false>>(a, grid, s);
    }
    return true;
}

bool cross_block_ok(const CrossBlockArgs &a, uint32_t embed_dim) {
    if ((embed_dim != 64u && embed_dim != 128u) || a.rows == 0u) return false;
    /* a head's columns are spread over neighbouring threads, four each */
    if (a.head_dim < 4u || a.head_dim > embed_dim || (a.head_dim & (a.head_dim - 1u)) != 0u) return false;
    for (const void *p : {(const void *)a.x, (const void *)a.norm_w, (const void *)a.wq, (const void *)a.k, (const void *)a.v,
                          (const void *)a.proj, (const void *)a.residual, (const void *)a.out})
        if ((reinterpret_cast<uintptr_t>(p) & 15u) != 0u) return false;
    return a.rows <= CROSS_ROWS;
}

bool cross_words_fill(CrossWords &w, const uint32_t *lo, const uint32_t *hi, size_t rows, const uint32_t *lens, size_t batch) {
    if (rows == 0 || batch + rows / 2 + 1 > CrossWords::WORDS) return false;
    bool alike = hi[0] > lo[0], tiling = true;
    uint32_t any = hi[rows - 1];
    for (size_t r = 0; r < rows; r++) {
        alike = alike && hi[r] - lo[r] == hi[0] - lo[0];
        tiling = tiling && (r + 1 == rows || hi[r] == lo[r + 1]);
        any |= lo[r];
    }
    if ((!alike && !tiling) || any > 0xFFFFu) return false;
    BLT_REQUIRE(!blt_stream_capturing(), "host data cannot be staged to the device while a graph is captured");
    w.rows = (uint32_t)rows, w.batch = (uint32_t)batch, w.span = alike ? hi[0] - lo[0] : 0u, w.reserved = 0;
    for (size_t b = 0; b < batch; b++) w.words[b] = lens[b];
    const auto start = [&](size_t r) { return r < rows ? lo[r] : hi[rows - 1]; };
    for (size_t r = 0; r <= rows; r += 2) w.words[batch + r / 2] = start(r) | start(r + 1) << 16;
    return true;
}

void cross_later_launch(CrossLater &later, uint32_t embed_dim, hipStream_t s) {
    matmul_later_launch(later, s);
    if (later.cross_waits) cross_block_launch(later.cross, embed_dim, s);
    later.cross_waits = false;
}

bool cross_block_launch(const CrossBlockArgs &a, uint32_t embed_dim, hipStream_t s) {
    if (!cross_block_ok(a, embed_dim)) return false;
    const dim3 grid((a.rows + 15u) / 16u);
    const auto launch = [&](auto narrow, auto wide, const auto &ranges) {
        if (embed_dim == 64u) blt_launch("cross_block", narrow, grid, dim3(256), 0, s, a, ranges);
        else blt_launch("cross_block", wide, grid, dim3(512), 0, s, a, ranges);
    };
    if (a.words) launch(cross_block_kernel<TailShape<64, 4, true>, CrossWords>, cross_block_kernel<TailShape<128, 8, true>, CrossWords>, *a.words);
    else launch(cross_block_kernel<TailShape<64, 4, true>, RangesThere>, cross_block_kernel<TailShape<128, 8, true>, RangesThere>, RangesThere());
    return true;
}

bool cross_qkv_launch(const CrossBlockArgs &a, const MatmulArgs &g, uint32_t embed_dim, hipStream_t s) {
    /* Three workgroups a row tile, as long as the chip holds them all at once (registers: one a CU for 128 columns, three for 64):
     * prompts of 1000 / 1360 / 1500 rows of 128 89.2 / 124.4 / 126.6 us as two launches a layer, 85.0 / 114.3 / 131.4 as one. */
    const uint32_t tiles = (a.rows + 15u) / 16u, most = embed_dim == 64u ? 768u : 256u;
    if (!cross_block_ok(a, embed_dim) || 3u * tiles > most || a.out == a.x || a.out == a.residual) return false; /* a row is read three times */
    if (g.norm_w == nullptr || g.b2 != nullptr || g.residual != nullptr || g.cross_k != nullptr || g.m != a.rows || g.k != embed_dim ||
        g.n != 3u * embed_dim || g.ldb % 4u != 0u || g.ldo % 4u != 0u || g.head_dim % 4u != 0u)
        return false;
    for (const void *p : {(const void *)g.b, (const void *)g.norm_w, (const void *)g.out, (const void *)g.stage_k, (const void *)g.stage_v})
        if ((reinterpret_cast<uintptr_t>(p) & 15u) != 0u) return false;
    const dim3 grid(3u, tiles);
    static_assert(sizeof(CrossBlockArgs) + sizeof(MatmulArgs) + sizeof(CrossWords) <= 4096, "kernel argument block");
    const auto launch = [&](auto narrow, auto wide, const auto &ranges) {
        if (embed_dim == 64u) blt_launch("cross_qkv", narrow, grid, dim3(256), 0, s, a, g, ranges);
        else blt_launch("cross_qkv", wide, grid, dim3(512), 0, s, a, g, ranges);
    };
    if (a.words) launch(cross_qkv_kernel<TailShape<64, 4, true>, CrossWords>, cross_qkv_kernel<TailShape<128, 8, true>, CrossWords>, *a.words);
    else launch(cross_qkv_kernel<TailShape<64, 4, true>, RangesThere>, cross_qkv_kernel<TailShape<128, 8, true>, RangesThere>, RangesThere());
    return true;
}
