/*
 * The whole incremental decoder step (csrc/infer/kv_cache.c:161-416) in ONE launch, for steps of
 * few rows: workgroups stay resident from the first layer to the LM head and hand the activations
 * to each other through device memory, where the launch-per-operation form runs 7 dependent
 * kernels per layer.
 *
 * What bounds such a step is neither bytes nor arithmetic (one row through two layers of 128
 * columns: 2.6 MB of weights, 1.6 MFLOP) but the chain of dependent stages: as launches each costs about
 * 4.6 us (launch boundary, cold argument block, one trip to memory, one drain), inside one launch 1 to 2 us from
 * the store to the reader's use and as much again for the stage.
 *
 * Groups.  The sequences of a step are independent, so they are dealt to up to eight groups of
 * workgroups that never talk to each other; group i is the workgroups with blockIdx % 8 == i, which
 * the dispatcher places on die i: a group's weights and activations then pass through one L2.  The
 * placement is a hint only, every hand-over is at device scope.
 *
 * Hand-over.  An activation is published as one 8-byte word {fp32 value, tag} with a device-scope
 * store; whoever needs it loads the word until the tag is the one of this launch and layer.  Value and
 * tag arrive together, so there is no barrier between workgroups, no counter and no fence: one
 * store and one load on the critical path (counter barriers with separate data measured 0.9 ... 1.5 us
 * per phase at 8 ... 32 workgroups).  Buffers are reused from layer to layer: a word of layer l+1 is
 * only written by a workgroup that has seen all of layer l's rows, and every stage depends on all words of the
 * stage before, so everything layer l's readers need has been read by then.  Words are laid out the
 * way the consumer's matrix fragments want them (64 consecutive words per instruction).
 *
 * A stage is a product of [rows, K] with 16-column tiles of a weight matrix, one tile (or an up / gate pair) per
 * workgroup, K split over its eight waves, v_mfma_f32_16x16x4_f32 on 16-row tiles, partial tiles added through
 * LDS; RMSNorm is folded in as in matmul.hip (the row statistic from the same loads, the scale after the product).
 * The self-attention stage gives a workgroup one (sequence, head, share of the keys): K and V rows are requested
 * before the query is there, coalesced and turned into fragments through the wave's LDS tile, exact online softmax per
 * wave, waves merged through LDS, shares merged by the reader.
 *
 * Fewer stages.  A hand-over costs more than a product of few rows with an [E, E] matrix does, so up to 128 columns the
 * stages that need all of a row's columns are not dealt out: every workgroup of the stage behind them does them again
 * (the output projection, by the up / gate tiles; the cross block over one sub-token, by the QKV tiles), four hand-overs a
 * layer instead of seven.  Of the cross block nothing but a row's scores has to wait for the row: see there.  At 256 columns
 * doing it again would take longer than the hand-over, and so would the products that each further sub-token adds.
 *
 * One workgroup of eight waves a compute unit does all stages, products and attention.  As two (one for each) a wave had
 * 128 registers, which held neither: 40 to 150 were spilled, every reload waited for every load before it, and four
 * waves a SIMD issued an instruction every nine cycles each.  What a load instruction costs a compute unit's memory path is
 * its lines, not its bytes: weights are read sixteen bytes a lane along rows, and turned in LDS where the fragments need
 * columns; a wait looks at one word until that is there, then at all of them, and takes along words written earlier.
 *
 * Who waits.  A launch is up to 256 workgroups, one per compute unit, and nothing promises that they all become
 * resident: another kernel may keep its place for as long as it likes, another process may run this very step.  So
 * nobody waits for a workgroup that has not started.  The workgroups of a group call the roll first: each has a word
 * in which it signs in, and who finds the time up before everybody has signs the others out.  If all are in, each has the
 * role its index gives it.  Else those that are in take all the work among them, stage by stage in the same order (any
 * number can: the first unfinished stage waits for nothing unfinished), and who finds itself signed out leaves.  The
 * fewer are in, the longer it is worth waiting: 5 us for the last one, 0.16 ms for the second.
 *
 * Every wait is bounded all the same (SPIN_LIMIT polls, then the wave raises a word in pinned host memory, stops
 * waiting for the rest of the launch, takes NaN for what it did not get and runs to its end; the host turns the word
 * into a fatal error at its next look).
 *
 * Measured, launches -> two workgroups a compute unit and seven stages -> this: one row, two layers of 128 columns, 356
 * keys 54 -> 38 -> 35 us; 64 such rows 62 -> 61 -> 44; 16 draft rows of one sequence 64 -> 62 -> 43; one row, E = 256, heads of 64
 * 90 -> 85 -> 55.  Error against float64 as before (logits of 12 rows, 128 columns 1.64e-7 -> 1.58e-7; 16 rows, 64 columns 1.42e-7
 * and 1.43e-7; 256 columns 1.97e-7 -> 1.71e-7).  Timeline of a layer (one row; clock read at the stages): QKV tiles 1.1 us for the scores and 0.9 for the
 * product, hand-over 1.2, attention 1.4, hand-over 1.5 ... 2.5 (the words of a row are read by 32 workgroups), output
 * projection 1.5 (0.85 of it fp32 matrix time of the 16-row tile), up / gate 0.8, hand-over 1.3, down projection 0.4,
 * hand-over 1.3, the folding of the next layer's cross block mostly behind the last two.
 */
#include "blt_hip.h"
#include "blt_fatal.h"
#include "hip_check.h"
#include "attn_device.h"
#include "attn_tile.h"
#include "lane_ops.h"
#include "launch.h"
#include "rope_device.h"
#include "step_resident.h"

#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <map>

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr uint32_t GROUPS = 8;      /* dies of the package */
constexpr uint32_t WAVES = 8;       /* per workgroup */
constexpr uint32_t MAX_LAYERS = 8;
constexpr uint32_t MAX_GROUP_ROWS = 32;
constexpr uint32_t MAX_ROWS = GROUPS * MAX_GROUP_ROWS;
constexpr uint32_t MAX_SPLITS_R = 2; /* shares of a (sequence, head)'s keys */
constexpr uint32_t SPIN_LIMIT = 1u << 22; /* polls, about half a microsecond each */
/* Ticks of 10 ns for the last one.  Steps on one or two streams never come to it; more streams' launches take each other's
 * compute units.  us a step of 8 / 16 / 64 sequences on four streams: 46.3 / 48.2 / 53.0 at 10 us, 43.8 / 46.4 / 51.4 at 5, no better at
 * 3, and at 2 steps on two streams come to it (8 sequences 33.4 -> 40.1).  (77 / 81 for 16 / 64 at 40 us.) */
constexpr uint32_t ROLL_LIMIT = 500;
constexpr uint32_t MAX_HIDDEN = 1024;

struct ResidentLayer {
    const float *xnorm, *xq, *xproj; /* cross block; xq == NULL: the layer has none */
    const float *xk, *xv;            /* tier-2 slabs */
    const float *norm1, *qkv, *proj, *norm2, *up, *gate, *down;
    float *ck, *cv; /* tier-1 slabs */
};

struct ResidentArgs {
    ResidentLayer layer[MAX_LAYERS];
    const float *d0; /* input rows: row r is d0 + in_row(r) * E */
    const float *lm;
    float *logits;
    const float *cos, *sin;
    uint64_t *words;   /* hand-over words, group_words per group */
    uint64_t *rolls;   /* a word per workgroup, WORKERS per group */
    uint32_t *timeout; /* pinned host word */
    uint64_t group_words;
    uint64_t max_seq, slab_x; /* rows per sequence of the tier-1 / tier-2 slabs */
    uint32_t L, E, H, hidden, V;
    uint32_t batch, n, per_group; /* sequences, rows per sequence, sequences per group */
    uint32_t splits;              /* shares of the keys */
    uint32_t subtokens, window, block_kind;
    uint32_t tag; /* tag of layer 0; layer l uses tag + l */
    uint32_t roll_limit, spin_limit;
    uint32_t indexed; /* rows come from d0 + row_index[r] * E and sit at position[r] (one sequence) */
    float scale;      /* log2(e) / sqrt(head_dim) */
    float xscale;     /* 1 / sqrt(head_dim) */
    uint32_t len[MAX_ROWS];    /* per sequence */
    uint16_t latent[MAX_ROWS]; /* per row */
    uint16_t row_index[MAX_GROUP_ROWS], position[MAX_GROUP_ROWS];
};
static_assert(sizeof(ResidentArgs) <= 4096, "kernel argument block");

/* The hand-over regions of one group, in words; RT 16-row tiles of rows, E columns, D of the hidden layer.
 *
 * A region that a product reads as its left operand holds element (row, k) in word (step * RT + row / 16) * 64 +
 * k / 4 % 4 * 16 + row % 16 of step k / 16 * 4 + k % 4: a wave's operand for the four k of a step, in the order of the
 * lanes of a 16x16x4 fragment, is 64 consecutive words, and lane (g, c) gets the terms 4 g ... 4 g + 3 of a block of
 * sixteen in its four steps.  Q and K of the new rows: per (row tile, head) and
 * s < HD / 4 the 64 words of the lanes (g, c) = element HD / 4 * g + s of row c.  V: rows of HD words. */
template <int E, int RT>
struct Regions {
    static constexpr uint32_t M = 16u * RT * E;
    static constexpr uint32_t cur0 = 0, cur1 = M, xcomb = 2 * M, mid = 3 * M, q = 4 * M, k = 5 * M, v = 6 * M, resid = 7 * M;
    static constexpr uint32_t comb = 8 * M, stat = (8 + MAX_SPLITS_R) * M, act = stat + MAX_SPLITS_R * 16u * RT * (E / 32u) * 2u;
    static constexpr uint32_t total(uint32_t hidden) { return act + 16u * RT * hidden; }
    static __device__ __forceinline__ uint32_t input(uint32_t layer) { return layer & 1u ? cur0 : cur1; }
    static __device__ __forceinline__ uint32_t output(uint32_t layer) { return layer & 1u ? cur1 : cur0; }
};

__device__ __forceinline__ uint64_t word_load(const uint64_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void word_store(uint64_t *p, float v, uint32_t tag) {
    __hip_atomic_store(p, ((uint64_t)tag << 32) | __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <int RT>
__host__ __device__ __forceinline__ constexpr uint32_t operand_at(uint32_t row, uint32_t k) {
    return ((((k >> 4) << 2) + (k & 3u)) * RT + (row >> 4)) * 64u + ((k >> 2) & 3u) * 16u + (row & 15u);
}
/* What lane (g, c) polls of row tile rt, counted from the step's first word: its own row's word, or the last row's where there
 * is no such row.  That one may lie in an earlier tile: of two row tiles the second has no row at all in a group of up to sixteen. */
__host__ __device__ __forceinline__ constexpr uint32_t polled_at(uint32_t rt, uint32_t g, uint32_t c, uint32_t rows) {
    const uint32_t own = 16u * rt + c, row = own < rows ? own : rows - 1u;
    return (row >> 4) * 64u + g * 16u + (row & 15u);
}
/* Stores are guarded by the rows a group has, so a wait ends only if every word it polls is one of a row below `rows`. */
template <int RT>
constexpr bool polled_words_are_stored() {
    for (uint32_t rows = 1u; rows <= 16u * RT; rows++)
        for (uint32_t lane = 0u; lane < 64u * RT; lane++) {
            const uint32_t g = lane >> 4 & 3u, word = polled_at(lane >> 6, g, lane & 15u, rows);
            bool stored = false;
            for (uint32_t row = 0u; row < rows && !stored; row++) stored = operand_at<RT>(row, 4u * g) == word;
            if (!stored) return false;
        }
    return true;
}
static_assert(polled_words_are_stored<1>() && polled_words_are_stored<2>(), "a wait for a word that nobody writes never ends");
/* the first lane group's term of a step; lane (g, c) has the one 4 g further */
__device__ __forceinline__ constexpr uint32_t term_of(uint32_t step) { return (step >> 2) * 16u + (step & 3u); }

/* A wave's waiting state: once one wait has run out, none of the wave's later ones wait. */
struct Waiter {
    uint32_t *timeout;
    uint32_t limit;
    bool expired;
};
__device__ __forceinline__ float not_there() { return __builtin_nanf(""); }

/* N words per lane, the one number i at(i), until every lane has them all.  A wave that
 * misses some looks again after a sleep: at all of them while they are few, else at the last one only
 * until that one is there.  Eight waves that poll twenty words each keep the compute unit's vector memory path
 * full, and it serves the oldest waves first -- a younger workgroup on the same unit that has to produce the
 * words then never gets a request in. */
/* Those from FIRST on carry the tag `tag` ^ `turn`: words written before the others could be, brought along because a wait of
 * their own would be another trip. */
template <int N, int FIRST, typename At>
__device__ __forceinline__ void await_mixed(Waiter &wt, At at, uint32_t tag, uint32_t turn, float (&out)[N], uint32_t line) {
    uint64_t t[N];
    for (uint32_t spin = 0;; spin++) {
        uint32_t off = 0;
#pragma unroll
        for (int i = 0; i < N; i++) t[i] = word_load(at(i));
#pragma unroll
        for (int i = 0; i < N; i++) off |= (uint32_t)(t[i] >> 32) ^ tag ^ (i < FIRST ? 0u : turn);
        if (__all(off == 0u) || wt.expired) break;
        __builtin_amdgcn_s_setprio(0);
        if (N > 4) {
            bool missing;
            do {
                __builtin_amdgcn_s_sleep(1);
                missing = (uint32_t)(word_load(at(FIRST - 1)) >> 32) != tag;
                spin++;
            } while (__any(missing) && spin < wt.limit);
        } else {
            __builtin_amdgcn_s_sleep(1);
        }
        __builtin_amdgcn_s_setprio(2);
        if (spin >= wt.limit) {
            wt.expired = true;
            __hip_atomic_store(wt.timeout, (blockIdx.x << 16) | line, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
#pragma unroll
    for (int i = 0; i < N; i++) out[i] = __uint_as_float((uint32_t)t[i]);
    out[0] = wt.expired ? not_there() : out[0]; /* one of a row's values is enough to make every sum of it NaN */
}
template <int N, typename At>
__device__ __forceinline__ void await_at(Waiter &wt, At at, uint32_t tag, float (&out)[N], uint32_t line) {
    await_mixed<N, N>(wt, at, tag, 0u, out, line);
}
/* word `index` of a region: a uniform base and a 32-bit byte offset per lane, which the load takes as they are */
__device__ __forceinline__ const uint64_t *word_of(const uint64_t *base, uint32_t index) {
    return reinterpret_cast<const uint64_t *>(reinterpret_cast<const char *>(base) + index * 8u);
}
template <int N, int STRIDE>
__device__ __forceinline__ void await(Waiter &wt, const uint64_t *base, uint32_t index, uint32_t tag, float (&out)[N],
                                      uint32_t line = __builtin_LINE()) {
    const uint64_t *p = word_of(base, index);
    await_at<N>(wt, [&](int i) { return p + i * STRIDE; }, tag, out, line);
}

/* The argument block is hidden from the optimiser once per stage: it would otherwise compute the addresses of
 * all stages ahead of the layer loop and spill them. */
typedef const __attribute__((address_space(4))) ResidentArgs *ArgsPtr;
__device__ __forceinline__ ArgsPtr hidden_args(ArgsPtr args) {
    uint32_t zero;
    asm volatile("s_mov_b32 %0, 0" : "=s"(zero));
    return (ArgsPtr)((const __attribute__((address_space(4))) char *)args + zero);
}

/* An array as a wave reads it: elements at an index all lanes share and an offset of the lane's own, which the load takes as
 * a scalar base and 32 bits -- no vector instruction and no register pair per address. */
struct LaneView {
    const char *base;
    uint32_t off; /* bytes */
    __device__ __forceinline__ LaneView(const float *p, uint32_t index) : base(reinterpret_cast<const char *>(p)), off(4u * index) {}
    __device__ __forceinline__ float operator[](size_t i) const { return *reinterpret_cast<const float *>(base + 4u * i + off); }
    __device__ __forceinline__ floatx4 four(size_t i) const { return *reinterpret_cast<const floatx4 *>(base + 4u * i + off); }
};
struct GroupView {
    uint64_t *words;
    uint32_t seq0, ns, row0, rows; /* the group's sequences and rows */
    uint32_t worker, wave;
};

constexpr uint32_t WORKERS = 32; /* workgroups of a group: one per compute unit of a die */
/* Tile 0 of a stage goes to this worker, tile 1 to the next: consecutive stages on different workgroups where there are few
 * tiles, so that the ones of a stage have its weights in registers when its operand comes. */
constexpr uint32_t FIRST_XQ = 24, FIRST_XPROJ = 0, FIRST_QKV = 0, FIRST_PROJ = 8, FIRST_UPGATE = 0, FIRST_DOWN = 24, FIRST_LM = 0;

/* Stages of a layer in their order, and the LM head behind the last layer */
enum Stage : uint32_t { STAGE_XQ, STAGE_XPROJ, STAGE_QKV, STAGE_ATTN, STAGE_PROJ, STAGE_UPGATE, STAGE_DOWN, STAGES, STAGE_LM = STAGES };
struct Standing {
    uint32_t rank, members; /* members == 0: the work is others' */
};
/* The roll call of a group.  A word per workgroup: 2 tag = in, 2 tag + 1 = out, less = not decided yet.  Words only grow and
 * each is decided once, so everybody comes to the same list. */
__device__ __forceinline__ void sign_in(uint64_t *roll, uint32_t index, uint32_t tag) {
    __hip_atomic_fetch_max(roll + index, 2ull * tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
/* by one wave of each workgroup; lane i and lane i + 32 look at workgroup i's word */
__device__ __forceinline__ Standing call_roll(uint64_t *roll, uint32_t index, uint32_t tag, uint32_t limit) {
    static_assert(WORKERS == 32u, "a half of the wave's lanes");
    const uint32_t lane = threadIdx.x & (WORKERS - 1u);
    const uint64_t in = 2ull * tag;
    const uint64_t begin = wall_clock64();
    for (;;) {
        uint64_t word = __hip_atomic_load(roll + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t present = (uint32_t)__ballot(word == in) & (uint32_t)(__ballot(word == in) >> 32);
        if (__all(word >= in)) {
            if ((present >> index & 1u) == 0u) return {0u, 0u};
            return {(uint32_t)__popc(present & ((1u << index) - 1u)), (uint32_t)__popc(present)};
        }
        /* only who is in for good signs others out: somebody always is */
        if ((present >> index & 1u) != 0u && (wall_clock64() - begin) * (uint64_t)__popc(present) >= (uint64_t)WORKERS * limit && word < in)
            __hip_atomic_compare_exchange_strong(roll + lane, &word, in + 1ull, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_s_sleep(1);
    }
}

/* What a run of a worker works on: one stage (STAGES of layer L: the LM head) ... */
struct OneStage {
    uint32_t layer, stage;
    __device__ __forceinline__ uint32_t begin() const { return layer; }
    __device__ __forceinline__ uint32_t end(uint32_t L) const { return min(layer + 1u, L); }
    __device__ __forceinline__ bool has(Stage st) const { return st == stage; }
    __device__ __forceinline__ bool all_here(uint32_t) { return true; }
};
/* ... or everything, if all workgroups of the group are there: it asks before its first wait and its first store, with
 * its first loads on their way, and returns if not.  All waves of a workgroup ask at the same place. */
struct WholeStep {
    ArgsPtr args;
    uint32_t group, index;
    Standing *standing; /* in LDS */
    bool asked;
    __device__ __forceinline__ uint32_t begin() const { return 0u; }
    __device__ __forceinline__ uint32_t end(uint32_t L) const { return L; }
    __device__ __forceinline__ bool has(Stage) const { return true; }
    __device__ __forceinline__ bool all_here(uint32_t wave) {
        if (asked) return true;
        asked = true;
        if (wave == 0u) {
            const Standing st = call_roll(args->rolls + group * WORKERS, index, args->tag, args->roll_limit);
            if ((threadIdx.x & 63u) == 0u) *standing = st;
        }
        __syncthreads();
        return __builtin_amdgcn_readfirstlane(standing->members) == WORKERS;
    }
};

/* FOLD: one sub-token a patch */
template <int E_, int HD_, int RT_, bool FOLD>
struct ResidentShape {
    static constexpr int E = E_, HD = HD_, RT = RT_, H = E / HD;
    /* up to 128 columns a wave has 16 of the terms of a product over E, and stages that need all of a row's columns are done
     * again by every workgroup of the stage behind them (see the head of the file) */
    static constexpr bool MERGED = E <= 128;
    /* the cross block among them, which is folded into the QKV stage.  Folding takes a product with W_q and one with W_proj for every
     * sub-token, a stage of its own only a dot product: one row, two layers of 128 columns, folded / not, us: one sub-token 34 / 36, two
     * 45 / 37, eight 105 / 41; 64 columns 24 / 28, 29 / 29, 54 / 34 */
    static constexpr bool FOLDED = MERGED && FOLD;
    static constexpr int AW = E < 128 ? E / 16 : 8; /* waves with a share of E */
    static constexpr int KB = E / 4 / AW;           /* four-term steps of a share */
    /* products over E whose whole row every workgroup needs: column groups of 64, a quarter of the terms a wave */
    static constexpr int CG = MERGED ? E / 64 : 1, QS = E / 16; /* at least four; four-term steps of a quarter */
    static constexpr int ROW = HD + 4, PITCH = E + 4, DT = HD / 16;
    static constexpr int NB = FOLDED || DT < 2 ? 2 : DT; /* column tiles of a product at once */
};
template <typename S>
struct ResidentLds {
    float part[2][WAVES][S::RT][S::NB][256]; /* partial tiles */
    float part_ss[2][16 * S::RT][WAVES];
    float keys[WAVES][16 * S::ROW]; /* attention: a wave's tile of key, value or output rows */
    float most[16][WAVES], sum[16][WAVES];
    float quarters[S::MERGED ? 4 : 1][S::MERGED ? 16 * S::RT * S::PITCH : 4]; /* products over E by quarters of the terms */
    float xkey[S::FOLDED ? 16 * S::RT * S::PITCH : 4], xvalue[S::FOLDED ? 16 * S::RT * S::PITCH : 4]; /* the sub-token of every row */
    float score[S::FOLDED ? WAVES : 1][S::FOLDED ? 16 * S::RT : 1][8];
    float xquery[S::FOLDED ? 1 : 16 * S::RT][S::HD];
    uint32_t len[MAX_GROUP_ROWS], latent[MAX_GROUP_ROWS]; /* of the group's sequences / rows */
    Standing standing;
};

/* One worker's part: every stage in its order, or one of them.  A stage of a product: its weights, the operand as soon as
 * it is there, the product over the wave's share of the terms, the waves' partial tiles through LDS, the results of 256 threads
 * per row tile. */
template <typename S, typename Share>
__device__ __forceinline__ void run_worker(ArgsPtr args, const GroupView gv, Share &sh, ResidentLds<S> &sm) {
    constexpr int E = S::E, HD = S::HD, RT = S::RT, H = S::H, KB = S::KB, AW = S::AW, DT = S::DT, QD = HD / 4, PITCH = S::PITCH, QS = S::QS;
    constexpr uint32_t CG = S::CG;
    using At = Regions<E, RT>;
    constexpr uint32_t RPW = 64 / HD; /* rows a wave attends at a time in the cross block */
    const uint32_t wave = gv.wave, rows = gv.rows;
    const bool sharing = wave < (uint32_t)AW; /* the wave has a share of a product over E */
    /* what this thread finishes: element (4 wave' + lane % 4, lane / 4) of row tile wave / 4 */
    const uint32_t f_rt = RT == 1 ? 0u : wave >> 2;
    const bool f_on = (RT == 2 || wave < 4u) && 16u * f_rt + 4u * (wave & 3u) < rows; /* the wave has rows to finish */
    uint32_t lane, g, c, f_row, f_col, f_safe;
    /* once per stage, hidden from the optimiser like the argument block */
    auto fresh_lane = [&]() __attribute__((always_inline)) {
        lane = threadIdx.x & 63u;
        asm volatile("" : "+v"(lane));
        g = lane >> 4, c = lane & 15u, f_col = lane >> 2;
        f_row = 16u * f_rt + 4u * (wave & 3u) + (lane & 3u), f_safe = min(f_row, rows - 1u);
    };
    fresh_lane();
    uint64_t *const words = gv.words;
    Waiter wt{args->timeout, args->spin_limit, false};
    uint32_t buf = 0;
    auto first = [&](uint32_t at) { return (gv.worker - at) & (WORKERS - 1u); };
    const uint32_t step0 = sharing ? KB * wave : 0u; /* the wave's share of E starts here (waves without one: anything in bounds) */

    /* this lane's word of a step, from the step's first word on */
    auto polled = [&](int rt) __attribute__((always_inline)) { return polled_at((uint32_t)rt, g, c, rows); };
    /* the left operand of this wave's N steps from step s0 on */
    auto operand = [&](auto kbn, uint32_t region, uint32_t s0, uint32_t tag, float (&av)[RT][decltype(kbn)::value])
                       __attribute__((always_inline)) {
        constexpr int N = decltype(kbn)::value;
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
            await<N, RT * 64>(wt, words + region + s0 * (RT * 64u), polled(rt), tag, av[rt]);
    };
    auto plain_row = [&](ArgsPtr ap, uint32_t row) { return ap->d0 + (size_t)(ap->indexed ? ap->row_index[row] : gv.row0 + row) * E; };
    /* ... of layer 0: the rows as the caller has them */
    auto operand_plain = [&](auto kbn, ArgsPtr ap, uint32_t s0, float (&av)[RT][decltype(kbn)::value]) __attribute__((always_inline)) {
        constexpr int N = decltype(kbn)::value;
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            const float *src = plain_row(ap, min(16u * rt + c, rows - 1u)) + 4u * g;
#pragma unroll
            for (int i = 0; i < N; i++) av[rt][i] = src[term_of(s0 + i)];
        }
    };
    /* this wave's partial tiles to LDS; buffers alternate, so one barrier per product is enough */
    auto leave = [&](auto nb, floatx4 (&acc)[RT][decltype(nb)::value], const float *ss) __attribute__((always_inline)) {
        constexpr int NB = decltype(nb)::value;
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
#pragma unroll
            for (int j = 0; j < NB; j++) *reinterpret_cast<floatx4 *>(&sm.part[buf][wave][rt][j][lane * 4u]) = acc[rt][j];
        if (ss != nullptr) {
#pragma unroll
            for (int rt = 0; rt < RT; rt++) {
                const float q = swap32(swap16(ss[rt], OpSum()), OpSum());
                if (g == 0) sm.part_ss[buf][16 * rt + c][wave] = q;
            }
        }
    };
    /* the finished element of column tile j of KS waves' parts */
    auto total = [&](auto ksn, uint32_t rt, uint32_t j) __attribute__((always_inline)) {
        constexpr uint32_t KS = decltype(ksn)::value;
        const float *p0 = &sm.part[buf][0][rt][j][(wave & 3u) * 64u + lane];
        float s0 = 0.f, s1 = 0.f;
#pragma unroll
        for (uint32_t v = 0; v < KS; v += 2) s0 += p0[v * (RT * S::NB * 256)], s1 += p0[(v + 1) * (RT * S::NB * 256)];
        return s0 + s1;
    };
    auto row_scale = [&](uint32_t row) __attribute__((always_inline)) {
        float s = 0.f;
#pragma unroll
        for (int v = 0; v < AW; v += 4) {
            const float4 x = *reinterpret_cast<const float4 *>(&sm.part_ss[buf][row][v]);
            s += (x.x + x.y) + (x.z + x.w);
        }
        return 1.0f / sqrtf(s * (1.0f / (float)E) + 1e-6f); /* reductions_cpu.c:345-346 */
    };
    using All = std::integral_constant<uint32_t, WAVES>;
    using Sharing = std::integral_constant<uint32_t, AW>;
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    using Steps = std::integral_constant<int, KB>;
    /* acc[rt] += the wave's share of a product with one column tile */
    auto product = [&](const float (&av)[RT][KB], const float (&b)[KB], floatx4 (&acc)[RT][1]) __attribute__((always_inline)) {
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            floatx4 a[4];
#pragma unroll
            for (int i = 0; i < 4; i++) a[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[rt][i], b[i], floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
            for (int i = 4; i < KB; i++) a[i & 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[rt][i], b[i], a[i & 3], 0, 0, 0);
            acc[rt][0] = (a[0] + a[1]) + (a[2] + a[3]);
        }
    };
    /* The attention's output as the left operand: its words, or the shares' sums, weighed with the common maximum and
     * divided by the common sum; a wave's columns are of one head where keys are shared out.  With it M words more, written
     * before the attention's output could be: waited for on their own they would be another trip. */
    auto attended = [&](auto sn, auto mn, uint32_t s_lo, bool shares, uint32_t tag, int rt, auto more, uint32_t more_tag,
                        float (&av)[decltype(sn)::value], float (&extra)[decltype(mn)::value ? decltype(mn)::value : 1]) __attribute__((always_inline)) {
        constexpr int KN = decltype(sn)::value, M = decltype(mn)::value;
        const uint32_t turn = more_tag ^ tag; /* all tags of a wait are compared with one */
        const uint64_t *p = word_of(words + At::comb + s_lo * (RT * 64u), polled(rt));
        if (!shares) {
            float all[KN + M];
            await_mixed<KN + M, KN>(wt, [&](int i) { return i < KN ? p + i * (RT * 64) : more(i - KN); }, tag, turn, all, __LINE__);
#pragma unroll
            for (int i = 0; i < KN; i++) av[i] = all[i];
#pragma unroll
            for (int i = 0; i < M; i++) extra[i] = all[KN + i];
            return;
        }
        const uint32_t head = 4u * s_lo / HD;
        float all[2 * KN + 4 + M];
        const uint64_t *st = word_of(words + At::stat + head * (32u * RT), min(16u * rt + c, rows - 1u) * 2u);
        await_mixed<2 * KN + 4 + M, 2 * KN + 4>(wt, [&](int i) {
            if (i < 2 * KN) return p + (i % KN) * (RT * 64) + (i < KN ? 0u : At::M);
            if (i < 2 * KN + 4) return st + ((i - 2 * KN) >> 1) * (H * 32 * RT) + (i & 1);
            return more(i - 2 * KN - 4);
        }, tag, turn, all, __LINE__);
        const float *s0 = all, *s1 = all + KN, *st0 = all + 2 * KN, *st1 = all + 2 * KN + 2;
        const float most = fmaxf(st0[0], st1[0]), base = most == neg_inf() ? 0.f : most;
        const float f0 = fast_exp2(st0[0] - base), f1 = fast_exp2(st1[0] - base), Lt = st0[1] * f0 + st1[1] * f1;
#pragma unroll
        for (int i = 0; i < KN; i++) av[i] = Lt == 0.f ? 0.f : (s0[i] * f0 + s1[i] * f1) / Lt;
#pragma unroll
        for (int i = 0; i < M; i++) extra[i] = all[2 * KN + 4 + i];
    };
    /* the wave's quarter of a product over E with its 64 columns, 16 rows: to LDS; and the quarter q of this wave's share, in
     * the layout of the operand */
    auto by_quarter = [&](int rt, const float (&x)[S::QS], const floatx4 (&w)[S::QS]) __attribute__((always_inline)) {
        /* chains of at most sixteen terms: with a quarter of 128 terms in one the step had 1.2 times the error */
        constexpr int CHAINS = S::QS == 4 ? 4 : 2;
        floatx4 acc[CHAINS][4];
#pragma unroll
        for (int i = 0; i < CHAINS; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i], w[i][j], floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
        for (int i = CHAINS; i < S::QS; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) acc[i % CHAINS][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i], w[i][j], acc[i % CHAINS][j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 4; j++) acc[0][j] = CHAINS == 4 ? (acc[0][j] + acc[1][j]) + (acc[CHAINS - 2][j] + acc[CHAINS - 1][j]) : acc[0][j] + acc[1][j];
        float *const to = sm.quarters[wave / S::CG & 3u] + 64u * (wave % S::CG) + 4u * c;
#pragma unroll
        for (int r = 0; r < 4; r++)
            *reinterpret_cast<floatx4 *>(to + (16u * rt + 4u * g + r) * PITCH) = floatx4{acc[0][0][r], acc[0][1][r], acc[0][2][r], acc[0][3][r]};
    };
    auto quarter_at = [&](int rt, int q) __attribute__((always_inline)) {
        return *reinterpret_cast<const floatx4 *>(sm.quarters[q] + (16u * rt + c) * PITCH + 4u * step0 + 4u * g);
    };
    /* [rows, E] products with one residual row added, as a stage of their own: cross projection, output projection */
    auto square = [&](ArgsPtr ap, const float *w, bool of_attention, uint32_t tag, bool res_plain, uint32_t res, uint32_t res_tag,
                      uint32_t to, uint32_t t) __attribute__((always_inline)) {
        fresh_lane();
        float b[KB], av[RT][KB], r1[1] = {0.f};
        const LaneView wp(w + t * 16u, 4u * g * E + c);
#pragma unroll
        for (int i = 0; i < KB; i++) b[i] = wp[term_of(step0 + i) * E];
        const uint32_t oc = t * 16u + f_col;
        if (f_on && res_plain) r1[0] = plain_row(ap, f_safe)[oc];
        if (!sh.all_here(wave)) return false;
        const uint64_t *const rp = word_of(words + res, operand_at<RT>(f_safe, oc));
        if (of_attention) {
#pragma unroll
            for (int rt = 0; rt < RT; rt++) {
                float none[1];
                if (res_plain) attended(Steps(), std::integral_constant<int, 0>(), step0, ap->splits > 1u, tag, rt, [&](int) { return rp; }, tag, av[rt], none);
                else attended(Steps(), One(), step0, ap->splits > 1u, tag, rt, [&](int) { return rp; }, res_tag, av[rt], r1);
            }
        } else {
            operand(Steps(), At::xcomb, step0, tag, av);
            if (f_on && !res_plain) /* written before this stage's operand could be: seen at the first look */
                await<1, 1>(wt, rp, 0u, res_tag, r1);
        }
        floatx4 acc[RT][1];
        product(av, b, acc);
        leave(One(), acc, nullptr);
        __syncthreads();
        if (f_on && f_row < rows) word_store(words + to + operand_at<RT>(f_row, oc), r1[0] + total(Sharing(), f_rt, 0), tag);
        buf ^= 1u;
        return true;
    };

    /* ---- units of the self-attention: one (sequence, head, share of the keys) each ---- */
    constexpr int NV = QD / 4, ROW = S::ROW, LPR = HD / 4, RPI = 64 / LPR;
    constexpr int T = HD == 32 ? 2 : 1; /* key tiles a wave has in registers as fragments, and as many on their way */
    struct Unit {
        uint32_t split, head, sq, len, t_lo, t_hi;
    };
    auto unit_of = [&](ArgsPtr ap, uint32_t u) __attribute__((always_inline)) {
        const uint32_t splits = ap->splits;
        Unit un;
        un.split = u % splits, un.head = (u / splits) % (uint32_t)H, un.sq = u / (splits * (uint32_t)H);
        un.len = __builtin_amdgcn_readfirstlane(sm.len[un.sq]);
        const bool windowed = ap->window > 0u && !ap->block_kind;
        const uint32_t lo = windowed && un.len + 1u > ap->window ? (un.len + 1u - ap->window) / 16u : 0u;
        const uint32_t cached = (un.len + 15u) / 16u; /* tiles of cached rows */
        const uint32_t share = (cached - min(lo, cached) + splits - 1u) / splits;
        un.t_lo = min(lo + un.split * share, cached), un.t_hi = min(un.t_lo + share, cached);
        return un;
    };
    const uint32_t L = args->L;
    for (uint32_t layer = sh.begin(); layer < sh.end(L); layer++) {
        ArgsPtr ap = hidden_args(args);
        const uint32_t tag = ap->tag + layer;
        const bool crossed = ap->layer[layer].xq != nullptr, plain = layer == 0u;
        const uint32_t in = At::input(layer);
        const uint32_t units = gv.ns * (uint32_t)H * ap->splits;
        const uint32_t unit0 = first(units < WORKERS ? WORKERS - units : 0u); /* few: where no tile of the stage before is */
        fresh_lane();
        floatx4 kg[T][NV], vg[T][NV]; /* rows of the wave's next key tiles on their way */
        auto request_keys = [&](ArgsPtr ap, uint32_t layer, const Unit &un, uint32_t tb) __attribute__((always_inline)) {
            const size_t slab = ((size_t)(gv.seq0 + un.sq) * ap->max_seq) * E + un.head * HD;
            const char *kb = reinterpret_cast<const char *>(ap->layer[layer].ck + slab);
            const char *vb = reinterpret_cast<const char *>(ap->layer[layer].cv + slab);
            const uint32_t prow = lane / LPR, pf = lane % LPR;
#pragma unroll
            for (int u2 = 0; u2 < T; u2++)
                if (tb + WAVES * u2 < un.t_hi) { /* wave-uniform */
#pragma unroll
                    for (int v = 0; v < NV; v++) {
                        const uint32_t off = min((tb + WAVES * u2) * 16u + prow + (uint32_t)(RPI * v), un.len - 1u) * (4u * E) + 16u * pf;
                        kg[u2][v] = *reinterpret_cast<const floatx4 *>(kb + off);
                        vg[u2][v] = *reinterpret_cast<const floatx4 *>(vb + off);
                    }
                }
        };
        bool keys_asked = !(sh.has(STAGE_ATTN) && unit0 < units);
        auto early_keys = [&]() __attribute__((always_inline)) { /* of the first unit, before the wait of the stage before */
            if (keys_asked) return;
            keys_asked = true;
            const Unit un = unit_of(ap, unit0);
            request_keys(ap, layer, un, un.t_lo + wave);
        };

        if constexpr (!S::FOLDED) {
            if (crossed && sh.has(STAGE_XQ) && first(FIRST_XQ) < (uint32_t)H) { /* ---- query projection of one cross head, its rows' cross attention ---- */
                const uint32_t head = first(FIRST_XQ);
                float b[DT][KB], av[RT][KB], ss[RT];
                const LaneView w(ap->layer[layer].xq + head * HD, 4u * g * E + c), nw(ap->layer[layer].xnorm, 4u * g);
#pragma unroll
                for (int i = 0; i < KB; i++) {
                    const uint32_t k = term_of(step0 + i);
                    const float n1 = nw[k];
#pragma unroll
                    for (int j = 0; j < DT; j++) b[j][i] = w[k * E + 16 * j] * n1;
                }
                /* the first sub-token of this lane's first row */
                const uint32_t xd = lane % HD;
                const float *xk = ap->layer[layer].xk, *xv = ap->layer[layer].xv;
                auto cell = [&](uint32_t row) {
                    return ((size_t)(gv.seq0 + row / ap->n) * ap->slab_x + (size_t)sm.latent[row] * ap->subtokens) * E + head * HD + xd;
                };
                const size_t cell0 = cell(min(wave * RPW + lane / HD, rows - 1u));
                const float early_k = xk[cell0], early_v = xv[cell0];
                if (plain) operand_plain(Steps(), ap, step0, av);
                if (!sh.all_here(wave)) return;
                if (sharing) {
                    if (!plain) operand(Steps(), in, step0, tag - 1u, av);
                    floatx4 acc[RT][DT];
#pragma unroll
                    for (int rt = 0; rt < RT; rt++) {
#pragma unroll
                        for (int j = 0; j < DT; j++) acc[rt][j] = floatx4{0.f, 0.f, 0.f, 0.f};
                        ss[rt] = 0.f;
#pragma unroll
                        for (int i = 0; i < KB; i++) {
#pragma unroll
                            for (int j = 0; j < DT; j++) acc[rt][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[rt][i], b[j][i], acc[rt][j], 0, 0, 0);
                            ss[rt] += av[rt][i] * av[rt][i];
                        }
                    }
                    leave(std::integral_constant<int, DT>(), acc, ss);
                }
                __syncthreads();
                if (f_on) {
                    const float scale = row_scale(f_row) * ap->xscale;
#pragma unroll
                    for (uint32_t j = 0; j < (uint32_t)DT; j++) sm.xquery[f_row][16u * j + f_col] = total(Sharing(), f_rt, j) * scale;
                }
                __syncthreads();
                /* the rows' cross attention over their few sub-tokens (kv_cache.c:303-324): HD lanes per row; maximum
                 * over finite scores, non-finite scores weigh nothing */
                for (uint32_t r0 = wave * RPW; r0 < rows; r0 += WAVES * RPW) {
                    const uint32_t row = min(r0 + lane / HD, rows - 1u);
                    const float qd = sm.xquery[row][xd];
                    const size_t at = cell(row);
                    const bool ahead = r0 == wave * RPW;
                    auto score = [&](float kd) __attribute__((always_inline)) {
                        float p = key_sum<32>(qd * kd);
                        if (HD == 64) p = swap32(p, OpSum());
                        return p;
                    };
                    float o;
                    if (ap->subtokens == 1u) { /* one key: all the weight, or none */
                        const float p = score(ahead ? early_k : xk[at]);
                        const float v = ahead ? early_v : xv[at];
                        o = isfinite(p) ? v : 0.f;
                    } else {
                        float mx = neg_inf(), sum = 0.f;
                        o = 0.f;
                        for (uint32_t j = 0; j < ap->subtokens; j++) {
                            const float p = score(xk[at + (size_t)j * E]);
                            mx = isfinite(p) ? fmaxf(mx, p) : mx;
                        }
                        for (uint32_t j = 0; j < ap->subtokens; j++) {
                            const float p = score(xk[at + (size_t)j * E]);
                            const float e = isfinite(p) ? expf(p - mx) : 0.f;
                            const float v = xv[at + (size_t)j * E];
                            sum += e;
                            o += e != 0.f ? e * v : 0.f;
                        }
                        o = sum > 0.f ? o / sum : 0.f;
                    }
                    if (r0 + lane / HD < rows) word_store(words + At::xcomb + operand_at<RT>(row, head * HD + xd), o, tag);
                }
                buf ^= 1u;
            }
            if (crossed && sh.has(STAGE_XPROJ) && first(FIRST_XPROJ) < (uint32_t)E / 16u &&
                !square(ap, ap->layer[layer].xproj, false, tag, plain, in, tag - 1u, At::mid, first(FIRST_XPROJ)))
                return;
        }

        ap = hidden_args(args);
        for (uint32_t t = first(FIRST_QKV); sh.has(STAGE_QKV) && t < 3u * E / 16u; t += WORKERS) { /* ---- cross block where merged; QKV: rotated, keys and values written through ---- */
            fresh_lane();
            float b[KB], av[RT][KB], ss[RT], cs = 0.f, sn = 0.f;
            const LaneView w(ap->layer[layer].qkv + t * 16u, 4u * g * (3u * E) + c), nw(ap->layer[layer].norm1, 4u * g);
#pragma unroll
            for (int i = 0; i < KB; i++) {
                const uint32_t k = term_of(step0 + i);
                b[i] = w[k * 3u * E] * nw[k];
            }
            const uint32_t part_of = t * 16u / E, cc = t * 16u + f_col - part_of * E, hh = cc / HD, dd = cc % HD;
            const uint32_t sq = f_safe / ap->n, slot = sm.len[sq] + f_safe % ap->n;
            if (f_on && part_of < 2u) { /* rotation of this thread's element */
                const uint32_t pos = ap->indexed ? ap->position[f_safe] : slot;
                cs = ap->cos[(size_t)pos * (HD / 2) + dd / 2u], sn = ap->sin[(size_t)pos * (HD / 2) + dd / 2u];
            }
            const uint32_t of_head = (f_rt * H + hh) * (HD * 16u);
            uint32_t to = part_of < 2u ? (part_of == 0u ? At::q : At::k) + of_head + (dd % QD) * 64u + (dd / QD) * 16u + (f_row & 15u)
                                       : At::v + of_head + (f_row & 15u) * HD + dd;
            float *cell = (part_of == 1u ? ap->layer[layer].ck : ap->layer[layer].cv) + ((size_t)(gv.seq0 + sq) * ap->max_seq + slot) * E + cc;
            asm volatile("" : "+v"(to), "+v"(cell)); /* here, not after the wait */
            const bool from_mid = crossed && !S::FOLDED; /* the cross block is stages of its own */
            if (plain && !from_mid && sharing) operand_plain(Steps(), ap, step0, av);

            if constexpr (S::FOLDED) {
                if (crossed) {
                    /* The cross block before its input is there.  A score is q . k = (x W_q) . k / rms = x . (n W_q k) / rms and the
                     * projected output the weighed sum of v W_proj: both vectors, per row and head, need weights and sub-tokens
                     * only.  The first comes out of the matrix instructions in the layout of the operand: element (k, row) in
                     * lane (k / 4 % 4, row); the second is made by quarters of its terms.  Weights come as whole lines of memory: a
                     * load whose lanes are on sixteen rows takes four times as long. */
                    constexpr int XR = (16 * RT * E / 4 + 64 * (int)WAVES - 1) / (64 * (int)WAVES), QB = QS / 4;
                    const uint32_t k0 = 4u * step0; /* the wave's sixteen columns */
                    const uint32_t prow = lane / LPR, pf = lane % LPR, cg = wave % CG, quarter = wave / CG & 3u;
                    floatx4 wq[H][NV], wp[QS], xr[2][XR];
                    auto request = [&](uint32_t l) __attribute__((always_inline)) { /* weights; the sub-token of every row */
#pragma unroll
                        for (int i = 0; i < XR; i++) {
                            const uint32_t at4 = min(threadIdx.x + 64u * WAVES * i, 16u * RT * E / 4u - 1u), row = min(at4 / (E / 4u), rows - 1u);
                            const size_t at = ((size_t)(gv.seq0 + row / ap->n) * ap->slab_x + sm.latent[row]) * E + 4u * (at4 % (E / 4u));
                            xr[0][i] = *reinterpret_cast<const floatx4 *>(ap->layer[l].xk + at), xr[1][i] = *reinterpret_cast<const floatx4 *>(ap->layer[l].xv + at);
                        }
                        const LaneView q(ap->layer[l].xq + k0 * E, prow * E + 4u * pf), pr(ap->layer[l].xproj + quarter * (E / 4u) * E + 64u * cg, 4u * g * E + 4u * c);
#pragma unroll
                        for (int h = 0; h < H; h++)
#pragma unroll
                            for (int v = 0; v < NV; v++) wq[h][v] = q.four(h * HD + RPI * v * E);
#pragma unroll
                        for (int i = 0; i < QS; i++) wp[i] = pr.four(term_of(i) * E);
                    };
                    auto park_rows = [&]() __attribute__((always_inline)) {
#pragma unroll
                        for (int i = 0; i < XR; i++) {
                            const uint32_t at4 = threadIdx.x + 64u * WAVES * i, to4 = at4 / (E / 4u) * PITCH + 4u * (at4 % (E / 4u));
                            if (at4 < 16u * RT * E / 4u)
                                *reinterpret_cast<floatx4 *>(sm.xkey + to4) = xr[0][i], *reinterpret_cast<floatx4 *>(sm.xvalue + to4) = xr[1][i];
                        }
                    };
                    floatx4 key[RT][H];
                    auto fold = [&]() __attribute__((always_inline)) {
                        const floatx4 nx = LaneView(ap->layer[layer].xnorm + k0, 4u * g).four(0);
                        float *const tile = sm.keys[wave];
#pragma unroll
                        for (int h = 0; h < H; h++) { /* rows -> fragments, through the wave's own LDS tile */
#pragma unroll
                            for (int v = 0; v < NV; v++) *reinterpret_cast<floatx4 *>(tile + (prow + (uint32_t)(RPI * v)) * ROW + 4u * pf) = wq[h][v];
                            floatx4 q[NV];
#pragma unroll
                            for (int v = 0; v < NV; v++) q[v] = *reinterpret_cast<const floatx4 *>(tile + c * ROW + QD * g + 4 * v);
#pragma unroll
                            for (int rt = 0; rt < RT; rt++) {
                                floatx4 u0 = floatx4{0.f, 0.f, 0.f, 0.f}, u1 = u0;
#pragma unroll
                                for (int v = 0; v < NV; v++) {
                                    const floatx4 kx = *reinterpret_cast<const floatx4 *>(sm.xkey + (16u * rt + c) * PITCH + h * HD + QD * g + 4 * v);
#pragma unroll
                                    for (int i = 0; i < 4; i += 2) {
                                        u0 = __builtin_amdgcn_mfma_f32_16x16x4f32(q[v][i], kx[i], u0, 0, 0, 0);
                                        u1 = __builtin_amdgcn_mfma_f32_16x16x4f32(q[v][i + 1], kx[i + 1], u1, 0, 0, 0);
                                    }
                                }
                                key[rt][h] = (u0 + u1) * nx;
                            }
                        }
#pragma unroll
                        for (int rt = 0; rt < RT; rt++) {
                            float vx[QS];
#pragma unroll
                            for (int b4 = 0; b4 < QB; b4++) {
                                const floatx4 x4 = *reinterpret_cast<const floatx4 *>(sm.xvalue + (16u * rt + c) * PITCH + quarter * (E / 4u) + 16 * b4 + 4u * g);
#pragma unroll
                                for (int i = 0; i < 4; i++) vx[4 * b4 + i] = x4[i];
                            }
                            by_quarter(rt, vx, wp);
                        }
                    };
                    /* d[h]: the rows' products with head h's key, d[4]: their sums of squares */
                    auto scores = [&](float (&d)[RT][5]) __attribute__((always_inline)) {
                        if (sharing) {
#pragma unroll
                            for (int rt = 0; rt < RT; rt++) {
                                float mine = 0.f, squares = 0.f;
#pragma unroll
                                for (int i = 0; i < 4; i++) squares += av[rt][i] * av[rt][i];
                                squares = swap32(swap16(squares, OpSum()), OpSum());
#pragma unroll
                                for (int h = 0; h < H; h++) {
                                    float p = (av[rt][0] * key[rt][h][0] + av[rt][1] * key[rt][h][1]) + (av[rt][2] * key[rt][h][2] + av[rt][3] * key[rt][h][3]);
                                    p = swap32(swap16(p, OpSum()), OpSum());
                                    mine = g == (uint32_t)h ? p : mine;
                                }
                                float *const to = sm.score[wave][16 * rt + c];
                                to[g] = mine;
                                if (g == 0u) to[4] = squares;
                            }
                        }
                        __syncthreads();
                        if (sharing) {
#pragma unroll
                            for (int rt = 0; rt < RT; rt++) { /* lane (g, c) adds up the waves g and g + 4 */
                                const float *from = sm.score[g][16 * rt + c];
                                floatx4 p = *reinterpret_cast<const floatx4 *>(from);
                                float q = from[4];
                                if constexpr (AW == 8) p += *reinterpret_cast<const floatx4 *>(from + 4 * 16 * RT * 8), q += from[4 * 16 * RT * 8 + 4];
#pragma unroll
                                for (int h = 0; h < H; h++) d[rt][h] = swap32(swap16(p[h], OpSum()), OpSum());
                                d[rt][4] = swap32(swap16(q, OpSum()), OpSum());
                            }
                        }
                    };
                    request(layer);
                    if (!sh.all_here(wave)) return;
                    park_rows();
                    __syncthreads();
                    if (sharing) {
                        fold();
                        if (!plain) operand(Steps(), in, step0, tag - 1u, av);
                    }
                    float d[RT][5], rms[RT];
                    scores(d);
                    floatx4 out[RT][H];
                    /* the projected value of head h, this wave's columns */
                    auto value = [&](int rt, int h) __attribute__((always_inline)) {
                        constexpr int QPH = 4 * HD / E; /* quarters of a head */
                        floatx4 z = quarter_at(rt, h * QPH);
#pragma unroll
                        for (int q = 1; q < QPH; q++) z += quarter_at(rt, h * QPH + q);
                        return z;
                    };
#pragma unroll
                    for (int rt = 0; rt < RT; rt++) {
                        rms[rt] = ap->xscale / sqrtf(d[rt][4] * (1.0f / (float)E) + 1e-6f); /* reductions_cpu.c:345-346 */
#pragma unroll
                        for (int h = 0; h < H; h++) { /* kv_cache.c:303-324: one key has all the weight, or none if its score is not finite */
                            const floatx4 z = value(rt, h);
#pragma unroll
                            for (int i = 0; i < 4; i++) out[rt][h][i] = isfinite(d[rt][h] * rms[rt]) ? z[i] : 0.f;
                        }
                    }
                    if (sharing) {
#pragma unroll
                        for (int rt = 0; rt < RT; rt++) {
#pragma unroll
                            for (int d = H / 2; d > 0; d /= 2) /* the heads' sums pairwise, then to the row */
#pragma unroll
                                for (int h = 0; h < d; h++) out[rt][h] += out[rt][h + d];
#pragma unroll
                            for (int i = 0; i < 4; i++) av[rt][i] += out[rt][0][i];
                            /* the residual of the output projection: each sixteen columns by one of the workgroups */
                            if (t == wave && 16u * rt + c < rows) {
#pragma unroll
                                for (int i = 0; i < 4; i++) word_store(words + At::mid + ((step0 + i) * RT + rt) * 64u + lane, av[rt][i], tag);
                            }
                        }
                    }
                }
            }
            if (!sh.all_here(wave)) return;
            floatx4 acc[RT][1];
            if (sharing) {
                if (!(S::FOLDED && crossed) && (!plain || from_mid)) operand(Steps(), from_mid ? At::mid : in, step0, from_mid ? tag : tag - 1u, av);
                product(av, b, acc);
#pragma unroll
                for (int rt = 0; rt < RT; rt++) {
                    ss[rt] = 0.f;
#pragma unroll
                    for (int i = 0; i < KB; i++) ss[rt] += av[rt][i] * av[rt][i];
                }
                leave(One(), acc, ss);
            }
            __syncthreads();
            if (f_on) {
                float v = total(Sharing(), f_rt, 0) * row_scale(f_row);
                if (part_of < 2u) { /* reductions_cpu.c:219-226; the pair's other element is four lanes away */
                    const float other = dpp_mov<0x1B>(dpp_mov<DPP_HALF_MIRROR>(v));
                    const float2 y = rope_rotate2(dd & 1u ? make_float2(other, v) : make_float2(v, other), cs, sn);
                    v = dd & 1u ? y.y : y.x;
                }
                if (f_row < rows) {
                    word_store(words + to, v, tag);
                    if (part_of != 0u) *cell = v;
                }
            }
            buf ^= 1u;
            if constexpr (S::MERGED) break; /* one tile a worker: no loop to carry values around */
        }

        early_keys();
        ap = hidden_args(args);
        if (sh.has(STAGE_ATTN)) { /* ---- self-attention ---- */
            if (!sh.all_here(wave)) return;
            float *const tile = sm.keys[wave];
            const uint32_t n = ap->n;
            for (uint32_t u = unit0; u < units; u += WORKERS) {
                ap = hidden_args(args);
                fresh_lane();
                const uint32_t splits = ap->splits;
                const Unit un = unit_of(ap, u);
                const uint32_t len = un.len, nk = len + n, head = un.head, sq = un.sq;
                const uint32_t prow = lane / LPR, pf = lane % LPR;
                const bool windowed = ap->window > 0u && !ap->block_kind;
                const bool fresh_here = un.split == splits - 1u && wave == WAVES - 1u; /* takes the new rows too */
                for (uint32_t qt = 0; qt * 16u < n; qt++) {
                    if (u != unit0 || qt != 0u) request_keys(ap, layer, un, un.t_lo + wave);
                    const bool qpad = 16u * qt + c >= n;
                    const uint32_t qrow = sq * n + min(16u * qt + c, n - 1u); /* row of the group */
                    uint32_t vis_lo = 0, vis_hi = nk;
                    if (!ap->block_kind) {
                        const uint32_t qpos = len + 16u * qt + c;
                        vis_hi = min(nk, qpos + 1u);
                        if (windowed && qpos + 1u > ap->window) vis_lo = qpos + 1u - ap->window;
                    }
                    if (qpad) vis_hi = 0;
                    float mx = neg_inf(), lsum = 0.f, qf[QD];
                    floatx4 oacc[DT];
#pragma unroll
                    for (int dd = 0; dd < DT; dd++) oacc[dd] = floatx4{0.f, 0.f, 0.f, 0.f};
                    /* one tile of keys j0 ..., exact online softmax: scores in lane (g, c) register r = key j0 + 4g + r of
                     * query c, then O^T += V^T P^T */
                    auto tile_step = [&](const float (&kf)[QD], const float (&vf)[DT][4], uint32_t j0, uint32_t j_end)
                                         __attribute__((always_inline)) {
                        floatx4 s0 = floatx4{0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
                        for (int s = 0; s < QD; s += 2) {
                            s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[s], qf[s], s0, 0, 0, 0);
                            s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[s + 1], qf[s + 1], s1, 0, 0, 0);
                        }
                        const uint32_t hi = min(vis_hi, j_end);
                        const uint32_t span = hi > vis_lo ? hi - vis_lo : 0u, rel = j0 + 4u * g - vis_lo;
                        float x[4], mt = mx;
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const float t = (s0[r] + s1[r]) * ap->scale;
                            x[r] = ((rel + r < span) & isfinite(t)) ? t : neg_inf();
                            mt = fmaxf(mt, x[r]);
                        }
                        mt = swap32(swap16(mt, OpMax()), OpMax());
                        const float ms = mt == neg_inf() ? 0.f : mt;
                        const float alpha = fast_exp2(mx - ms);
                        mx = mt;
                        float ps = 0.f;
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            x[r] = fast_exp2(x[r] - ms);
                            ps += x[r];
                        }
                        lsum = lsum * alpha + ps;
#pragma unroll
                        for (int dd = 0; dd < DT; dd++) {
#pragma unroll
                            for (int r = 0; r < 4; r++) oacc[dd][r] *= alpha;
                        }
#pragma unroll
                        for (int r = 0; r < 4; r++)
#pragma unroll
                            for (int dd = 0; dd < DT; dd++)
                                oacc[dd] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[dd][r], x[r], oacc[dd], 0, 0, 0);
                    };
                    const uint64_t *const q_words = word_of(words + At::q + head * (HD * 16u), (qrow >> 4) * (H * HD * 16u) + g * 16u + (qrow & 15u));
                    /* the new rows of key tile kt, with the query if that is not there yet: one trip for both */
                    auto fresh_tile = [&](uint32_t kt, bool with_q) __attribute__((always_inline)) {
                        const uint32_t krow = sq * n + min(16u * kt + c, n - 1u);
                        /* this lane's key row as a K fragment, its part of four value rows */
                        float kf[QD], vf[DT][4];
                        const uint64_t *of_head = words + At::k + head * (HD * 16u), *kp = word_of(of_head, (krow >> 4) * (H * HD * 16u) + g * 16u + (krow & 15u));
                        const uint64_t *vp[4];
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const uint32_t vrow = sq * n + min(16u * kt + 4u * g + (uint32_t)r, n - 1u);
                            vp[r] = word_of(of_head + (At::v - At::k), (vrow >> 4) * (H * HD * 16u) + (vrow & 15u) * HD + DT * c);
                        }
                        if constexpr (HD == 32) {
                            float kv[2 * QD + DT * 4];
                            await_at<2 * QD + DT * 4>(wt, [&](int i) {
                                return i < QD ? q_words + i * 64 : i < 2 * QD ? kp + (i - QD) * 64 : vp[((i - 2 * QD) / DT) & 3] + (i - 2 * QD) % DT;
                            }, tag, kv, __LINE__);
                            if (with_q) {
#pragma unroll
                                for (int s = 0; s < QD; s++) qf[s] = kv[s];
                            }
#pragma unroll
                            for (int s = 0; s < QD; s++) kf[s] = kv[QD + s];
#pragma unroll
                            for (int i = 0; i < DT * 4; i++) vf[i % DT][i / DT] = kv[2 * QD + i];
                        } else { /* the registers do not hold all at once: 150 would be spilled */
                            float v4[DT * 4];
                            if (with_q) await_at<QD>(wt, [&](int i) { return q_words + i * 64; }, tag, qf, __LINE__);
                            await_at<QD>(wt, [&](int i) { return kp + i * 64; }, tag, kf, __LINE__);
                            await_at<DT * 4>(wt, [&](int i) { return vp[(i / DT) & 3] + i % DT; }, tag, v4, __LINE__);
#pragma unroll
                            for (int i = 0; i < DT * 4; i++) vf[i % DT][i / DT] = v4[i];
                        }
                        tile_step(kf, vf, len + 16u * kt, nk);
                    };
                    /* before the cached rows become fragments: the registers do not hold both */
                    if (fresh_here) fresh_tile(0u, true);
                    bool have_q = fresh_here;
                    for (uint32_t tb = un.t_lo + wave; tb < un.t_hi; tb += WAVES * T) {
                        float kf[T][QD], vf[T][DT][4];
#pragma unroll
                        for (int u2 = 0; u2 < T; u2++) { /* rows -> fragments, through the wave's own LDS tile */
                            if (tb + WAVES * u2 >= un.t_hi) continue;
#pragma unroll
                            for (int v = 0; v < NV; v++)
                                *reinterpret_cast<floatx4 *>(tile + (prow + (uint32_t)(RPI * v)) * ROW + 4u * pf) = kg[u2][v];
#pragma unroll
                            for (int s = 0; s < QD; s += 4) {
                                const float4 t = *reinterpret_cast<const float4 *>(tile + c * ROW + g * QD + s);
                                kf[u2][s + 0] = t.x, kf[u2][s + 1] = t.y, kf[u2][s + 2] = t.z, kf[u2][s + 3] = t.w;
                            }
#pragma unroll
                            for (int v = 0; v < NV; v++)
                                *reinterpret_cast<floatx4 *>(tile + (prow + (uint32_t)(RPI * v)) * ROW + 4u * pf) = vg[u2][v];
#pragma unroll
                            for (int r = 0; r < 4; r++) {
                                const float *vrow = tile + (4u * g + r) * ROW + DT * c;
#pragma unroll
                                for (int dd = 0; dd < DT; dd++) vf[u2][dd][r] = vrow[dd];
                            }
                        }
                        if (tb + WAVES * T < un.t_hi) request_keys(ap, layer, un, tb + WAVES * T);
                        if (!have_q) {
                            await_at<QD>(wt, [&](int i) { return q_words + i * 64; }, tag, qf, __LINE__);
                            have_q = true;
                        }
#pragma unroll
                        for (int u2 = 0; u2 < T; u2++)
                            if (tb + WAVES * u2 < un.t_hi) tile_step(kf[u2], vf[u2], (tb + WAVES * u2) * 16u, len);
                    }
                    if (RT == 2 && fresh_here)
                        for (uint32_t kt = 1; kt * 16u < n; kt++) fresh_tile(kt, false);
                    lsum = swap32(swap16(lsum, OpSum()), OpSum());
                    if (wt.expired) lsum = not_there(); /* scores that are not finite would just weigh nothing */
                    if (g == 0) sm.most[c][wave] = mx, sm.sum[c][wave] = lsum;
                    /* lane (g, c) holds columns DT (4g + r) + dd of query row c */
#pragma unroll
                    for (int r = 0; r < 4; r++)
#pragma unroll
                        for (int dd = 0; dd < DT; dd++) tile[c * ROW + DT * (4u * g + r) + dd] = oacc[dd][r];
                    __syncthreads();
                    /* a thread per (row, column): the waves' partials, scaled to the common maximum */
                    const uint32_t live = min(16u, n - 16u * qt);
                    for (uint32_t cell = threadIdx.x; cell < live * HD; cell += 64u * WAVES) {
                        const uint32_t mr = cell / HD, mc = cell % HD;
                        float wm[WAVES], ws[WAVES], o[WAVES];
#pragma unroll
                        for (uint32_t v = 0; v < WAVES; v += 4u) {
                            const float4 x = *reinterpret_cast<const float4 *>(&sm.most[mr][v]), y = *reinterpret_cast<const float4 *>(&sm.sum[mr][v]);
                            wm[v] = x.x, wm[v + 1] = x.y, wm[v + 2] = x.z, wm[v + 3] = x.w;
                            ws[v] = y.x, ws[v + 1] = y.y, ws[v + 2] = y.z, ws[v + 3] = y.w;
                        }
#pragma unroll
                        for (uint32_t v = 0; v < WAVES; v++) o[v] = sm.keys[v][mr * ROW + mc];
                        float M = wm[0];
#pragma unroll
                        for (uint32_t v = 1; v < WAVES; v++) M = fmaxf(M, wm[v]);
                        const float Ms = M == neg_inf() ? 0.f : M;
                        float Lt = 0.f, sum = 0.f;
#pragma unroll
                        for (uint32_t v = 0; v < WAVES; v++) {
                            const float f = fast_exp2(wm[v] - Ms);
                            Lt += ws[v] * f, sum += o[v] * f;
                        }
                        const uint32_t R = sq * n + 16u * qt + mr, col = head * HD + mc;
                        if (splits > 1u) {
                            word_store(words + At::comb + un.split * At::M + operand_at<RT>(R, col), sum, tag);
                            if (mc < 2u) word_store(words + At::stat + (un.split * H + head) * (32u * RT) + R * 2u + mc, mc == 0u ? M : Lt, tag);
                        } else {
                            word_store(words + At::comb + operand_at<RT>(R, col), Lt == 0.f ? 0.f : sum / Lt, tag);
                        }
                    }
                    __syncthreads(); /* the tiles may be written again */
                }
            }
        }

        ap = hidden_args(args);
        const bool res_plain = plain && !crossed; /* the residual of the output projection */
        const uint32_t res = crossed ? At::mid : in, res_tag = crossed ? tag : tag - 1u;
        if constexpr (!S::MERGED) {
            if (sh.has(STAGE_PROJ) && first(FIRST_PROJ) < (uint32_t)E / 16u &&
                !square(ap, ap->layer[layer].proj, true, tag, res_plain, res, res_tag, At::resid, first(FIRST_PROJ)))
                return;
        }

        ap = hidden_args(args);
        fresh_lane();
        const uint32_t hidden = ap->hidden, t_first = first(FIRST_UPGATE);
        const bool gated_here = sh.has(STAGE_UPGATE) && t_first < hidden / 16u;
        const uint32_t steps = hidden / 32u; /* of a wave in the down projection */
        const bool down_here = sh.has(STAGE_DOWN) && first(FIRST_DOWN) < (uint32_t)E / 16u;
        constexpr int CH = RT == 1 ? 16 : 8; /* its steps in flight together */
        float bd[CH];
        const LaneView wd(ap->layer[layer].down + first(FIRST_DOWN) * 16u, 4u * g * E + c);
        if (down_here) { /* on their way while this workgroup is busy with the stage before */
#pragma unroll
            for (int i = 0; i < CH; i++) bd[i] = (uint32_t)i < steps ? wd[term_of(steps * wave + i) * E] : 0.f;
        }
        if (gated_here) { /* ---- output projection where merged; up, gate, activation ---- */
            float rv[RT][KB]; /* the rows behind the attention, this wave's columns, as the left operand */
            float ss[RT];
            bool have_rows = false;
            for (uint32_t t = t_first; t < hidden / 16u; t += WORKERS) {
                fresh_lane();
                float b[2][KB];
                const LaneView up(ap->layer[layer].up + t * 16u, 4u * g * hidden + c), gate(ap->layer[layer].gate + t * 16u, 4u * g * hidden + c);
                const LaneView nw(ap->layer[layer].norm2, 4u * g);
#pragma unroll
                for (int i = 0; i < KB; i++) {
                    const uint32_t k = term_of(step0 + i);
                    const float n1 = nw[k];
                    b[0][i] = up[k * hidden] * n1, b[1][i] = gate[k * hidden] * n1;
                }
                if (!have_rows) {
                    have_rows = true;
                    if (!sh.all_here(wave)) return;
                    if constexpr (S::MERGED) {
                        /* output projection, by quarters of the terms */
                        if (sharing) {
                            const uint32_t quarter = wave / S::CG & 3u;
                            floatx4 wo[S::QS];
                            const LaneView w(ap->layer[layer].proj + quarter * (E / 4u) * E + 64u * (wave % S::CG), 4u * g * E + 4u * c);
#pragma unroll
                            for (int i = 0; i < S::QS; i++) wo[i] = w.four(term_of(i) * E);
#pragma unroll
                            for (int rt = 0; rt < RT; rt++) {
                                float x[S::QS], none[1];
                                using Quarter = std::integral_constant<int, S::QS>;
                                if (res_plain) {
                                    const float *src = plain_row(ap, min(16u * rt + c, rows - 1u)) + 4u * step0 + 4u * g;
#pragma unroll
                                    for (int i = 0; i < 4; i++) rv[rt][i] = src[i];
                                    attended(Quarter(), std::integral_constant<int, 0>(), quarter * S::QS, ap->splits > 1u, tag, rt, [&](int) { return (const uint64_t *)words; }, tag, x, none);
                                } else {
                                    const uint64_t *rp = word_of(words + res + step0 * (RT * 64u), polled(rt));
                                    attended(Quarter(), Steps(), quarter * S::QS, ap->splits > 1u, tag, rt, [&](int i) { return rp + i * (RT * 64); }, res_tag, x, rv[rt]);
                                }
                                by_quarter(rt, x, wo);
                            }
                        }
                        __syncthreads();
                        if (sharing) {
#pragma unroll
                            for (int rt = 0; rt < RT; rt++) {
                                const floatx4 p = (quarter_at(rt, 0) + quarter_at(rt, 1)) + (quarter_at(rt, 2) + quarter_at(rt, 3));
#pragma unroll
                                for (int i = 0; i < 4; i++) rv[rt][i] += p[i];
                                /* the residual of the down projection: each sixteen columns by one of the workgroups */
                                if (t == wave % (hidden / 16u) && 16u * rt + c < rows) {
#pragma unroll
                                    for (int i = 0; i < 4; i++) word_store(words + At::resid + ((step0 + i) * RT + rt) * 64u + lane, rv[rt][i], tag);
                                }
                            }
                        }
                    } else {
                        operand(Steps(), At::resid, step0, tag, rv);
                    }
#pragma unroll
                    for (int rt = 0; rt < RT; rt++) {
                        ss[rt] = 0.f;
#pragma unroll
                        for (int i = 0; i < KB; i++) ss[rt] += rv[rt][i] * rv[rt][i];
                    }
                }
                if (sharing) {
                    floatx4 acc[RT][2];
#pragma unroll
                    for (int rt = 0; rt < RT; rt++) {
                        floatx4 odd[2];
#pragma unroll
                        for (int j = 0; j < 2; j++) acc[rt][j] = odd[j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int i = 0; i < KB; i += 2)
#pragma unroll
                            for (int j = 0; j < 2; j++) {
                                acc[rt][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(rv[rt][i], b[j][i], acc[rt][j], 0, 0, 0);
                                odd[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(rv[rt][i + 1], b[j][i + 1], odd[j], 0, 0, 0);
                            }
#pragma unroll
                        for (int j = 0; j < 2; j++) acc[rt][j] += odd[j];
                    }
                    leave(Two(), acc, ss);
                }
                __syncthreads();
                if (f_on && f_row < rows) {
                    const float scale = row_scale(f_row), v = total(Sharing(), f_rt, 0) * scale, gt = total(Sharing(), f_rt, 1) * scale;
                    word_store(words + At::act + operand_at<RT>(f_row, t * 16u + f_col), gt / (1.0f + expf(-gt)) * v, tag);
                }
                buf ^= 1u;
            }
        }

        ap = hidden_args(args);
        if (down_here) { /* ---- down projection + residual ---- */
            if (!sh.all_here(wave)) return;
            fresh_lane();
            const uint32_t oc = first(FIRST_DOWN) * 16u + f_col;
            const uint64_t *const rp = word_of(words + At::resid, operand_at<RT>(f_safe, oc));
            float r1 = 0.f;
            floatx4 acc[RT][2];
#pragma unroll
            for (int rt = 0; rt < RT; rt++) acc[rt][0] = acc[rt][1] = floatx4{0.f, 0.f, 0.f, 0.f};
            for (uint32_t k0 = 0; k0 < steps; k0 += CH) {
                if (k0) {
#pragma unroll
                    for (int i = 0; i < CH; i++) bd[i] = k0 + i < steps ? wd[term_of(steps * wave + k0 + i) * E] : 0.f;
                }
#pragma unroll
                for (int rt = 0; rt < RT; rt++) {
                    float av[CH + 1]; /* past the wave's last step: repeats, against weights of zero; and the residual */
                    const uint64_t *p = word_of(words + At::act + (steps * wave + k0) * (RT * 64u), polled(rt));
                    await_at<CH + 1>(wt, [&](int i) { return i < CH ? p + min((uint32_t)i, steps - 1u - k0) * (RT * 64u) : rp; }, tag, av, __LINE__);
#pragma unroll
                    for (int i = 0; i < CH; i++) acc[rt][i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i], bd[i], acc[rt][i & 1], 0, 0, 0);
                    r1 = av[CH];
                }
            }
            floatx4 sum[RT][1];
#pragma unroll
            for (int rt = 0; rt < RT; rt++) sum[rt][0] = acc[rt][0] + acc[rt][1];
            leave(One(), sum, nullptr);
            __syncthreads();
            if (f_on && f_row < rows) word_store(words + At::output(layer) + operand_at<RT>(f_row, oc), r1 + total(All(), f_rt, 0), tag);
            buf ^= 1u;
        }
    }

    if (!sh.has(STAGE_LM)) return;
    ArgsPtr ap = hidden_args(args);
    const uint32_t V = ap->V;
    for (uint32_t t = first(FIRST_LM); t < V / 16u; t += WORKERS) { /* ---- LM head ---- */
        fresh_lane();
        float b[KB], av[RT][KB];
        const LaneView w(ap->lm + t * 16u, 4u * g * V + c);
#pragma unroll
        for (int i = 0; i < KB; i++) b[i] = w[(size_t)term_of(step0 + i) * V];
        if (!sh.all_here(wave)) return;
        if (sharing) {
            operand(Steps(), At::output(L - 1u), step0, ap->tag + L - 1u, av);
            floatx4 acc[RT][1];
            product(av, b, acc);
            leave(One(), acc, nullptr);
        }
        __syncthreads();
        if (f_on && f_row < rows) ap->logits[(size_t)(gv.row0 + f_row) * V + t * 16u + f_col] = total(Sharing(), f_rt, 0);
        buf ^= 1u;
    }
    (void)sh.all_here(wave); /* a workgroup without any tile may have to stand in for others */
}

template <typename S>
__global__ __launch_bounds__(64 * WAVES, 2) void kv_step_resident_kernel(ResidentArgs a) {
    __shared__ __attribute__((aligned(16))) ResidentLds<S> sm;
    GroupView gv;
    const uint32_t group = blockIdx.x % GROUPS, index = blockIdx.x / GROUPS;
    gv.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    gv.seq0 = group * a.per_group;
    if (gv.seq0 >= a.batch) return;
    if (threadIdx.x == 0u) sign_in(a.rolls + group * WORKERS, index, a.tag);
    gv.ns = min(a.per_group, a.batch - gv.seq0);
    gv.rows = gv.ns * a.n, gv.row0 = gv.seq0 * a.n;
    gv.words = a.words + (size_t)group * a.group_words;
    const ArgsPtr ap = (ArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
    if (threadIdx.x < MAX_GROUP_ROWS) {
        sm.len[threadIdx.x] = a.len[gv.seq0 + min(threadIdx.x, gv.ns - 1u)];
        sm.latent[threadIdx.x] = a.latent[gv.row0 + min(threadIdx.x, gv.rows - 1u)];
    }
    __syncthreads();
    gv.worker = index;
    WholeStep whole{ap, group, index, &sm.standing, false};
    run_worker<S>(ap, gv, whole, sm);
    const uint32_t rank = __builtin_amdgcn_readfirstlane(sm.standing.rank), members = __builtin_amdgcn_readfirstlane(sm.standing.members);
    if (members == WORKERS) return;

    if (members == 0u) return;
    for (uint32_t stage = 0; stage <= a.L * STAGES; stage++) {
        OneStage one{stage / STAGES, stage < a.L * STAGES ? stage % STAGES : (uint32_t)STAGE_LM};
        for (gv.worker = rank; gv.worker < WORKERS; gv.worker += members) {
            run_worker<S>(ap, gv, one, sm);
            __syncthreads(); /* the shared areas may be written again */
        }
    }
}

__global__ void clear_hand_over_kernel(uint64_t *w, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256u + threadIdx.x;
    if (i < n) w[i] = 0u;
}

typedef void (*ResidentKernel)(ResidentArgs);
template <bool FOLD>
ResidentKernel kernel_of(size_t E, size_t hd, uint32_t row_tiles) {
    if (E == 64 && hd == 32)
        return row_tiles == 2u ? kv_step_resident_kernel<ResidentShape<64, 32, 2, FOLD>> : kv_step_resident_kernel<ResidentShape<64, 32, 1, FOLD>>;
    if (E == 64) return kv_step_resident_kernel<ResidentShape<64, 64, 1, FOLD>>;
    if (E == 128) return hd == 32 ? kv_step_resident_kernel<ResidentShape<128, 32, 1, FOLD>> : kv_step_resident_kernel<ResidentShape<128, 64, 1, FOLD>>;
    return hd == 32 ? kv_step_resident_kernel<ResidentShape<256, 32, 1, false>> : kv_step_resident_kernel<ResidentShape<256, 64, 1, false>>;
}
constexpr uint32_t group_words(size_t E, uint32_t row_tiles, uint32_t hidden) {
    return (E == 64 ? row_tiles == 2u ? Regions<64, 2>::total(hidden) : Regions<64, 1>::total(hidden)
                    : E == 128 ? Regions<128, 1>::total(hidden) : Regions<256, 1>::total(hidden)) + 63u & ~63u;
}

/* Hand-over words and roll calls of one (thread, stream), like the library's other scratch: launches on one stream follow
 * each other, launches on two streams never share them.  Tags of successive launches differ, so the words are cleared
 * only when they are new or the tags have run through.  Sized for every shape the kernel takes (3.7 MB). */
struct HandOver {
    static constexpr size_t WORDS = GROUPS * (size_t)std::max(group_words(64, 2, MAX_HIDDEN), group_words(256, 1, MAX_HIDDEN));
    static constexpr size_t COUNT = WORDS + GROUPS * WORKERS; /* and the roll calls */
    uint64_t *words = nullptr;
    uint32_t next_tag = 0;
};
struct HandOvers {
    std::map<std::pair<int, hipStream_t>, HandOver> by_stream;
    ~HandOvers() { /* a thread that ends gives them back; when the process does, the runtime may have ended first */
        if (gettid() != getpid())
            for (auto &entry : by_stream) (void)hipFree(entry.second.words); /* waits for what still uses them */
    }
};

/* pinned, written by a kernel whose waits ran out */
uint32_t *timeout_word() {
    static uint32_t *const word = [] {
        uint32_t *w = nullptr;
        HIP_CHECK(hipHostMalloc((void **)&w, 64, hipHostMallocPortable));
        *w = 0u;
        return w;
    }();
    return word;
}
std::atomic<bool> g_launched{false};

/* BLT_HIP_STEP_TEST=team|giveup|wrap (test hook): who looks signs out whoever is not in yet / no wait lasts
 * / the tags run through at the third launch of a stream */
enum TestPin { TEST_NONE, TEST_TEAM, TEST_GIVEUP, TEST_WRAP };
TestPin test_pin() {
    static const TestPin pin = [] {
        const char *e = getenv("BLT_HIP_STEP_TEST");
        if (e && std::strcmp(e, "team") == 0) return TEST_TEAM;
        if (e && std::strcmp(e, "giveup") == 0) return TEST_GIVEUP;
        if (e && std::strcmp(e, "wrap") == 0) return TEST_WRAP;
        return TEST_NONE;
    }();
    return pin;
}

/* Do `blocks` workgroups of the kernel fit the compute units this stream may use, all at once?  The launch would be right
 * otherwise too (see the roll call), but the launches would be faster. */
bool can_be_resident(ResidentKernel kernel, uint32_t blocks, int dev, hipStream_t s) {
    struct Fit {
        uint32_t per_unit = 0, units = 0;
    };
    static thread_local std::map<std::pair<ResidentKernel, int>, Fit> fits;
    Fit &fit = fits[{kernel, dev}];
    if (fit.units == 0u) {
        int per_unit = 0, units = 0;
        HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_unit, reinterpret_cast<const void *>(kernel), 64 * WAVES, 0));
        HIP_CHECK(hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, dev));
        fit.per_unit = (uint32_t)per_unit, fit.units = (uint32_t)units;
    }
    uint32_t mask[32], open = 0;
    const uint32_t mask_words = (fit.units + 31u) / 32u;
    if (mask_words > 32u) return false;
    if (hipExtStreamGetCUMask(s, mask_words, mask) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    for (uint32_t i = 0; i < mask_words; i++) open += (uint32_t)__builtin_popcount(mask[i]);
    return (uint64_t)fit.per_unit * std::min(open, fit.units) >= blocks;
}

} // namespace

void kv_step_resident_check() {
    if (!g_launched.load(std::memory_order_relaxed)) return;
    const uint32_t word = __atomic_load_n(timeout_word(), __ATOMIC_RELAXED);
    if (word != 0u)
        BLT_FATAL("blt_kv_decode_step: workgroup %u of the resident step gave up waiting (step_resident.hip:%u)", word >> 16, word & 0xFFFFu);
}

bool kv_step_resident(const StepResident &st) {
    const blt_kv_cache *cache = st.cache;
    const blt_local_decoder *dec = cache->decoder;
    const blt_local_decoder_config *cfg = &dec->config;
    const size_t E = cache->embed_dim, L = cfg->num_layers, H = cfg->num_heads, V = cfg->vocab_size, hd = E / H;
    if ((hd != 32 && hd != 64) || cfg->cross_attn_heads != H || (E != 64 && E != 128 && E != 256) || L < 1 || L > MAX_LAYERS ||
        V % 16 != 0 || V == 0 || V > (size_t)1 << 26 || blt_stream_capturing())
        return false;
    const size_t per_group = (st.batch + GROUPS - 1) / GROUPS, group_rows = per_group * st.n;
    if (group_rows > MAX_GROUP_ROWS || st.batch > MAX_ROWS) return false;
    /* Where the launches win, measured over E, heads, layers, rows and lengths (us, launches -> resident, two layers).  Up to 16
     * rows a group and heads of 32: everywhere (one row of 356 keys, E = 64 / 128 / 256: 47 -> 25, 54 -> 34, 76 -> 48; 16 rows of 800 keys 61 -> 34, 69 -> 44,
     * 93 -> 73; 64 sequences 52 -> 31, 62 -> 42, 95 -> 74).
     * 17 to 32 rows: narrow models with heads of 32 only (E = 64: 75 -> 45 at 30 draft rows); others would need the
     * registers of two row tiles.  Heads of 64: one sequence (E = 128: 68 -> 39 at two rows, 78 -> 46 at 16 draft rows; E = 256: 91 -> 55, 102 ->
     * 85) and single rows of up to four sequences a group (E = 256, 24 sequences: 101 -> 63).  No crossover lies there: the step
     * would gain beyond it too (E = 128, 16 sequences of four rows: 74 -> 44; E = 256, 64 single rows 96 -> 77) up to 128 single
     * rows (106 -> 112); these shapes are not taken because no test has run them in one launch. */
    if (group_rows > 16 && (E > 64 || hd == 64)) return false;
    if (hd == 64 && st.batch > 1 && (st.n > 1 || per_group > 4)) return false;
    if (st.row_index != nullptr && st.batch != 1) return false;
    const size_t hidden = dec->layers[0].ffn_up_w.shape[1];
    if (hidden % 32 != 0 || hidden == 0 || hidden > MAX_HIDDEN) return false;
    for (size_t l = 0; l < L; l++)
        if (dec->layers[l].ffn_up_w.shape[1] != hidden) return false;
    if (cache->max_seq_len > 0xFFFFFFFFu || cache->max_subtokens > 0xFFFFFFFFu || (uint64_t)cache->max_seq_len * E * 4u > 0xFFFFFFFFu)
        return false;

    ResidentArgs a;
    __builtin_memset(&a, 0, sizeof(a));
    auto f32 = [](const blt_tensor &t) { return (const float *)t.data; };
    const bool folds = E <= 128 && cache->k == 1;
    uintptr_t bits = 0;
    for (size_t l = 0; l < L; l++) {
        const blt_local_layer_storage *s = &dec->layers[l];
        ResidentLayer &r = a.layer[l];
        if (st.crosses[l]) {
            r.xnorm = f32(s->cross_norm_weight), r.xq = f32(s->cross_weight_q), r.xproj = f32(s->cross_weight_proj);
            r.xk = f32(cache->cross_k[l]), r.xv = f32(cache->cross_v[l]);
        }
        r.norm1 = f32(s->norm1_weight), r.qkv = f32(s->attn_qkv_w), r.proj = f32(s->attn_proj_w);
        r.norm2 = f32(s->norm2_weight), r.up = f32(s->ffn_up_w), r.gate = f32(s->ffn_gate_w), r.down = f32(s->ffn_down_w);
        r.ck = (float *)cache->self_k[l].data, r.cv = (float *)cache->self_v[l].data;
        const auto also = [&bits](const float *p) { bits |= reinterpret_cast<uintptr_t>(p); };
        also(r.ck), also(r.cv);
        if (E <= 128) also(r.proj); /* by the merged stage */
        if (folds) also(r.xk), also(r.xv), also(r.xq), also(r.xnorm), also(r.xproj);
    }
    if (bits & 15u) return false; /* read sixteen bytes at a time; the other weights by the word */
    a.d0 = st.d0_rows, a.lm = f32(dec->lm_head_weight), a.logits = st.logits;
    a.cos = f32(dec->rope_cos_cache), a.sin = f32(dec->rope_sin_cache);
    a.max_seq = cache->max_seq_len, a.slab_x = cache->max_subtokens;
    a.L = (uint32_t)L, a.E = (uint32_t)E, a.H = (uint32_t)H, a.hidden = (uint32_t)hidden, a.V = (uint32_t)V;
    a.batch = (uint32_t)st.batch, a.n = (uint32_t)st.n, a.per_group = (uint32_t)per_group;
    a.subtokens = (uint32_t)cache->k, a.window = (uint32_t)st.window, a.block_kind = st.block_kind ? 1u : 0u;
    a.xscale = 1.0f / sqrtf((float)hd);
    a.scale = a.xscale * LOG2E;
    size_t longest = 0;
    for (size_t b = 0; b < st.batch; b++) {
        a.len[b] = (uint32_t)st.base[b];
        longest = std::max(longest, st.base[b]);
    }
    if (longest + st.n > cfg->max_seq_len || longest + st.n > cache->max_seq_len) return false; /* the per-launch form has the message */
    for (size_t r = 0; r < st.batch * st.n; r++) {
        if (st.latent[r] > 0xFFFFu) return false;
        a.latent[r] = (uint16_t)st.latent[r];
    }
    if (st.row_index != nullptr || st.positions != nullptr) {
        a.indexed = 1u;
        for (size_t r = 0; r < st.n; r++) {
            const size_t pos = st.positions ? st.positions[r] : st.base[0] + r, row = st.row_index ? st.row_index[r] : r;
            if (pos > 0xFFFFu || row > 0xFFFFu) return false;
            a.position[r] = (uint16_t)pos, a.row_index[r] = (uint16_t)row;
        }
    }
    /* Workgroups per group: one per compute unit of a die; the widest stage (hidden / 16 tiles) fills them.
     * Keys are shared out while there are workgroups without a (sequence, head) and a share keeps every
     * wave of a workgroup a tile. */
    const uint32_t pairs = (uint32_t)(per_group * H);
    a.splits = 1u;
    if (hd % (E / 8) == 0)
        while (a.splits < MAX_SPLITS_R && pairs * a.splits * 2u <= WORKERS && longest >= 128u * a.splits) a.splits *= 2u;
    const uint32_t rt = group_rows > 16 ? 2u : 1u;
    a.group_words = group_words(E, rt, a.hidden);

    int dev = 0;
    HIP_CHECK(hipGetDevice(&dev));
    const hipStream_t s = blt_stream();
    /* recorded by the caller's own capture of the stream, a replay would find the words of the launch before it under its
     * own tag */
    if (blt_stream_captured_by_caller(s)) return false;
    const ResidentKernel kernel = folds ? kernel_of<true>(E, hd, rt) : kernel_of<false>(E, hd, rt);
    const uint32_t groups = (uint32_t)((st.batch + per_group - 1) / per_group);
    if (!can_be_resident(kernel, groups * WORKERS, dev, s)) return false;
    kv_step_resident_check();
    static thread_local HandOvers hand_overs;
    HandOver &ho = hand_overs.by_stream[{dev, s}];
    const TestPin pin = test_pin();
    if (ho.next_tag == 0u || ho.next_tag > 0xFFFFFFFFu - 2u * MAX_LAYERS) {
        const bool fresh = ho.words == nullptr;
        if (fresh) HIP_CHECK(hipMalloc((void **)&ho.words, HandOver::COUNT * sizeof(uint64_t)));
        blt_launch("kv_step_clear", clear_hand_over_kernel, dim3((unsigned)((HandOver::COUNT + 255) / 256)), dim3(256), 0, s, ho.words,
                   HandOver::COUNT);
        ho.next_tag = fresh && pin == TEST_WRAP ? 0xFFFFFFFFu - 2u * MAX_LAYERS - (uint32_t)L : 1u;
    }
    a.words = ho.words;
    a.rolls = ho.words + HandOver::WORDS;
    a.timeout = timeout_word();
    a.roll_limit = pin == TEST_TEAM ? 0u : ROLL_LIMIT;
    a.spin_limit = pin == TEST_GIVEUP ? 0u : SPIN_LIMIT;
    a.tag = ho.next_tag;
    ho.next_tag += (uint32_t)L;
    blt_launch("kv_step_resident", kernel, dim3(GROUPS * WORKERS), dim3(64 * WAVES), 0, s, a);
    g_launched.store(true, std::memory_order_relaxed);
    return true;
}
