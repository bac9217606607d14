/*
 * The whole incremental decoder step (csrc/infer/kv_cache.c:161-416) in ONE launch, for steps of
 * few rows: workgroups stay resident from the first layer to the LM head and hand the activations
 * to each other through device memory, where the launch-per-operation form runs 7 dependent
 * kernels per layer.
 *
 * What bounds such a step is neither bytes nor arithmetic (one row through two layers of 128
 * columns: 2.6 MB of weights, 1.6 MFLOP) but the chain of dependent stages, 15 of them here: as
 * launches each costs about 4.6 us (launch boundary, cold argument block, one trip to memory, one
 * drain), inside one launch about 1 us (a store, the poll that sees it, a K-split product, one
 * barrier).
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
 * A stage is a product of [rows, K] with 16-column tiles of a weight matrix, one tile (or an up / gate
 * pair, or a cross head) per workgroup, K split over its eight waves, v_mfma_f32_16x16x4_f32 on 16-row tiles,
 * partial tiles added through LDS; RMSNorm is folded in as in matmul.hip (the row statistic from the
 * same loads, the scale after the product).  The self-attention stage gives a workgroup one (sequence,
 * head, share of the keys): K and V rows are requested before the query is there, coalesced and turned into
 * fragments through the wave's LDS tile, exact online softmax per wave, waves merged through LDS, shares merged by the
 * reader.
 *
 * Who waits.  A launch is up to 512 workgroups, two per compute unit, and nothing promises that they all become
 * resident: another kernel may keep its place for as long as it likes, another process may run this very step.  So
 * nobody waits for a workgroup that has not started.  The workgroups of a group call the roll first: each has a word
 * in which it signs in, and who finds the time up before everybody has signs the others out.  If all are in, each has the
 * role its index gives it.  Else those that are in take all the work among them, stage by stage in the same order (any
 * number can: the first unfinished stage waits for nothing unfinished), and who finds itself signed out leaves.  The
 * fewer are in, the longer it is worth waiting: 20 us for the last one, 1.3 ms for the second.
 *
 * Every wait is bounded all the same (SPIN_LIMIT polls, then the wave raises a word in pinned host memory, stops
 * waiting for the rest of the launch, takes NaN for what it did not get and runs to its end; the host turns the word
 * into a fatal error at its next look).
 *
 * Measured, launches -> this kernel: one row, two layers of 128 columns, 300 keys 69 -> 38 us; 64 such rows 78 ->
 * 61 us; 16 draft rows of one sequence 80 -> 61 us.  The roll call is a quarter of a microsecond of that where the first
 * loads of a workgroup are on their way meanwhile, and 1.5 us in front of everything.  What is left is the chain: a
 * hand-over takes about 1 us from the store to the reader's first use, and a wave that shares its SIMD with three
 * others issues an instruction every nine cycles, so the 100 ... 200 instructions of a stage between its operand and
 * its result are another.  Two workgroups of eight waves on a compute unit leave a wave 128 registers, which do not hold
 * either role: about 40 are spilled at heads of 32, about 150 at heads of 64, and a reload waits for every load before it.
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
constexpr uint32_t ROLL_LIMIT = 2000; /* ticks of 10 ns */
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
    uint64_t *rolls;   /* a word per workgroup, 2 WORKERS per group */
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
 * A region that a product reads as its left operand holds element (row, k) in word
 * (k / 4 * RT + row / 16) * 64 + k % 4 * 16 + row % 16, the order of the lanes of a 16x16x4 fragment: a
 * wave's operand for four k is 64 consecutive words.  Q and K of the new rows: per (row tile, head) and
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
__device__ __forceinline__ uint32_t operand_at(uint32_t row, uint32_t k) {
    return ((k >> 2) * RT + (row >> 4)) * 64u + (k & 3u) * 16u + (row & 15u);
}

/* A wave's waiting state: once one wait has run out, none of the wave's later ones wait. */
struct Waiter {
    uint32_t *timeout;
    uint32_t limit;
    bool expired;
};
__device__ __forceinline__ float not_there() { return __builtin_nanf(""); }

/* N words per lane, the one number i at(i), until every lane that is not `pad` has them all.  A wave that
 * misses some looks again after a sleep: at all of them while they are few, else at the last one only
 * until that one is there.  Eight waves that poll twenty words each keep the compute unit's vector memory path
 * full, and it serves the oldest waves first -- a younger workgroup on the same unit that has to produce the
 * words then never gets a request in. */
template <int N, typename At>
__device__ __forceinline__ void await_at(Waiter &wt, At at, bool pad, uint32_t tag, float (&out)[N], uint32_t line) {
    uint64_t t[N];
    for (uint32_t spin = 0;; spin++) {
        uint32_t off = 0;
#pragma unroll
        for (int i = 0; i < N; i++) t[i] = word_load(at(i));
#pragma unroll
        for (int i = 0; i < N; i++) off |= (uint32_t)(t[i] >> 32) ^ tag;
        if (__all((off == 0u) | pad) || wt.expired) break;
        __builtin_amdgcn_s_setprio(0);
        if (N > 4) {
            bool missing;
            do {
                __builtin_amdgcn_s_sleep(1);
                missing = ((uint32_t)(word_load(at(N - 1)) >> 32) != tag) & !pad;
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
    for (int i = 0; i < N; i++) out[i] = __uint_as_float((uint32_t)t[i]); /* pad lanes: anything */
    out[0] = wt.expired ? not_there() : out[0]; /* one of a row's values is enough to make every sum of it NaN */
}
/* word `index` of a region: a uniform base and a 32-bit byte offset per lane, which the load takes as they are */
__device__ __forceinline__ const uint64_t *word_of(const uint64_t *base, uint32_t index) {
    return reinterpret_cast<const uint64_t *>(reinterpret_cast<const char *>(base) + index * 8u);
}
template <int N, int STRIDE>
__device__ __forceinline__ void await(Waiter &wt, const uint64_t *base, uint32_t index, bool pad, uint32_t tag, float (&out)[N],
                                      uint32_t line = __builtin_LINE()) {
    const uint64_t *p = word_of(base, index);
    await_at<N>(wt, [&](int i) { return p + i * STRIDE; }, pad, tag, out, line);
}

/* The argument block is hidden from the optimiser once per stage: it would otherwise compute the addresses of
 * all stages ahead of the layer loop and spill them. */
typedef const __attribute__((address_space(4))) ResidentArgs *ArgsPtr;
__device__ __forceinline__ ArgsPtr hidden_args(ArgsPtr args) {
    uint32_t zero;
    asm volatile("s_mov_b32 %0, 0" : "=s"(zero));
    return (ArgsPtr)((const __attribute__((address_space(4))) char *)args + zero);
}

struct GroupView {
    uint64_t *words;
    uint32_t seq0, ns, row0, rows; /* the group's sequences and rows */
    uint32_t worker, wave;         /* worker: among the workgroups of its role */
};

template <int HD, int RT>
struct ResidentShape {
    static constexpr int ROW = HD + 4;
    static constexpr int PART = WAVES * RT * 2 * 256; /* floats of one buffer of partial tiles */
    static constexpr int ATTN = WAVES * 16 * ROW + 2 * 16 * WAVES;
    static constexpr int AREA = 2 * PART > ATTN ? 2 * PART : ATTN;
};

constexpr uint32_t WORKERS = 32; /* workgroups of a group for the products, and as many for the self-attention: one of each per compute unit of a die */
/* Tile 0 of a stage goes to this worker, tile 1 to the next: consecutive stages on different workgroups, so
 * that the ones of a stage have its weights in registers and are looking for its operand when the stage before
 * finishes. */
constexpr uint32_t FIRST_XQ = 24, FIRST_XPROJ = 0, FIRST_QKV = 8, FIRST_PROJ = 0, FIRST_UPGATE = 16, FIRST_DOWN = 8, FIRST_LM = 16;

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
/* by one wave of each workgroup; lane i looks at workgroup i's word */
__device__ __forceinline__ Standing call_roll(uint64_t *roll, uint32_t index, uint32_t tag, uint32_t limit) {
    static_assert(2u * WORKERS == 64u, "a lane per workgroup");
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t in = 2ull * tag;
    const uint64_t begin = wall_clock64();
    for (;;) {
        uint64_t word = __hip_atomic_load(roll + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint64_t present = __ballot(word == in);
        if (__all(word >= in)) {
            if ((present >> index & 1ull) == 0ull) return {0u, 0u};
            return {(uint32_t)__popcll(present & ((1ull << index) - 1ull)), (uint32_t)__popcll(present)};
        }
        /* only who is in for good signs others out: somebody always is */
        if ((present >> index & 1ull) != 0ull && (wall_clock64() - begin) * __popcll(present) >= 64ull * limit && word < in)
            __hip_atomic_compare_exchange_strong(roll + lane, &word, in + 1ull, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_s_sleep(1);
    }
}

/* What a call of a role works on: one stage (STAGES of layer L: the LM head) ... */
struct OneStage {
    uint32_t layer, stage;
    __device__ __forceinline__ uint32_t begin() const { return layer; }
    __device__ __forceinline__ uint32_t end(uint32_t L) const { return min(layer + 1u, L); }
    __device__ __forceinline__ bool has(Stage st) const { return st == stage; }
    __device__ __forceinline__ bool all_here(uint32_t) { return true; }
};
/* ... or everything, if all workgroups of the group are there: a role asks before its first wait and its first store, with
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
            const Standing st = call_roll(args->rolls + group * (2u * WORKERS), index, args->tag, args->roll_limit);
            if ((threadIdx.x & 63u) == 0u) *standing = st;
        }
        __syncthreads();
        return __builtin_amdgcn_readfirstlane(standing->members) == 2u * WORKERS;
    }
};

/* The workgroups that run the products: every stage but the self-attention.  A stage of a worker: its weights,
 * the operand as soon as it is there, the product over the wave's share of K, the waves' partial tiles through
 * LDS, the results of 256 threads per row tile. */
template <int E, int HD, int RT, typename Share>
__device__ __forceinline__ void product_role(ArgsPtr args, const GroupView gv, Share sh, float *area,
                                             float (*part_ss)[16 * RT][WAVES], float (*xquery)[HD]) {
    using At = Regions<E, RT>;
    using Shape = ResidentShape<HD, RT>;
    constexpr int QD = HD / 4, DT = HD / 16, H = E / HD;
    constexpr int KB = E / 32;               /* four-row steps of K = E per wave */
    constexpr uint32_t RPW = 64 / HD;        /* rows a wave attends at a time in the cross block */
    constexpr int XKB = KB * (DT / 2);       /* steps of a wave in a cross head's projection: two of its column tiles */
    constexpr uint32_t XKS = WAVES / (DT / 2);
    const uint32_t wave = gv.wave, rows = gv.rows;
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

    /* the left operand of this wave's KBN steps from step kb_lo on */
    auto operand = [&](auto kbn, uint32_t region, uint32_t kb_lo, uint32_t tag, float (&av)[RT][decltype(kbn)::value])
                       __attribute__((always_inline)) {
        constexpr int N = decltype(kbn)::value;
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
            await<N, RT * 64>(wt, words + region + (kb_lo * RT + (uint32_t)rt) * 64u, lane, 16u * rt + c >= rows, tag, av[rt]);
    };
    /* ... of layer 0: the rows as the caller has them */
    auto operand_plain = [&](auto kbn, ArgsPtr ap, uint32_t kb_lo, float (&av)[RT][decltype(kbn)::value]) __attribute__((always_inline)) {
        constexpr int N = decltype(kbn)::value;
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            const uint32_t row = min(16u * rt + c, rows - 1u);
            const float *src = ap->d0 + (size_t)(ap->indexed ? ap->row_index[row] : gv.row0 + row) * E + 4u * kb_lo + g;
#pragma unroll
            for (int i = 0; i < N; i++) av[rt][i] = src[4 * i];
        }
    };
    auto plain_row = [&](ArgsPtr ap, uint32_t row) { return ap->d0 + (size_t)(ap->indexed ? ap->row_index[row] : gv.row0 + row) * E; };
    /* partial tiles and row statistics of all waves meet; buffers alternate, so one barrier per product is enough */
    auto meet = [&](auto nb, floatx4 (&acc)[RT][decltype(nb)::value], const float *ss) __attribute__((always_inline)) {
        constexpr int NB = decltype(nb)::value;
        float *const part = area + buf * Shape::PART;
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
#pragma unroll
            for (int j = 0; j < NB; j++)
                *reinterpret_cast<floatx4 *>(part + ((wave * RT + rt) * 2 + j) * 256 + lane * 4u) = acc[rt][j];
        if (ss != nullptr) {
#pragma unroll
            for (int rt = 0; rt < RT; rt++) {
                const float s = swap32(swap16(ss[rt], OpSum()), OpSum());
                if (g == 0) part_ss[buf][16 * rt + c][wave] = s;
            }
        }
        __syncthreads();
    };
    /* the finished element of column tile j (of KS K parts; waves of tile pair j / 2) */
    auto total = [&](auto ksn, uint32_t rt, uint32_t j) __attribute__((always_inline)) {
        constexpr uint32_t KS = decltype(ksn)::value;
        const float *p0 = area + buf * Shape::PART + (((j >> 1) * KS * RT + rt) * 2 + (j & 1u)) * 256 + (wave & 3u) * 64u + lane;
        float s0 = 0.f, s1 = 0.f;
#pragma unroll
        for (uint32_t v = 0; v < KS; v += 2) s0 += p0[v * (RT * 2 * 256)], s1 += p0[(v + 1) * (RT * 2 * 256)];
        return s0 + s1;
    };
    auto row_scale = [&](auto ksn, uint32_t row) __attribute__((always_inline)) {
        constexpr uint32_t KS = decltype(ksn)::value;
        float s = 0.f; /* where two groups of waves hold the whole row, the first is enough */
#pragma unroll
        for (uint32_t v = 0; v < KS; v += 4) {
            const float4 x = *reinterpret_cast<const float4 *>(&part_ss[buf][row][v]);
            s += (x.x + x.y) + (x.z + x.w);
        }
        return 1.0f / sqrtf(s * (1.0f / (float)E) + 1e-6f); /* reductions_cpu.c:345-346 */
    };
    using All = std::integral_constant<uint32_t, WAVES>;
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    using Steps = std::integral_constant<int, KB>;

    /* [rows, E] products with one residual row added: cross projection, output projection */
    auto square = [&](ArgsPtr ap, const float *w, uint32_t src, bool shares, uint32_t tag, bool res_plain, uint32_t res, uint32_t res_tag,
                      uint32_t to, uint32_t t) __attribute__((always_inline)) {
        fresh_lane();
        float b[KB], av[RT][KB], r1[1] = {0.f};
        const float *wp = w + (4u * KB * wave + g) * E + t * 16u + c;
#pragma unroll
        for (int i = 0; i < KB; i++) b[i] = wp[4 * i * E];
        const uint32_t oc = t * 16u + f_col;
        if (f_on && res_plain) r1[0] = plain_row(ap, f_safe)[oc];
        if (!sh.all_here(wave)) return false;
        if (shares) { /* the shares' sums, weighed with the common maximum and divided by the common sum; a wave's columns are of one head */
            const uint32_t head = 4u * KB * wave / HD;
#pragma unroll
            for (int rt = 0; rt < RT; rt++) {
                float all[2 * KB + 4];
                const uint64_t *p = word_of(words + src + (KB * wave * RT + (uint32_t)rt) * 64u, lane);
                const uint64_t *st = word_of(words + At::stat + head * (32u * RT), min(16u * rt + c, rows - 1u) * 2u);
                await_at<2 * KB + 4>(wt, [&](int i) {
                    if (i < 2 * KB) return p + (i % KB) * (RT * 64) + (i < KB ? 0u : At::M);
                    return st + ((i - 2 * KB) >> 1) * (H * 32 * RT) + (i & 1);
                }, 16u * rt + c >= rows, tag, all, __LINE__);
                const float *s0 = all, *s1 = all + KB, *st0 = all + 2 * KB, *st1 = all + 2 * KB + 2;
                const float M = fmaxf(st0[0], st1[0]), Ms = M == neg_inf() ? 0.f : M;
                const float f0 = fast_exp2(st0[0] - Ms), f1 = fast_exp2(st1[0] - Ms), Lt = st0[1] * f0 + st1[1] * f1;
#pragma unroll
                for (int i = 0; i < KB; i++) av[rt][i] = Lt == 0.f ? 0.f : (s0[i] * f0 + s1[i] * f1) / Lt;
            }
        } else {
            operand(Steps(), src, KB * wave, tag, av);
        }
        floatx4 acc[RT][1];
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            floatx4 a0 = floatx4{0.f, 0.f, 0.f, 0.f}, a1 = a0;
#pragma unroll
            for (int i = 0; i < KB; i += 2) {
                a0 = __builtin_amdgcn_mfma_f32_16x16x4f32(av[rt][i], b[i], a0, 0, 0, 0);
                a1 = __builtin_amdgcn_mfma_f32_16x16x4f32(av[rt][i + 1], b[i + 1], a1, 0, 0, 0);
            }
            acc[rt][0] = a0 + a1;
        }
        if (f_on && !res_plain) /* written before this stage's operand could be: seen at the first look */
            await<1, 1>(wt, words + res, operand_at<RT>(f_safe, oc), false, res_tag, r1);
        meet(One(), acc, nullptr);
        if (f_on && f_row < rows) word_store(words + to + operand_at<RT>(f_row, oc), r1[0] + total(All(), f_rt, 0), tag);
        buf ^= 1u;
        return true;
    };
    auto first = [&](uint32_t at) { return (gv.worker - at) & (WORKERS - 1u); };

    const uint32_t L = args->L;
    for (uint32_t layer = sh.begin(); layer < sh.end(L); layer++) {
        ArgsPtr ap = hidden_args(args);
        const uint32_t tag = ap->tag + layer;
        const bool crossed = ap->layer[layer].xq != nullptr, plain = layer == 0u;
        const uint32_t in = At::input(layer);

        if (crossed && sh.has(STAGE_XQ) && first(FIRST_XQ) < (uint32_t)H) { /* ---- query projection of one cross head, its rows' cross attention ---- */
            fresh_lane();
            const uint32_t head = first(FIRST_XQ), kpart = wave % XKS, tpart = wave / XKS;
            float b[2][XKB], av[RT][XKB], ss[RT];
            const float *w = ap->layer[layer].xq + (4u * XKB * kpart + g) * E + head * HD + 32u * tpart + c;
            const float *nw = ap->layer[layer].xnorm + 4u * XKB * kpart + g;
#pragma unroll
            for (int i = 0; i < XKB; i++) {
                const float n1 = nw[4 * i];
                b[0][i] = w[4 * i * E] * n1, b[1][i] = w[4 * i * E + 16] * n1;
            }
            /* the first sub-token of this lane's first row */
            const uint32_t xd = lane % HD;
            const float *xk = ap->layer[layer].xk, *xv = ap->layer[layer].xv;
            auto cell = [&](uint32_t row) {
                return ((size_t)(gv.seq0 + row / ap->n) * ap->slab_x + (size_t)ap->latent[gv.row0 + row] * ap->subtokens) * E + head * HD + xd;
            };
            const size_t cell0 = cell(min(wave * RPW + lane / HD, rows - 1u));
            const float early_k = xk[cell0], early_v = xv[cell0];
            if (plain) operand_plain(std::integral_constant<int, XKB>(), ap, XKB * kpart, av);
            if (!sh.all_here(wave)) return;
            if (!plain) operand(std::integral_constant<int, XKB>(), in, XKB * kpart, tag - 1u, av);
            floatx4 acc[RT][2];
#pragma unroll
            for (int rt = 0; rt < RT; rt++) {
                acc[rt][0] = acc[rt][1] = floatx4{0.f, 0.f, 0.f, 0.f};
                ss[rt] = 0.f;
#pragma unroll
                for (int i = 0; i < XKB; i++) {
                    acc[rt][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[rt][i], b[0][i], acc[rt][0], 0, 0, 0);
                    acc[rt][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[rt][i], b[1][i], acc[rt][1], 0, 0, 0);
                    ss[rt] += av[rt][i] * av[rt][i];
                }
            }
            meet(Two(), acc, ss);
            if (f_on) {
                const float scale = row_scale(std::integral_constant<uint32_t, XKS>(), f_row) * ap->xscale;
#pragma unroll
                for (uint32_t j = 0; j < (uint32_t)DT; j++)
                    xquery[f_row][16u * j + f_col] = total(std::integral_constant<uint32_t, XKS>(), f_rt, j) * scale;
            }
            __syncthreads();
            /* the rows' cross attention over their few sub-tokens (kv_cache.c:303-324): HD lanes per row; maximum
             * over finite scores, non-finite scores weigh nothing */
            for (uint32_t r0 = wave * RPW; r0 < rows; r0 += WAVES * RPW) {
                const uint32_t row = min(r0 + lane / HD, rows - 1u);
                const float qd = xquery[row][xd];
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
            !square(ap, ap->layer[layer].xproj, At::xcomb, false, tag, plain, in, tag - 1u, At::mid, first(FIRST_XPROJ)))
            return;

        ap = hidden_args(args);
        for (uint32_t t = first(FIRST_QKV); sh.has(STAGE_QKV) && t < 3u * E / 16u; t += WORKERS) { /* ---- QKV: rotated, keys and values written through ---- */
            fresh_lane();
            float b[KB], av[RT][KB], ss[RT], cs = 0.f, sn = 0.f;
            const float *w = ap->layer[layer].qkv + (4u * KB * wave + g) * (3u * E) + t * 16u + c;
            const float *nw = ap->layer[layer].norm1 + 4u * KB * wave + g;
#pragma unroll
            for (int i = 0; i < KB; i++) b[i] = w[4 * i * 3 * E] * nw[4 * i];
            const uint32_t part_of = t * 16u / E, cc = t * 16u + f_col - part_of * E, hh = cc / HD, dd = cc % HD;
            const uint32_t sq = f_safe / ap->n, slot = ap->len[gv.seq0 + sq] + f_safe % ap->n;
            if (f_on && part_of < 2u) { /* rotation of this thread's element */
                const uint32_t pos = ap->indexed ? ap->position[f_safe] : slot;
                cs = ap->cos[(size_t)pos * (HD / 2) + dd / 2u], sn = ap->sin[(size_t)pos * (HD / 2) + dd / 2u];
            }
            const uint32_t of_head = (f_rt * H + hh) * (HD * 16u);
            uint32_t to = part_of < 2u ? (part_of == 0u ? At::q : At::k) + of_head + (dd % QD) * 64u + (dd / QD) * 16u + (f_row & 15u)
                                       : At::v + of_head + (f_row & 15u) * HD + dd;
            float *cell = (part_of == 1u ? ap->layer[layer].ck : ap->layer[layer].cv) + ((size_t)(gv.seq0 + sq) * ap->max_seq + slot) * E + cc;
            asm volatile("" : "+v"(to), "+v"(cell)); /* here, not after the wait */
            if (plain && !crossed) operand_plain(Steps(), ap, KB * wave, av);
            if (!sh.all_here(wave)) return;
            if (!plain || crossed) operand(Steps(), crossed ? At::mid : in, KB * wave, crossed ? tag : tag - 1u, av);
            floatx4 acc[RT][1];
#pragma unroll
            for (int rt = 0; rt < RT; rt++) {
                floatx4 a0 = floatx4{0.f, 0.f, 0.f, 0.f}, a1 = a0;
                ss[rt] = 0.f;
#pragma unroll
                for (int i = 0; i < KB; i += 2) {
                    a0 = __builtin_amdgcn_mfma_f32_16x16x4f32(av[rt][i], b[i], a0, 0, 0, 0);
                    a1 = __builtin_amdgcn_mfma_f32_16x16x4f32(av[rt][i + 1], b[i + 1], a1, 0, 0, 0);
                    ss[rt] += av[rt][i] * av[rt][i] + av[rt][i + 1] * av[rt][i + 1];
                }
                acc[rt][0] = a0 + a1;
            }
            meet(One(), acc, ss);
            if (f_on) {
                float v = total(All(), f_rt, 0) * row_scale(All(), f_row);
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
        }

        ap = hidden_args(args);
        if (sh.has(STAGE_PROJ) && first(FIRST_PROJ) < (uint32_t)E / 16u &&
            !square(ap, ap->layer[layer].proj, At::comb, ap->splits > 1u, tag, plain && !crossed, crossed ? At::mid : in,
                    crossed ? tag : tag - 1u, At::resid, first(FIRST_PROJ)))
            return;

        ap = hidden_args(args);
        fresh_lane();
        const uint32_t hidden = ap->hidden, steps = hidden / 32u; /* steps: of a wave in the down projection */
        const bool down_here = sh.has(STAGE_DOWN) && first(FIRST_DOWN) < (uint32_t)E / 16u;
        constexpr int CH = RT == 1 ? 16 : 8; /* its steps in flight together */
        float bd[CH];
        const float *wd = ap->layer[layer].down + (4u * steps * wave + g) * E + first(FIRST_DOWN) * 16u + c;
        if (down_here) { /* on their way while this workgroup is busy with the stage before */
#pragma unroll
            for (int i = 0; i < CH; i++) bd[i] = (uint32_t)i < steps ? wd[i * 4u * E] : 0.f;
        }
        for (uint32_t t = first(FIRST_UPGATE); sh.has(STAGE_UPGATE) && t < hidden / 16u; t += WORKERS) { /* ---- up, gate, activation ---- */
            fresh_lane();
            float b[2][KB], av[RT][KB], ss[RT];
            const uint32_t off = (4u * KB * wave + g) * hidden + t * 16u + c;
            const float *up = ap->layer[layer].up + off, *gate = ap->layer[layer].gate + off;
            const float *nw = ap->layer[layer].norm2 + 4u * KB * wave + g;
#pragma unroll
            for (int i = 0; i < KB; i++) {
                const float n1 = nw[4 * i];
                b[0][i] = up[4 * i * hidden] * n1, b[1][i] = gate[4 * i * hidden] * n1;
            }
            if (!sh.all_here(wave)) return;
            operand(Steps(), At::resid, KB * wave, tag, av);
            floatx4 acc[RT][2];
#pragma unroll
            for (int rt = 0; rt < RT; rt++) {
                acc[rt][0] = acc[rt][1] = floatx4{0.f, 0.f, 0.f, 0.f};
                ss[rt] = 0.f;
#pragma unroll
                for (int i = 0; i < KB; i++) {
                    acc[rt][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[rt][i], b[0][i], acc[rt][0], 0, 0, 0);
                    acc[rt][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[rt][i], b[1][i], acc[rt][1], 0, 0, 0);
                    ss[rt] += av[rt][i] * av[rt][i];
                }
            }
            meet(Two(), acc, ss);
            if (f_on && f_row < rows) {
                const float scale = row_scale(All(), f_row), v = total(All(), f_rt, 0) * scale, gt = total(All(), f_rt, 1) * scale;
                word_store(words + At::act + operand_at<RT>(f_row, t * 16u + f_col), gt / (1.0f + expf(-gt)) * v, tag);
            }
            buf ^= 1u;
        }

        ap = hidden_args(args);
        if (down_here) { /* ---- down projection + residual ---- */
            if (!sh.all_here(wave)) return;
            fresh_lane();
            const uint32_t oc = first(FIRST_DOWN) * 16u + f_col;
            float r1[1] = {0.f};
            floatx4 acc[RT][2];
#pragma unroll
            for (int rt = 0; rt < RT; rt++) acc[rt][0] = acc[rt][1] = floatx4{0.f, 0.f, 0.f, 0.f};
            for (uint32_t k0 = 0; k0 < steps; k0 += CH) {
                if (k0) {
#pragma unroll
                    for (int i = 0; i < CH; i++) bd[i] = k0 + i < steps ? wd[(k0 + i) * 4u * E] : 0.f;
                }
#pragma unroll
                for (int rt = 0; rt < RT; rt++) {
                    float av[CH]; /* past the wave's last step: repeats, against weights of zero */
                    const uint64_t *p = word_of(words + At::act + ((steps * wave + k0) * RT + (uint32_t)rt) * 64u, lane);
                    await_at<CH>(wt, [&](int i) { return p + min((uint32_t)i, steps - 1u - k0) * (RT * 64u); }, 16u * rt + c >= rows, tag, av,
                                 __LINE__);
#pragma unroll
                    for (int i = 0; i < CH; i++) acc[rt][i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i], bd[i], acc[rt][i & 1], 0, 0, 0);
                }
            }
            if (f_on) await<1, 1>(wt, words + At::resid, operand_at<RT>(f_safe, oc), false, tag, r1);
            floatx4 sum[RT][1];
#pragma unroll
            for (int rt = 0; rt < RT; rt++) sum[rt][0] = acc[rt][0] + acc[rt][1];
            meet(One(), sum, nullptr);
            if (f_on && f_row < rows) word_store(words + At::output(layer) + operand_at<RT>(f_row, oc), r1[0] + total(All(), f_rt, 0), tag);
            buf ^= 1u;
        }
    }

    if (!sh.has(STAGE_LM)) return;
    ArgsPtr ap = hidden_args(args);
    const uint32_t V = ap->V;
    for (uint32_t t = first(FIRST_LM); t < V / 16u; t += WORKERS) { /* ---- LM head ---- */
        fresh_lane();
        float b[KB], av[RT][KB];
        const float *w = ap->lm + (size_t)(4u * KB * wave + g) * V + t * 16u + c;
#pragma unroll
        for (int i = 0; i < KB; i++) b[i] = w[(size_t)(4 * i) * V];
        if (!sh.all_here(wave)) return;
        operand(Steps(), At::output(L - 1u), KB * wave, ap->tag + L - 1u, av);
        floatx4 acc[RT][1];
#pragma unroll
        for (int rt = 0; rt < RT; rt++) {
            acc[rt][0] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < KB; i++) acc[rt][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[rt][i], b[i], acc[rt][0], 0, 0, 0);
        }
        meet(One(), acc, nullptr);
        if (f_on && f_row < rows) ap->logits[(size_t)(gv.row0 + f_row) * V + t * 16u + f_col] = total(All(), f_rt, 0);
        buf ^= 1u;
    }
    (void)sh.all_here(wave); /* a workgroup without any tile may have to stand in for others */
}

/* The workgroups that run the self-attention stages: units of one (sequence, head, share of the keys).  The first
 * key and value tiles of a wave are requested and turned into fragments before the query is there. */
template <int E, int HD, int RT, typename Share>
__device__ __forceinline__ void attention_role(ArgsPtr args, const GroupView gv, Share sh, float *area) {
    using At = Regions<E, RT>;
    constexpr int QD = HD / 4, NV = QD / 4, DT = HD / 16, ROW = HD + 4, H = E / HD;
    constexpr int LPR = HD / 4, RPI = 64 / LPR;
    constexpr int T = HD == 32 ? 2 : 1; /* key tiles a wave has in registers */
    const uint32_t tid = threadIdx.x, wave = gv.wave;
    uint64_t *const words = gv.words;
    Waiter wt{args->timeout, args->spin_limit, false};
    float *const sm_max = area, *const sm_sum = area + 16 * WAVES;
    float *const tiles = area + 2 * 16 * WAVES;
    float *const tile = tiles + wave * (16 * ROW);
    const uint32_t splits = args->splits, units = gv.ns * (uint32_t)H * splits, n = args->n;
    if (!sh.all_here(wave)) return;

    for (uint32_t layer = sh.begin(); layer < sh.end(args->L); layer++)
    for (uint32_t u = gv.worker; u < units; u += WORKERS) {
        const ArgsPtr ap = hidden_args(args);
        uint32_t lane = tid & 63u;
        asm volatile("" : "+v"(lane));
        const uint32_t g = lane >> 4, c = lane & 15u, prow = lane / LPR, pf = lane % LPR;
        const uint32_t tag = ap->tag + layer;
        const uint32_t split = u % splits, head = (u / splits) % (uint32_t)H, sq = u / (splits * (uint32_t)H);
        const uint32_t len = ap->len[gv.seq0 + sq], nk = len + n;
        const bool windowed = ap->window > 0u && !ap->block_kind;
        const uint32_t first = windowed && len + 1u > ap->window ? (len + 1u - ap->window) / 16u : 0u;
        const uint32_t cached = (len + 15u) / 16u; /* tiles of cached rows */
        const uint32_t share = (cached - min(first, cached) + splits - 1u) / splits;
        const uint32_t t_lo = min(first + split * share, cached), t_hi = min(t_lo + share, cached);
        const size_t slab = ((size_t)(gv.seq0 + sq) * ap->max_seq) * E + head * HD;
        const char *kb = reinterpret_cast<const char *>(ap->layer[layer].ck + slab);
        const char *vb = reinterpret_cast<const char *>(ap->layer[layer].cv + slab);
        const bool fresh_here = split == splits - 1u && wave == WAVES - 1u; /* takes the new rows too */
        for (uint32_t qt = 0; qt * 16u < n; qt++) {
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
            bool have_q = false;
            for (uint32_t tb = t_lo + wave; tb < t_hi || (fresh_here && !have_q); tb += WAVES * T) {
                float kf[T][QD], vf[T][DT][4];
                {
                    floatx4 kg[T][NV], vg[T][NV];
#pragma unroll
                    for (int u2 = 0; u2 < T; u2++)
                        if (tb + WAVES * u2 < t_hi) { /* wave-uniform */
#pragma unroll
                            for (int v = 0; v < NV; v++) {
                                const uint32_t off = min((tb + WAVES * u2) * 16u + prow + (uint32_t)(RPI * v), len - 1u) * (4u * E) + 16u * pf;
                                kg[u2][v] = *reinterpret_cast<const floatx4 *>(kb + off);
                                vg[u2][v] = *reinterpret_cast<const floatx4 *>(vb + off);
                            }
                        }
#pragma unroll
                    for (int u2 = 0; u2 < T; u2++) { /* rows -> fragments, through the wave's own LDS tile */
                        if (tb + WAVES * u2 >= t_hi) continue;
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
                }
                if (!have_q) {
                    await<QD, 64>(wt, words + At::q + head * (HD * 16u), (qrow >> 4) * (H * HD * 16u) + g * 16u + (qrow & 15u), qpad, tag, qf);
                    have_q = true;
                }
#pragma unroll
                for (int u2 = 0; u2 < T; u2++)
                    if (tb + WAVES * u2 < t_hi) tile_step(kf[u2], vf[u2], (tb + WAVES * u2) * 16u, len);
            }
            if (fresh_here) {
                for (uint32_t kt = 0; kt * 16u < n; kt++) {
                    const uint32_t krow = sq * n + min(16u * kt + c, n - 1u);
                    /* this lane's key row as a K fragment, its part of four value rows */
                    float kf[QD], vf[DT][4], kv[QD + DT * 4];
                    const uint64_t *of_head = words + At::k + head * (HD * 16u), *kp = word_of(of_head, (krow >> 4) * (H * HD * 16u) + g * 16u + (krow & 15u));
                    const uint64_t *vp[4];
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const uint32_t vrow = sq * n + min(16u * kt + 4u * g + (uint32_t)r, n - 1u);
                        vp[r] = word_of(of_head + (At::v - At::k), (vrow >> 4) * (H * HD * 16u) + (vrow & 15u) * HD + DT * c);
                    }
                    await_at<QD + DT * 4>(wt, [&](int i) { return i < QD ? kp + i * 64 : vp[((i - QD) / DT) & 3] + (i - QD) % DT; }, false, tag, kv,
                                          __LINE__);
#pragma unroll
                    for (int s = 0; s < QD; s++) kf[s] = kv[s];
#pragma unroll
                    for (int r = 0; r < 4; r++)
#pragma unroll
                        for (int dd = 0; dd < DT; dd++) vf[dd][r] = kv[QD + r * DT + dd];
                    tile_step(kf, vf, len + 16u * kt, nk);
                }
            }
            lsum = swap32(swap16(lsum, OpSum()), OpSum());
            if (wt.expired) lsum = not_there(); /* scores that are not finite would just weigh nothing */
            if (g == 0) sm_max[c * WAVES + wave] = mx, sm_sum[c * WAVES + wave] = lsum;
            /* lane (g, c) holds columns DT (4g + r) + dd of query row c */
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int dd = 0; dd < DT; dd++) tile[c * ROW + DT * (4u * g + r) + dd] = oacc[dd][r];
            __syncthreads();
            /* a thread per (row, column): the waves' partials, scaled to the common maximum */
            const uint32_t live = min(16u, n - 16u * qt);
            for (uint32_t cell = tid; cell < live * HD; cell += 64u * WAVES) {
                const uint32_t mr = cell / HD, mc = cell % HD;
                float wm[WAVES], ws[WAVES], o[WAVES];
#pragma unroll
                for (uint32_t v = 0; v < WAVES; v += 4u) {
                    const float4 x = *reinterpret_cast<const float4 *>(sm_max + mr * WAVES + v), y = *reinterpret_cast<const float4 *>(sm_sum + mr * WAVES + v);
                    wm[v] = x.x, wm[v + 1] = x.y, wm[v + 2] = x.z, wm[v + 3] = x.w;
                    ws[v] = y.x, ws[v + 1] = y.y, ws[v + 2] = y.z, ws[v + 3] = y.w;
                }
#pragma unroll
                for (uint32_t v = 0; v < WAVES; v++) o[v] = tiles[v * (16 * ROW) + mr * ROW + mc];
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
                    word_store(words + At::comb + split * At::M + operand_at<RT>(R, col), sum, tag);
                    if (mc < 2u) word_store(words + At::stat + (split * H + head) * (32u * RT) + R * 2u + mc, mc == 0u ? M : Lt, tag);
                } else {
                    word_store(words + At::comb + operand_at<RT>(R, col), Lt == 0.f ? 0.f : sum / Lt, tag);
                }
            }
            __syncthreads(); /* the area may be written again */
        }
    }
}

template <int E, int HD, int RT>
__global__ __launch_bounds__(64 * WAVES, 4) void kv_step_resident_kernel(ResidentArgs a) {
    __shared__ __attribute__((aligned(16))) float area[ResidentShape<HD, RT>::AREA];
    __shared__ __attribute__((aligned(16))) float part_ss[2][16 * RT][WAVES];
    __shared__ float xquery[16 * RT][HD];
    __shared__ Standing standing;
    GroupView gv;
    const uint32_t group = blockIdx.x % GROUPS, index = blockIdx.x / GROUPS;
    gv.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    gv.seq0 = group * a.per_group;
    if (gv.seq0 >= a.batch) return;
    if (threadIdx.x == 0u) sign_in(a.rolls + group * (2u * WORKERS), index, a.tag);
    gv.ns = min(a.per_group, a.batch - gv.seq0);
    gv.rows = gv.ns * a.n, gv.row0 = gv.seq0 * a.n;
    gv.words = a.words + (size_t)group * a.group_words;
    const ArgsPtr ap = (ArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
    gv.worker = index & (WORKERS - 1u);
    const WholeStep whole{ap, group, index, &standing, false};
    if (index < WORKERS) product_role<E, HD, RT>(ap, gv, whole, area, part_ss, xquery);
    else attention_role<E, HD, RT>(ap, gv, whole, area);
    const uint32_t rank = __builtin_amdgcn_readfirstlane(standing.rank), members = __builtin_amdgcn_readfirstlane(standing.members);
    if (members == 2u * WORKERS) return;

    const uint32_t stride = min(members, WORKERS);
    if (rank >= stride) return;
    for (uint32_t stage = 0; stage <= a.L * STAGES; stage++) {
        const OneStage one{stage / STAGES, stage < a.L * STAGES ? stage % STAGES : (uint32_t)STAGE_LM};
        for (gv.worker = rank; gv.worker < WORKERS; gv.worker += stride) {
            if (one.stage == STAGE_ATTN) attention_role<E, HD, RT>(ap, gv, one, area);
            else product_role<E, HD, RT>(ap, gv, one, area, part_ss, xquery);
            __syncthreads(); /* the shared areas may be written again */
        }
    }
}

__global__ void clear_hand_over_kernel(uint64_t *w, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256u + threadIdx.x;
    if (i < n) w[i] = 0u;
}

typedef void (*ResidentKernel)(ResidentArgs);
ResidentKernel kernel_of(size_t E, size_t hd, uint32_t row_tiles) {
    if (E == 64 && hd == 32) return row_tiles == 2u ? kv_step_resident_kernel<64, 32, 2> : kv_step_resident_kernel<64, 32, 1>;
    if (E == 64) return kv_step_resident_kernel<64, 64, 1>;
    if (E == 128) return hd == 32 ? kv_step_resident_kernel<128, 32, 1> : kv_step_resident_kernel<128, 64, 1>;
    return hd == 32 ? kv_step_resident_kernel<256, 32, 1> : kv_step_resident_kernel<256, 64, 1>;
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
    static constexpr size_t COUNT = WORDS + GROUPS * 2u * WORKERS; /* and the roll calls */
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
        V % 16 != 0 || V == 0 || blt_stream_capturing())
        return false;
    const size_t per_group = (st.batch + GROUPS - 1) / GROUPS, group_rows = per_group * st.n;
    if (group_rows > MAX_GROUP_ROWS || st.batch > MAX_ROWS) return false;
    /* Where the launches win, measured over E, heads, layers, rows and lengths (us, launches -> resident, four
     * layers).  Up to 16 rows a group and heads of 32: everywhere (E = 64: 113 -> 50 at one row, 133 -> 82 at 96;
     * E = 256: 155 -> 93, 254 -> 231 at 64 rows of 900 keys).  17 to 32 rows: narrow models only (E = 64: 140 ->
     * 126), the products of wide ones have all compute units in the launches (E = 256: 25 rows 227 -> 247, eight
     * groups of 32 rows 229 -> 282).  Heads of 64 have half the keys per wave in flight and spill four
     * times as many registers: single rows of few sequences a group (E = 256, 20 sequences: 187 -> 162; 64 of 900 keys: 251
     * -> 343). */
    if (group_rows > 16 && E > 64) return false;
    if (hd == 64 && (st.n > 1 || per_group > 4)) return false;
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
        bits |= reinterpret_cast<uintptr_t>(r.ck) | reinterpret_cast<uintptr_t>(r.cv);
    }
    if (bits & 15u) return false; /* rows are read sixteen bytes at a time */
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
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (s != nullptr) HIP_CHECK(hipStreamIsCapturing(s, &capture));
    if (capture != hipStreamCaptureStatusNone) return false;
    const ResidentKernel kernel = kernel_of(E, hd, rt);
    const uint32_t groups = (uint32_t)((st.batch + per_group - 1) / per_group);
    if (!can_be_resident(kernel, groups * 2u * WORKERS, dev, s)) return false;
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
    blt_launch("kv_step_resident", kernel, dim3(GROUPS * 2u * WORKERS), dim3(64 * WAVES), 0, s, a);
    g_launched.store(true, std::memory_order_relaxed);
    return true;
}
