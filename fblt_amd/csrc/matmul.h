/* Launch interface of the fp32 matrix product kernels (matmul.hip). */
#ifndef FBLT_AMD_MATMUL_H
#define FBLT_AMD_MATMUL_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "blt_abi.h"
#include "rope_device.h"

/* out[m, n] = a[m, k] * b[k, n], leading dimensions in elements.  With
 * rope_cos / rope_sin set ([m, head_dim/2] tables, row r = position of output
 * row r), pairs (2i, 2i+1) of every head_dim-wide block of the first
 * rope_cols output columns are rotated before they are stored; head_dim and
 * rope_cols must be multiples of 4. */
struct MatmulArgs {
    const float *a;
    const float *b;
    const float *b2;       /* optional second weight matrix [k, n] (same ldb): out = silu(a*b2) .* (a*b), the gated
                              feed-forward activation (csrc/ops/elementwise_cpu.c:86-99) in one pass          */
    float *out2;           /* with b2: store a*b2 here (same ldo) instead of gating the first product with it  */
    const float *residual; /* optional [m, n] (leading dimension ldo) added to the result                     */
    const float *norm_w;   /* optional [k]: the rows of a are RMS-normalised with this weight first, i.e. the
                              product is taken of blt_rmsnorm_forward(a, norm_w) (csrc/ops/reductions_cpu.c:
                              327-352) without materialising it; the row statistic is accumulated from the
                              same loads (fp32 tolerance: the scale is applied after the product)              */
    float *out;
    const float *rope_cos;
    const float *rope_sin;
    uint32_t m, k, n;
    uint32_t lda, ldb, ldo;
    uint32_t rope_cols, head_dim;
    /* Optional cross-attention epilogue (matmul_takes_cross): the product is the query projection
     * of a cross block with heads cross_head_dim wide; instead of being stored, each projected row
     * attends, head by head, over the sub-tokens [cross_lo[row], cross_hi[row]) of its sequence's
     * tier-2 slab (sequence = row / cross_rows_per_seq) and the weighted V row goes to
     * cross_out[row, head columns] (csrc/infer/kv_cache.c:303-324).  More than 32 rows: split-K
     * kernel, 32-wide heads (a 32x32 output tile is one head of 32 rows).  Up to 32 rows: the exact
     * kernel with n <= 256, whose single workgroup per row group holds whole projected rows.
     * out may be null. */
    const float *cross_k;
    const float *cross_v;
    float *cross_out;
    const uint32_t *cross_lo;
    const uint32_t *cross_hi;
    uint32_t cross_rows_per_seq, cross_slab_rows, cross_head_dim;
    float cross_scale;
    /* Optional destination of a packed QKV product (n = 3 E, rope_cols = 2 E): row stage_n * b + r is the new row r of
     * sequence b, at position stage_len[b] + r of the rotary tables (which then have a row per position, not per row).  The
     * rotated Q rows go to out (ldo = E), the rotated K rows and the V rows to the slabs [batch, stage_slab_rows, E]; all
     * 16-byte aligned. */
    float *stage_k;
    float *stage_v;
    const uint32_t *stage_len;
    uint64_t stage_slab_rows;
    uint32_t stage_n;
    /* Products of up to 32 rows normally run on the thread-per-column kernel, whose sums follow the
     * reference's order (bit-identical results) at the price of a serial chain of k additions.
     * tolerant != 0: the caller accepts fp32-tolerance results for such shapes too, and they go to
     * the matrix cores with K split over the waves (the whole decoder step sets it: a one-row
     * step takes 72 us instead of 112). */
    uint32_t tolerant;
    /* Set by the launcher, never by callers.  slices > 1: the K range is also split over slices
     * workgroups per output tile (grid z); each leaves its tile's sums in slice_sums
     * [tile][slice][1024, or 4096 of the 64x64 tile] and the one that draws the last of the tile's tickets adds them in slice
     * order and runs the epilogue. */
    uint32_t slices;
    float *slice_sums;
    uint32_t *slice_tickets;
};

/* Four consecutive results of row `row`, position pos of sequence b, rotated where they are of Q or K: to Q or to the slabs. */
__device__ __forceinline__ void matmul_stage4(const MatmulArgs &g, uint32_t row, uint32_t b, uint32_t pos, uint32_t col, float4 v) {
    const uint32_t E = g.n / 3u, part = col / E, at = col % E;
    if (part < 2u) {
        const size_t turn = (size_t)pos * (g.head_dim / 2u) + (at % g.head_dim) / 2u;
        v = rope_rotate4(v, g.rope_cos + turn, g.rope_sin + turn);
    }
    float *const to = part == 0u ? g.out + (size_t)row * E : (part == 1u ? g.stage_k : g.stage_v) + ((size_t)b * g.stage_slab_rows + pos) * E;
    *reinterpret_cast<float4 *>(to + at) = v;
}
/* Four consecutive results of output row `row` starting at column `col`:
 * optional rotation, optional residual, store with bounds. */
template <bool ROPE>
__device__ __forceinline__ void matmul_store4(const MatmulArgs &g, uint32_t row, uint32_t col, float4 v, bool vec_ok) {
    if (ROPE && g.stage_k) { /* new rows of a cache: no residual */
        if (col >= g.n) return;
        const uint32_t b = row / g.stage_n;
        matmul_stage4(g, row, b, g.stage_len[b] + row % g.stage_n, col, v);
        return;
    }
    if (ROPE && col < g.rope_cols) {
        /* columns col..col+3 are pairs (col % head_dim)/2 and the next one of the row's position */
        const size_t at = (size_t)row * (g.head_dim / 2u) + (col % g.head_dim) / 2u;
        v = rope_rotate4(v, g.rope_cos + at, g.rope_sin + at);
    }
    float *orow = g.out + (size_t)row * g.ldo;
    const float *rrow = g.residual ? g.residual + (size_t)row * g.ldo : nullptr;
    if (vec_ok) {
        if (col < g.n) {
            if (rrow) {
                const float4 r = *reinterpret_cast<const float4 *>(rrow + col);
                v.x = r.x + v.x, v.y = r.y + v.y, v.z = r.z + v.z, v.w = r.w + v.w;
            }
            *reinterpret_cast<float4 *>(orow + col) = v;
        }
    } else {
        const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (col + i < g.n) orow[col + i] = rrow ? rrow[col + i] + e[i] : e[i];
    }
}

void matmul_f32_launch(const MatmulArgs &g, hipStream_t s);
/* MatmulArgs::tolerant of whole steps, blocks and forward passes: their projections are taken on the matrix cores whatever the
 * row count (fp32 tolerance, as they always are above 32 rows; us, exact / this: a one-row decoder step 112 / 72, a block of 16
 * rows of 128 columns 56.6 / 17.5, of 30 rows of 512 175 / 42, a forward of 64 bytes 278 / 156; error of those blocks against float64
 * 3.5e-7 / 1.7e-7 and 6.5e-7 / 2.3e-7).  BLT_HIP_EXACT_STEP=1 keeps the exact kernel up to 32 rows (results bit-identical
 * to the CPU reference's). */
uint32_t matmul_tolerant();
__device__ __forceinline__ float silu_times(float gate, float up) {
    const float silu = gate / (1.0f + expf(-gate));
    return silu * up;
}
/* Room for `floats` partial sums and `count` zeroed tickets of one launch on the stream, per (thread, stream): launches on one
 * stream follow each other, launches on two never share them.  Every launch leaves its tickets at zero.  false: the
 * buffers would have to grow while a graph capture is open, or the capture is the caller's own: a replay may run beside later
 * launches that use the same sums and tickets. */
bool matmul_slice_scratch(size_t floats, size_t count, hipStream_t s, float **sums, uint32_t **tickets);
/* What of a transformer block is behind its attention, in one launch (block_tail.hip): out = r + SwiGLU(RMSNorm(r)) * down
 * with r = x + comb * proj.  All row-major and dense; out may be x. */
struct BlockTailArgs {
    const float *comb, *x, *proj, *norm_w, *up, *gate, *down;
    float *out, *resid; /* resid: room for r */
    uint32_t rows, hidden;
    uint64_t *sums; /* set by the launcher */
    uint32_t *tickets;
};
/* A cross block past its K and V rows, in one launch (block_tail.hip): out = residual + combined * proj, where row r of
 * `combined` attends, head by head, from RMSNorm(x) * wq (x * wq without norm_w) over rows lo[r] .. hi[r] - 1 of k and v,
 * counted from slab_rows * (r / rows_per_seq); no rows: zeros.  All dense rows of embed_dim; out may be x. */
/* Key ranges on their way: a pass's first cross block brings them in its arguments and leaves them, and the lengths of the sequences,
 * where later launches look for them.  words: the lengths, then the ranges' starts, two in each, and after them, if a range ends where
 * the next one starts (span 0; else all are that long), the last one's end. */
struct CrossWords {
    static constexpr uint32_t WORDS = 880; /* with the other arguments of the largest launch, a block of 4096 bytes */
    uint32_t *lo, *hi, *lens;
    uint32_t rows, batch, span, reserved;
    uint32_t words[WORDS];
};
/* false: not of this kind, the caller uploads them.  lens: batch of them (none: of no use to later launches). */
bool cross_words_fill(CrossWords &w, const uint32_t *lo, const uint32_t *hi, size_t rows, const uint32_t *lens, size_t batch);
struct CrossBlockArgs {
    const float *x, *norm_w, *wq, *k, *v, *proj, *residual; /* norm_w, residual: optional */
    float *out;
    const uint32_t *lo, *hi;
    uint64_t slab_rows;
    uint32_t rows, rows_per_seq, head_dim;
    float scale;
    const CrossWords *words; /* the launcher's: what lo and hi are to hold (null: they do) */
};
/* false: not for this shape, nothing was launched.  cross_block_ok: the same answer before lo and hi are there. */
bool cross_block_ok(const CrossBlockArgs &a, uint32_t embed_dim);
bool cross_block_launch(const CrossBlockArgs &a, uint32_t embed_dim, hipStream_t s);
/* The same, and the packed QKV product g of its output rows, RMS-normalised (g.norm_w; g.a is not looked at), in one launch. */
bool cross_qkv_launch(const CrossBlockArgs &a, const MatmulArgs &g, uint32_t embed_dim, hipStream_t s);
/* A cross block put off until launches of the next layer, which has nothing to do with it, can take it along: the product of its
 * keys and values beside that layer's first product, the rest beside its tail. */
struct CrossLater {
    MatmulArgs kv;
    CrossBlockArgs cross;
    bool kv_waits = false, cross_waits = false;
    bool feeds = false; /* unlike that, the block is what the next layer starts from: it goes along with its QKV product or before */
};
/* What the cross blocks of one forward pass, which have their mask in common, leave each other. */
struct CrossPass {
    const uint32_t *lo = nullptr, *hi = nullptr; /* the mask's key ranges on the device; lo null: not there (yet) */
    uint32_t span = 0;
    CrossWords words;
    CrossLater *later = nullptr; /* a block may be left there instead of launched */
    /* K and V weights of the next block over the same rows: its keys and values may be made in this block's launch ... */
    const blt_tensor *next_k = nullptr, *next_v = nullptr;
    float *made_k = nullptr, *made_v = nullptr; /* ... and are here then */
};
/* what still waits, in launches of its own: the product only, or both */
void matmul_later_launch(CrossLater &later, hipStream_t s);
void cross_later_launch(CrossLater &later, uint32_t embed_dim, hipStream_t s);
/* false: not for this shape, nothing was launched.  later: what waits may go along. */
bool block_tail_launch(BlockTailArgs a, uint32_t embed_dim, hipStream_t s, CrossLater *later = nullptr);
/* g0 (plain, rotated, or like g1) and g1 (two weight matrices, two outputs) in one launch; only when matmul_pair_ok says so */
bool matmul_pair_ok(const MatmulArgs &g0, const MatmulArgs &g1);
void matmul_f32_launch_pair(const MatmulArgs &g0, const MatmulArgs &g1, hipStream_t s);
/* the cross-attention epilogue for this shape and g.cross_head_dim, no other epilogue set */
bool matmul_takes_cross(const MatmulArgs &g);
/* norm_w likewise */
bool matmul_takes_norm(const MatmulArgs &g);

#endif
