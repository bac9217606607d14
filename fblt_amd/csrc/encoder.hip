/*
 * The local encoder's forward pass on the device, and the three tensor ops it
 * needs beyond the attention blocks (reference: csrc/models/local_encoder.c:193-281,
 * csrc/models/hash_ngram.c:142-207, csrc/models/byte_embedding.c:16-53,
 * csrc/ops/gather_scatter_cpu.c:41-61, csrc/ops/elementwise_cpu.c:31-40,
 * csrc/ops/patch_pool_cpu.c:3-48):
 *
 *   e_0 = (byte_embedding[b_i] + sum_n table_n[hash_n(b_{i-n+1..i})]) / (K + 1)
 *   P_0 = pool(e_0, patches), repeated over the k sub-token column blocks
 *   per layer: h = transformer_block(h); where the cross block fires,
 *              P = P + cross_attention(RMSNorm(P), h)
 *
 * Hashing runs on the device too, in the launch that embeds and pools.  The small
 * kernels keep the reference's order of additions, so they are bit-identical to the
 * CPU ops: the embedding sum adds the tables in their order and scales last, the mean
 * pool adds a patch's rows first to last and multiplies by 1 / len.
 */
#include "blt_hip.h"
#include "blt_fatal.h"
#include "hip_check.h"
#include "launch.h"
#include "matmul.h"

#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <vector>

/* blt_cross_attention_forward_hip with the steps either side of it in a caller's layer folded in
 * (mha.hip): norm_w, when set, is the weight of the RMSNorm that makes query_in's rows the queries
 * (taken inside the query projection), residual [rows, embed] is added to the projected output.
 * pass: kept between the layers of one forward pass, whose cross blocks share a mask. */
void blt_cross_attention_run(const blt_tensor *query_in, const blt_tensor *kv_in,
                             const blt_cross_attention_weights *weights, blt_tensor *output,
                             const blt_cross_attention_config *config, blt_arena *arena, const float *norm_w,
                             const float *residual, CrossPass *pass);
/* blt_transformer_forward_hip (mha.hip); later: a cross block that waits for launches to go along with, all of it launched on return */
void blt_transformer_run(const blt_tensor *input, const blt_transformer_weights *w, blt_tensor *output,
                         const blt_transformer_config *config, blt_arena *arena, CrossLater *later);

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int IDX_PER_LAUNCH = 512; /* index entries a launch carries in its arguments */
struct IndexChunk {
    uint32_t v[IDX_PER_LAUNCH];
};

/* io[row0 + i, :] += table[idx[i], :] for every i whose index is not the sentinel */
__global__ __launch_bounds__(256) void rows_accumulate_kernel(const float *__restrict__ table, float *__restrict__ io,
                                                              uint64_t row_len, IndexChunk idx) {
    const uint32_t at = idx.v[blockIdx.x];
    if (at == BLT_IDX_SENTINEL) return;
    const float *s = table + (uint64_t)at * row_len;
    float *d = io + (uint64_t)blockIdx.x * row_len;
    for (uint64_t t = threadIdx.x; t < row_len; t += 256u) d[t] += s[t];
}

__global__ __launch_bounds__(256) void scale_kernel(float *__restrict__ x, uint64_t n, float scalar) {
    for (uint64_t t = (uint64_t)blockIdx.x * 256u + threadIdx.x; t < n; t += (uint64_t)gridDim.x * 256u) x[t] *= scalar;
}

constexpr int PATCHES_PER_LAUNCH = 256;
struct PatchChunk {
    uint32_t start[PATCHES_PER_LAUNCH];
    uint32_t len[PATCHES_PER_LAUNCH];
};

/* One workgroup per patch, one thread per column: the patch's rows first to last (the reference's
 * order of additions), written into `copies` column blocks of the output row. */
__global__ __launch_bounds__(256) void patch_pool_kernel(const float *__restrict__ h, float *__restrict__ out,
                                                         uint32_t embed_dim, uint32_t out_stride, uint32_t copies,
                                                         int take_max, PatchChunk p) {
    const uint32_t start = p.start[blockIdx.x], len = p.len[blockIdx.x];
    float *dst = out + (uint64_t)blockIdx.x * out_stride;
    for (uint32_t d = threadIdx.x; d < embed_dim; d += 256u) {
        const float *src = h + (uint64_t)start * embed_dim + d;
        float acc;
        if (take_max) {
            acc = src[0];
            for (uint32_t i = 1; i < len; i++) {
                const float v = src[(uint64_t)i * embed_dim];
                if (v > acc) acc = v;
            }
        } else {
            acc = 0.0f;
            for (uint32_t i = 0; i < len; i++) acc += src[(uint64_t)i * embed_dim];
            acc *= 1.0f / (float)len;
        }
        for (uint32_t c = 0; c < copies; c++) dst[c * embed_dim + d] = acc;
    }
}

constexpr int MAX_TABLES = BLT_MAX_NGRAM_SIZES;
constexpr uint32_t EMBED_RUNS = 256;   /* patches of a launch */
constexpr uint32_t EMBED_BYTES = 2560; /* bytes of text that travel in the arguments */
constexpr uint32_t EMBED_ROWS = 8;     /* rows of a patch at a time */
constexpr uint32_t EMBED_COLS = 512;   /* columns of a workgroup */
struct EmbedArgs {
    const float *byte_table;
    const float *table[MAX_TABLES]; /* [modulus, embed_dim] each */
    const uint8_t *bytes;           /* null: text */
    float *h;                       /* [all rows, embed_dim] */
    float *pooled;                  /* of the launch's patches, copies blocks of columns of each row (null: rows only) */
    uint64_t modulus, power[8];     /* prime^i mod modulus */
    uint32_t ngram[MAX_TABLES], tables, embed_dim, out_stride, copies;
    int scaled, take_max;
    float scale;
    uint32_t start[EMBED_RUNS + 1]; /* patches follow each other */
    uint8_t text[EMBED_BYTES];
};
static_assert(sizeof(EmbedArgs) <= 4096, "kernel argument block");

/* h[i, :] = (byte_table[byte i, :] + table_0[index_0 of i, :] + ...) * scale, the tables in order; an index is the reference's rolling
 * polynomial hash (csrc/models/hash_ngram.c:16-79) in closed form: position i >= n - 1 hashes bytes b[i-n+1..i] as sum b[j] *
 * prime^(i-j) mod modulus, earlier positions have no n-gram.  And the mean or maximum of a patch's rows, first to last (the
 * reference's order).
 * A workgroup is a patch, eight rows at a time: one wave hashes their n-grams while the others wait, then a thread has four columns of
 * a row (one where VEC is false), all its table rows requested before the first is added, and the rows of the eight meet in LDS.
 * Bound: latency (byte, hash, table row, row sums).  A forward of 512 bytes, one layer of 128 columns each: 100.4 us, from 116.1 with the
 * indices made on the host, uploaded and the patches pooled in three launches, and 171 with the bytes on the device. */
template <bool VEC>
__global__ __launch_bounds__(256) void embed_pool_kernel(EmbedArgs a) {
    constexpr uint32_t W = VEC ? 4u : 1u;
    __shared__ uint32_t index[EMBED_ROWS][MAX_TABLES + 1];
    __shared__ __attribute__((aligned(16))) float sum[EMBED_ROWS][EMBED_COLS];
    const uint32_t tid = threadIdx.x, E = a.embed_dim;
    const uint32_t first = a.start[blockIdx.x], end = a.start[blockIdx.x + 1u];
    const uint32_t col0 = blockIdx.y * EMBED_COLS, cols = min(EMBED_COLS, E - col0), pieces = cols / W;
    const uint8_t *const bytes = a.bytes;
    const auto byte_at = [&](uint32_t i) -> uint64_t { return bytes ? bytes[i] : a.text[i]; };
    float pooled[EMBED_COLS / 256u] = {0.f, 0.f};
    for (uint32_t row0 = first; row0 < end; row0 += EMBED_ROWS) {
        const uint32_t rows = min(EMBED_ROWS, end - row0);
        if (tid < 8u * EMBED_ROWS) {
            const uint32_t r = tid >> 3, t = tid & 7u, i = row0 + r; /* lane 0: the byte itself, 1 ...: the tables */
            if (r < rows && t <= a.tables) {
                const uint32_t n = t == 0u ? 1u : a.ngram[t - 1u];
                uint32_t at = BLT_IDX_SENTINEL;
                if (i + 1u >= n) {
                    uint64_t hash = 0; /* below 8 * 255 * modulus; no table has 2^50 rows */
                    for (uint32_t j = 0; j < n; j++) hash += byte_at(i - j) * (t == 0u ? 1u : a.power[j]);
                    at = (uint32_t)hash;
                    if (t != 0u) at = (hash | a.modulus) >> 32 ? (uint32_t)(hash % a.modulus) : (uint32_t)hash % (uint32_t)a.modulus;
                }
                index[r][t] = at;
            }
        }
        __syncthreads();
        for (uint32_t item = tid; item < rows * pieces; item += 256u) {
            const uint32_t r = item / pieces, d = col0 + W * (item % pieces);
            const auto add_up = [&](auto zero) {
                typedef decltype(zero) Vec;
                Vec acc = *reinterpret_cast<const Vec *>(a.byte_table + (uint64_t)index[r][0] * E + d), v[MAX_TABLES];
#pragma unroll
                for (uint32_t t = 0; t < MAX_TABLES; t++) {
                    if (t >= a.tables) break;
                    const uint32_t at = index[r][t + 1u];
                    v[t] = *reinterpret_cast<const Vec *>(a.table[t] + (uint64_t)(at == BLT_IDX_SENTINEL ? 0u : at) * E + d);
                }
#pragma unroll
                for (uint32_t t = 0; t < MAX_TABLES; t++) {
                    if (t >= a.tables) break;
                    if (index[r][t + 1u] != BLT_IDX_SENTINEL) acc += v[t];
                }
                if (a.scaled) acc *= a.scale;
                *reinterpret_cast<Vec *>(a.h + (uint64_t)(row0 + r) * E + d) = acc;
                *reinterpret_cast<Vec *>(&sum[r][d - col0]) = acc;
            };
            if constexpr (VEC) add_up(floatx4{0.f, 0.f, 0.f, 0.f});
            else add_up(0.f);
        }
        __syncthreads();
        if (a.pooled) {
#pragma unroll
            for (uint32_t c = 0; c < EMBED_COLS / 256u; c++) {
                const uint32_t d = tid + 256u * c;
                if (d >= cols) break;
                if (a.take_max) {
                    if (row0 == first) pooled[c] = sum[0][d];
                    for (uint32_t r = row0 == first ? 1u : 0u; r < rows; r++)
                        if (sum[r][d] > pooled[c]) pooled[c] = sum[r][d];
                } else {
                    for (uint32_t r = 0; r < rows; r++) pooled[c] += sum[r][d];
                }
            }
            __syncthreads(); /* before the next eight */
        }
    }
    if (!a.pooled) return;
#pragma unroll
    for (uint32_t c = 0; c < EMBED_COLS / 256u; c++) {
        const uint32_t d = tid + 256u * c;
        if (d >= cols) break;
        if (!a.take_max) pooled[c] *= 1.0f / (float)(end - first);
        for (uint32_t copy = 0; copy < a.copies; copy++) a.pooled[(uint64_t)blockIdx.x * a.out_stride + copy * E + col0 + d] = pooled[c];
    }
}

void check_2d(const blt_tensor *t, size_t rows, size_t cols, const char *msg) {
    BLT_REQUIRE(t != NULL && t->data != NULL && t->ndim == 2 && t->dtype == BLT_DTYPE_FP32 &&
                    t->backend == BLT_BACKEND_HIP && (rows == 0 || t->shape[0] == rows) &&
                    (cols == 0 || t->shape[1] == cols),
                "%s", msg);
}

blt_tensor view_2d(void *data, size_t rows, size_t cols) {
    blt_tensor t;
    std::memset(&t, 0, sizeof(t));
    t.data = data;
    t.shape[0] = rows, t.shape[1] = cols;
    t.strides[0] = cols, t.strides[1] = 1;
    t.ndim = 2;
    t.numel = rows * cols;
    t.dtype = BLT_DTYPE_FP32;
    t.backend = BLT_BACKEND_HIP;
    t.is_view = true;
    return t;
}

void pool_launch(const float *h, size_t seq_len, size_t embed_dim, const blt_patch_info *patches, size_t num_patches,
                 blt_patch_pool_type pool_type, float *out, size_t out_stride, size_t copies) {
    BLT_REQUIRE(pool_type == BLT_POOL_MEAN || pool_type == BLT_POOL_MAX, "patch_pool: unknown pool_type");
    BLT_REQUIRE(seq_len <= 0xFFFFFFFFu && embed_dim <= 0xFFFFFFFFu && out_stride <= 0xFFFFFFFFu,
                "patch_pool: sizes exceed 2^32-1");
    for (size_t j0 = 0; j0 < num_patches; j0 += PATCHES_PER_LAUNCH) {
        const size_t n = std::min<size_t>(PATCHES_PER_LAUNCH, num_patches - j0);
        PatchChunk c;
        std::memset(&c, 0, sizeof(c));
        for (size_t j = 0; j < n; j++) {
            const blt_patch_info &pi = patches[j0 + j];
            BLT_REQUIRE(pi.length >= 1, "patch_pool: empty patch");
            BLT_REQUIRE(pi.start_idx + pi.length <= seq_len, "patch_pool: patch out of range");
            c.start[j] = (uint32_t)pi.start_idx, c.len[j] = (uint32_t)pi.length;
        }
        blt_launch("patch_pool", patch_pool_kernel, dim3((unsigned)n), dim3(256), 0, blt_stream(), h, out + j0 * out_stride,
                   (uint32_t)embed_dim, (uint32_t)out_stride, (uint32_t)copies,
                   pool_type == BLT_POOL_MAX ? 1 : 0, c);
        HIP_CHECK_LAUNCH("blt_patch_pool_forward");
    }
}

/* Do the patches follow each other over all rows?  Then the launch that makes the rows pools them, but for long ones, whose rows it
 * would make eight after eight: a forward of 512 bytes, some patches of 8 / 64 / 256 rows, 98.7 / 121.6 / 157.7 us so, 101.1 / 125.2 /
 * 158.4 with the pooling as a launch. */
bool patches_tile(const blt_patch_info *patches, size_t num_patches, size_t seq_len) {
    size_t at = 0;
    for (size_t j = 0; j < num_patches; j++) {
        if (patches[j].start_idx != at || patches[j].length < 1 || patches[j].length > std::min<size_t>(256, seq_len - at))
            return false;
        at += patches[j].length;
    }
    return at == seq_len;
}

} // namespace

/* Replaces blt_indexed_row_accumulate_cuda (contract csrc/ops/gather_scatter.h:23-28,
 * gather_scatter_cpu.c:41-61): io[i, :] += table[idx_host[i], :], sentinel entries skipped. */
extern "C" void blt_indexed_row_accumulate_hip(const blt_tensor *table, const uint32_t *idx_host, blt_tensor *io) {
    BLT_REQUIRE(table != NULL && idx_host != NULL && io != NULL, "blt_indexed_row_accumulate: arguments cannot be NULL");
    check_2d(table, 0, 0, "blt_indexed_row_accumulate: HIP implementation needs 2D FP32 device tensors");
    check_2d(io, 0, 0, "blt_indexed_row_accumulate: HIP implementation needs 2D FP32 device tensors");
    const size_t rows = io->shape[0], embed_dim = io->shape[1];
    BLT_REQUIRE(table->shape[1] == embed_dim, "blt_indexed_row_accumulate: embed_dim mismatch");
    if (embed_dim == 0) return;
    for (size_t r0 = 0; r0 < rows; r0 += IDX_PER_LAUNCH) {
        const size_t n = std::min<size_t>(IDX_PER_LAUNCH, rows - r0);
        IndexChunk c;
        for (size_t i = 0; i < (size_t)IDX_PER_LAUNCH; i++) {
            c.v[i] = i < n ? idx_host[r0 + i] : BLT_IDX_SENTINEL;
            BLT_REQUIRE(c.v[i] == BLT_IDX_SENTINEL || c.v[i] < table->shape[0],
                        "blt_indexed_row_accumulate: index out of range");
        }
        blt_launch("rows_accumulate", rows_accumulate_kernel, dim3((unsigned)n), dim3(256), 0, blt_stream(),
                   (const float *)table->data, (float *)io->data + r0 * embed_dim, (uint64_t)embed_dim, c);
        HIP_CHECK_LAUNCH("blt_indexed_row_accumulate");
    }
}

/* Replaces blt_scale_cuda (csrc/ops/elementwise.h:10, elementwise_cpu.c:31-40): t *= scalar in place. */
extern "C" void blt_scale_hip(blt_tensor *t, float scalar) {
    BLT_REQUIRE(t != NULL, "blt_scale: tensor must not be null");
    BLT_REQUIRE(t->dtype == BLT_DTYPE_FP32, "blt_scale: only supports FP32 tensors");
    BLT_REQUIRE(t->backend == BLT_BACKEND_HIP, "blt_scale: HIP implementation called with non-HIP backend");
    if (t->numel == 0) return;
    const unsigned blocks = (unsigned)std::min<size_t>((t->numel + 255u) / 256u, 4096u);
    blt_launch("scale", scale_kernel, dim3(blocks), dim3(256), 0, blt_stream(), (float *)t->data, (uint64_t)t->numel,
               scalar);
    HIP_CHECK_LAUNCH("blt_scale");
}

/* Replaces blt_patch_pool_forward_cuda (contract csrc/ops/patch_pool.h:18-21, patch_pool_cpu.c:3-48):
 * out[j, :] = mean or per-column maximum of byte_hidden rows [start_j, start_j + len_j); the
 * patch table is a HOST array. */
extern "C" void blt_patch_pool_forward_hip(const blt_tensor *byte_hidden, const blt_patch_info *patches,
                                           size_t num_patches, blt_patch_pool_type pool_type, blt_tensor *out) {
    BLT_REQUIRE(byte_hidden != NULL && out != NULL, "patch_pool: NULL tensor");
    BLT_REQUIRE(patches != NULL || num_patches == 0, "patch_pool: NULL patches");
    check_2d(byte_hidden, 0, 0, "patch_pool: byte_hidden must be 2D FP32");
    const size_t seq_len = byte_hidden->shape[0], embed_dim = byte_hidden->shape[1];
    check_2d(out, num_patches, embed_dim, "patch_pool: out must be [num_patches, embed_dim] FP32");
    if (num_patches == 0 || embed_dim == 0) return;
    pool_launch((const float *)byte_hidden->data, seq_len, embed_dim, patches, num_patches, pool_type,
                (float *)out->data, embed_dim, 1);
}

/* csrc/models/local_encoder.c:193-281 on device tensors.  bytes_in may live on either side (on the
 * host it may change on return, on the device it is read in stream order); weights, outputs and the
 * arena are device memory.  Mask metadata is a host allocation of this call. */
extern "C" void blt_local_encoder_forward_hip(const blt_local_encoder *model, const blt_tensor *bytes_in,
                                              const blt_patch_info *patches, size_t num_patches,
                                              const size_t *doc_boundaries, size_t num_docs, blt_tensor *patch_out,
                                              blt_tensor *byte_hidden_out, blt_arena *arena) {
    BLT_REQUIRE(model != NULL && bytes_in != NULL && arena != NULL,
                "blt_local_encoder: model, bytes_in and arena cannot be NULL");
    BLT_REQUIRE(arena->backend == BLT_BACKEND_HIP, "blt_local_encoder: HIP implementation needs a device arena");
    BLT_REQUIRE(patches != NULL && num_patches >= 1, "blt_local_encoder: need at least one patch");
    BLT_REQUIRE(bytes_in->ndim == 1 && bytes_in->dtype == BLT_DTYPE_UINT8,
                "blt_local_encoder: bytes_in must be 1D UINT8 [seq_len]");
    const blt_local_encoder_config &cfg = model->config;
    const size_t seq_len = bytes_in->shape[0];
    BLT_REQUIRE(seq_len >= 1 && seq_len <= cfg.max_seq_len, "blt_local_encoder: seq_len must be in [1, max_seq_len]");
    BLT_REQUIRE(patch_out != NULL && byte_hidden_out != NULL,
                "blt_local_encoder_forward: patch_out and byte_hidden_out cannot be NULL");
    const size_t E = cfg.embed_dim;
    const size_t patch_dim = cfg.patch_dim == 0 ? E : cfg.patch_dim;
    BLT_REQUIRE(E > 0 && patch_dim % E == 0, "blt_local_encoder_forward: patch_dim must be a multiple of embed_dim");
    const size_t k = patch_dim / E;
    check_2d(patch_out, num_patches, patch_dim, "blt_local_encoder_forward: patch_out must be [num_patches, patch_dim] FP32");
    check_2d(byte_hidden_out, seq_len, E, "blt_local_encoder_forward: byte_hidden_out must be [seq_len, embed_dim] FP32");
    check_2d(&model->byte_embedding_weight, 256, E, "blt_local_encoder_forward: byte_embedding_weight must be [256, embed_dim]");
    BLT_REQUIRE(cfg.num_heads >= 1 && E % cfg.num_heads == 0 && (E / cfg.num_heads) % 2 == 0,
                "blt_local_encoder_forward: embed_dim must split into heads of even width");
    const size_t half = E / cfg.num_heads / 2;
    check_2d(&model->rope_cos_cache, 0, half, "blt_local_encoder_forward: rope caches must be [max_seq_len, head_dim/2]");
    check_2d(&model->rope_sin_cache, 0, half, "blt_local_encoder_forward: rope caches must be [max_seq_len, head_dim/2]");
    BLT_REQUIRE(model->rope_cos_cache.shape[0] >= seq_len && model->rope_sin_cache.shape[0] >= seq_len,
                "blt_local_encoder_forward: rope caches are shorter than the sequence");
    BLT_REQUIRE(model->layers != NULL && cfg.num_layers >= 1, "blt_local_encoder_forward: layers cannot be NULL");
    const blt_hash_ngram_config &ng = cfg.ngram_config;
    BLT_REQUIRE(ng.num_ngram_sizes <= BLT_MAX_NGRAM_SIZES && ng.embed_dim == E,
                "blt_local_encoder_forward: ngram_config does not fit the encoder");

    /* ---- byte rows with their n-grams, and P_0: pooled rows in every sub-token column block (local_encoder.c:237-245) ---- */
    /* The patches belong to the bytes and are part of a recording, so the bytes have to be, too: host bytes in a capture of the caller's
     * own are, device bytes would be read by the replay. */
    BLT_REQUIRE(!blt_stream_capturing(), "blt_local_encoder_forward: mask metadata cannot be staged while a graph capture is open");
    BLT_REQUIRE(bytes_in->backend != BLT_BACKEND_HIP || !blt_stream_captured_by_caller(),
                "blt_local_encoder_forward: a replay would read other bytes than the recorded patches belong to; record it with the bytes "
                "on the host");
    const size_t byte_shape[2] = {seq_len, E}, patch_shape[2] = {num_patches, patch_dim};
    EmbedArgs em;
    std::memset(&em, 0, offsetof(EmbedArgs, start));
    em.byte_table = (const float *)model->byte_embedding_weight.data;
    em.modulus = ng.per_ngram_vocab;
    for (size_t t = 0; t < ng.num_ngram_sizes; t++) {
        const size_t n = ng.ngram_sizes[t];
        if (n == 0 || n > seq_len) continue; /* hash_ngram.c:178-180 */
        check_2d(&model->ngram_weights.tables[t], ng.per_ngram_vocab, E, "blt_hash_ngram_forward: weights->tables");
        BLT_REQUIRE(n <= 8, "blt_rolling_hash_init: n must be in [1, 8]");
        BLT_REQUIRE(em.modulus > 1, "blt_rolling_hash_init: modulus must be > 1");
        BLT_REQUIRE(ng.hash_prime > 0 && ng.hash_prime <= ((UINT64_MAX - 255) / em.modulus),
                    "blt_rolling_hash_init: prime * modulus would overflow uint64");
        em.table[em.tables] = (const float *)model->ngram_weights.tables[t].data;
        em.ngram[em.tables++] = (uint32_t)n;
    }
    if (em.tables != 0) {
        em.power[0] = 1;
        for (int i = 1; i < 8; i++) em.power[i] = em.power[i - 1] * ng.hash_prime % em.modulus;
    }
    if (bytes_in->backend == BLT_BACKEND_HIP) {
        em.bytes = (const uint8_t *)bytes_in->data;
    } else if (seq_len <= EMBED_BYTES) {
        std::memcpy(em.text, bytes_in->data, seq_len);
    } else {
        uint8_t *dev = (uint8_t *)blt_arena_alloc(arena, seq_len, 64);
        blt_hip_memcpy_h2d(dev, bytes_in->data, seq_len);
        em.bytes = dev;
    }
    blt_tensor h = blt_tensor_create_uninit(arena, byte_shape, 2, BLT_DTYPE_FP32);
    blt_tensor p = blt_tensor_create_uninit(arena, patch_shape, 2, BLT_DTYPE_FP32);
    em.h = (float *)h.data, em.embed_dim = (uint32_t)E;
    em.scaled = ng.normalize ? 1 : 0, em.scale = 1.0f / (float)(ng.num_ngram_sizes + 1);
    em.out_stride = (uint32_t)patch_dim, em.copies = (uint32_t)k, em.take_max = cfg.pool_type == BLT_POOL_MAX ? 1 : 0;
    const bool tile = patches_tile(patches, num_patches, seq_len) && (cfg.pool_type == BLT_POOL_MEAN || cfg.pool_type == BLT_POOL_MAX);
    const size_t runs = tile ? num_patches : (seq_len + EMBED_ROWS - 1) / EMBED_ROWS;
    bool vec = E % 4 == 0 && (reinterpret_cast<uintptr_t>(em.byte_table) & 15u) == 0;
    for (uint32_t t = 0; t < em.tables; t++) vec = vec && (reinterpret_cast<uintptr_t>(em.table[t]) & 15u) == 0;
    for (size_t j0 = 0; j0 < runs; j0 += EMBED_RUNS) {
        const size_t n = std::min<size_t>(EMBED_RUNS, runs - j0);
        for (size_t j = 0; j < n; j++) em.start[j] = (uint32_t)(tile ? patches[j0 + j].start_idx : (j0 + j) * EMBED_ROWS);
        em.start[n] = (uint32_t)(j0 + n == runs ? seq_len : tile ? patches[j0 + n].start_idx : (j0 + n) * EMBED_ROWS);
        em.pooled = tile ? (float *)p.data + j0 * patch_dim : nullptr;
        const dim3 grid((unsigned)n, (unsigned)((E + EMBED_COLS - 1) / EMBED_COLS));
        blt_launch("embed_pool", vec ? embed_pool_kernel<true> : embed_pool_kernel<false>, grid, dim3(256), 0, blt_stream(), em);
    }
    HIP_CHECK_LAUNCH("blt_local_encoder_forward: embedding");
    if (!tile) pool_launch((const float *)h.data, seq_len, E, patches, num_patches, cfg.pool_type, (float *)p.data, patch_dim, k);

    /* ---- masks (local_encoder.c:52-113): host metadata ---- */
    std::vector<size_t> q_groups(num_patches), kv_groups(seq_len), q_groups_split;
    blt_patch_build_group_ids(patches, num_patches, seq_len, q_groups.data(), kv_groups.data());
    blt_mask_config local_mask, cross_mask;
    std::memset(&local_mask, 0, sizeof(local_mask));
    std::memset(&cross_mask, 0, sizeof(cross_mask));
    local_mask.seq_len_q = local_mask.seq_len_kv = seq_len;
    local_mask.sliding_window = cfg.local_window;
    local_mask.doc_boundaries = doc_boundaries;
    local_mask.num_docs = num_docs;
    local_mask.is_causal = true;
    cross_mask.seq_len_q = num_patches * k;
    cross_mask.seq_len_kv = seq_len;
    cross_mask.kv_group_ids = kv_groups.data();
    cross_mask.bidirectional_within_group = true;
    if (k == 1) {
        cross_mask.query_group_ids = q_groups.data();
    } else {
        q_groups_split.resize(num_patches * k);
        blt_patch_expand_group_ids(q_groups.data(), num_patches, k, q_groups_split.data());
        cross_mask.query_group_ids = q_groups_split.data();
    }
    blt_tensor cos_view = view_2d(model->rope_cos_cache.data, seq_len, half);
    blt_tensor sin_view = view_2d(model->rope_sin_cache.data, seq_len, half);

    blt_transformer_config layer_cfg;
    std::memset(&layer_cfg, 0, sizeof(layer_cfg));
    layer_cfg.attn_config.embed_dim = E;
    layer_cfg.attn_config.num_heads = cfg.num_heads;
    layer_cfg.attn_config.is_causal = true;
    layer_cfg.attn_config.use_rope = true;
    layer_cfg.attn_config.rope_theta = cfg.rope_theta;
    layer_cfg.attn_config.rope_cos_cache = &cos_view;
    layer_cfg.attn_config.rope_sin_cache = &sin_view;
    layer_cfg.attn_config.mask_config = &local_mask;
    layer_cfg.hidden_dim = cfg.hidden_dim;
    layer_cfg.norm_type = BLT_NORM_RMSNORM;
    layer_cfg.activation_type = BLT_ACTIVATION_SWIGLU;
    blt_cross_attention_config cross_cfg;
    std::memset(&cross_cfg, 0, sizeof(cross_cfg));
    cross_cfg.embed_dim = E;
    cross_cfg.patch_dim = patch_dim;
    cross_cfg.split_mode = k == 1 ? BLT_CROSS_ATTN_NO_SPLIT : BLT_CROSS_ATTN_SPLIT_QUERY;
    cross_cfg.num_heads = cfg.cross_attn_heads;
    cross_cfg.mask_config = &cross_mask;

    /* ---- layers; the last results land in the caller's tensors ---- */
    /* A layer's cross block takes nothing from the next layer and gives nothing to it: but for the last one it goes along with that
     * layer's launches.  512 bytes through an encoder and a decoder of two layers of 128 columns with four patch layers between them, us: with
     * the decoder's keys in pairs 240 -> 230, three layers each 256 -> 239. */
    CrossPass cross_pass;
    CrossLater later;
    size_t last_cross = cfg.num_layers; /* none */
    for (size_t l = 0; l < cfg.num_layers; l++)
        if (blt_local_cross_attn_fires(cfg.cross_attn_placement, cfg.cross_attn_all_layers, cfg.num_layers, l)) last_cross = l;
    for (size_t l = 0; l < cfg.num_layers; l++) {
        const blt_local_layer_storage *s = &model->layers[l];
        blt_transformer_weights w;
        std::memset(&w, 0, sizeof(w));
        w.norm1_weight = &s->norm1_weight, w.attn_qkv_w = &s->attn_qkv_w, w.attn_proj_w = &s->attn_proj_w;
        w.norm2_weight = &s->norm2_weight, w.ffn_up_w = &s->ffn_up_w, w.ffn_gate_w = &s->ffn_gate_w;
        w.ffn_down_w = &s->ffn_down_w;
        blt_tensor h_next = l + 1 == cfg.num_layers ? view_2d(byte_hidden_out->data, seq_len, E)
                                                    : blt_tensor_create_uninit(arena, byte_shape, 2, BLT_DTYPE_FP32);
        blt_transformer_run(&h, &w, &h_next, &layer_cfg, arena, &later);
        h = h_next;
        if (!blt_local_cross_attn_fires(cfg.cross_attn_placement, cfg.cross_attn_all_layers, cfg.num_layers, l)) continue;

        /* P_{l+1} = P_l + cross(RMSNorm(P_l), h) (local_encoder.c:255-272), the norm inside the query
         * projection and the sum in the epilogue of the output projection: three launches */
        blt_tensor p_rows = view_2d(p.data, num_patches * k, E);
        blt_cross_attention_weights xw;
        xw.weight_q = &s->cross_weight_q, xw.weight_k = &s->cross_weight_k, xw.weight_v = &s->cross_weight_v;
        xw.weight_proj = &s->cross_weight_proj;
        blt_tensor p_next = l == last_cross ? view_2d(patch_out->data, num_patches, patch_dim)
                                            : blt_tensor_create_uninit(arena, patch_shape, 2, BLT_DTYPE_FP32);
        blt_tensor next_rows = view_2d(p_next.data, num_patches * k, E);
        cross_pass.later = l + 1 < cfg.num_layers ? &later : nullptr;
        blt_cross_attention_run(&p_rows, &h, &xw, &next_rows, &cross_cfg, arena,
                                (const float *)s->cross_norm_weight.data, (const float *)p.data, &cross_pass);
        p = p_next;
    }
    if (last_cross == cfg.num_layers) /* no cross block fired: P_0 is the result */
        blt_strided_copy_hip(BLT_BACKEND_HIP, (float *)patch_out->data, num_patches * patch_dim, (const float *)p.data,
                             num_patches * patch_dim, 1, num_patches * patch_dim);
    /* the host index arrays of the masks are consumed by the calls above (ranges are staged, dense
     * masks are built before the attention launch is issued): nothing outlives this call */
}

/*
 * blt_local_decoder_forward_ext without D_0 options and loss (reference: csrc/models/
 * local_decoder.c:233-351).  D_0 is byte_hidden_in itself; per layer B = D + cross(RMSNorm(D),
 * patch sub-tokens) where the cross block fires (norm inside the query projection, sum in the
 * output projection's epilogue: three launches), D = byte block(B) under the causal, windowed,
 * per-document mask (five launches); logits = D_final * lm_head.  A byte reads the latent the
 * paper's rule gives it (blt_patch_decoder_latent_at, the last byte of the window its own patch's
 * when trailing_closed): one sub-token group per row, so the cross mask travels as key ranges.
 */
extern "C" void blt_local_decoder_forward_ext_hip(const blt_local_decoder *model, const blt_tensor *byte_hidden_in,
                                                  const blt_tensor *patch_in, const blt_patch_info *patches,
                                                  size_t num_patches, const size_t *doc_boundaries, size_t num_docs,
                                                  int trailing_closed, blt_tensor *logits_out, blt_arena *arena) {
    BLT_REQUIRE(model != NULL && byte_hidden_in != NULL && patch_in != NULL && patches != NULL && arena != NULL,
                "blt_local_decoder_forward_ext: model, byte_hidden_in, patch_in, patches and arena cannot be NULL");
    BLT_REQUIRE(logits_out != NULL, "blt_local_decoder_forward_ext: logits_out cannot be NULL");
    BLT_REQUIRE(arena->backend == BLT_BACKEND_HIP, "blt_local_decoder_forward_ext: HIP implementation needs a device arena");
    const blt_local_decoder_config &cfg = model->config;
    const size_t E = cfg.embed_dim, V = cfg.vocab_size;
    BLT_REQUIRE(cfg.num_heads != 0 && E % cfg.num_heads == 0 && (E / cfg.num_heads) % 2 == 0,
                "blt_local_decoder_forward_ext: embed_dim / num_heads must be an even head width");
    BLT_REQUIRE(byte_hidden_in->ndim == 2 && byte_hidden_in->dtype == BLT_DTYPE_FP32 && byte_hidden_in->shape[1] == E &&
                    byte_hidden_in->backend == BLT_BACKEND_HIP,
                "blt_local_decoder_forward_ext: byte_hidden_in must be [seq_len, embed_dim] FP32");
    const size_t seq_len = byte_hidden_in->shape[0];
    BLT_REQUIRE(seq_len >= 1 && seq_len <= cfg.max_seq_len,
                "blt_local_decoder_forward_ext: seq_len must be in [1, max_seq_len]");
    BLT_REQUIRE(num_patches >= 1, "blt_local_decoder_forward_ext: num_patches must be >= 1");
    const size_t patch_dim = cfg.patch_dim == 0 ? E : cfg.patch_dim;
    BLT_REQUIRE(patch_dim % E == 0, "blt_local_decoder_forward_ext: patch_dim must be a multiple of embed_dim");
    const size_t k = patch_dim / E, half = E / cfg.num_heads / 2;
    check_2d(patch_in, num_patches, patch_dim, "blt_local_decoder_forward_ext: patch_in must be [num_patches, patch_dim] FP32");
    check_2d(logits_out, seq_len, V, "blt_local_decoder_forward_ext: logits_out must be [seq_len, vocab_size] FP32");
    check_2d(&model->lm_head_weight, E, V, "blt_local_decoder_forward_ext: lm_head_weight must be [embed_dim, vocab_size] FP32");
    check_2d(&model->rope_cos_cache, cfg.max_seq_len, half, "blt_local_decoder_forward_ext: rope_cos_cache");
    check_2d(&model->rope_sin_cache, cfg.max_seq_len, half, "blt_local_decoder_forward_ext: rope_sin_cache");
    size_t covered = 0;
    for (size_t j = 0; j < num_patches; j++) { /* patches tile [0, seq_len) (patch_pool_cpu.c:98-118) */
        BLT_REQUIRE(patches[j].start_idx == covered && patches[j].length >= 1,
                    "blt_local_decoder_forward_ext: patches must tile the window without gaps");
        covered += patches[j].length;
    }
    BLT_REQUIRE(covered == seq_len, "blt_local_decoder_forward_ext: patches must tile [0, seq_len) exactly");

    /* ---- masks (local_decoder.c:64-121): host metadata ---- */
    std::vector<size_t> byte_groups(seq_len), kv_groups(num_patches * k);
    for (size_t i = 0; i < seq_len; i++) byte_groups[i] = blt_patch_decoder_latent_at(patches, num_patches, i);
    if (trailing_closed) byte_groups[seq_len - 1] = num_patches - 1;
    for (size_t j = 0; j < num_patches * k; j++) kv_groups[j] = j / k;
    blt_mask_config local_mask, cross_mask;
    std::memset(&local_mask, 0, sizeof(local_mask));
    std::memset(&cross_mask, 0, sizeof(cross_mask));
    local_mask.seq_len_q = local_mask.seq_len_kv = seq_len;
    local_mask.sliding_window = cfg.local_window;
    local_mask.doc_boundaries = doc_boundaries;
    local_mask.num_docs = num_docs;
    local_mask.is_causal = true;
    cross_mask.seq_len_q = seq_len;
    cross_mask.seq_len_kv = num_patches * k;
    cross_mask.query_group_ids = byte_groups.data();
    cross_mask.kv_group_ids = kv_groups.data();
    cross_mask.bidirectional_within_group = true;
    blt_tensor cos_view = view_2d(model->rope_cos_cache.data, seq_len, half);
    blt_tensor sin_view = view_2d(model->rope_sin_cache.data, seq_len, half);
    blt_transformer_config layer_cfg;
    std::memset(&layer_cfg, 0, sizeof(layer_cfg));
    layer_cfg.attn_config.embed_dim = E;
    layer_cfg.attn_config.num_heads = cfg.num_heads;
    layer_cfg.attn_config.is_causal = true;
    layer_cfg.attn_config.use_rope = true;
    layer_cfg.attn_config.rope_theta = cfg.rope_theta;
    layer_cfg.attn_config.rope_cos_cache = &cos_view;
    layer_cfg.attn_config.rope_sin_cache = &sin_view;
    layer_cfg.attn_config.mask_config = &local_mask;
    layer_cfg.hidden_dim = cfg.hidden_dim;
    layer_cfg.norm_type = BLT_NORM_RMSNORM;
    layer_cfg.activation_type = BLT_ACTIVATION_SWIGLU;
    blt_cross_attention_config cross_cfg;
    std::memset(&cross_cfg, 0, sizeof(cross_cfg));
    cross_cfg.embed_dim = E;
    cross_cfg.patch_dim = patch_dim;
    cross_cfg.split_mode = k == 1 ? BLT_CROSS_ATTN_NO_SPLIT : BLT_CROSS_ATTN_SPLIT_KV;
    cross_cfg.num_heads = cfg.cross_attn_heads;
    cross_cfg.mask_config = &cross_mask;

    /* ---- layers ---- */
    CrossPass cross_pass;
    CrossLater first; /* a layer's cross block, for the launch of its QKV product */
    first.feeds = true;
    cross_pass.later = &first;
    const size_t byte_shape[2] = {seq_len, E};
    blt_tensor latents = view_2d(patch_in->data, num_patches * k, E);
    blt_tensor d = view_2d(byte_hidden_in->data, seq_len, E);
    for (size_t l = 0; l < cfg.num_layers; l++) {
        blt_local_layer_storage *s = &model->layers[l];
        blt_tensor b = d;
        if (blt_local_cross_attn_fires(cfg.cross_attn_placement, cfg.cross_attn_all_layers, cfg.num_layers, l)) {
            blt_cross_attention_weights xw;
            xw.weight_q = &s->cross_weight_q, xw.weight_k = &s->cross_weight_k, xw.weight_v = &s->cross_weight_v;
            xw.weight_proj = &s->cross_weight_proj;
            b = blt_tensor_create_uninit(arena, byte_shape, 2, BLT_DTYPE_FP32);
            /* every layer's keys and values come from the same latents: those of two layers in one launch */
            cross_pass.next_k = cross_pass.next_v = nullptr;
            for (size_t n = l + 1; n < cfg.num_layers && cross_pass.next_k == nullptr; n++)
                if (blt_local_cross_attn_fires(cfg.cross_attn_placement, cfg.cross_attn_all_layers, cfg.num_layers, n))
                    cross_pass.next_k = &model->layers[n].cross_weight_k, cross_pass.next_v = &model->layers[n].cross_weight_v;
            blt_cross_attention_run(&d, &latents, &xw, &b, &cross_cfg, arena, (const float *)s->cross_norm_weight.data,
                                    (const float *)d.data, &cross_pass);
        }
        blt_transformer_weights w;
        std::memset(&w, 0, sizeof(w));
        w.norm1_weight = &s->norm1_weight, w.norm2_weight = &s->norm2_weight;
        w.attn_qkv_w = &s->attn_qkv_w, w.attn_proj_w = &s->attn_proj_w;
        w.ffn_up_w = &s->ffn_up_w, w.ffn_gate_w = &s->ffn_gate_w, w.ffn_down_w = &s->ffn_down_w;
        blt_tensor d_next = blt_tensor_create_uninit(arena, byte_shape, 2, BLT_DTYPE_FP32);
        blt_transformer_run(&b, &w, &d_next, &layer_cfg, arena, &first);
        d = d_next;
    }
    blt_matmul_hip(&d, &model->lm_head_weight, logits_out);
}
