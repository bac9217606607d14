"""The calls a byte-level language model's host program makes on this library, as timed cases.

`listed()` names twelve of them, `draw(rng)` gives more of the same ranges, `prepare` makes what the
program holds before the call (inputs on the GPU, weights, cache, plan, work arena), `run` makes the
call, `work` says what it cannot do without and `tolerance` how far another correct fp32
implementation may be off.  Everything is fp32, the only compute type of the library.

Kinds, each an entry point (or the two or three that belong together) of include/blt_hip.h:

  heads   blt_build_attention_mask, then one blt_attention_head_core per head with the dense mask and
          weights_out: what an unchanged caller of the per-head op issues for one sequence
  attn    blt_attention_plan_run_hip: causal self-attention of a batch of sequences
  cross   the same for patch queries over the bytes of their own patch (row ranges)
  kv      the attention of a KV-cache step for a batch: one new row each (decode), a chunk or a
          block (verify); lengths on the host or on the device, rows rotated before or inside
  step    blt_kv_decode_step / _batched_hip: the whole decoder step, one new row each (decode), a few
          (verify of a draft) or, from an empty cache, a whole prompt with its patches
  draft   blt_kv_block_step_hip: one denoising pass of a block of masked rows over a cached prefix
  model   blt_local_encoder_forward, blt_transformer_forward per layer, blt_local_decoder_forward_ext:
          the whole inference forward of one byte window
  block   blt_transformer_forward: one layer of the patch transformer over packed documents
"""
import ctypes as C
import math

import numpy as np
import torch

from fblt_amd import abi, api, decoder, encoder

VOCAB = 256           # byte logits
NGRAMS = (3, 4, 5)    # hashed n-gram tables of the encoder
NGRAM_VOCAB = 2048
THETA = 500000.0
MB = 1 << 20


def listed():
    return [
        # an unchanged per-head caller at the local decoder's window: 512 bytes, 4 heads
        {"name": "heads_512", "kind": "heads", "T": 512, "H": 4, "hd": 32},
        # patch transformer's self-attention: 16 windows of 128 patches
        {"name": "attn_patches", "kind": "attn", "batch": 16, "T": 128, "H": 8, "hd": 64, "window": 0},
        # long byte windows in one batch, the largest prefill: compute bound
        {"name": "attn_long", "kind": "attn", "batch": 8, "T": 4096, "H": 4, "hd": 32, "window": 0},
        # local encoder's cross-attention: 16 windows of 512 bytes in 128 patches
        {"name": "cross_patches", "kind": "cross", "batch": 16, "T": 512, "P": 128, "H": 4, "hd": 32},
        # serving: one new byte for each of 128 sequences over long caches, bandwidth bound
        {"name": "kv_decode_long", "kind": "kv", "batch": 128, "n": 1, "len_lo": 1024, "len_hi": 2032, "H": 4, "hd": 32,
         "block": False, "lens": "host", "rope": False, "window": 0},
        # verify of an 8-row block for 64 sequences
        {"name": "kv_verify_8", "kind": "kv", "batch": 64, "n": 8, "len_lo": 64, "len_hi": 508, "H": 4, "hd": 32,
         "block": True, "lens": "device", "rope": False, "window": 0},
        # interactive generation: the next byte of one sequence, the smallest whole step
        {"name": "step_one", "kind": "step", "batch": 1, "n": 1, "len_lo": 356, "len_hi": 356, "E": 128, "H": 4,
         "hidden": 512, "L": 2, "window": 0},
        # serving: the next byte of 64 sequences
        {"name": "step_batch", "kind": "step", "batch": 64, "n": 1, "len_lo": 1, "len_hi": 512, "E": 128, "H": 4,
         "hidden": 512, "L": 2, "window": 0},
        # the prompt: 512 bytes into an empty cache
        {"name": "step_prompt", "kind": "step", "batch": 1, "n": 512, "len_lo": 0, "len_hi": 0, "E": 128, "H": 4,
         "hidden": 512, "L": 2, "window": 0},
        # one denoising pass of a block of 16
        {"name": "draft_16", "kind": "draft", "R": 16, "N": 356, "E": 128, "H": 4, "hidden": 512, "L": 2},
        # one byte window through encoder, patch transformer and decoder
        {"name": "model_512", "kind": "model", "T": 512, "E": 128, "H": 4, "hidden": 512, "L": 2, "G": 4, "docs": 1,
         "window": 0, "bytes": "host"},
        # a wide patch-transformer layer over eight packed documents
        {"name": "block_2048", "kind": "block", "T": 2048, "E": 512, "H": 8, "hidden": 2048, "docs": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["heads", "attn", "attn", "cross", "kv", "kv", "step", "step", "step", "draft", "model", "block"])
    H, hd = rng.randint(1, 8), rng.choice([32, 64])
    E, heads = rng.choice([(64, 2), (128, 4), (128, 4), (256, 8), (256, 4)])
    if kind == "heads":
        return {"kind": kind, "T": _log(rng, 16, 1024), "H": H, "hd": hd}
    if kind == "attn":
        T = _log(rng, 32, 4096)
        most = int(3.2e10 // (2.0 * hd * H * T * T))     # no more arithmetic than the largest listed case
        return {"kind": kind, "batch": max(1, min(most, _log(rng, 1, 64))), "T": T, "H": H, "hd": hd,
                "window": T // 4 if rng.random() < 0.25 else 0}
    if kind == "cross":
        T = _log(rng, 64, 2048)
        return {"kind": kind, "batch": _log(rng, 1, 64), "T": T, "P": max(16, T // rng.randint(3, 5)), "H": H, "hd": hd}
    if kind == "kv":
        n = 1 if rng.random() < 0.5 else rng.randint(2, 32)
        hi = _log(rng, 16, 2032)
        batch = max(1, min(_log(rng, 1, 256), int(2.5e8 // (8 * H * hd * hi))))
        return {"kind": kind, "batch": batch, "n": n, "len_lo": max(1, hi // rng.choice([1, 2, 8])), "len_hi": hi, "H": H,
                "hd": hd, "block": n > 1 and rng.random() < 0.6, "lens": rng.choice(["host", "device"]),
                "rope": rng.random() < 0.5, "window": hi // 2 if rng.random() < 0.2 else 0}
    if kind == "step":
        form = rng.choice(["one", "batch", "prompt"])
        c = {"kind": kind, "E": E, "H": heads, "hidden": 4 * E, "L": rng.randint(1, 4), "window": 0}
        if form == "prompt":
            return dict(c, batch=1, n=_log(rng, 16, 1024), len_lo=0, len_hi=0, window=128 if rng.random() < 0.25 else 0)
        hi = _log(rng, 16, 1024)
        return dict(c, batch=1 if form == "one" else _log(rng, 2, 64), n=1 if rng.random() < 0.7 else rng.randint(2, 16),
                    len_lo=hi if form == "one" else max(1, hi // 8), len_hi=hi)
    if kind == "draft":
        return {"kind": kind, "R": rng.randint(2, 32), "N": _log(rng, 16, 1024), "E": E, "H": heads, "hidden": 4 * E,
                "L": rng.randint(1, 4)}
    if kind == "model":
        return {"kind": kind, "T": _log(rng, 32, 1024), "E": E, "H": heads, "hidden": 4 * E, "L": rng.randint(1, 3),
                "G": rng.randint(1, 6), "docs": rng.randint(1, 3), "window": 64 if rng.random() < 0.25 else 0,
                "bytes": rng.choice(["host", "device"])}
    E, heads = rng.choice([(128, 4), (256, 8), (256, 4), (512, 8)])
    return {"kind": kind, "T": _log(rng, 16, 2048), "E": E, "H": heads, "hidden": 4 * E, "docs": rng.randint(1, 8)}


# ---- what the program holds ------------------------------------------------------------------------

class _State:
    """What one kind's preparation leaves behind; `call()` is the timed pass (it holds no reference to
    the state, so that dropping the state gives its memory back at once)."""

    def __init__(self, seed):
        self.lib = api.load()
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.rs = np.random.RandomState(seed % (1 << 31))
        self.keep, self.arenas, self.plan, self.call = [], [], None, None

    def randn(self, *shape, scale=1.0):
        return torch.randn(*shape, generator=self.gen, device="cuda", dtype=torch.float32) * scale

    def arena(self, nbytes):
        a = self.lib.blt_arena_create(nbytes, abi.BLT_BACKEND_HIP)
        self.arenas.append(a)
        return a

    def view(self, t, dtype=abi.BLT_DTYPE_FP32):
        self.keep.append(t)
        return abi.tensor_view(t.data_ptr(), tuple(t.shape), abi.BLT_BACKEND_HIP, dtype=dtype)

    def rope(self, positions, hd):
        """Device rotation tables as blt_rope_precompute fills them."""
        cos, sin = (torch.zeros(positions, hd // 2, device="cuda") for _ in range(2))
        vc, vs = self.view(cos), self.view(sin)
        self.lib.blt_rope_precompute(positions, C.byref(abi.BltRopeConfig(THETA, hd)), C.byref(vc), C.byref(vs))
        return cos, sin, vc, vs

    def patch_lengths(self, total, count=None):
        """Geometric patch lengths (mean 4, 1..16) that tile `total` bytes, `count` of them if given."""
        if count is None:
            lens = []
            while sum(lens) < total:
                lens.append(min(int(np.clip(self.rs.geometric(0.25), 1, 16)), total - sum(lens)))
            return lens
        lens = np.clip(self.rs.geometric(0.25, size=count), 1, 16)
        while lens.sum() != total:
            i = self.rs.randint(count)
            lens[i] = np.clip(lens[i] + (1 if lens.sum() < total else -1), 1, 16)
        return lens.tolist()

    def __del__(self):
        if self.plan is not None:
            self.lib.blt_attention_plan_destroy_hip(self.plan)
        for a in self.arenas:
            self.lib.blt_arena_destroy(a)


def _scale(hd):
    return float(np.float32(1.0) / np.sqrt(np.float32(hd)))


def _packed_heads(qkv, out, batch, T, H, hd, weights=None):
    """blt_attention_head_args of every (sequence, head) of packed [batch*T, 3E] rows."""
    E = H * hd
    return [api.head_args(qkv.data_ptr() + 4 * (b * T * 3 * E + h * hd), qkv.data_ptr() + 4 * (b * T * 3 * E + E + h * hd),
                          qkv.data_ptr() + 4 * (b * T * 3 * E + 2 * E + h * hd), out.data_ptr() + 4 * b * T * E, T, T, hd,
                          _scale(hd), 3 * E, 3 * E, 3 * E, E, h * hd, weights=weights) for b in range(batch)
            for h in range(H)]


def _heads(s, c):
    lib = s.lib
    T, H, hd = c["T"], c["H"], c["hd"]
    qkv, out = s.randn(T, 3 * H * hd), torch.zeros(T, H * hd, device="cuda")
    weights = torch.zeros(T, T, device="cuda")   # one score matrix, every head's in turn
    s.keep += [qkv, out, weights]
    arena = s.arena(4 * T * T + MB)
    cfg = abi.BltMaskConfig()
    cfg.seq_len_q = cfg.seq_len_kv = T
    cfg.is_causal = True
    args, mask = _packed_heads(qkv, out, 1, T, H, hd, weights.data_ptr()), abi.BltTensor()
    refs = [C.byref(a) for a in args]

    def call():
        arena.contents.offset = 0
        lib.blt_build_attention_mask(C.byref(cfg), C.byref(mask), arena)
        for a, ref in zip(args, refs):
            a.mask = mask.data
            lib.blt_attention_head_core(abi.BLT_BACKEND_HIP, ref)
        return out, weights
    return call


def _attn(s, c):
    lib = s.lib
    batch, T, H, hd = c["batch"], c["T"], c["H"], c["hd"]
    qkv, out = s.randn(batch * T, 3 * H * hd), torch.zeros(batch * T, H * hd, device="cuda")
    s.keep += [qkv, out]
    probs = [api.problem(a, api.BLT_ATTN_MASK_CAUSAL, 0, c["window"]) for a in _packed_heads(qkv, out, batch, T, H, hd)]
    plan = s.plan = lib.blt_attention_plan_create_hip(api.problem_array(probs), len(probs))

    def call():
        lib.blt_attention_plan_run_hip(plan)
        return out
    return call


def _cross(s, c):
    lib = s.lib
    batch, T, P, H, hd = c["batch"], c["T"], c["P"], c["H"], c["hd"]
    E = H * hd
    q, k, v = s.randn(batch * P, E), s.randn(batch * T, E), s.randn(batch * T, E)
    out = torch.zeros(batch * P, E, device="cuda")
    lens = np.stack([s.patch_lengths(T, P) for _ in range(batch)])
    hi = np.cumsum(lens, axis=1).astype(np.int32)
    lo = (hi - lens).astype(np.int32)
    lo, hi = torch.from_numpy(lo).cuda(), torch.from_numpy(hi).cuda()
    s.keep += [q, k, v, out, lo, hi]
    probs = []
    for b in range(batch):
        for h in range(H):
            a = api.head_args(q.data_ptr() + 4 * (b * P * E + h * hd), k.data_ptr() + 4 * (b * T * E + h * hd),
                              v.data_ptr() + 4 * (b * T * E + h * hd), out.data_ptr() + 4 * b * P * E, P, T, hd, _scale(hd), E,
                              E, E, E, h * hd)
            probs.append(api.problem(a, api.BLT_ATTN_MASK_ROW_RANGE, row_lo=lo.data_ptr() + 4 * b * P,
                                     row_hi=hi.data_ptr() + 4 * b * P, row_span=16))
    plan = s.plan = lib.blt_attention_plan_create_hip(api.problem_array(probs), len(probs))

    def call():
        lib.blt_attention_plan_run_hip(plan)
        return out
    return call


def _kv(s, c):
    lib = s.lib
    batch, n, H, hd = c["batch"], c["n"], c["H"], c["hd"]
    E, max_len = H * hd, c["len_hi"] + 32
    lens = s.rs.randint(c["len_lo"], c["len_hi"] + 1, size=batch).astype(np.uint32)
    ck, cv = s.randn(batch * max_len, E), s.randn(batch * max_len, E)
    q, k, v = (s.randn(batch * n, E) for _ in range(3))
    out, dev_lens = torch.zeros(batch * n, E, device="cuda"), torch.from_numpy(lens.astype(np.int32)).cuda()
    s.keep += [ck, cv, q, k, v, out, lens, dev_lens]
    cache = api.BltKvAttnCache(ck.data_ptr(), cv.data_ptr(), dev_lens.data_ptr(), batch, max_len, E, H, c["window"])
    ref, kind = C.byref(cache), api.BLT_KV_STEP_BLOCK if c["block"] else api.BLT_KV_STEP_CAUSAL
    cos = sin = None
    if c["rope"]:
        cos, sin = (t.data_ptr() for t in s.rope(max_len, hd)[:2])
    rows = (q.data_ptr(), E, k.data_ptr(), E, v.data_ptr(), E)
    hint = int(lens.max()) + n
    if c["lens"] == "host":
        args = (ref, lens.ctypes.data_as(C.POINTER(C.c_uint32))) + rows + (cos, sin, max_len if c["rope"] else 0,
                                                                             out.data_ptr(), E, n, kind)
        fn = lib.blt_kv_attend_step_lens_hip
    elif c["rope"]:
        args = (ref,) + rows + (cos, sin, max_len, out.data_ptr(), E, n, kind, 0, hint)
        fn = lib.blt_kv_rope_attend_step_hip
    else:
        args = (ref,) + rows + (out.data_ptr(), E, n, kind, 0, hint)
        fn = lib.blt_kv_attend_step_hip

    def call():
        fn(*args)
        return out, ck, cv
    return call


class _Decoder:
    """A local decoder's weights and its two-tier cache over device tensors."""

    def __init__(self, s, c, max_len, batch):
        E, H, L = c["E"], c["H"], c["L"]
        self.max_len, self.batch = max_len, batch
        w = decoder.random_weights(E, c["hidden"], L, VOCAB, int(s.rs.randint(1 << 30)))
        cos, sin = (t.cpu().numpy() for t in s.rope(max_len, E // H)[:2])
        self.bound = decoder.bind(w, cos, sin, abi.BLT_BACKEND_HIP, decoder.device_place, E, H, H, c["hidden"], VOCAB, max_len,
                                  window=c.get("window", 0))
        self.tiers = {n: [s.randn(batch * max_len, E) for _ in range(L)] for n in ("self_k", "self_v", "cross_k", "cross_v")}
        self.handles = {n: (abi.BltTensor * L)(*(s.view(t) for t in ts)) for n, ts in self.tiers.items()}
        self.patch_table = (abi.BltPatchInfo * (batch * max_len))()
        self.cache = abi.BltKvCache()
        self.cache.decoder = self.bound.ptr
        self.cache.max_seq_len, self.cache.batch_size, self.cache.max_subtokens = max_len, batch, max_len
        self.cache.embed_dim, self.cache.k, self.cache.patch_dim = E, 1, E
        for n, h in self.handles.items():
            setattr(self.cache, n, C.cast(h, C.POINTER(abi.BltTensor)))
        self.cache.cached_patches = C.cast(self.patch_table, C.POINTER(abi.BltPatchInfo))
        self.ref = C.byref(self.cache)
        s.keep += [self.bound, self.tiers, self.handles, self.patch_table]

    def slabs(self):
        return [t for n in ("self_k", "self_v") for t in self.tiers[n]]


def _step(s, c):
    lib = s.lib
    batch, n, E = c["batch"], c["n"], c["E"]
    d = _Decoder(s, c, c["len_hi"] + n + 8, batch)
    lens = s.rs.randint(c["len_lo"], c["len_hi"] + 1, size=batch)
    x, logits = s.randn(batch * n, E), torch.zeros(batch * n, VOCAB, device="cuda")
    vx, vl = s.view(x), s.view(logits)
    work = s.arena(64 * MB + 64 * batch * n * (4 * E + c["hidden"]))
    outs = [logits] + d.slabs()
    lengths = [s.patch_lengths(int(v) + n) for v in lens]
    tables = [decoder.patch_table(p) for p in lengths]
    if batch == 1:
        pin = s.randn(len(lengths[0]), E)
        vp, P, base = s.view(pin), len(lengths[0]), int(lens[0])
        lib.blt_kv_cache_refresh_cross(d.ref, C.byref(vp), tables[0], P, 0, work)

        def call():
            work.contents.offset = 0
            # back to the prefix, as after a rejected draft; a prompt brings its patches along
            lib.blt_kv_cache_truncate(d.ref, base, P if base else 0)
            if not base:
                lib.blt_kv_cache_refresh_cross(d.ref, C.byref(vp), tables[0], P, 0, work)
            lib.blt_kv_decode_step(d.ref, C.byref(vp), tables[0], P, C.byref(vx), 0, C.byref(vl), work)
            return outs
        d.cache.self_len = base
        return call
    for b in range(batch):
        vp = s.view(s.randn(len(lengths[b]), E))
        lib.blt_kv_cache_refresh_cross_seq_hip(d.ref, b, C.byref(vp), tables[b], len(lengths[b]), 0, work)
        work.contents.offset = 0
    ptrs = (C.POINTER(abi.BltPatchInfo) * batch)(*(C.cast(t, C.POINTER(abi.BltPatchInfo)) for t in tables))
    num, self_len = abi.size_array([len(p) for p in lengths]), abi.size_array(lens)
    base = bytes(self_len)
    s.keep += [tables, ptrs, num]

    def call():
        work.contents.offset = 0
        C.memmove(self_len, base, len(base))
        lib.blt_kv_decode_step_batched_hip(d.ref, self_len, ptrs, num, None, C.byref(vx), C.byref(vl), work)
        return outs
    return call


def _draft(s, c):
    lib = s.lib
    R, N, E = c["R"], c["N"], c["E"]
    d = _Decoder(s, c, N + 40, 1)
    lengths = s.patch_lengths(N)
    P, patches = len(lengths), decoder.patch_table(lengths)
    vp, work = s.view(s.randn(P, E)), s.arena(96 * MB)
    lib.blt_kv_cache_refresh_cross(d.ref, C.byref(vp), patches, P, 0, work)
    d.cache.self_len = N
    tokens = [int(t) if u < 0.5 else abi.BLT_MASK_TOKEN_ID for t, u in zip(s.rs.randint(0, 256, R), s.rs.rand(R))]
    batch = decoder.BlockBatch(N, R, P, tokens=tokens)
    logits = torch.zeros(R, VOCAB, device="cuda")
    vl, outs = s.view(logits), [logits] + d.slabs()
    s.keep += [batch, patches]
    bref = batch.ptr

    def call():
        work.contents.offset = 0
        lib.blt_kv_block_step_hip(d.ref, P, bref, abi.BLT_D0_LEARNED, C.byref(vl), work)
        return outs
    return call


def _doc_starts(T, docs):
    """Starts of documents 1, 2, ... of `docs` nearly equal ones over T rows."""
    return [T * d // docs for d in range(1, docs) if 0 < T * d // docs < T]


def _transformer(s, T, E, H, hidden, docs, layers):
    """Weights of `layers` blocks and their configuration: rotary attention, causal within documents."""
    cos, sin, vc, vs = s.rope(T, E // H)
    mc = abi.BltMaskConfig()
    mc.seq_len_q = mc.seq_len_kv = T
    mc.is_causal = True
    if docs:
        bounds = abi.size_array(docs)
        mc.doc_boundaries, mc.num_docs = bounds, len(docs) + 1
        s.keep.append(bounds)
    ac = abi.BltAttentionConfig()
    ac.embed_dim, ac.num_heads, ac.head_dim, ac.is_causal = E, H, E // H, True
    ac.use_rope, ac.rope_theta = True, THETA
    ac.rope_cos_cache, ac.rope_sin_cache, ac.mask_config = C.pointer(vc), C.pointer(vs), C.pointer(mc)
    cfg = abi.BltTransformerConfig()
    cfg.attn_config = ac
    cfg.hidden_dim, cfg.norm_type, cfg.activation_type = hidden, abi.BLT_NORM_RMSNORM, abi.BLT_ACTIVATION_SWIGLU
    weights = []
    for _ in range(layers):
        t = [1 + s.randn(E, scale=0.1), s.randn(E, 3 * E, scale=E ** -0.5), s.randn(E, E, scale=E ** -0.5),
             1 + s.randn(E, scale=0.1), s.randn(E, hidden, scale=E ** -0.5), s.randn(E, hidden, scale=E ** -0.5),
             s.randn(hidden, E, scale=hidden ** -0.5)]
        v = [s.view(x) for x in t]
        w = abi.BltTransformerWeights()
        w.norm1_weight, w.attn_qkv_w, w.attn_proj_w, w.norm2_weight = (C.pointer(x) for x in v[:4])
        w.ffn_up_w, w.ffn_gate_w, w.ffn_down_w = (C.pointer(x) for x in v[4:])
        s.keep.append(v)
        weights.append(w)
    s.keep += [vc, vs, mc, ac]
    return cfg, weights


def _block(s, c):
    lib = s.lib
    T, E = c["T"], c["E"]
    cfg, (w,) = _transformer(s, T, E, c["H"], c["hidden"], _doc_starts(T, c["docs"]), 1)
    x, out = s.randn(T, E), torch.zeros(T, E, device="cuda")
    vx, vo, work = s.view(x), s.view(out), s.arena(16 * MB + 64 * T * (4 * E + c["hidden"]))

    def call():
        work.contents.offset = 0
        lib.blt_transformer_forward(C.byref(vx), C.byref(w), C.byref(vo), C.byref(cfg), work)
        return out
    return call


def _model(s, c):
    lib = s.lib
    T, E, H, hidden, L = c["T"], c["E"], c["H"], c["hidden"], c["L"]
    cos, sin = (t.cpu().numpy() for t in s.rope(T, E // H)[:2])
    ew = encoder.random_weights(E, hidden, L, NGRAMS, NGRAM_VOCAB, int(s.rs.randint(1 << 30)))
    enc = encoder.bind(ew, cos, sin, abi.BLT_BACKEND_HIP, decoder.device_place, E, H, H, hidden, T, NGRAMS, NGRAM_VOCAB,
                       1000003, window=c["window"])
    dw = decoder.random_weights(E, hidden, L, VOCAB, int(s.rs.randint(1 << 30)))
    dec = decoder.bind(dw, cos, sin, abi.BLT_BACKEND_HIP, decoder.device_place, E, H, H, hidden, VOCAB, T, window=c["window"])
    P = -(-T // 4)
    lengths = s.patch_lengths(T, P)
    patches = decoder.patch_table(lengths)
    starts = np.concatenate([[0], np.cumsum(lengths)[:-1]])
    patch_docs = _doc_starts(P, c["docs"])
    byte_docs = abi.size_array([starts[p] for p in patch_docs]) if patch_docs else None
    num_docs = len(patch_docs) + 1 if patch_docs else 0
    cfg, layers = _transformer(s, P, E, H, hidden, patch_docs, c["G"])
    text = s.rs.randint(0, 256, size=T).astype(np.uint8)
    if c["bytes"] == "host":
        vb = abi.tensor_view(text.ctypes.data, text.shape, abi.BLT_BACKEND_CPU, dtype=abi.BLT_DTYPE_UINT8)
    else:
        vb = s.view(torch.from_numpy(text).cuda(), abi.BLT_DTYPE_UINT8)
    pool = [torch.zeros(P, E, device="cuda") for _ in range(2)]
    hid, logits = torch.zeros(T, E, device="cuda"), torch.zeros(T, VOCAB, device="cuda")
    vp, vh, vl = [s.view(t) for t in pool], s.view(hid), s.view(logits)
    work = s.arena(64 * MB + 64 * T * (4 * E + hidden))
    s.keep += [enc, dec, patches, text, byte_docs]

    def call():
        work.contents.offset = 0
        lib.blt_local_encoder_forward(enc.ptr, C.byref(vb), patches, P, byte_docs, num_docs, C.byref(vp[0]), C.byref(vh), work)
        at = 0
        for w in layers:
            work.contents.offset = 0
            lib.blt_transformer_forward(C.byref(vp[at]), C.byref(w), C.byref(vp[1 - at]), C.byref(cfg), work)
            at = 1 - at
        work.contents.offset = 0
        lib.blt_local_decoder_forward_ext(dec.ptr, C.byref(vh), C.byref(vp[at]), patches, P, None, None, byte_docs, num_docs,
                                            None, 0, C.byref(vl), None, work)
        return logits, hid, pool[at]
    return call


_KINDS = {"heads": _heads, "attn": _attn, "cross": _cross, "kv": _kv, "step": _step, "draft": _draft, "model": _model,
          "block": _block}


def prepare(case, seed):
    s = _State(seed)
    s.call = _KINDS[case["kind"]](s, case)
    return s


def run(state):
    return state.call()


# ---- what a pass cannot do without -----------------------------------------------------------------

def _causal_pairs(T, window=0):
    if not window or window >= T:
        return T * (T + 1) / 2
    return window * (window + 1) / 2 + (T - window) * window


def _layer(rows, E, hidden, pairs):
    """(flops, weight floats) of one transformer block over `rows` rows, `pairs` visible pairs per head."""
    w = 4 * E * E + 3 * E * hidden
    return 2.0 * rows * w + 4.0 * E * pairs, w


def work(case):
    c, kind = case, case["kind"]
    if kind == "heads":
        E, T = c["H"] * c["hd"], c["T"]
        # the dense mask is written and read, every head writes its weights
        return {"bytes": 4.0 * (4 * T * E + (2 + c["H"]) * T * T), "flops": 4.0 * E * T * (T + 1) / 2}
    if kind == "attn":
        E = c["H"] * c["hd"]
        return {"bytes": 4.0 * 4 * c["batch"] * c["T"] * E, "flops": 4.0 * E * c["batch"] * _causal_pairs(c["T"], c["window"])}
    if kind == "cross":
        E = c["H"] * c["hd"]
        return {"bytes": 4.0 * c["batch"] * (2 * c["T"] * E + 2 * c["P"] * E + 2 * c["P"]),
                "flops": 4.0 * E * c["batch"] * c["T"]}
    if kind == "kv":
        E, mean = c["H"] * c["hd"], (c["len_lo"] + c["len_hi"]) / 2
        seen = min(mean + c["n"], c["window"] + c["n"]) if c["window"] else mean + c["n"]
        pairs = c["n"] * (min(mean, c["window"]) if c["window"] else mean) + (c["n"] ** 2 if c["block"] else _causal_pairs(c["n"]))
        return {"bytes": 4.0 * c["batch"] * E * (2 * seen + 6 * c["n"]), "flops": 4.0 * E * c["batch"] * pairs}
    E, hidden = c["E"], c["hidden"]
    if kind == "block":
        d, T = c["docs"], c["T"]
        f, w = _layer(T, E, hidden, d * _causal_pairs(max(1, T / d)))
        return {"bytes": 4.0 * (w + 2 * T * E), "flops": f}
    if kind == "step" or kind == "draft":
        batch, n = (c["batch"], c["n"]) if kind == "step" else (1, c["R"])
        mean = (c["len_lo"] + c["len_hi"]) / 2 if kind == "step" else c["N"]
        rows, prompt = batch * n, kind == "step" and c["len_hi"] == 0
        pairs = batch * (n * mean + (_causal_pairs(n, c["window"]) if kind == "step" else n * n))
        f, w = _layer(rows, E, hidden, pairs)
        patches = n / 4 if prompt else 0   # a prompt's patches become keys and values of the cross block
        f += 2.0 * E * E * 2 * (rows + patches) + 4.0 * E * rows
        w += 2 * E * E + (2 * E * E if prompt else 0)
        # weights, the cached rows, the new rows written, a latent's key and value for every new row
        byt = c["L"] * (w + 2 * E * batch * (mean + n) + 2 * E * max(rows / 4, batch)) + E * VOCAB + rows * (E + VOCAB)
        return {"bytes": 4.0 * byt, "flops": c["L"] * f + 2.0 * rows * E * VOCAB}
    T, P, d = c["T"], c["T"] / 4, c["docs"]
    pairs = d * _causal_pairs(max(1, T / d), c["window"])
    f, w = _layer(T, E, hidden, pairs)
    fe = f + 2.0 * E * E * 2 * (T + P) + 4.0 * E * T        # cross block of a local layer, either direction
    fg, wg = _layer(P, E, hidden, d * _causal_pairs(max(1, P / d)))
    flops = 2 * c["L"] * fe + c["G"] * fg + 2.0 * T * E * VOCAB
    byt = 2 * c["L"] * (w + 4 * E * E) + c["G"] * wg + E * VOCAB + T * (E * (2 + len(NGRAMS)) + VOCAB) + P * E
    return {"bytes": 4.0 * byt, "flops": flops}


def tolerance(case):
    # fp32 sums in another order; whole steps and forwards pass the difference through several layers
    return {"rel": 1e-5}
