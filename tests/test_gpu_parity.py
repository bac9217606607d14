"""GPU parity: the HIP library against the CPU checker on identical seeded inputs.

Every compute call goes through the C-ABI of libfblt_hip.so.  Tolerance for
fp32 attention outputs and weights (stated by the task): |got - ref| <=
1e-5 + 1e-4 * |ref| element-wise; integer/boolean work (masks, cache slots,
lengths) must be bit-exact.
"""
import ctypes as C

import numpy as np
import pytest

from tests import lse_check
from fblt_amd import abi, api, workloads
from oracle import binding, runner as orunner

pytestmark = pytest.mark.gpu

ATOL, RTOL = 1e-5, 1e-4


def assert_close(got, ref, what=""):
    got = np.asarray(got, dtype=np.float64)
    ref = np.asarray(ref, dtype=np.float64)
    assert got.shape == ref.shape, (what, got.shape, ref.shape)
    with np.errstate(invalid="ignore"):
        err = np.abs(got - ref)
        bound = ATOL + RTOL * np.abs(ref)
        # nothing compares with NaN: it is right only where the reference has it, an infinity where that has the same one
        bad = ~((err <= bound) & np.isfinite(ref)) & (got != ref) & ~(np.isnan(got) & np.isnan(ref))
    assert not bad.any(), "%s: %d/%d out of tolerance, max abs err %.3e at %s (got %r ref %r)" % (
        what, int(bad.sum()), bad.size, float(err.max()), np.unravel_index(int(err.argmax()), err.shape),
        float(got.flat[int(err.argmax())]), float(ref.flat[int(err.argmax())]))
    return float(err.max())


@pytest.fixture(scope="module")
def dev():
    from fblt_amd import runner
    return runner


def _oracle_out(w, orc, weights=None):
    for n in w.outputs:
        w.buffers[n][:] = 0
    orunner.run(w, lib=orc, weights=weights)
    return {n: w.buffers[n].copy() for n in w.outputs}


def _families(monkeypatch, fam):
    # the override is read once per process; tests pin it through a reload of the cache
    pass


# ---------------------------------------------------------------------------
# configs 1-3 through every entry point
# ---------------------------------------------------------------------------
SMALL = {
    "c1_small": lambda: workloads.config1(batch=1, T=96, H=2, hd=32),
    "c1_ragged": lambda: workloads.config1(batch=2, T=77, H=2, hd=32),
    "c2_small": lambda: workloads.config2(batch=2, P=48, H=2, hd=64, T_bytes=192),
    "c3_small": lambda: workloads.config3(batch=2, T=128, P=32, H=2, hd=32),
    "c1_hd16": lambda: workloads.config1(batch=1, T=50, H=3, hd=16),
    "c1_hd128": lambda: workloads.config1(batch=1, T=40, H=1, hd=128),
    "c1_hd8": lambda: workloads.config1(batch=1, T=33, H=2, hd=8),
}
FULL = {
    "c1_full": lambda: workloads.config1(),
    "c2_full": lambda: workloads.config2(),
    "c3_full": lambda: workloads.config3(),
}


@pytest.mark.parametrize("name", list(SMALL) + list(FULL))
@pytest.mark.parametrize("entry", ["per_head_dense", "per_head_flag", "batch_descriptor", "batch_dense", "plan"])
def test_dense_configs(name, entry, oracle, dev):
    w = (SMALL.get(name) or FULL[name])()
    if entry == "per_head_flag" and w.heads[0].mask != "causal":
        pytest.skip("is_causal flag only describes causal problems")
    ref = _oracle_out(w, oracle)
    d = dev.DeviceWorkload(w)
    try:
        d.zero_outputs()
        if entry == "per_head_dense":
            d.run_per_head("dense", with_weights=True)
        elif entry == "per_head_flag":
            d.run_per_head("flag", with_weights=False)
        elif entry == "batch_descriptor":
            d.run_batch("descriptor")
        elif entry == "batch_dense":
            d.run_batch("dense")
        else:
            plan = d.make_plan("descriptor")
            d.lib.blt_attention_plan_run_hip(plan)
            d.lib.blt_backend_pass_sync_hip()
            d.lib.blt_attention_plan_destroy_hip(plan)
        got = d.output("out")
    finally:
        d.close()
    assert_close(got, ref["out"], "%s/%s" % (name, entry))


@pytest.mark.parametrize("name", ["c1_small", "c1_ragged", "c2_small", "c3_small"])
@pytest.mark.parametrize("mask_mode", ["descriptor", "dense"])
def test_weights_and_lse(name, mask_mode, oracle, dev):
    """weights_out holds the post-softmax weights (zeros where masked); lse_out holds (max, sum)."""
    import torch
    w = SMALL[name]()
    host_w = [np.zeros(h.nq * h.nk, dtype=np.float32) for h in w.heads]
    ref = _oracle_out(w, oracle, weights=host_w)
    d = dev.DeviceWorkload(w)
    try:
        d.zero_outputs()
        wbufs = [torch.full((h.nq * h.nk,), 7.0, dtype=torch.float32, device="cuda") for h in w.heads]
        lbufs = [torch.full((h.nq * 2,), 7.0, dtype=torch.float32, device="cuda") for h in w.heads]
        arr = d.problems(mask_mode, [t.data_ptr() for t in wbufs], [t.data_ptr() for t in lbufs])
        d.lib.blt_attention_batch_hip(arr, len(w.heads))
        d.lib.blt_backend_pass_sync_hip()
        got = d.output("out")
        assert_close(got, ref["out"], name)
        for t, h in enumerate(w.heads):
            gw = wbufs[t].cpu().numpy()
            assert_close(gw, host_w[t], "%s weights head %d" % (name, t))
            assert ((gw == 0) == (host_w[t] == 0)).all(), "masked pattern differs"
        # (m, l) in natural units: the weights rebuilt from the pair must be the checker's weights
        cache = {}
        lse_check.check_workload(w, [t.cpu().numpy() for t in lbufs], host_w,
                                 lambda h: orunner._mask_for(oracle, w, h, cache))
    finally:
        d.close()


def test_lse_pair_single_head(oracle, dev):
    """lse_out alone (the reference's BLT_FLASH_ATTN output mode) and together with weights_out:
    dead rows, additive biases, causal flag, no mask."""
    lse_check.run_single_head_cases(api.load(), oracle, api, abi, binding)


# ---------------------------------------------------------------------------
# per-head call: the reference's own vectors and edge cases
# ---------------------------------------------------------------------------
def _run_single(lib, q, k, v, nq, nk, hd, scale, q_stride, k_stride, v_stride, out_cols, col, q_off=0, k_off=0,
                v_off=0, mask=None, causal=False, want_weights=True):
    import torch
    tq, tk, tv = (torch.from_numpy(x).cuda() for x in (q, k, v))
    out = torch.full((nq * out_cols,), 5.0, dtype=torch.float32, device="cuda")
    wts = torch.full((max(nq * nk, 1),), 9.0, dtype=torch.float32, device="cuda")
    tm = torch.from_numpy(mask).cuda() if mask is not None else None
    a = api.head_args(tq.data_ptr() + 4 * q_off, tk.data_ptr() + 4 * k_off, tv.data_ptr() + 4 * v_off,
                      out.data_ptr(), nq, nk, hd, scale, q_stride, k_stride, v_stride, out_cols, col,
                      weights=wts.data_ptr() if want_weights else None,
                      scratch=None if want_weights else wts.data_ptr(),
                      mask=tm.data_ptr() if tm is not None else None, causal=causal)
    lib.blt_attention_head_core_hip(abi.BLT_BACKEND_HIP, C.byref(a))
    lib.blt_backend_pass_sync_hip()
    return out.cpu().numpy().reshape(nq, out_cols), wts.cpu().numpy()[:nq * nk].reshape(nq, nk)


def test_reference_identity_vector(dev):
    """tests/unit/models/unit_attention.c:24-88: identity projections, 2 tokens, 2 heads of dim 2."""
    lib = api.load()
    qkv = np.zeros((2, 12), dtype=np.float32)
    x = np.array([[1, 0, 1, 0], [0, 1, 0, 1]], dtype=np.float32)
    qkv[:, 0:4] = x
    qkv[:, 4:8] = x
    qkv[:, 8:12] = x
    scale = float(1.0 / np.sqrt(np.float32(2.0)))
    want = np.array([[0.6697615, 0.3302385, 0.6697615, 0.3302385], [0.3302385, 0.6697615, 0.3302385, 0.6697615]])
    got = np.zeros((2, 4))
    for h in range(2):
        o, _ = _run_single(lib, qkv.reshape(-1), qkv.reshape(-1), qkv.reshape(-1), 2, 2, 2, scale, 12, 12, 12, 4,
                           2 * h, q_off=2 * h, k_off=4 + 2 * h, v_off=8 + 2 * h)
        got[:, 2 * h:2 * h + 2] = o[:, 2 * h:2 * h + 2]
        # columns of the other head are left alone (sentinel 5.0)
        other = [c for c in range(4) if c // 2 != h]
        assert (o[:, other] == 5.0).all()
    assert np.abs(got - want).max() < 1e-6
    # causal variant (unit_attention.c:160-171): row 0 sees only itself
    want_c = np.array([[1, 0, 1, 0], [0.3302385, 0.6697615, 0.3302385, 0.6697615]])
    for h in range(2):
        o, wts = _run_single(lib, qkv.reshape(-1), qkv.reshape(-1), qkv.reshape(-1), 2, 2, 2, scale, 12, 12, 12, 4,
                             2 * h, q_off=2 * h, k_off=4 + 2 * h, v_off=8 + 2 * h, causal=True)
        assert np.abs(o[:, 2 * h:2 * h + 2] - want_c[:, 2 * h:2 * h + 2]).max() < 1e-6
        assert wts[0, 1] == 0.0 and abs(wts[0, 0] - 1.0) < 1e-6


@pytest.mark.parametrize("nq,nk,hd", [(1, 1, 32), (1, 300, 32), (5, 7, 32), (31, 33, 64), (64, 65, 32),
                                      (17, 129, 128), (3, 40, 20), (40, 40, 6), (2, 5, 200)])
@pytest.mark.parametrize("masked", ["none", "causal", "dense_random"])
def test_single_head_shapes(nq, nk, hd, masked, oracle, dev):
    """Ragged shapes, odd head dims and unaligned strides through the per-head call."""
    lib = api.load()
    rs = np.random.RandomState(1000 * nq + nk + hd)
    stride = hd + 3  # not a multiple of 4: forces the scalar access path
    q = rs.randn(nq, stride).astype(np.float32)
    k = rs.randn(nk, stride).astype(np.float32)
    v = rs.randn(nk, stride).astype(np.float32)
    scale = float(1.0 / np.sqrt(np.float32(hd)))
    mask = None
    causal = masked == "causal"
    if masked == "dense_random":
        mask = np.where(rs.rand(nq, nk) < 0.4, -np.inf, 0.0).astype(np.float32)
        mask[0, :] = -np.inf  # an all-masked row must give zeros
        if nq > 1:
            mask[1, :] = 0.0
    out_ref = np.zeros((nq, hd + 1), dtype=np.float32)
    w_ref = np.zeros((nq, nk), dtype=np.float32)
    a = binding.head_args(q.reshape(-1), k.reshape(-1), v.reshape(-1), out_ref.reshape(-1), nq, nk, hd, scale,
                          stride, stride, stride, hd + 1, 1, weights=w_ref.reshape(-1),
                          mask=None if mask is None else mask.reshape(-1), causal=causal)
    assert oracle.orc_attention_head_core(C.byref(a)) == 0
    got, gw = _run_single(lib, q.reshape(-1), k.reshape(-1), v.reshape(-1), nq, nk, hd, scale, stride, stride, stride,
                          hd + 1, 1, mask=None if mask is None else mask.reshape(-1), causal=causal)
    assert (got[:, 0] == 5.0).all(), "column outside the head slice was written"
    assert_close(got[:, 1:], out_ref[:, 1:], "out")
    assert_close(gw, w_ref, "weights")
    if mask is not None:
        assert (got[0, 1:] == 0).all() and (gw[0] == 0).all()


@pytest.mark.parametrize("seed", range(40))
def test_single_head_randomised(seed, oracle, dev):
    """Seeded draws of everything the per-head call leaves open: ragged sizes, head widths with and
    without the 16-byte fast paths, padded row strides, a column offset in the output, the mask given
    as nothing / the causal flag / a dense additive mask with -inf, finite biases and dead rows, and
    the scale."""
    lib = api.load()
    rs = np.random.RandomState(7000 + seed)
    nq = int(rs.choice([1, 2, 7, 31, 32, 33, 64, 100, 129, 200]))
    nk = int(rs.choice([1, 3, 31, 32, 33, 65, 128, 257, 400]))
    hd = int(rs.choice([4, 8, 12, 16, 32, 48, 64, 96, 128]))
    pad = int(rs.choice([0, 0, 4, 3]))
    qs, ks, vs = hd + pad, hd + int(rs.choice([0, 4, 5])), hd + int(rs.choice([0, 8, 1]))
    col = int(rs.choice([0, 4, 1]))
    os_ = hd + col + int(rs.choice([0, 4, 2]))
    kind = rs.choice(["none", "causal", "dense"])
    q = rs.randn(nq, qs).astype(np.float32)
    k = rs.randn(nk, ks).astype(np.float32)
    v = rs.randn(nk, vs).astype(np.float32)
    scale = float(rs.choice([1.0 / np.sqrt(np.float32(hd)), 0.05, 1.0]))
    mask = None
    if kind == "dense":
        mask = np.where(rs.rand(nq, nk) < 0.5, -np.inf, 0.0).astype(np.float32)
        bias = rs.rand(nq, nk) < 0.2
        mask[bias & np.isfinite(mask)] = rs.randn(int((bias & np.isfinite(mask)).sum())).astype(np.float32)
        mask[rs.randint(nq), :] = -np.inf
    out_ref = np.zeros((nq, os_), dtype=np.float32)
    w_ref = np.zeros((nq, nk), dtype=np.float32)
    flat = None if mask is None else mask.reshape(-1)
    a = binding.head_args(q.reshape(-1), k.reshape(-1), v.reshape(-1), out_ref.reshape(-1), nq, nk, hd, scale,
                          qs, ks, vs, os_, col, weights=w_ref.reshape(-1), mask=flat, causal=kind == "causal")
    assert oracle.orc_attention_head_core(C.byref(a)) == 0
    got, gw = _run_single(lib, q.reshape(-1), k.reshape(-1), v.reshape(-1), nq, nk, hd, scale, qs, ks, vs, os_, col,
                          mask=flat, causal=kind == "causal")
    what = "seed %d nq %d nk %d hd %d strides %d/%d/%d out %d+%d %s" % (seed, nq, nk, hd, qs, ks, vs, os_, col, kind)
    assert (got[:, :col] == 5.0).all() and (got[:, col + hd:] == 5.0).all(), "columns outside the head slice: " + what
    assert_close(got[:, col:col + hd], out_ref[:, col:col + hd], "out " + what)
    assert_close(gw, w_ref, "weights " + what)


def test_additive_mask_values(oracle, dev):
    """A dense mask is additive: finite biases shift the scores, +inf / nan entries drop the key."""
    lib = api.load()
    rs = np.random.RandomState(7)
    nq, nk, hd = 37, 70, 32
    q, k, v = (rs.randn(n, hd).astype(np.float32) for n in (nq, nk, nk))
    mask = (rs.randn(nq, nk) * 2).astype(np.float32)
    mask[rs.rand(nq, nk) < 0.2] = -np.inf
    mask[2, 3] = np.inf
    mask[4, 5] = np.nan
    scale = 0.25
    out_ref = np.zeros((nq, hd), dtype=np.float32)
    w_ref = np.zeros((nq, nk), dtype=np.float32)
    a = binding.head_args(q.reshape(-1), k.reshape(-1), v.reshape(-1), out_ref.reshape(-1), nq, nk, hd, scale, hd, hd,
                          hd, hd, 0, weights=w_ref.reshape(-1), mask=mask.reshape(-1))
    assert oracle.orc_attention_head_core(C.byref(a)) == 0
    got, gw = _run_single(lib, q.reshape(-1), k.reshape(-1), v.reshape(-1), nq, nk, hd, scale, hd, hd, hd, hd, 0,
                          mask=mask.reshape(-1))
    assert_close(got, out_ref, "out")
    assert_close(gw, w_ref, "weights")
    assert gw[2, 3] == 0 and gw[4, 5] == 0


# ---------------------------------------------------------------------------
# dense mask builders on the device: bit-exact
# ---------------------------------------------------------------------------
def _variants():
    sq, skv = 19, 23
    docs = [7, 15, 15]
    qg = [i % 3 for i in range(sq)]
    kg = [j % 3 for j in range(skv)]
    # the variant matrix of tests/parity/parity_cuda_composites.c:66-105
    table = [(True, 0, False, False, False), (False, 5, False, False, False), (True, 4, True, False, False),
             (False, 0, True, False, False), (True, 0, False, True, True), (True, 0, False, True, False),
             (True, 6, True, True, True)]
    for causal, window, use_docs, use_groups, bidir in table:
        yield sq, skv, causal, window, docs if use_docs else None, (qg, kg) if use_groups else None, bidir, 0
    # sizes past one block, causal offsets, sorted groups (cross-attention)
    yield 300, 517, True, 0, None, None, False, 217
    yield 300, 517, True, 64, None, None, False, 217
    yield 128, 512, False, 0, None, ([p for p in range(128)], [j // 4 for j in range(512)]), True, 0


@pytest.mark.parametrize("case", list(_variants()), ids=lambda c: "q%d_k%d_c%d_w%d_d%d_g%d_b%d_o%d" % (
    c[0], c[1], c[2], c[3], c[4] is not None, c[5] is not None, c[6], c[7]))
def test_attention_mask_bit_exact(case, oracle, dev):
    sq, skv, causal, window, docs, groups, bidir, off = case
    lib = api.load()
    cfg = abi.BltMaskConfig()
    cfg.seq_len_q, cfg.seq_len_kv = sq, skv
    cfg.is_causal, cfg.sliding_window, cfg.causal_offset = causal, window, off
    keep = []
    if docs is not None:
        arr = abi.size_array(docs)
        keep.append(arr)
        cfg.doc_boundaries, cfg.num_docs = arr, len(docs) + 1
    if groups is not None:
        qa, ka = abi.size_array(groups[0]), abi.size_array(groups[1])
        keep += [qa, ka]
        cfg.query_group_ids, cfg.kv_group_ids = qa, ka
        cfg.bidirectional_within_group = bidir
    want = np.empty(sq * skv, dtype=np.float32)
    assert oracle.orc_build_attention_mask(C.byref(cfg), binding.fptr(want)) == 0
    arena = lib.blt_arena_create(8 << 20, abi.BLT_BACKEND_HIP)
    t = abi.BltTensor()
    lib.blt_build_attention_mask(C.byref(cfg), C.byref(t), arena)  # public dispatcher -> HIP twin
    assert t.backend == abi.BLT_BACKEND_HIP and t.shape[0] == sq and t.shape[1] == skv and t.numel == sq * skv
    got = np.empty(sq * skv, dtype=np.float32)
    lib.blt_tensor_download(C.byref(t), got.ctypes.data, got.nbytes)
    lib.blt_arena_destroy(arena)
    assert got.tobytes() == want.tobytes()
    # the row-range reduction describes the same visibility whenever it claims to
    lo = (C.c_uint32 * sq)()
    hi = (C.c_uint32 * sq)()
    if lib.blt_mask_config_row_ranges(C.byref(cfg), lo, hi):
        allowed = want.reshape(sq, skv) == 0
        for i in range(sq):
            row = np.zeros(skv, dtype=bool)
            row[lo[i]:hi[i]] = True
            assert (row == allowed[i]).all(), i
    else:
        assert groups is not None  # only unsorted group ids are not interval-shaped


@pytest.mark.parametrize("mode,S,N,B,starts", [
    (abi.BLT_BDM_TRAIN, 14, 6, 4, [2, 4]),
    (abi.BLT_BDM_INFER, 7, 3, 0, None),
    (abi.BLT_BDM_TRAIN, 24, 12, 2, [0, 4, 1, 7, 3, 11]),
    (abi.BLT_BDM_INFER, 24, 12, 2, None),
    (abi.BLT_BDM_INFER, 524, 508, 16, None),
    (abi.BLT_BDM_TRAIN, 9 + 3 * 4, 9, 3, [1, 3, 5, 8]),
])
def test_block_diffusion_mask_bit_exact(mode, S, N, B, starts, oracle, dev):
    lib = api.load()
    cfg = abi.BltBlockDiffusionConfig()
    cfg.mode, cfg.seq_len, cfg.num_clean, cfg.block_size = mode, S, N, B
    keep = None
    if starts is not None:
        keep = abi.size_array(starts)
        cfg.block_starts, cfg.num_blocks = keep, len(starts)
    want = np.empty(S * S, dtype=np.float32)
    assert oracle.orc_build_block_diffusion_mask(C.byref(cfg), binding.fptr(want)) == 0
    arena = lib.blt_arena_create(8 << 20, abi.BLT_BACKEND_HIP)
    t = abi.BltTensor()
    lib.blt_build_block_diffusion_mask(C.byref(cfg), C.byref(t), arena)
    got = np.empty(S * S, dtype=np.float32)
    lib.blt_tensor_download(C.byref(t), got.ctypes.data, got.nbytes)
    lib.blt_arena_destroy(arena)
    assert got.tobytes() == want.tobytes()


# ---------------------------------------------------------------------------
# KV-cache step (config 4) and block verify (config 5)
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("batch,steps,H,hd,len_hi", [(3, 5, 4, 32, 70), (64, 6, 4, 32, 512), (5, 4, 2, 64, 100),
                                                     (4, 3, 8, 16, 40), (2, 40, 4, 32, 3),
                                                     (64, 256, 4, 32, 512)])   # the last: config 4 at full size
@pytest.mark.parametrize("lens_mode", ["device", "host"])
def test_kv_decode_steps(batch, steps, H, hd, len_hi, lens_mode, oracle, dev):
    """lens_mode host: blt_kv_attend_step_lens_hip, the lengths kept by the caller as the reference
    keeps them (kv_cache.h:56-60) and carried in the kernel arguments."""
    kw = workloads.config4(batch=batch, steps=steps, H=H, hd=hd, len_hi=len_hi)
    ref_out, ref_k, ref_v = orunner.run_kv(kw, lib=oracle)
    d = dev.DeviceKvWorkload(kw, lens=lens_mode)
    d.run()
    out, ck, cv, lens = d.results()
    assert (lens == kw.lens.astype(np.int64) + steps).all()          # slot bookkeeping: exact
    assert ck.tobytes() == ref_k.tobytes() and cv.tobytes() == ref_v.tobytes()  # write-through: bit-exact rows
    assert_close(out, ref_out, "kv decode")


@pytest.mark.parametrize("lens_mode", ["device", "host"])
def test_kv_decode_window(lens_mode, oracle, dev):
    kw = workloads.config4(batch=6, steps=4, H=4, hd=32, len_hi=200)
    kw.window = 48
    ref_out, ref_k, ref_v = orunner.run_kv(kw, lib=oracle)
    d = dev.DeviceKvWorkload(kw, lens=lens_mode)
    d.run()
    out, ck, cv, lens = d.results()
    assert ck.tobytes() == ref_k.tobytes()
    assert_close(out, ref_out, "kv decode window")


@pytest.mark.parametrize("lens_mode", ["device", "host"])
@pytest.mark.parametrize("batch,H,hd,len_lo,len_hi,window,rope", [
    (64, 4, 32, 0, 300, 0, False),     # from empty caches
    (64, 4, 32, 100, 700, 0, True),    # rotation fused in
    (40, 4, 32, 1, 900, 130, False),   # window that skips whole rounds of keys
    (32, 8, 16, 1, 400, 0, True),
    (64, 2, 64, 1, 500, 77, True),
    (128, 1, 128, 1, 260, 0, False),
    (70, 2, 8, 0, 200, 0, False),
    (140, 1, 4, 1, 150, 5, False),
    (300, 1, 32, 1, 140, 0, True),     # host lengths: more sequences than one launch carries
    (130, 2, 32, 1000, 2040, 0, False),
    (34, 4, 32, 2000, 4090, 0, False),  # long caches, 136 (sequence, head) pairs: still one workgroup per pair
    (120, 4, 32, 1500, 2900, 600, True),
    (32, 4, 32, 6000, 8180, 0, False),   # the longest caches the single-row kernel is routed
])
def test_kv_single_row_steps(batch, H, hd, len_lo, len_hi, window, rope, lens_mode, oracle, dev):
    """One new row per sequence at batch sizes that give one workgroup per (sequence, head): every
    head width, empty caches, windows, fused rotation, three committing steps in a row; lengths
    in device memory or in the caller's hands."""
    steps = 3
    kw = workloads.config4(batch=batch, steps=steps, H=H, hd=hd, len_lo=len_lo, len_hi=len_hi,
                           max_seq_len=len_hi + steps, rope=rope)
    kw.window = window
    ref_out, ref_k, ref_v = orunner.run_kv(kw, lib=oracle)
    d = dev.DeviceKvWorkload(kw, lens=lens_mode)
    d.run()
    out, ck, cv, lens = d.results()
    assert (lens == kw.lens.astype(np.int64) + steps).all()
    assert ck.tobytes() == ref_k.tobytes() and cv.tobytes() == ref_v.tobytes()
    assert_close(out, ref_out, "kv single rows")


@pytest.mark.parametrize("lens_mode", ["device", "host"])
@pytest.mark.parametrize("n", [2, 3, 8, 20])
def test_kv_prefill_chunk(n, lens_mode, oracle, dev):
    """n > 1 rows per step, chunk-causal (kv_cache.c:229-236): same kernel, causal kind."""
    kw = workloads.config4(batch=5, steps=3, H=4, hd=32, len_hi=90, max_seq_len=90 + 3 * n)
    rs = np.random.RandomState(n)
    kw.n = n
    kw.q_new, kw.k_new, kw.v_new = (rs.randn(kw.steps, kw.batch * n, kw.E).astype(np.float32) for _ in range(3))
    ref_out, ref_k, ref_v = orunner.run_kv(kw, lib=oracle)
    d = dev.DeviceKvWorkload(kw, lens=lens_mode)
    d.run()
    out, ck, cv, lens = d.results()
    assert (lens == kw.lens.astype(np.int64) + n * kw.steps).all()
    assert ck.tobytes() == ref_k.tobytes() and cv.tobytes() == ref_v.tobytes()
    assert_close(out, ref_out, "kv chunk n=%d" % n)


@pytest.mark.parametrize("lens_mode", ["device", "host"])
@pytest.mark.parametrize("B", [4, 8, 16, 32])
@pytest.mark.parametrize("batch", [3, 64])
def test_block_verify(B, batch, lens_mode, oracle, dev):
    kw = workloads.config5(batch=batch, B=B)
    ref_out, ref_k, ref_v = orunner.run_kv(kw, lib=oracle)
    d = dev.DeviceKvWorkload(kw, lens=lens_mode)
    d.run()
    out, ck, cv, lens = d.results()
    assert (lens == kw.lens).all()   # verify does not commit
    assert ck.tobytes() == ref_k.tobytes() and cv.tobytes() == ref_v.tobytes()
    assert_close(out, ref_out, "block verify B=%d" % B)


@pytest.mark.parametrize("kind", ["block", "causal_chunk"])
def test_block_step_long_unequal_sequences(kind, oracle, dev):
    """More (sequence, head) pairs than compute units, prefixes of 300 ... 1100 keys, lengths on the
    host: the block step hands the pairs out as workgroups of their own, longest sequence first
    (blt_kv_attend_step_lens_hip).  Same results as the checker; the caches take the new rows bit
    for bit; the device-length entry point, which cannot reorder, agrees."""
    kw = workloads.config5(batch=72, B=16, len_lo=300, len_hi=1100, max_seq_len=1152)
    if kind == "causal_chunk":
        kw.kind = "causal"
        kw.commit = True
    ref_out, ref_k, ref_v = orunner.run_kv(kw, lib=oracle)
    for lens_mode in ("host", "device"):
        d = dev.DeviceKvWorkload(kw, lens=lens_mode)
        d.run()
        out, ck, cv, lens = d.results()
        assert (lens == kw.lens.astype(np.int64) + (16 if kw.commit else 0)).all()
        assert ck.tobytes() == ref_k.tobytes() and cv.tobytes() == ref_v.tobytes()
        assert_close(out, ref_out, "block step by length, %s, %s lengths" % (kind, lens_mode))


@pytest.mark.parametrize("B,nseq", [(4, 12), (8, 12), (16, 64)])
def test_diffusion_self_attention_call_pattern(B, nseq, oracle, dev):
    """The reference's own route to config 5 (csrc/models/block_diffusion.c:196-204, 293-319): the whole
    [prefix ; block] sequence of S = N + B rows through one blt_attention_head_core call per head with
    nq = nk = S and the dense INFER mask blt_build_block_diffusion_mask builds on the device.  All S rows
    against the checker; the block rows also against what the cached-prefix block kernel returns
    for the same sequence (blt_kv_attend_step_hip, BLT_KV_STEP_BLOCK)."""
    import torch
    lib = api.load()
    kw = workloads.config5(B=B)
    d = dev.DeviceKvWorkload(kw)
    d.run()
    step_out = d.results()[0][0]                      # [batch * B, E] of the single step
    E, H, hd = kw.E, kw.H, kw.hd
    scale = float(np.float32(1.0) / np.sqrt(np.float32(hd)))
    arena = lib.blt_arena_create(16 << 20, abi.BLT_BACKEND_HIP)
    rs = np.random.RandomState(B)
    for b in range(nseq):
        N = int(kw.lens[b])
        S = N + B
        slab = slice(b * kw.max_seq_len, b * kw.max_seq_len + N)
        k = np.concatenate([kw.cache_k[slab], kw.k_new[0, b * B:(b + 1) * B]]).astype(np.float32)
        v = np.concatenate([kw.cache_v[slab], kw.v_new[0, b * B:(b + 1) * B]]).astype(np.float32)
        q = np.concatenate([rs.randn(N, E).astype(np.float32), kw.q_new[0, b * B:(b + 1) * B]])
        cfg = abi.BltBlockDiffusionConfig()
        cfg.mode, cfg.seq_len, cfg.num_clean, cfg.block_size = abi.BLT_BDM_INFER, S, N, B
        # checker: restated mask builder + one core call per head
        mask = np.empty(S * S, dtype=np.float32)
        assert oracle.orc_build_block_diffusion_mask(C.byref(cfg), binding.fptr(mask)) == 0
        ref = np.zeros((S, E), dtype=np.float32)
        scratch = np.empty(S * S, dtype=np.float32)
        for h in range(H):
            a = binding.head_args(q.reshape(-1), k.reshape(-1), v.reshape(-1), ref.reshape(-1), S, S, hd, scale, E, E,
                                  E, E, h * hd, q_off=h * hd, k_off=h * hd, v_off=h * hd, scratch=scratch, mask=mask)
            assert oracle.orc_attention_head_core(C.byref(a)) == 0
        # device: the reference caller's statements on this library's ops
        arena.contents.offset = 0
        t = abi.BltTensor()
        lib.blt_build_block_diffusion_mask(C.byref(cfg), C.byref(t), arena)
        got_mask = np.empty(S * S, dtype=np.float32)
        lib.blt_tensor_download(C.byref(t), got_mask.ctypes.data, got_mask.nbytes)
        assert got_mask.tobytes() == mask.tobytes()
        tq, tk, tv = (torch.from_numpy(x).cuda() for x in (q, k, v))
        comb = torch.zeros((S, E), dtype=torch.float32, device="cuda")
        scores = torch.empty(S * S, dtype=torch.float32, device="cuda")
        for h in range(H):
            a = api.head_args(tq.data_ptr() + 4 * h * hd, tk.data_ptr() + 4 * h * hd, tv.data_ptr() + 4 * h * hd,
                              comb.data_ptr(), S, S, hd, scale, E, E, E, E, h * hd, weights=scores.data_ptr(),
                              mask=t.data)
            lib.blt_attention_head_core(abi.BLT_BACKEND_HIP, C.byref(a))
        lib.blt_backend_pass_sync_hip()
        got = comb.cpu().numpy()
        assert_close(got, ref, "sequence %d: [prefix ; block] rows" % b)
        assert_close(step_out[b * B:(b + 1) * B], ref[N:], "sequence %d: block kernel against the dense route" % b)
    lib.blt_arena_destroy(arena)


def test_zero_weight_key_with_non_finite_value_row(oracle, dev):
    """Documents the one place where results can differ from the reference: the reference's weighted
    sum skips keys whose weight is exactly zero (csrc/ops/attn_core_cpu.c:47-50), so a masked key
    whose V row holds inf / NaN leaves the output finite; the kernels here multiply (0 * inf = NaN).
    What is guaranteed and checked: (1) only the columns that are non-finite in that V row can
    differ; (2) wherever the reference's output is non-finite, so is this library's; (3) rows whose
    key range ends before the bad key's 32-key tile (the kernels never load tiles no row of a
    32-row query tile can see) are untouched; (4) elsewhere in those columns the value is either
    the reference's (within tolerance) or NaN."""
    lib = api.load()
    rs = np.random.RandomState(11)
    nq = nk = 160
    hd = 32
    q, k, v = (rs.randn(n, hd).astype(np.float32) for n in (nq, nk, nk))
    bad_key, bad_col = 100, 5
    v[bad_key, bad_col] = np.inf
    scale = float(np.float32(1.0) / np.sqrt(np.float32(hd)))
    out_ref = np.zeros((nq, hd), dtype=np.float32)
    w_ref = np.zeros((nq, nk), dtype=np.float32)
    a = binding.head_args(q.reshape(-1), k.reshape(-1), v.reshape(-1), out_ref.reshape(-1), nq, nk, hd, scale, hd, hd,
                          hd, hd, 0, weights=w_ref.reshape(-1), causal=True)
    assert oracle.orc_attention_head_core(C.byref(a)) == 0
    assert np.isfinite(out_ref[:bad_key]).all() and not np.isfinite(out_ref[bad_key:, bad_col]).any()
    got, _ = _run_single(lib, q.reshape(-1), k.reshape(-1), v.reshape(-1), nq, nk, hd, scale, hd, hd, hd, hd, 0,
                         causal=True)
    other = [c for c in range(hd) if c != bad_col]
    assert_close(got[:, other], out_ref[:, other], "columns the bad value is not in")          # (1)
    assert not np.isfinite(got[bad_key:, bad_col]).any()                                       # (2)
    first_tile_row = (bad_key // 32) * 32
    assert_close(got[:first_tile_row, bad_col], out_ref[:first_tile_row, bad_col], "rows before the key's tile")  # (3)
    mid = got[first_tile_row:bad_key, bad_col]                                                 # (4)
    fin = np.isfinite(mid)
    assert np.isnan(mid[~fin]).all()
    if fin.any():
        assert_close(mid[fin], out_ref[first_tile_row:bad_key, bad_col][fin], "finite cells of the key's tile")


@pytest.mark.parametrize("mode", ["hint", "slab", "tables", "graph"])
def test_kv_step_length_beyond_capacity_is_reported(mode):
    """The lengths of the KV step live on the device; the host sizes the launch from a hint.  A
    sequence that outgrew the hint, its slab or the rotation tables is left alone by the kernels
    (which all exit normally) and the next synchronising call ends with the reference's "exceeds
    cache capacity" error (csrc/infer/kv_cache.c:191).  "graph": the same for a committing step that is
    replayed from a HIP graph past its captured hint.  Runs in its own process: the error is fatal."""
    import os
    import subprocess
    import sys
    here = os.path.dirname(os.path.abspath(__file__))
    p = subprocess.run([sys.executable, "-u", os.path.join(here, "kv_guard_case.py"), mode], capture_output=True,
                       text=True, timeout=300)
    assert "CHECKED" in p.stdout and "NOT REACHED" not in p.stdout, p.stdout[-2000:] + p.stderr[-2000:]
    assert mode != "graph" or "REPLAY 1 QUIET" in p.stdout, p.stdout[-2000:]
    assert p.returncode == 1 and "exceeds cache capacity" in p.stderr, (p.returncode, p.stderr[-2000:])


@pytest.mark.parametrize("lens_mode", ["device", "host"])
@pytest.mark.parametrize("seed", range(24))
def test_kv_step_randomised(seed, lens_mode, oracle, dev):
    """Seeded draws over the KV step's free choices: sequences, heads, head width, cached lengths
    (from empty to long), rows per step (single rows, blocks, chunks longer than one launch takes),
    step kind, window, rotation fused in or not, committing steps in a row."""
    rs = np.random.RandomState(9100 + seed)
    batch = int(rs.choice([1, 2, 5, 17]))
    H, hd = int(rs.choice([1, 2, 4])), int(rs.choice([8, 16, 32, 64]))
    len_hi = int(rs.choice([1, 6, 40, 130, 300]))
    kind = "causal" if rs.rand() < 0.6 else "block"
    n = int(rs.choice([1, 2, 5, 16, 17, 32] + ([33, 40] if kind == "causal" else [])))
    steps = int(rs.choice([1, 2, 3])) if kind == "causal" else 1
    rope = bool(rs.rand() < 0.4)
    kw = workloads.config4(batch=batch, steps=steps, H=H, hd=hd, len_lo=0 if rs.rand() < 0.3 else 1, len_hi=len_hi,
                           max_seq_len=len_hi + steps * n + int(rs.choice([0, 3])), rope=rope)
    kw.n, kw.kind, kw.commit = n, kind, kind == "causal"
    if kind == "causal" and rs.rand() < 0.4:
        kw.window = int(rs.choice([1, 7, 48]))
    kw.q_new, kw.k_new, kw.v_new = (rs.randn(kw.steps, kw.batch * n, kw.E).astype(np.float32) for _ in range(3))
    ref_out, ref_k, ref_v = orunner.run_kv(kw, lib=oracle)
    d = dev.DeviceKvWorkload(kw, lens=lens_mode)
    d.run()
    out, ck, cv, lens = d.results()
    what = "seed %d batch %d H %d hd %d len<=%d n %d %s steps %d window %s rope %s" % (
        seed, batch, H, hd, len_hi, n, kind, steps, getattr(kw, "window", 0), rope)
    assert (lens == kw.lens.astype(np.int64) + (n * steps if kw.commit else 0)).all(), what
    assert ck.tobytes() == ref_k.tobytes() and cv.tobytes() == ref_v.tobytes(), what
    assert_close(out, ref_out, "kv step " + what)


# ---------------------------------------------------------------------------
# small device utilities
# ---------------------------------------------------------------------------
def test_strided_copy_softmax_dot(oracle, dev):
    import torch
    lib = api.load()
    rs = np.random.RandomState(3)
    src = rs.randn(9, 24).astype(np.float32)
    tsrc = torch.from_numpy(src).cuda()
    for cols, off in [(8, 4), (5, 3)]:
        dst = torch.zeros((9, 16), dtype=torch.float32, device="cuda")
        lib.blt_strided_copy(abi.BLT_BACKEND_HIP, dst.data_ptr() + 4 * 2, 16, tsrc.data_ptr() + 4 * off, 24, 9, cols)
        lib.blt_backend_pass_sync(abi.BLT_BACKEND_HIP)
        want = np.zeros((9, 16), dtype=np.float32)
        want[:, 2:2 + cols] = src[:, off:off + cols]
        assert (dst.cpu().numpy() == want).all()
    for n, causal, use_mask in [(1, False, False), (300, True, False), (1000, False, True)]:
        row = rs.randn(n).astype(np.float32) * 3
        mask = np.where(rs.rand(n) < 0.3, -np.inf, 0).astype(np.float32) if use_mask else None
        ref = row.copy()
        oracle.orc_softmax_masked_row_inplace(binding.fptr(ref), n, n // 2, causal, binding.fptr(mask), 0.5)
        t = torch.from_numpy(row).cuda()
        tm = torch.from_numpy(mask).cuda() if use_mask else None
        lib.blt_softmax_masked_row_inplace(abi.BLT_BACKEND_HIP, t.data_ptr(), n, n // 2, causal,
                                           tm.data_ptr() if use_mask else None, 0.5)
        lib.blt_backend_pass_sync(abi.BLT_BACKEND_HIP)
        assert_close(t.cpu().numpy(), ref, "softmax row")
    a, b = rs.randn(777).astype(np.float32), rs.randn(777).astype(np.float32)
    ta, tb = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    got = lib.blt_vec_dot(abi.BLT_BACKEND_HIP, ta.data_ptr(), tb.data_ptr(), 777)
    assert abs(got - float(np.dot(a.astype(np.float64), b.astype(np.float64)))) < 1e-3


DEAD_ROW_SNIPPETS = {
    # ranges exist: the host answers, no read-back (rows 7.. of a 10 x 5 causal window have no key left)
    "host_ranges": """
cfg = abi.BltMaskConfig(); cfg.seq_len_q, cfg.seq_len_kv = 10, 5
cfg.is_causal, cfg.sliding_window = True, 2
""",
    # interleaved groups: no ranges, the kernel flags live rows and the count is read back
    "device_flags": """
cfg = abi.BltMaskConfig(); cfg.seq_len_q, cfg.seq_len_kv = 3, 4
qg, kg = abi.size_array([0, 1, 2]), abi.size_array([0, 1, 0, 1])
cfg.query_group_ids, cfg.kv_group_ids, cfg.bidirectional_within_group = qg, kg, True
""",
}


@pytest.mark.parametrize("name", list(DEAD_ROW_SNIPPETS))
def test_mask_builder_dead_row_is_fatal(name, dev):
    """A query row without any allowed key ends the process with the reference's message
    (csrc/ops/mask_builder_cpu.c:93), on both ways the device builder has of finding it."""
    import subprocess
    import sys
    import os
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    code = ("import ctypes as C, sys\nsys.path.insert(0, %r)\nimport torch\nfrom fblt_amd import abi, api\n"
            "lib = api.load()\n" % root) + DEAD_ROW_SNIPPETS[name] + (
            "arena = lib.blt_arena_create(1 << 20, abi.BLT_BACKEND_HIP)\nt = abi.BltTensor()\n"
            "lib.blt_build_attention_mask(C.byref(cfg), C.byref(t), arena)\nlib.blt_backend_pass_sync_hip()\n"
            "print('SURVIVED')\n")
    p = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert p.returncode == 1, (p.returncode, p.stdout, p.stderr)
    assert "query position has no valid key" in p.stderr and "SURVIVED" not in p.stdout


@pytest.mark.parametrize("rows,src_rows,row_len", [(1, 7, 16), (5, 40, 33), (130, 512, 16), (300, 64, 64)])
def test_rows_gather(rows, src_rows, row_len, dev):
    """blt_rows_gather (csrc/ops/gather_scatter.h:41-42): dst[i, :] = src[pos[i], :], positions a host
    array, repeats allowed, more rows than one launch carries, row lengths that are not a multiple
    of four.  Copies are bit-exact."""
    import torch
    lib = api.load()
    rs = np.random.RandomState(rows + row_len)
    src = rs.randn(src_rows, row_len).astype(np.float32)
    pos = rs.randint(0, src_rows, size=rows)
    pos[-1] = src_rows - 1
    tsrc = torch.from_numpy(src).cuda()
    tdst = torch.full((rows, row_len), 7.0, dtype=torch.float32, device="cuda")
    vs, vd = _dev_tensor(tsrc), _dev_tensor(tdst)
    lib.blt_rows_gather(C.byref(vs), (C.c_size_t * rows)(*pos.tolist()), C.byref(vd))
    lib.blt_backend_pass_sync_hip()
    assert (tdst.cpu().numpy() == src[pos]).all()


def test_rope_position_gather(dev):
    """blt_rope_position_gather (csrc/infer/rope_gather.c:5-35): table rows of the given absolute
    positions as two new [n, half] arena tensors."""
    import torch
    lib = api.load()
    rs = np.random.RandomState(11)
    cos, sin = rs.randn(96, 16).astype(np.float32), rs.randn(96, 16).astype(np.float32)
    tc, ts = torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda()
    vc, vs = _dev_tensor(tc), _dev_tensor(ts)
    arena = lib.blt_arena_create(1 << 20, abi.BLT_BACKEND_HIP)
    pos = [40, 41, 42, 95, 0]
    oc, os_ = abi.BltTensor(), abi.BltTensor()
    lib.blt_rope_position_gather(C.byref(vc), C.byref(vs), (C.c_size_t * 5)(*pos), 5, C.byref(oc), C.byref(os_), arena)
    lib.blt_backend_pass_sync_hip()
    assert (oc.ndim, oc.shape[0], oc.shape[1], oc.backend) == (2, 5, 16, abi.BLT_BACKEND_HIP)
    got_c, got_s = np.empty((5, 16), dtype=np.float32), np.empty((5, 16), dtype=np.float32)
    lib.blt_hip_memcpy_d2h(got_c.ctypes.data, oc.data, got_c.nbytes)
    lib.blt_hip_memcpy_d2h(got_s.ctypes.data, os_.data, got_s.nbytes)
    lib.blt_arena_destroy(arena)
    assert (got_c == cos[pos]).all() and (got_s == sin[pos]).all()


@pytest.mark.parametrize("lens", ["host", "device"])
@pytest.mark.parametrize("batch,H,hd,n,lo,hi,kind,window,kernel", [
    (3, 4, 32, 17, 1, 3, "block", 0, "kv_block_once"), (9, 4, 32, 32, 0, 150, "causal", 0, "kv_block_once"),
    (5, 1, 32, 31, 20, 300, "causal", 40, "kv_block_once"), (9, 4, 32, 18, 0, 150, "causal", 9, "kv_block_once"),
    (2, 2, 64, 25, 100, 380, "block", 0, "kv_block_once"), (70, 4, 64, 17, 10, 70, "causal", 0, "kv_block_once"),
    (33, 4, 32, 20, 500, 690, "block", 0, "kv_block_once"), (33, 4, 32, 20, 500, 760, "block", 0, "kv_block_mfma"),   # past 48 tiles
    (32, 4, 32, 20, 500, 960, "block", 0, "kv_block_once"), (32, 4, 32, 17, 500, 1100, "causal", 700, "kv_block16_mfma"),
    (3, 1, 64, 32, 300, 700, "causal", 0, "kv_block16_mfma"), (33, 4, 64, 32, 400, 600, "block", 0, "kv_block_mfma"),
    (66, 4, 64, 32, 150, 200, "causal", 0, "kv_block_mfma"), (1, 3, 32, 32, 2000, 2300, "causal", 0, "kv_block_mfma")])
def test_kv_steps_of_two_row_tiles(batch, H, hd, n, lo, hi, kind, window, kernel, lens, dev, oracle):
    """Steps of 17 to 32 rows: a sequence's rows as two halves, a workgroup each, or all in one, by the rule's lines.  Two steps that
    commit, rows rotated inside; outputs against the restated step, the cache's rows bit for bit (either half stores), and the
    lengths that the last of a sequence's workgroups advances."""
    kw = workloads.config5(batch=batch, B=n, H=H, hd=hd, len_lo=lo, len_hi=hi, max_seq_len=hi + 2 * n, steps=2, rope=True)
    kw.kind, kw.window, kw.commit = kind, window, True
    ref_out, ref_k, ref_v = orunner.run_kv(kw, lib=oracle)
    d = dev.DeviceKvWorkload(kw, lens=lens)
    lib = api.load()
    lib.blt_hip_profile_begin()
    d.run()
    names = [name for name in api.profile_end() if name.startswith("kv_block")]
    out, ck, cv, got_lens = d.results()
    assert kernel in names, names  # the second step sees more keys
    assert_close(out, ref_out, "step rows")
    assert ck.tobytes() == ref_k.tobytes() and cv.tobytes() == ref_v.tobytes()
    assert (np.asarray(got_lens).astype(np.int64) == kw.lens.astype(np.int64) + 2 * n).all()


@pytest.mark.parametrize("kernel", ["valu", "mfma", "mfma_once", "mfma_loop", "mfma32"])
def test_kv_step_kernel_families_agree(kernel):
    """The kernels behind the KV step entry points (VALU; matrix-core as routed; the all-at-once kernel
    wherever it takes the shape; the looping kernels only -- 4x4x1 tiles up to four rows, 16-wide tiles
    up to 16; 32-wide tiles only) on the same cases -- block rows, prefill chunks, rotation fused in or
    not -- pinned through BLT_HIP_BLOCK_KERNEL / BLT_HIP_BLOCK_TILE in a fresh process (the hooks are
    read once)."""
    import subprocess
    import sys
    import os
    here = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, BLT_HIP_BLOCK_KERNEL=kernel[:4])
    tile = {"mfma32": "32", "mfma_once": "once", "mfma_loop": "4"}.get(kernel)
    if tile:
        env["BLT_HIP_BLOCK_TILE"] = tile
    p = subprocess.run([sys.executable, "-u", os.path.join(here, "kv_family_cases.py")], capture_output=True,
                       text=True, timeout=600, env=env)
    assert p.returncode == 0 and "OK" in p.stdout, p.stdout[-2000:] + p.stderr[-2000:]


@pytest.mark.parametrize("family", ["rows", "mfma", "wide", "fine", "fine16", "fine128", "once"])
def test_attention_kernel_families(family):
    """Every attention kernel family on the same cases (causal, chunked prefill, sliding window,
    dense masks, lse output), pinned through BLT_HIP_ATTN_FAMILY in a fresh process; the fine
    kernel in its workgroup shapes (BLT_HIP_FINE_ROWS: 32 rows and eight waves, 16 rows and
    sixteen waves wherever the batch is strided, whole problems of up to 128 rows on four waves
    wherever the batch is strided and the keys fit one fill)."""
    import subprocess
    import sys
    import os
    here = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, BLT_HIP_ATTN_FAMILY=family)
    shape = family
    if family.startswith("fine"):
        env["BLT_HIP_ATTN_FAMILY"] = "fine"
        env["BLT_HIP_FINE_ROWS"] = {"fine": "32", "fine16": "16", "fine128": "128"}[family]
        family = "fine"
    p = subprocess.run([sys.executable, "-u", os.path.join(here, "family_cases.py")], capture_output=True, text=True,
                       timeout=600, env=env)
    assert p.returncode == 0 and "OK" in p.stdout, p.stdout[-2000:] + p.stderr[-2000:]
    kernels = [ln for ln in p.stdout.splitlines() if ln.startswith("KERNELS")][0].split()[1]
    assert kernels == family, kernels
    launched = [ln for ln in p.stdout.splitlines() if ln.startswith("LAUNCHED")][0].split()[1].split(",")
    if family == "fine":
        assert ("attn_whole" in launched) == (shape == "fine128"), launched


@pytest.mark.parametrize("kernel,batch,H,hd,nq,nk,window", [
    ("wide", 24, 4, 32, 1025, 1025, 0), ("wide", 24, 4, 32, 1281, 1313, 0),   # eight waves: a group of one row, an offset diagonal
    ("wide", 32, 5, 32, 520, 520, 0), ("wide", 64, 2, 64, 513, 600, 40),      # four waves: ragged last group; short windows
    ("wide", 24, 8, 64, 300, 300, 0),
    ("mfma", 3, 2, 32, 777, 777, 0), ("mfma", 3, 4, 64, 801, 801, 100), ("mfma", 3, 2, 128, 225, 300, 0),
    ("mfma", 3, 2, 40, 130, 130, 0)])                                          # heads of 40: elements with a guard
def test_attention_on_split_operands(kernel, batch, H, hd, nq, nk, window, dev):
    """The kernels that work on bf16 parts against float64, then with values that are not finite in one problem: a key with
    such a score leaves the softmax, the other columns of a bad value row and all other problems stay as they were."""
    import torch
    w = workloads.offset_causal(batch=batch, nq=nq, nk=nk, H=H, hd=hd, window=window)
    d = dev.DeviceWorkload(w)
    lib = api.load()
    E = H * hd
    i, j = torch.arange(nq, device="cuda")[:, None], torch.arange(nk, device="cuda")[None, :]
    seen = j <= i + nk - nq
    if window:
        seen &= j > i + nk - nq - window

    def run():
        d.zero_outputs()
        plan = d.make_plan("descriptor")
        assert lib.blt_attention_plan_kernel_hip(plan) == kernel.encode()
        lib.blt_attention_plan_run_hip(plan)
        lib.blt_backend_pass_sync_hip()
        lib.blt_attention_plan_destroy_hip(plan)
        return torch.from_numpy(d.output("out").copy()).cuda().view(batch, nq, H, hd)

    def want(b, head, dropped=None):
        q, k, v = (d.dev[n].view(batch, -1, H, hd)[b, :, head].double() for n in ("q", "k", "v"))
        s = (q @ k.T.contiguous()) * w.heads[0].scale
        keep = seen if dropped is None else seen & (j != dropped)
        p = torch.softmax(s.masked_fill(~keep, float("-inf")), dim=1)
        return (p @ v.nan_to_num(0.0, 0.0, 0.0)).float()

    try:
        first = run()
        for b, head in ((0, 0), (batch - 1, H - 1), (batch // 2, H // 2)):
            assert_close(first[b, :, head].cpu().numpy(), want(b, head).cpu().numpy(), "problem %d/%d" % (b, head))
        d.dev["k"].view(batch, nk, H, hd)[1, 7, 1, 3] = float("nan")
        d.dev["v"].view(batch, nk, H, hd)[2, 40, 0, 5] = float("inf")
        torch.cuda.synchronize()
        got = run()
        assert_close(got[1, :, 1].cpu().numpy(), want(1, 1, dropped=7).cpu().numpy(), "a key that is not finite")
        rows = seen[:, 40]
        assert torch.isinf(got[2, rows, 0, 5]).all() and (got[2, rows, 0, 5] > 0).all()
        others = [c for c in range(hd) if c != 5]
        assert_close(got[2, :, 0][:, others].cpu().numpy(), want(2, 0)[:, others].cpu().numpy(), "columns beside the bad one")
        got[1, :, 1], got[2, :, 0] = first[1, :, 1], first[2, :, 0]
        assert torch.equal(got, first)
    finally:
        d.close()


@pytest.mark.parametrize("batch,H,hd,nq,nk", [(24, 4, 32, 1025, 1025), (64, 2, 32, 513, 600), (24, 8, 64, 300, 300)])
def test_attention_on_halves_out_of_range(batch, H, hd, nq, nk, dev):
    """The large-batch kernel takes K and V apart into f16 parts where runs of them lie within 2^-17 .. 4094, and a group of rows
    whose keys do not is run again on bf16 parts: below, above, at zero, with one value or one column outside, within at both
    ends.  Each column against float64 in the 2-norm: a value is within 2^-23, a product within 2^-21, scores of at most 8 in
    log2 units double that in a weight; 2^-19 in all."""
    import torch
    w = workloads.offset_causal(batch=batch, nq=nq, nk=nk, H=H, hd=hd)
    d = dev.DeviceWorkload(w)
    lib = api.load()
    try:
        q, k, v = (d.dev[n].view(batch, -1, H, hd) for n in ("q", "k", "v"))
        v[1] *= 1e-7                                 # all of V below
        q[2] *= 1e-5
        k[2] *= 1e5                                  # all of K above
        v[3, nk // 2, :, 1] = 3e4                    # one value above, met half way
        k[4] = 0.0
        v[5, :, :, 2] *= 1e-8                        # a column below, the others not
        k[6] *= 2.0 ** -6
        v[6] *= 2.0 ** -8                            # within
        v[7] *= 500.0
        k[8, :, 1] *= 1e-9                           # the keys of one head below
        torch.cuda.synchronize()
        d.zero_outputs()
        plan = d.make_plan("descriptor")
        assert lib.blt_attention_plan_kernel_hip(plan) == b"wide"
        lib.blt_attention_plan_run_hip(plan)
        lib.blt_backend_pass_sync_hip()
        lib.blt_attention_plan_destroy_hip(plan)
        got = torch.from_numpy(d.output("out").copy()).cuda().view(batch, nq, H, hd).double()
        i, j = torch.arange(nq, device="cuda")[:, None], torch.arange(nk, device="cuda")[None, :]
        for b in range(10):
            for head in (0, 1):
                s = (q[b, :, head].double() @ k[b, :, head].double().T.contiguous()) * w.heads[0].scale
                want = torch.softmax(s.masked_fill(j > i + nk - nq, float("-inf")), dim=1) @ v[b, :, head].double()
                error = (got[b, :, head] - want).norm(dim=0) / want.norm(dim=0)
                assert error.max().item() < 2.0 ** -19, (b, head, error.max().item())
    finally:
        d.close()


@pytest.mark.parametrize("batch,H,hd,nq,nk", [(32, 4, 32, 1025, 1025), (24, 8, 64, 300, 300), (64, 4, 32, 300, 300)])
def test_attention_whose_small_values_carry_the_result(batch, H, hd, nq, nk, dev):
    """f16 parts hold weights, keys and values to a fraction of the largest, so a group of rows whose output hangs on small ones
    beside large ones runs again on bf16 parts: a first key of nearly all the weight and no value, a row whose one key is far
    smaller than its neighbours, queries whose large columns meet small ones of the keys.  Each row against float64 in the
    2-norm, relative to the sum of its terms' magnitudes: scores of up to 42 in log2 units that fp32 rounds twelve times are off by
    42 sqrt(12) 2^-24 typically and three times that at most, 2^-16 in a weight; nothing else comes near that."""
    import torch
    w = workloads.offset_causal(batch=batch, nq=nq, nk=nk, H=H, hd=hd)
    d = dev.DeviceWorkload(w)
    lib = api.load()
    scale = w.heads[0].scale
    try:
        q, k, v = (d.dev[n].view(batch, -1, H, hd) for n in ("q", "k", "v"))
        for b, bits in ((1, 14.0), (2, 24.0), (3, 36.0)):  # the first key ahead of the others by so many powers of two
            q[b, :, :, 0], k[b, :, :, 0] = 4.0, 0.0
            k[b, 0, :, 0] = bits * 0.6931 / (4.0 * scale)
            v[b, 0] = 0.0
        v[4, 0] *= 1e-8
        v[5, 0] *= 1e-11
        q[6, :, :, 1:] *= 1e8
        k[6, :, :, 1:] *= 1e-8
        q[6, :, :, 0], k[6, :, :, 0] = 0.0, 1.0
        q[7, :, 0, 1:] *= 1e-8
        k[7, :, 0, 1:] *= 1e8
        k[7, :, 0, 0] = 0.0
        torch.cuda.synchronize()
        d.zero_outputs()
        plan = d.make_plan("descriptor")
        assert lib.blt_attention_plan_kernel_hip(plan) == b"wide"
        lib.blt_attention_plan_run_hip(plan)
        lib.blt_backend_pass_sync_hip()
        lib.blt_attention_plan_destroy_hip(plan)
        got = torch.from_numpy(d.output("out").copy()).cuda().view(batch, nq, H, hd).double()
        i, j = torch.arange(nq, device="cuda")[:, None], torch.arange(nk, device="cuda")[None, :]
        for b in range(9):
            for head in (0, H - 1):
                s = (q[b, :, head].double() @ k[b, :, head].double().T.contiguous()) * scale
                p, x = torch.softmax(s.masked_fill(j > i + nk - nq, float("-inf")), dim=1), v[b, :, head].double()
                off, size = (got[b, :, head] - p @ x).norm(dim=1), (p @ x.abs()).norm(dim=1)
                worst = (off / size.clamp_min(1e-300)).max().item()
                assert worst <= 2.0 ** -16, (b, head, worst)
    finally:
        d.close()


@pytest.mark.parametrize("batch,H,hd,nq,nk,window", [
    (32, 4, 32, 1025, 1025, 0), (64, 4, 32, 300, 333, 0), (64, 4, 32, 520, 520, 65),       # eight waves, four, windows
    (64, 4, 32, 520, 520, 255), (64, 4, 32, 520, 520, 256), (32, 4, 32, 390, 411, 64),     # both sides of the line for windows
    (48, 4, 64, 510, 510, 0), (48, 4, 64, 512, 512, 0), (32, 2, 64, 1030, 1061, 0),        # both sides of the line for heads of 64
    (48, 4, 64, 640, 640, 319), (48, 4, 64, 640, 640, 320)])
def test_attention_weighed_before_its_maximum(batch, H, hd, nq, nk, window, dev):
    """The large-batch kernel weighs a tile against the maximum so far and looks for a new one only where the weights add up to
    too much: scores that rise all along a row, stand still, fall, jump near its end, or are the same everywhere; a window that
    some rows of a tile enter later than others; and a column of V that is nothing but zeros until values too small for f16
    parts come.  Against float64, column by column in the 2-norm, relative to the sum of the terms' magnitudes: scores of up to 42 in
    log2 units that fp32 rounds twelve times are off by 42 sqrt(12) 2^-24 typically and three times that at most, 2^-16 in a weight."""
    import torch
    w = workloads.offset_causal(batch=batch, nq=nq, nk=nk, H=H, hd=hd, window=window)
    d = dev.DeviceWorkload(w)
    lib = api.load()
    scale = w.heads[0].scale
    try:
        q, k, v = (d.dev[n].view(batch, -1, H, hd) for n in ("q", "k", "v"))
        ramp = torch.arange(nk, device="cuda", dtype=torch.float32)[:, None] / nk
        for b, column in ((1, ramp * 40), (2, -ramp * 40), (3, torch.zeros_like(ramp)), (4, (ramp > 0.7) * 30.0), (5, (ramp > 0.98) * 3.5)):
            q[b, :, :, 0], k[b, :, :, 0] = 1.0, column * (0.6931 / scale)
            q[b, :, :, 1:] *= 0.0 if b == 3 else 0.3
        v[6, : nk - 50, :, 3] = 0.0
        v[6, nk - 50 :, :, 3] *= 1e-8
        torch.cuda.synchronize()
        d.zero_outputs()
        plan = d.make_plan("descriptor")
        assert lib.blt_attention_plan_kernel_hip(plan) == b"wide"
        lib.blt_attention_plan_run_hip(plan)
        lib.blt_backend_pass_sync_hip()
        lib.blt_attention_plan_destroy_hip(plan)
        got = torch.from_numpy(d.output("out").copy()).cuda().view(batch, nq, H, hd).double()
        i, j = torch.arange(nq, device="cuda")[:, None] + nk - nq, torch.arange(nk, device="cuda")[None, :]
        keep = (j <= i) & (j > i - window) if window else j <= i
        for b in range(8):
            for head in (0, H - 1):
                s = (q[b, :, head].double() @ k[b, :, head].double().T.contiguous()) * scale
                p, x = torch.softmax(s.masked_fill(~keep, float("-inf")), dim=1), v[b, :, head].double()
                off, size = (got[b, :, head] - p @ x).norm(dim=0), (p @ x.abs()).norm(dim=0)
                worst = (off / size.clamp_min(1e-300)).max().item()
                assert worst <= 2.0 ** -16, (b, head, worst)
    finally:
        d.close()


@pytest.mark.parametrize("batch,T,window,hd,mixed,kernel", [
    (65, 129, 0, 32, False, "attn_wide_brief"), (64, 129, 0, 32, False, "attn_wide"), (65, 129, 0, 64, False, "attn_wide"),
    (22, 700, 128, 32, False, "attn_wide_brief"), (22, 700, 129, 32, False, "attn_wide"), (44, 383, 0, 32, True, "attn_wide_brief"),
    (44, 385, 0, 32, False, "attn_wide"), (48, 300, 1, 32, True, "attn_wide_brief"), (70, 200, 33, 32, True, "attn_wide_brief")])
def test_attention_of_many_short_rows(batch, T, window, hd, mixed, kernel, dev):
    """Causal launches of many short or windowed rows take the large-batch kernel's bf16 form at once: both sides of its lines, in
    strided batches and in batches of two lengths, with values that no f16 holds, against float64."""
    import torch
    lib, H = api.load(), 4
    lengths = [T - (3 if mixed and b % 2 else 0) for b in range(batch)]
    q, k, v = (torch.randn(batch, T, H, hd, device="cuda") for _ in range(3))
    v[1], k[2] = v[1] * 1e30, k[2] * 1e-30
    out = torch.full_like(q, 7.0)
    probs = [api.problem(api.head_args(*(t[b, :, h].data_ptr() for t in (q, k, v, out)), n, n, hd, float(hd) ** -0.5, H * hd, H * hd,
                                       H * hd, H * hd, 0), api.BLT_ATTN_MASK_CAUSAL, window=window)
             for b, n in enumerate(lengths) for h in range(H)]
    torch.cuda.synchronize()
    lib.blt_hip_profile_begin()
    lib.blt_attention_batch_hip(api.problem_array(probs), len(probs))
    lib.blt_backend_pass_sync_hip()
    assert [name for name in api.profile_end() if name.startswith("attn")] == [kernel]
    i = torch.arange(T, device="cuda")
    keep = (i[None] <= i[:, None]) & ((i[None] + window > i[:, None]) if window else True)
    for b in (0, 1, 2, batch // 2, batch - 1):
        n, size = lengths[b], 1e30 if b == 1 else 1.0
        for h in (0, H - 1):
            s = (q[b, :n, h].double() @ k[b, :n, h].double().T.contiguous()) * float(hd) ** -0.5
            want = torch.softmax(s.masked_fill(~keep[:n, :n], float("-inf")), dim=1) @ v[b, :n, h].double()
            assert_close((out[b, :n, h].double() / size).cpu().numpy(), (want / size).cpu().numpy(), "problem %d/%d" % (b, h))
    if mixed:
        assert bool((out[1, T - 3:] == 7.0).all())


@pytest.mark.parametrize("family", ["auto", "rows", "mfma", "wide", "fine", "fine16", "fine128", "once"])
def test_attention_random_shapes(family):
    """72 randomly shaped strided batches per routing (automatic, and every family / workgroup shape
    pinned wherever the shape allows it) through the one-shot batch entry and a plan, against the
    checker (tests/random_cases.py, fresh process: the routing hooks are read once)."""
    import subprocess
    import sys
    import os
    here = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ)
    if family.startswith("fine"):
        env["BLT_HIP_ATTN_FAMILY"] = "fine"
        env["BLT_HIP_FINE_ROWS"] = {"fine": "32", "fine16": "16", "fine128": "128"}[family]
    elif family != "auto":
        env["BLT_HIP_ATTN_FAMILY"] = family
    p = subprocess.run([sys.executable, "-u", os.path.join(here, "random_cases.py"), "11", "12", "13", "14", "15", "16"],
                       capture_output=True, text=True, timeout=600, env=env)
    assert p.returncode == 0 and "OK" in p.stdout, p.stdout[-2000:] + p.stderr[-2000:]
    launched = [ln for ln in p.stdout.splitlines() if ln.startswith("LAUNCHED")][0].split()[1].split(",")
    if family == "fine128":
        assert "attn_whole" in launched, launched
    if family == "once":
        assert "attn_once" in launched, launched


@pytest.mark.parametrize("case", ["decode", "chunk5", "block16", "packed"])
def test_kv_rope_step(case, oracle, dev):
    """blt_kv_rope_attend_step_hip: rotation of the new Q/K rows fused into the step.  Rotated K rows
    land in the cache bit for bit as the reference's blt_rope_apply writes them."""
    import torch
    if case == "decode":
        kw = workloads.config4(batch=11, steps=6, len_hi=300, rope=True)
    elif case == "chunk5":
        kw = workloads.config4(batch=6, steps=3, len_hi=100, max_seq_len=100 + 15, rope=True)
        rs = np.random.RandomState(5)
        kw.n = 5
        kw.q_new, kw.k_new, kw.v_new = (rs.randn(kw.steps, kw.batch * 5, kw.E).astype(np.float32) for _ in range(3))
    elif case == "block16":
        kw = workloads.config5(batch=8, B=16, rope=True)
    else:
        kw = workloads.config4(batch=4, steps=1, len_hi=60, rope=True)
    ref_out, ref_k, ref_v = orunner.run_kv(kw, lib=oracle)
    d = dev.DeviceKvWorkload(kw)
    if case == "packed":
        # the three column blocks of one packed [batch*n, 3E] buffer, row stride 3E
        E = kw.E
        qkv = torch.from_numpy(np.concatenate([kw.q_new[0], kw.k_new[0], kw.v_new[0]], axis=1)).cuda()
        d.lib.blt_kv_rope_attend_step_hip(C.byref(d.c), qkv.data_ptr(), 3 * E, qkv.data_ptr() + 4 * E, 3 * E,
                                          qkv.data_ptr() + 8 * E, 3 * E, d.rope[0].data_ptr(), d.rope[1].data_ptr(),
                                          d.rope[0].shape[0], d.out[0].data_ptr(), E, kw.n, d.kind, 1,
                                          d.host_max_len + kw.n)
        d.lib.blt_backend_pass_sync_hip()
    else:
        d.run()
    out, ck, cv, lens = d.results()
    assert ck.tobytes() == ref_k.tobytes() and cv.tobytes() == ref_v.tobytes()
    assert_close(out, ref_out, "rope " + case)
    if kw.commit:
        assert (lens == kw.lens + kw.n * kw.steps).all()


# ---------------------------------------------------------------------------
# projections, rotation and the attention block
# ---------------------------------------------------------------------------
def _dev_tensor(t, shape=None):
    return abi.tensor_view(t.data_ptr(), tuple(t.shape) if shape is None else shape, abi.BLT_BACKEND_HIP)


@pytest.mark.parametrize("m,n", [(2048, 1536), (2049, 1537), (1024, 512), (1030, 515), (640, 512), (577, 450)])
@pytest.mark.parametrize("k", [20, 32, 64, 70, 96, 128, 160, 186, 384, 448, 455, 512])
def test_matmul_whole_steps(m, n, k):
    """The tile kernels' loop takes whole steps of K (32 or 64) in pairs: none, one, odd and even counts, with and without a rest,
    on both tiles and both forms of the operands, and the 32 x 32 tiles below them.  Against float64: a sum of k fp32 products is within k 2^-24 of the
    sum of their magnitudes whatever its order, and rounding to fp32 adds less."""
    import torch
    lib = api.load()
    rs = np.random.RandomState(m + 3 * n + 7 * k)
    a, b = rs.randn(m, k).astype(np.float32), (rs.randn(k, n) / np.sqrt(k)).astype(np.float32)
    ta, tb, to = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda(), torch.full((m, n), 7.0, device="cuda")
    va, vb, vo = _dev_tensor(ta), _dev_tensor(tb), _dev_tensor(to)
    lib.blt_matmul(C.byref(va), C.byref(vb), C.byref(vo))
    a, b = a.astype(np.float64), b.astype(np.float64)
    off = np.abs(to.cpu().numpy() - a @ b)
    assert (off <= (k + 1) * 2.0 ** -24 * (np.abs(a) @ np.abs(b))).all()


def _product_kernel(m, k, n):
    """The kernel that a plain product of more than 64 rows is to take, and over how many slices of K."""
    tiles, small = -(-m // 64) * -(-n // 64), -(-m // 32) * -(-n // 32)
    whole = "matmul_mfma" if tiles >= 112 else "matmul_splitk"
    if k < 1024 or not 16 <= tiles <= 128 or tiles * k < 80 * 1024 or (tiles < 112 and small <= 128):
        return whole, 1
    least = 2 if tiles >= 112 else 3 if k <= 2560 else 4
    for slices in range(min(256 // tiles if tiles >= 112 else max(256 // tiles, least), k // 384), least - 1, -1):
        run = -(-(-(-k // slices)) // 64) * 64
        if k - (slices - 1) * run >= 384:
            return "matmul_mfma_slices", slices
    return whole, 1


@pytest.mark.parametrize("m,n", [(65, 1025), (301, 512), (641, 449), (1000, 512), (1024, 515), (577, 450), (897, 508), (290, 460)])
@pytest.mark.parametrize("k", [1023, 1024, 1025, 1530, 2048, 2049, 2500, 5200])
def test_matmul_tiles_in_slices(m, n, k):
    """16 to 128 tiles of 64 x 64 and a long K: up to six workgroups a tile, each with its run of K, odd rests among them, and the shapes
    beside the rule's lines that stay whole; the bound of test_matmul_whole_steps (one more rounding a slice).  The same bits whoever
    comes last and wherever the output lies, and an infinity in one slice is one in the result."""
    import torch
    lib = api.load()
    rs = np.random.RandomState(m + 3 * n + 7 * k)
    a, b = rs.randn(m, k).astype(np.float32), (rs.randn(k, n) / np.sqrt(k)).astype(np.float32)
    ta, tb = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    outs = [torch.full((m, n), 7.0, device="cuda") for _ in range(2)]
    outs.append(torch.full((m * n + 1,), 7.0, device="cuda")[1:].view(m, n))     # off a 16-byte boundary
    va, vb = _dev_tensor(ta), _dev_tensor(tb)
    torch.cuda.synchronize()
    lib.blt_hip_profile_begin()
    for out in outs:
        vo = _dev_tensor(out)
        lib.blt_matmul(C.byref(va), C.byref(vb), C.byref(vo))
    launched = api.profile_end()
    launched.pop("matmul_clear_words", None)
    assert {name: v[0] for name, v in launched.items()} == {_product_kernel(m, k, n)[0]: 3}, launched
    got = [out.cpu().numpy() for out in outs]
    assert got[0].tobytes() == got[1].tobytes() == got[2].tobytes()
    a, b = a.astype(np.float64), b.astype(np.float64)
    assert (np.abs(got[0] - a @ b) <= (k + 16) * 2.0 ** -24 * (np.abs(a) @ np.abs(b))).all()
    ta[5, k - 3] = float("inf")
    lib.blt_matmul(C.byref(va), C.byref(vb), C.byref(vo))
    row = outs[2].cpu().numpy()
    assert (row[5] == np.where(tb[k - 3].cpu().numpy() > 0, np.inf, -np.inf)).all()
    assert np.isfinite(np.delete(row, 5, 0)).all()


@pytest.mark.parametrize("m,k,n,exact", [(1, 128, 384, True), (5, 33, 17, True), (32, 512, 512, True),
                                          (3, 1100, 70, True), (1, 7, 300, True), (9, 528, 257, True),
                                          (16, 128, 512, True), (33, 64, 64, False), (64, 128, 384, False),
                                          (512, 128, 384, False), (100, 70, 50, False), (513, 129, 130, False),
                                          (2048, 512, 1536, False), (4100, 70, 2050, False), (4096, 96, 2048, False),
                                          (1500, 300, 600, False), (1100, 257, 1030, False), (2048, 2048, 512, False),
                                          (118, 2048, 512, False), (64, 4096, 256, False), (100, 3000, 70, False), (33, 1025, 40, False)])
def test_matmul(m, k, n, exact, oracle, dev):
    """blt_matmul: up to 32 rows bit-identical to the reference loop, above that fp32 tolerance."""
    import torch
    lib = api.load()
    rs = np.random.RandomState(m + k + n)
    a = rs.randn(m, k).astype(np.float32)
    b = (rs.randn(k, n) / np.sqrt(k)).astype(np.float32)
    ref = np.zeros((m, n), dtype=np.float32)
    oracle.orc_matmul(binding.fptr(a.reshape(-1)), binding.fptr(b.reshape(-1)), binding.fptr(ref.reshape(-1)), m, k, n)
    ta, tb = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    to = torch.full((m, n), 7.0, dtype=torch.float32, device="cuda")
    va, vb, vo = _dev_tensor(ta), _dev_tensor(tb), _dev_tensor(to)
    lib.blt_matmul(C.byref(va), C.byref(vb), C.byref(vo))
    lib.blt_backend_pass_sync_hip()
    got = to.cpu().numpy()
    if exact:
        assert got.tobytes() == ref.tobytes()
    else:
        assert_close(got, ref, "matmul %dx%dx%d" % (m, k, n))


@pytest.mark.parametrize("m,k,n", [(512, 256, 512), (513, 256, 512), (511, 300, 544), (33, 256, 4064), (200, 1000, 1150), (384, 380, 1020)])
def test_matmul_of_two_small_tiles_a_compute_unit(m, k, n, dev):
    """Products of 256 small tiles and of more, that share compute units, against float64."""
    import torch
    lib = api.load()
    a, b = torch.randn(m, k, device="cuda"), torch.randn(k, n, device="cuda")
    out = torch.full((m, n), 7.0, device="cuda")
    va, vb, vo = _dev_tensor(a), _dev_tensor(b), _dev_tensor(out)
    torch.cuda.synchronize()
    lib.blt_hip_profile_begin()
    lib.blt_matmul(C.byref(va), C.byref(vb), C.byref(vo))
    assert set(api.profile_end()) == {"matmul_splitk"}
    lib.blt_backend_pass_sync_hip()
    assert _relative(out, a.double() @ b.double()) <= 3 * 2.0 ** -24 * k ** 0.5   # as of products on parts


@pytest.mark.parametrize("m,k,n", [(769, 1, 769), (800, 33, 772), (1025, 512, 1540), (2049, 96, 2050), (770, 130, 771)])
def test_matmul_on_split_operands(m, k, n, dev):
    """Both tile sizes of the product on bf16 parts at ragged edges against float64, then with values that are not finite:
    what they take part in is what fp32 sums give, everything else stays."""
    import torch
    lib = api.load()
    a, b = torch.randn(m, k, device="cuda"), torch.randn(k, n, device="cuda") / k ** 0.5
    out = torch.full((m, n), 7.0, device="cuda")

    def product():
        va, vb, vo = _dev_tensor(a), _dev_tensor(b), _dev_tensor(out)
        torch.cuda.synchronize()
        lib.blt_matmul(C.byref(va), C.byref(vb), C.byref(vo))
        lib.blt_backend_pass_sync_hip()
        return out.clone()

    first = product()
    assert_close(first.cpu().numpy(), (a.double() @ b.double()).float().cpu().numpy(), "matmul %dx%dx%d" % (m, k, n))
    a[5, k - 1], a[m - 1, 0], b[0, n - 1] = float("inf"), float("nan"), 3.4e38
    got = product()
    inf = (a[5, :, None].cpu() * b.cpu()).sum(dim=0)  # one infinity in each sum: infinite with its sign
    assert torch.equal(got[5, :n - 1].cpu(), inf[:n - 1]) and torch.isnan(got[m - 1]).all()
    want = torch.outer(a[:, 0].cpu(), b[0, n - 1:].cpu())[:, 0] if k == 1 else (a.cpu() @ b[:, n - 1].cpu())
    big = [i for i in range(m) if i not in (5, m - 1)]
    last = got[big, n - 1].cpu()
    assert torch.equal(torch.isinf(last), torch.isinf(want[big])) and torch.equal(torch.sign(last), torch.sign(want[big]))
    assert_close(got[big][:, :n - 1].cpu().numpy(), first[big][:, :n - 1].cpu().numpy(), "beside the bad values")


@pytest.mark.parametrize("T,hd,dense", [(300, 48, False), (300, 128, False), (1200, 32, True), (1200, 64, False), (130, 2, False)])
def test_weights_and_output_share_their_scores(T, hd, dense, dev):
    """Weights taken after the output: they sum to one even where scores are large (a score of a thousand has a rounding
    error of 6e-5, which cancels only if maximum, sum and weight use the same score), and an output stored in place of the
    queries does not change them."""
    import torch
    lib = api.load()
    q, k, v = (torch.randn(T, hd, device="cuda") * s for s in (30.0, 3.0, 1.0))
    out, weights = torch.full_like(q, 7.0), torch.full((2, T, T), 7.0, device="cuda")
    mask = torch.triu(torch.full((T, T), -float("inf"), device="cuda"), 1) if dense else None
    scale = float(hd) ** -0.5

    def run(to, w):
        a = api.head_args(q.data_ptr(), k.data_ptr(), v.data_ptr(), to.data_ptr(), T, T, hd, scale, hd, hd, hd, hd, 0,
                          weights=w.data_ptr(), mask=mask.data_ptr() if dense else None, causal=not dense)
        torch.cuda.synchronize()
        lib.blt_attention_head_core(abi.BLT_BACKEND_HIP, C.byref(a))
        lib.blt_backend_pass_sync_hip()

    run(out, weights[0])
    # nk roundings of 2^-24 of weights that sum to one, at random, and the exponentials' own
    assert float((weights[0].double().sum(-1) - 1).abs().max()) <= 6e-7
    run(q, weights[1])
    assert torch.equal(weights[0], weights[1]) and torch.equal(out, q)


@pytest.mark.parametrize("T,H,hd,batch", [(256, 4, 32, 80), (256, 4, 64, 80), (2304, 4, 32, 16), (300, 1, 128, 1)])
def test_second_run_reads_queries_in_place_of_the_output(T, H, hd, batch, dev):
    """One query row that is not finite sends its group through the kernels' second run; with the output in place of the
    queries it gives what it gives beside them."""
    import torch
    lib = api.load()
    q, k, v = (torch.randn(batch, H, T, hd, device="cuda") for _ in range(3))
    q[0, 0, T // 2 + 3, 1] = float("inf")
    got = []
    for to in (torch.full_like(q, 7.0), q):
        probs = [api.problem(api.head_args(*(t[b, h].data_ptr() for t in (q, k, v, to)), T, T, hd, float(hd) ** -0.5, hd, hd, hd,
                                           hd, 0), api.BLT_ATTN_MASK_CAUSAL) for b in range(batch) for h in range(H)]
        torch.cuda.synchronize()
        lib.blt_attention_batch_hip(api.problem_array(probs), len(probs))
        lib.blt_backend_pass_sync_hip()
        got.append(to)
    assert torch.equal(got[0], got[1]) and bool(torch.isfinite(got[0]).all())


def _relative(got, ref):
    return float((got.double() - ref).norm() / ref.norm())


@pytest.mark.parametrize("scale_a,scale_b", [(1.0, 1.0), (1e-36, 1.0), (1.0, 1e-38), (1e-40, 1e33), (1e-37, 1e30), (1e16, 1e16)])
@pytest.mark.parametrize("m,k,n", [(1024, 6, 1024), (1030, 512, 1026), (2048, 33, 2048)])
def test_matmul_over_the_range_of_fp32(m, k, n, scale_a, scale_b, dev):
    """Products on bf16 parts hold their operands in all 24 bits down to subnormals, and results too large for the
    scaled sums are as close: within what a chain of k fp32 additions gives (2^-24 sqrt(k) and a factor of three for
    the roundings of the operands' products)."""
    import torch
    lib = api.load()
    a, b = torch.randn(m, k, device="cuda") * scale_a, torch.randn(k, n, device="cuda") * scale_b
    out = torch.full((m, n), 7.0, device="cuda")
    va, vb, vo = _dev_tensor(a), _dev_tensor(b), _dev_tensor(out)
    torch.cuda.synchronize()
    lib.blt_matmul(C.byref(va), C.byref(vb), C.byref(vo))
    lib.blt_backend_pass_sync_hip()
    assert _relative(out, a.double() @ b.double()) <= 3 * 2.0 ** -24 * max(k, 4) ** 0.5


@pytest.mark.parametrize("m,k,n", [(700, 400, 720), (2048, 160, 1290), (2050, 514, 2049)])
@pytest.mark.parametrize("what", ["both", "one row", "one column", "zeros"])
def test_matmul_whose_small_values_carry_the_result(m, k, n, what, dev):
    """f16 parts hold an operand to a fraction of its largest, so a tile in which a row or a column of the product comes from small
    values against large ones only -- [1, x] . [x, 1] -- starts again on bf16 parts; rows and columns of nothing but zeros
    beside it are zeros.  Each row and each column against float64 in the 2-norm: 2^-24 for each of the sqrt(K) roundings that
    count, and 2^-22 for the parts."""
    import torch
    lib = api.load()
    x = 1e-9
    a, b = torch.randn(m, k, device="cuda"), torch.randn(k, n, device="cuda")
    small, large = torch.arange(k, device="cuda") % 2 == 1, torch.arange(k, device="cuda") % 2 == 0
    if what == "both":
        a[:, small] *= x
        b[large] *= x
    elif what == "one row":
        a[m - 2, small] *= x
        b[large] *= x
    elif what == "one column":
        a[:, small] *= x
        b[large, n - 2] *= x
    else:
        a[3:9], a[m - 1], b[:, 5], b[:, n - 40:] = 0.0, 0.0, 0.0, 0.0
    out = torch.full((m, n), 7.0, device="cuda")
    va, vb, vo = _dev_tensor(a), _dev_tensor(b), _dev_tensor(out)
    torch.cuda.synchronize()
    lib.blt_hip_profile_begin()
    lib.blt_matmul(C.byref(va), C.byref(vb), C.byref(vo))
    lib.blt_backend_pass_sync_hip()
    assert list(api.profile_end()) == ["matmul_mfma"]
    want = a.double() @ b.double()
    for dim in (0, 1):
        off, size = (out.double() - want).norm(dim=dim), want.norm(dim=dim)
        worst = (off / size.clamp_min(1e-300)).max().item()
        assert worst <= 2.0 ** -24 * k ** 0.5 + 2.0 ** -22, (dim, worst)


@pytest.mark.parametrize("m,k,n", [
    (640, 2048, 512), (301, 2048, 512), (420, 1536, 512), (577, 2309, 500), (513, 4099, 320),    # 64 x 64 tiles in slices
    (700, 2048, 512), (513, 3071, 512), (640, 2048, 640), (820, 1300, 500),                      # more than 256 workgroups
    (800, 1024, 512), (300, 4096, 256),                                                          # too few slices, too few tiles
    (580, 512, 512), (180, 512, 1520), (645, 386, 512), (512, 768, 540), (448, 1000, 960)])      # more than 256 tiles of 32 x 32
def test_matmul_below_the_tiles_keeps_every_bit(m, k, n, dev):
    """Products of fewer than 112 tiles of 64 x 64 hold every bit of their operands, whatever stands beside a value: one result of
    sixteen terms that are a billionth of their row and column's others, a one-hot row, and the same on the other side.  A sum of
    sixteen is sixteen roundings of products and as many of sums, at most 2^-24 of the terms' magnitudes each; the zeros
    between them add nothing."""
    import torch
    sliced = {(640, 2048, 512): 3, (301, 2048, 512): 4, (420, 1536, 512): 4, (577, 2309, 500): 3, (513, 4099, 320): 5,
              (700, 2048, 512): 3, (513, 3071, 512): 4, (640, 2048, 640): 3, (820, 1300, 500): 3}
    assert _product_kernel(m, k, n) == (("matmul_mfma_slices", sliced[m, k, n]) if (m, k, n) in sliced else ("matmul_splitk", 1))
    lib = api.load()
    torch.manual_seed(m + n + k)
    a, b = torch.randn(m, k, device="cuda"), torch.randn(k, n, device="cuda")
    for x, y in ((a, b), (b.T, a.T)):       # views: row 7 of a and column 9 of b, then column 7 and row 9
        at = torch.arange(16, device="cuda") * (k // 16) + k // 32
        few = y[at, 9].clone()
        y[:, 9] = 0.0
        y[at, 9] = few
        x[7, at] *= 1e-9
        x[11] = 0.0
        x[11, k - 5] = 1.0
    a[11, :], b[:, 11] = 0.0, 0.0
    a[11, k - 5] = b[k - 5, 11] = 1.0
    out = torch.full((m, n), 7.0, device="cuda")
    va, vb, vo = _dev_tensor(a), _dev_tensor(b), _dev_tensor(out)
    torch.cuda.synchronize()
    lib.blt_matmul(C.byref(va), C.byref(vb), C.byref(vo))
    torch.cuda.synchronize()
    for row, column in ((7, 9), (9, 7)):
        x, y = a[row].double(), b[:, column].double()
        assert int((x * y != 0).sum()) == 16
        off = abs(out[row, column].item() - float(x @ y))
        assert off <= 32 * 2.0 ** -24 * float(x.abs() @ y.abs()), (row, column, off / float(x.abs() @ y.abs()))
    assert torch.equal(out[11], b[k - 5]) and torch.equal(out[:, 11], a[:, k - 5])


@pytest.mark.parametrize("m,k,n", [(700, 400, 720), (2048, 160, 1290), (70, 384, 4000), (1500, 385, 700)])
def test_matmul_on_halves_out_of_range(m, k, n, dev):
    """The matrix-core product takes its operands apart into f16 parts up to 4094 (a) and 1023 (b), and from 2^-15 and 2^-17 on in
    the first step, and a tile that meets others starts again on bf16 parts: below, above, at zero, one value outside in
    the last step, NaN and infinity.  Each against float64 in the 2-norm of a row: 2^-24 for each of at most
    sqrt(K) roundings that count, and 2^-22 for the parts."""
    import ctypes as C
    import torch
    lib = api.load()
    gen = torch.Generator(device="cuda").manual_seed(k)
    view = lambda t: abi.tensor_view(t.data_ptr(), tuple(t.shape), abi.BLT_BACKEND_HIP)
    bound = 2.0 ** -24 * k ** 0.5 + 2.0 ** -22

    def product(a, b):
        out = torch.zeros(m, n, device="cuda")
        va, vb, vo = view(a), view(b), view(out)
        torch.cuda.synchronize()
        lib.blt_hip_profile_begin()
        lib.blt_matmul(C.byref(va), C.byref(vb), C.byref(vo))
        torch.cuda.synchronize()
        assert list(api.profile_end()) == ["matmul_mfma"]
        return out.double()

    a0 = torch.randn(m, k, device="cuda", generator=gen)
    b0 = torch.randn(k, n, device="cuda", generator=gen)
    for what in ("as drawn", "a below", "b above", "a zero", "one late", "rows apart", "ends"):
        a, b = a0.clone(), b0.clone()
        if what == "a below":
            a *= 1e-9
        elif what == "b above":
            b *= 1e4
        elif what == "a zero":
            a.zero_()
        elif what == "one late":
            a[m // 2, k - 1] = 1e5
        elif what == "rows apart":
            a[::3] *= 1e-8
            b[:, ::5] *= 1e6
        elif what == "ends":
            a *= 2.0 ** -7
            b *= 100.0
        want = a.double() @ b.double()
        error = (product(a, b) - want).norm(dim=1)
        if what == "rows apart":                     # columns of two scales: each by itself
            for cols in (slice(0, None, 5), slice(1, None, 5)):
                part = (product(a, b) - want)[:, cols].norm(dim=1) / want[:, cols].norm(dim=1)
                assert part.max().item() < bound, (what, part.max().item())
        else:
            assert (error <= bound * want.norm(dim=1)).all(), (what, (error / want.norm(dim=1)).max().item())
    a, b = a0.clone(), b0.clone()
    a[3, 5] = float("nan")
    b[k - 2, 9] = float("inf")
    got, clean = product(a, b), product(a0, b0)
    assert torch.isnan(got[3]).all()
    rows = torch.arange(m, device="cuda") != 3
    assert torch.equal(got[rows, 9], a0[rows, k - 2].double().sign() * float("inf"))
    cols = torch.arange(n, device="cuda") != 9
    assert ((got - clean)[rows][:, cols].norm() / clean.norm()).item() < bound


@pytest.mark.parametrize("m,k,n", [(1024, 1, 1024), (1500, 2, 700), (2048, 3, 2048), (1024, 4, 1024)])
def test_matmul_of_few_products(m, k, n, dev):
    """One and two products an element are as close as fp32 makes them: a single one correctly rounded (uniform rounding
    errors have a root mean square of 2^-24 / sqrt(12) of the power of two below the value, less over random values: 2.6e-8
    is what correct rounding of a normal product gives), two 3.2e-8; three and four on parts no worse than two roundings."""
    import torch
    lib = api.load()
    a, b = torch.randn(m, k, device="cuda"), torch.randn(k, n, device="cuda")
    out = torch.full((m, n), 7.0, device="cuda")
    va, vb, vo = _dev_tensor(a), _dev_tensor(b), _dev_tensor(out)
    torch.cuda.synchronize()
    lib.blt_matmul(C.byref(va), C.byref(vb), C.byref(vo))
    lib.blt_backend_pass_sync_hip()
    if k == 1:
        assert torch.equal(out, a * b)
    assert _relative(out, a.double() @ b.double()) <= (2.6e-8 if k == 1 else 3.2e-8 if k == 2 else 3.6e-8)


@pytest.mark.parametrize("scale_q,scale_k,scale_v", [(1.0, 1.0, 1.0), (1.0, 1.0, 1e-36), (1e-33, 1e33, 1.0), (1e-36, 1e36, 1.0),
                                                     (1e36, 1e-36, 1.0), (1e28, 1e-28, 1.0), (1e-40, 1e37, 1e25), (1.0, 1.0, 1e33), (0.0, 0.0, 1.0)])
@pytest.mark.parametrize("T,H,hd,batch", [(300, 1, 1, 1), (300, 1, 2, 1), (300, 1, 48, 1), (300, 1, 128, 1), (256, 4, 32, 80), (256, 4, 64, 80), (2304, 4, 32, 16)])
def test_attention_over_the_range_of_fp32(T, H, hd, batch, scale_q, scale_k, scale_v, dev):
    """Attention on bf16 parts (the latency kernel, the throughput kernel with four and eight waves) with tiny and huge
    operands, outputs and scores too large for the scaled sums: within ten times 2^-24 sqrt(hd), the rounding of a score of
    a few units.  Scale 0: all scores -1e30, every visible key weighs the same."""
    import torch
    lib = api.load()
    qkv = [torch.randn(batch, H, T, hd, device="cuda") * s for s in (scale_q, scale_k, scale_v)]
    if scale_q == 0.0:
        qkv[0].fill_(1e15)
        qkv[1].fill_(-1e15)
    q, k, v = qkv
    out = torch.full_like(q, 7.0)
    scale = float(np.float32(hd) ** np.float32(-0.5))
    probs = [api.problem(api.head_args(*(t[b, h].data_ptr() for t in (q, k, v, out)), T, T, hd, scale, hd, hd, hd, hd, 0),
                         api.BLT_ATTN_MASK_CAUSAL) for b in range(batch) for h in range(H)]
    plan = lib.blt_attention_plan_create_hip(api.problem_array(probs), len(probs))
    name = lib.blt_attention_plan_kernel_hip(plan).decode()
    torch.cuda.synchronize()
    lib.blt_attention_plan_run_hip(plan)
    lib.blt_backend_pass_sync_hip()
    lib.blt_attention_plan_destroy_hip(plan)
    assert ("mfma" if batch == 1 else "wide") in name, name
    hidden = torch.triu(torch.ones(T, T, dtype=torch.bool, device="cuda"), 1)
    for b in range(0, batch, 15):
        s = (q[b].double() @ k[b].double().transpose(1, 2).contiguous()) * scale
        ref = torch.softmax(s.masked_fill(hidden, -float("inf")), -1) @ v[b].double()
        assert _relative(out[b], ref) <= 10 * 2.0 ** -24 * hd ** 0.5, (b, name)


@pytest.mark.parametrize("m,k,n", [(40, 33, (1 << 25) + 64), (33, 1, (1 << 27) + 5), (40, 5, (1 << 27) + 5),
                                   ((1 << 22) + 70, 2, 64)])
def test_matmul_of_very_wide_matrices(m, k, n, dev):
    """More than 2^25 columns: the rows of b of one K step lie more than 2^32 bytes apart; more than 2^27 columns or 2^20
    rows go in several launches.  A sample of columns, the first and the last against float64."""
    import torch
    lib = api.load()
    a, b = torch.randn(m, k, device="cuda"), torch.randn(k, n, device="cuda")
    out = torch.full((m, n), 7.0, device="cuda")
    va, vb, vo = _dev_tensor(a), _dev_tensor(b), _dev_tensor(out)
    torch.cuda.synchronize()
    lib.blt_matmul(C.byref(va), C.byref(vb), C.byref(vo))
    lib.blt_backend_pass_sync_hip()
    cols = torch.cat([torch.arange(64), torch.randint(0, n, (4096,)), (1 << 25) + torch.arange(-64, 64),
                      torch.arange(n - 64, n)]).clamp_(0, n - 1).unique().cuda()
    assert_close(out[:, cols].cpu().numpy(), (a.double() @ b[:, cols].double()).cpu().numpy(), "matmul %dx%dx%d" % (m, k, n))


def test_attention_over_rows_far_apart(dev):
    """Batches large enough for the throughput kernel whose K and V rows are more than 2^27 bytes apart (a tile of 32 rows
    spans more than 2^32)."""
    import torch
    lib = api.load()
    nq, nk, hd, count, stride = 160, 40, 32, 330, (1 << 25) + 4
    slab = torch.empty(nk * stride, device="cuda")
    rows = slab.view(nk, stride)[:, :2 * hd]
    rows.copy_(torch.randn(nk, 2 * hd, device="cuda"))
    q, out = torch.randn(count, nq, hd, device="cuda"), torch.full((count, nq, hd), 7.0, device="cuda")
    scale = float(hd) ** -0.5
    probs = [api.problem(api.head_args(q[i].data_ptr(), slab.data_ptr(), slab.data_ptr() + 4 * hd, out[i].data_ptr(), nq, nk, hd,
                                       scale, hd, stride, stride, hd, 0, lse=None), api.BLT_ATTN_MASK_CAUSAL)
             for i in range(count)]
    torch.cuda.synchronize()
    lib.blt_attention_batch_hip(api.problem_array(probs), count)
    lib.blt_backend_pass_sync_hip()
    k, v = rows[:, :hd].double().cpu(), rows[:, hd:].double().cpu()
    s = (q.double().cpu() @ k.T) * scale
    s.masked_fill_(torch.triu(torch.ones(nq, nk, dtype=torch.bool), 1), -float("inf"))
    assert_close(out.cpu().numpy(), (torch.softmax(s, -1) @ v).numpy(), "rows far apart")


@pytest.mark.parametrize("nq,nk,masked,weighed,kernel", [(513, 513, True, True, "attn_once"), (17, 1024, True, False, "attn_once"),
                                                         (1000, 1001, False, True, "attn_once"), (33, 1024, False, False, "attn_once"),
                                                         (40, 689, False, False, "attn_once"), (40, 688, False, False, "attn_mfma"),
                                                         (16, 1025, True, True, "attn_mfma")])
def test_wide_heads_over_many_keys(nq, nk, masked, weighed, kernel, dev):
    """Heads of 64 over more keys than a wave's registers hold at once, with a dense mask that closes rows and whole tiles, with
    weights, with neither (from 689 keys on), against the sums in 64 bits."""
    import torch
    lib = api.load()
    rs = np.random.RandomState(nq + nk)
    q, k, v = (rs.randn(n, 64).astype(np.float32) for n in (nq, nk, nk))
    mask = np.where(rs.rand(nq, nk) < 0.3, -np.inf, rs.randn(nq, nk)).astype(np.float32)
    mask[:, 32:90], mask[:, 300:333], mask[nq - 1] = -np.inf, -np.inf, -np.inf
    x = q.astype(np.float64) @ k.T.astype(np.float64) / 8.0 + (mask if masked else 0.0)
    if masked:
        x[nq - 1] = 0.0
    w = np.exp(x - x.max(axis=1, keepdims=True))
    w /= w.sum(axis=1, keepdims=True)
    if masked:
        w[nq - 1] = 0.0
    dq, dk, dv, dm = (torch.from_numpy(t).cuda() for t in (q, k, v, mask))
    out, weights = torch.full((nq, 64), 7.0, device="cuda"), torch.full((nq, nk), 7.0, device="cuda")
    a = api.head_args(dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), out.data_ptr(), nq, nk, 64, 0.125, 64, 64, 64, 64, 0)
    a.mask, a.weights_out = (dm.data_ptr() if masked else None), (weights.data_ptr() if weighed else None)
    torch.cuda.synchronize()
    lib.blt_hip_profile_begin()
    lib.blt_attention_batch_hip(api.problem_array([api.problem(a)]), 1)
    names = set(api.profile_end())
    lib.blt_backend_pass_sync_hip()
    assert kernel in names, names
    assert_close(out.cpu().numpy(), (w @ v).astype(np.float32), "output")
    if weighed:
        assert_close(weights.cpu().numpy(), w.astype(np.float32), "weights")


@pytest.mark.parametrize("lens,H,hd,window,gap,kernel,staged", [
    ([100, 61, 7, 1, 130], 3, 32, 0, 0, "attn_once", False), ([17, 200], 2, 64, 50, 0, "attn_once", False),
    ([300, 211, 170], 8, 64, 0, 0, "attn_mfma", False), ([250, 131, 380], 8, 32, 0, 0, "attn_mfma", False),
    ([900, 33, 470], 8, 32, 0, 0, "attn_mfma", False), ([60, 50, 61, 33] * 8, 8, 64, 0, 0, "attn_fine", False),
    ([190, 131, 181], 16, 32, 0, 0, "attn_fine", False),
    ([5, 3, 12, 9], 2, 64, 0, 0, "attn_rows", False), ([1, 2, 15], 3, 24, 4, 0, "attn_rows", False),
    ([40, 41] * 16, 1, 32, 0, 0, "attn_once", False), ([40, 41] * 16 + [8], 1, 32, 0, 0, "attn_once", True),   # one document more
    ([2560, 2559], 1, 32, 90, 0, "attn_once", False), ([2560, 2561], 1, 32, 90, 0, "attn_once", True),           # one item more
    ([100, 61], 2, 32, 0, 5, "attn_once", True), ([100, 61], 2, 48, 0, 0, "attn_mfma", True)])   # rows between; heads of no own kernel
def test_attention_over_unequal_documents(lens, H, hd, window, gap, kernel, staged, dev):
    """Packed documents of unequal lengths in one call, at the most documents and work items that the kernel arguments hold and
    beyond, from each kernel, against the sums in 64 bits."""
    import torch
    lib = api.load()
    starts = np.concatenate([[0], np.cumsum(np.array(lens) + gap)])
    T, E, scale = int(starts[-1]), H * hd, 1.0 / np.sqrt(hd)
    rs = np.random.RandomState(T)
    qkv = rs.randn(T, 3 * E).astype(np.float32)
    rows, want = qkv.astype(np.float64), np.full((T, E), 7.0)
    tq, to = torch.from_numpy(qkv).cuda(), torch.full((T, E), 7.0, dtype=torch.float32, device="cuda")
    probs = []
    for first, n in zip(starts[:-1].tolist(), lens):
        back = np.arange(n)[:, None] - np.arange(n)[None, :]
        hidden = (back < 0) | ((back >= window) if window else False)
        for h in range(H):
            q, k, v = (rows[first:first + n, i * E + h * hd:i * E + (h + 1) * hd] for i in range(3))
            x = np.where(hidden, -np.inf, q @ k.T * scale)
            w = np.exp(x - x.max(axis=1, keepdims=True))
            want[first:first + n, h * hd:(h + 1) * hd] = w / w.sum(axis=1, keepdims=True) @ v
            a = abi.BltAttentionHeadArgs()
            a.q, a.k, a.v = (tq.data_ptr() + 4 * (first * 3 * E + i * E + h * hd) for i in range(3))
            a.q_stride = a.k_stride = a.v_stride = 3 * E
            a.combined, a.combined_stride, a.combined_col_offset = to.data_ptr() + 4 * first * E, E, h * hd
            a.nq = a.nk = n
            a.head_dim, a.scale = hd, scale
            probs.append(api.problem(a, api.BLT_ATTN_MASK_CAUSAL, window=window))
    lib.blt_hip_profile_begin()
    lib.blt_attention_batch_hip(api.problem_array(probs), len(probs))
    names = set(api.profile_end())
    lib.blt_backend_pass_sync_hip()
    assert names == ({kernel, "upload_words"} if staged else {kernel}), names
    assert_close(to.cpu().numpy(), want.astype(np.float32), "documents of %s rows" % lens)


@pytest.mark.parametrize("T,H,hd,docs", [(200, 2, 32, [0, 7, 90, 150]), (512, 4, 32, [0, 300]), (128, 8, 64, [0]),
                                         (96, 2, 64, [0, 20, 40, 60, 80])])
def test_document_causal_ranges_take_the_matrix_cores(T, H, hd, docs, oracle, dev):
    """Row-range problems whose caller states a long row_span (document-causal self-attention: row i sees
    [start of its document, i]) run on the matrix-core family, short or unstated spans one row per wave; both
    against the restated core under the equivalent dense mask (csrc/ops/mask_builder_cpu.c:21-98)."""
    import torch
    lib = api.load()
    rs = np.random.RandomState(T + hd)
    E = H * hd
    qkv = rs.randn(T, 3 * E).astype(np.float32)
    start = np.zeros(T, dtype=np.uint32)
    for d0 in docs:
        start[d0:] = d0
    lo, hi = start, (np.arange(T) + 1).astype(np.uint32)
    mask = np.full((T, T), -np.inf, dtype=np.float32)
    for i in range(T):
        mask[i, lo[i]:hi[i]] = 0.0
    ref = np.zeros((T, E), dtype=np.float32)
    wts = np.zeros((T, T), dtype=np.float32)
    flat = qkv.reshape(-1)
    for h in range(H):
        a = binding.head_args(flat, flat, flat, ref.reshape(-1), T, T, hd, 1.0 / np.sqrt(hd), 3 * E, 3 * E, 3 * E, E,
                              h * hd, q_off=h * hd, k_off=E + h * hd, v_off=2 * E + h * hd, weights=wts.reshape(-1),
                              mask=mask.reshape(-1))
        assert oracle.orc_attention_head_core(C.byref(a)) == 0
    tq = torch.from_numpy(qkv).cuda()
    dlo, dhi = torch.from_numpy(lo.view(np.int32)).cuda(), torch.from_numpy(hi.view(np.int32)).cuda()
    span = int((hi - lo).max())
    for stated, kernel in ((span, "attn_mfma" if span >= 24 else "attn_rows"), (0, "attn_rows")):
        to = torch.zeros((T, E), dtype=torch.float32, device="cuda")
        probs = []
        for h in range(H):
            a = abi.BltAttentionHeadArgs()
            a.q, a.k, a.v = tq.data_ptr() + 4 * h * hd, tq.data_ptr() + 4 * (E + h * hd), tq.data_ptr() + 4 * (2 * E + h * hd)
            a.q_stride = a.k_stride = a.v_stride = 3 * E
            a.combined, a.combined_stride, a.combined_col_offset = to.data_ptr(), E, h * hd
            a.nq = a.nk = T
            a.head_dim, a.scale = hd, 1.0 / np.sqrt(hd)
            probs.append(api.problem(a, api.BLT_ATTN_MASK_ROW_RANGE, row_lo=dlo.data_ptr(), row_hi=dhi.data_ptr(),
                                     row_span=stated))
        lib.blt_hip_profile_begin()
        lib.blt_attention_batch_hip(api.problem_array(probs), H)
        launched = api.profile_end()
        assert list(launched) == [kernel], (launched, stated)
        assert_close(to.cpu().numpy(), ref, "document-causal ranges T=%d span stated %d" % (T, stated))


def test_matmul_k_slices_back_to_back(dev):
    """Long-K products over few output tiles split K over several workgroups per tile, which meet through
    per-stream sums and tickets: launches of different shapes issued back to back, without a wait in between,
    must each find the tickets re-armed and must give the same bits every time (the slices are added in slice
    order whichever workgroup comes last)."""
    import torch
    lib = api.load()
    torch.manual_seed(5)
    shapes = [(118, 2048, 512), (64, 4096, 256), (100, 3000, 70), (40, 1024, 2048), (118, 2048, 512)]
    ops = []
    for m, k, n in shapes:
        a = torch.randn(m, k, device="cuda")
        b = torch.randn(k, n, device="cuda") / k ** 0.5
        outs = [torch.full((m, n), 3.0, device="cuda") for _ in range(3)]
        ops.append((a, b, outs))
    for rnd in range(3):
        for a, b, outs in ops:
            va, vb, vo = _dev_tensor(a), _dev_tensor(b), _dev_tensor(outs[rnd])
            lib.blt_matmul(C.byref(va), C.byref(vb), C.byref(vo))
    lib.blt_backend_pass_sync_hip()
    for (m, k, n), (a, b, outs) in zip(shapes, ops):
        want = (a.double() @ b.double()).float().cpu().numpy()
        got = [o.cpu().numpy() for o in outs]
        assert_close(got[0], want, "sliced matmul %dx%dx%d" % (m, k, n))
        assert got[0].tobytes() == got[1].tobytes() == got[2].tobytes(), (m, k, n)


def test_rope_apply_bit_exact(oracle, dev):
    import torch
    lib = api.load()
    rs = np.random.RandomState(77)
    T, H, hd = 45, 3, 32
    half = hd // 2
    x = rs.randn(T, H, hd).astype(np.float32)
    cos, sin = np.empty(T * half, dtype=np.float32), np.empty(T * half, dtype=np.float32)
    assert oracle.orc_rope_precompute(T, 500000.0, hd, binding.fptr(cos), binding.fptr(sin)) == 0
    # tables: the device dispatcher computes them on the host with the same formula
    tc = torch.zeros((T, half), dtype=torch.float32, device="cuda")
    ts = torch.zeros((T, half), dtype=torch.float32, device="cuda")
    vc, vs = _dev_tensor(tc), _dev_tensor(ts)
    cfg = abi.BltRopeConfig(500000.0, hd)
    lib.blt_rope_precompute(T, C.byref(cfg), C.byref(vc), C.byref(vs))
    assert tc.cpu().numpy().tobytes() == cos.tobytes() and ts.cpu().numpy().tobytes() == sin.tobytes()
    ref = np.empty_like(x)
    oracle.orc_rope_apply(binding.fptr(x.reshape(-1)), T, H, hd, binding.fptr(cos), binding.fptr(sin),
                          binding.fptr(ref.reshape(-1)))
    tx = torch.from_numpy(x).cuda()
    to = torch.zeros_like(tx)
    vx, vo = _dev_tensor(tx), _dev_tensor(to)
    lib.blt_rope_apply(C.byref(vx), C.byref(vc), C.byref(vs), C.byref(vo))
    lib.blt_backend_pass_sync_hip()
    assert to.cpu().numpy().tobytes() == ref.tobytes()
    # packed, in place, one head block of [T, 3E] rows
    E = H * hd
    qkv = rs.randn(T, 3 * E).astype(np.float32)
    want = qkv.copy()
    oracle.orc_rope_apply_packed(binding.fptr(want.reshape(-1)), 3 * E, E + hd, T, hd, binding.fptr(cos),
                                 binding.fptr(sin))
    tq = torch.from_numpy(qkv).cuda()
    lib.blt_rope_apply_packed(tq.data_ptr(), 3 * E, E + hd, T, hd, tc.data_ptr(), ts.data_ptr(), abi.BLT_BACKEND_HIP)
    lib.blt_backend_pass_sync_hip()
    assert tq.cpu().numpy().tobytes() == want.tobytes()


IMPLS = ["library", "reference_callers"]


def _entry(impl, lib):
    """Where the block-level calls go: the library's own entry points, or the reference's caller
    code (models/attention.c, cross_attention.c, infer/kv_cache.c compiled unmodified) whose tensor
    ops are served by the library -- the drop-in arrangement itself."""
    if impl == "library":
        return lib
    callers = binding.load_ref_callers()
    if callers is None:
        pytest.skip("oracle/_ref/libblt_ref_callers.so was not built (needs the reference sources)")
    return callers


@pytest.mark.parametrize("impl", IMPLS)
@pytest.mark.parametrize("T,E,H,causal,rope,mask,cached", [
    (2, 4, 2, False, False, None, False),          # the reference's identity-weight block
    (20, 32, 4, True, True, None, False),          # few rows: exact products, separate rotation pass
    (96, 64, 2, True, True, None, True),
    (512, 128, 4, False, True, "causal_cfg", True),  # the local decoder's call at C1 size
    (300, 128, 4, False, True, "window", False),
    (70, 48, 3, False, False, "docs", False),        # dense mask from the device builder
    (128, 512, 8, False, False, "causal_cfg", False),  # the patch transformer's call at C2 size
])
def test_multihead_attention_block(T, E, H, causal, rope, mask, cached, impl, oracle, dev):
    """blt_multihead_attention on device tensors against the restated block."""
    import torch
    lib = api.load()
    entry = _entry(impl, lib)
    rs = np.random.RandomState(T + E)
    hd, half = E // H, E // H // 2
    if (T, E, H) == (2, 4, 2):
        x = np.array([[1, 0, 1, 0], [0, 1, 0, 1]], dtype=np.float32)
        wqkv = np.zeros((4, 12), dtype=np.float32)
        for i in range(4):
            wqkv[i, i] = wqkv[i, 4 + i] = wqkv[i, 8 + i] = 1.0
        wproj = np.eye(4, dtype=np.float32)
    else:
        x = rs.randn(T, E).astype(np.float32)
        wqkv = (rs.randn(E, 3 * E) / np.sqrt(E)).astype(np.float32)
        wproj = (rs.randn(E, E) / np.sqrt(E)).astype(np.float32)
    cfg, keep = None, None
    if mask is not None:
        cfg = abi.BltMaskConfig()
        cfg.seq_len_q = cfg.seq_len_kv = T
        if mask == "window":
            cfg.is_causal, cfg.sliding_window = True, 40
        elif mask == "docs":
            keep = abi.size_array([21, 50])
            cfg.doc_boundaries, cfg.num_docs = keep, 3
        else:
            cfg.is_causal = True
    ref = np.zeros((T, E), dtype=np.float32)
    assert oracle.orc_multihead_attention(
        binding.fptr(x.reshape(-1)), binding.fptr(wqkv.reshape(-1)), binding.fptr(wproj.reshape(-1)),
        binding.fptr(ref.reshape(-1)), T, E, H, int(causal), int(rope), 500000.0, None, None,
        C.byref(cfg) if cfg is not None else None) == 0
    if (T, E, H) == (2, 4, 2):   # tests/unit/models/unit_attention.c:82-88
        assert abs(ref[0, 0] - 0.6697615) < 1e-6 and abs(ref[0, 1] - 0.3302385) < 1e-6
    tx, tq, tp = (torch.from_numpy(v).cuda() for v in (x, wqkv, wproj))
    to = torch.full((T, E), 7.0, dtype=torch.float32, device="cuda")
    ac = abi.BltAttentionConfig()
    ac.embed_dim, ac.num_heads, ac.head_dim = E, H, hd
    ac.is_causal, ac.use_rope, ac.rope_theta = causal, rope, 500000.0
    if cfg is not None:
        ac.mask_config = C.pointer(cfg)
    tables = None
    if rope and cached:
        cos, sin = np.empty(T * half, dtype=np.float32), np.empty(T * half, dtype=np.float32)
        oracle.orc_rope_precompute(T, 500000.0, hd, binding.fptr(cos), binding.fptr(sin))
        tables = (torch.from_numpy(cos.reshape(T, half)).cuda(), torch.from_numpy(sin.reshape(T, half)).cuda())
        vc, vs = _dev_tensor(tables[0]), _dev_tensor(tables[1])
        ac.rope_cos_cache, ac.rope_sin_cache = C.pointer(vc), C.pointer(vs)
    arena = lib.blt_arena_create(64 << 20, abi.BLT_BACKEND_HIP)
    try:
        vx, vq, vp, vo = _dev_tensor(tx), _dev_tensor(tq), _dev_tensor(tp), _dev_tensor(to)
        entry.blt_multihead_attention(C.byref(vx), C.byref(vq), C.byref(vp), C.byref(vo), C.byref(ac), arena)
        lib.blt_backend_pass_sync_hip()
        got = to.cpu().numpy()
    finally:
        lib.blt_arena_destroy(arena)
    assert_close(got, ref, "attention block T=%d E=%d H=%d" % (T, E, H))


@pytest.mark.parametrize("impl", IMPLS)
@pytest.mark.parametrize("P,T,E,H,kind", [
    (2, 4, 4, 2, "identity"),          # tests/unit/models/unit_cross_attention.c:24-117
    (9, 70, 32, 4, "groups"),          # few rows: exact products
    (128, 512, 128, 4, "groups"),      # the encoder's call at C3 size: split-K products, two outputs in one pass
    (128, 512, 128, 4, "even"),        # 4 bytes per patch, the shape the bench uses
    (40, 4099, 128, 2, "groups"),      # long, ragged groups; K and V through the 64x64 product kernel
    (33, 100, 48, 3, "interleaved"),   # groups not contiguous: dense mask from the device builder
    (64, 200, 64, 2, "window"),        # no groups: window-only visibility
])
def test_cross_attention_block(P, T, E, H, kind, impl, oracle, dev):
    """blt_cross_attention_forward on device tensors against the restated block."""
    import torch
    lib = api.load()
    entry = _entry(impl, lib)
    rs = np.random.RandomState(P + T + E)
    if kind == "identity":
        xq = np.array([[1, 0, 1, 0], [0, 1, 0, 1]], dtype=np.float32)
        xkv = np.array([[1, 0, 1, 0], [0, 1, 0, 1], [1, 0, 1, 0], [0, 1, 0, 1]], dtype=np.float32)
        ws = [np.eye(4, dtype=np.float32) for _ in range(4)]
    else:
        xq, xkv = rs.randn(P, E).astype(np.float32), rs.randn(T, E).astype(np.float32)
        ws = [(rs.randn(E, E) / np.sqrt(E)).astype(np.float32) for _ in range(4)]
    cfg = abi.BltMaskConfig()
    cfg.seq_len_q, cfg.seq_len_kv = P, T
    keep = None
    if kind == "window":
        cfg.sliding_window = 90
    else:
        if kind == "identity":
            groups = np.array([0, 0, 1, 1])
        elif kind == "even":
            groups = np.arange(T) // (T // P)
        else:
            groups = np.sort(np.concatenate([np.arange(P), rs.randint(0, P, size=T - P)]))
            if kind == "interleaved":
                groups = rs.permutation(groups)
        keep = (abi.size_array(list(range(P))), abi.size_array(groups.tolist()))
        cfg.query_group_ids, cfg.kv_group_ids = keep
        cfg.bidirectional_within_group = True
    ref = np.zeros((P, E), dtype=np.float32)
    assert oracle.orc_cross_attention_forward(*(binding.fptr(a.reshape(-1)) for a in (xq, xkv, *ws, ref)), P, T, E, H,
                                              C.byref(cfg)) == 0
    if kind == "identity":
        assert abs(ref[0, 0] - 0.6697615) < 1e-6 and abs(ref[1, 0] - 0.3302385) < 1e-6
    dev_in = [torch.from_numpy(a).cuda() for a in (xq, xkv, *ws)]
    to = torch.full((P, E), 7.0, dtype=torch.float32, device="cuda")
    views = [_dev_tensor(t) for t in dev_in]
    vo = _dev_tensor(to)
    wts = abi.BltCrossAttentionWeights(*(C.pointer(v) for v in views[2:]))
    cc = abi.BltCrossAttentionConfig()
    cc.embed_dim, cc.num_heads, cc.head_dim = E, H, 0   # 0 = embed_dim / num_heads
    cc.mask_config = C.pointer(cfg)
    arena = lib.blt_arena_create(64 << 20, abi.BLT_BACKEND_HIP)
    try:
        entry.blt_cross_attention_forward(C.byref(views[0]), C.byref(views[1]), C.byref(wts), C.byref(vo), C.byref(cc),
                                        arena)
        lib.blt_backend_pass_sync_hip()
        got = to.cpu().numpy()
    finally:
        lib.blt_arena_destroy(arena)
    assert_close(got, ref, "cross attention P=%d T=%d E=%d H=%d %s" % (P, T, E, H, kind))


@pytest.mark.parametrize("P,T,E,H,longest,fused", [
    (33, 60, 64, 16, 4, True), (40, 300, 64, 1, 17, True), (50, 90, 128, 32, 9, True), (63, 1500, 128, 1, 64, True),
    (65, 400, 128, 4, 33, True),
    (40, 300, 128, 4, 65, False), (32, 60, 128, 4, 4, False), (40, 60, 96, 3, 4, False)])   # each past one of its limits
def test_cross_attention_in_one_launch_past_its_keys(P, T, E, H, longest, fused, oracle, dev):
    """The launch from the query's norm to the residual at the edges of its shapes, against the restated block; then with a key
    that is not finite, which drops out of its own patch's softmax and changes no other row."""
    import torch
    lib = api.load()
    rs = np.random.RandomState(P + T + H)
    xq, xkv = rs.randn(P, E).astype(np.float32), rs.randn(T, E).astype(np.float32)
    ws = [(rs.randn(E, E) / np.sqrt(E)).astype(np.float32) for _ in range(4)]
    sizes = np.ones(P, dtype=int)
    sizes[P // 2] = longest
    while sizes.sum() < T:                          # the rest at random, none past the longest
        sizes[rs.choice(np.flatnonzero(sizes < min(longest, T)))] += 1
        if (sizes >= longest).all():
            break
    T = int(sizes.sum())
    xkv = np.ascontiguousarray(np.resize(xkv, (T, E)))
    cfg = abi.BltMaskConfig()
    cfg.seq_len_q, cfg.seq_len_kv = P, T
    keep = (abi.size_array(list(range(P))), abi.size_array(np.repeat(np.arange(P), sizes).tolist()))
    cfg.query_group_ids, cfg.kv_group_ids = keep
    cfg.bidirectional_within_group = True

    def run(kv):
        tensors = [torch.from_numpy(a).cuda() for a in (xq, kv, *ws)]
        to = torch.full((P, E), 7.0, dtype=torch.float32, device="cuda")
        views = [_dev_tensor(t) for t in tensors]
        vo = _dev_tensor(to)
        wts = abi.BltCrossAttentionWeights(*(C.pointer(v) for v in views[2:]))
        cc = abi.BltCrossAttentionConfig()
        cc.embed_dim, cc.num_heads, cc.head_dim = E, H, 0
        cc.mask_config = C.pointer(cfg)
        arena = lib.blt_arena_create(64 << 20, abi.BLT_BACKEND_HIP)
        try:
            lib.blt_hip_profile_begin()
            lib.blt_cross_attention_forward(C.byref(views[0]), C.byref(views[1]), C.byref(wts), C.byref(vo), C.byref(cc), arena)
            assert ("cross_block" in api.profile_end()) == fused
            lib.blt_backend_pass_sync_hip()
            return to.cpu().numpy()
        finally:
            lib.blt_arena_destroy(arena)

    ref = np.zeros((P, E), dtype=np.float32)
    assert oracle.orc_cross_attention_forward(*(binding.fptr(a.reshape(-1)) for a in (xq, xkv, *ws, ref)), P, T, E, H,
                                              C.byref(cfg)) == 0
    got = run(xkv)
    assert_close(got, ref, "cross block")
    if fused:
        bad = xkv.copy()
        patch = P // 2
        bad[int(sizes[:patch].sum()) + longest - 1] = np.nan      # the last byte of the longest patch
        out = run(bad)
        others = np.arange(P) != patch
        assert np.array_equal(out[others], got[others])
        short = sizes.copy()
        short[patch] -= 1
        cut = np.delete(xkv, int(sizes[:patch].sum()) + longest - 1, axis=0)
        cfg.seq_len_kv = T - 1
        keep2 = (keep[0], abi.size_array(np.repeat(np.arange(P), short).tolist()))
        cfg.query_group_ids, cfg.kv_group_ids = keep2
        assert oracle.orc_cross_attention_forward(*(binding.fptr(np.ascontiguousarray(a).reshape(-1)) for a in (xq, cut, *ws)),
                                                  binding.fptr(ref.reshape(-1)), P, T - 1, E, H, C.byref(cfg)) == 0
        assert_close(out[patch], ref[patch], "without the key that is not finite")


def test_cross_attention_in_one_launch_with_faded_keys(dev):
    """Keys that lose all their weight to keys further on (scores of -120 ... 0 in steps, so that no single step makes it zero)
    have no part in the result, their infinite value rows either; rows that see none of it keep their bits."""
    import torch
    lib = api.load()
    P, E, longest = 40, 64, 17
    rs = np.random.RandomState(3)
    xq = rs.randn(P, E).astype(np.float32)
    wq, wk, wv, wo = ((rs.randn(E, E) / np.sqrt(E)).astype(np.float32) for _ in range(4))
    wk[0], wv[0], wv[0, 5] = 0.0, 0.0, 1e30          # column 0 of a byte: nothing to its key, to its value 1e30 a unit
    sizes = np.full(P, 2)
    patch = P // 2
    sizes[patch] = longest
    at, T = int(sizes[:patch].sum()), int(sizes.sum())
    xkv = rs.randn(T, E).astype(np.float32)
    xkv[:, 0] = 0.0
    along = (wk.astype(np.float64) @ (xq[patch].astype(np.float64) @ wq))
    along[0] = 0.0
    along /= (along @ (wk.astype(np.float64) @ (xq[patch].astype(np.float64) @ wq))) / np.sqrt(E)   # a score of one
    scores = -120.0 + 120.0 / (longest - 1) * np.arange(longest)
    xkv[at:at + longest] = (scores[:, None] * along).astype(np.float32)
    cfg = abi.BltMaskConfig()
    cfg.seq_len_q, cfg.seq_len_kv = P, T
    keep = (abi.size_array(list(range(P))), abi.size_array(np.repeat(np.arange(P), sizes).tolist()))
    cfg.query_group_ids, cfg.kv_group_ids = keep
    cfg.bidirectional_within_group = True

    def run(kv):
        tensors = [torch.from_numpy(a).cuda() for a in (xq, kv, wq, wk, wv, wo)]
        to = torch.full((P, E), 7.0, dtype=torch.float32, device="cuda")
        views = [_dev_tensor(t) for t in tensors]
        vo = _dev_tensor(to)
        wts = abi.BltCrossAttentionWeights(*(C.pointer(v) for v in views[2:]))
        cc = abi.BltCrossAttentionConfig()
        cc.embed_dim, cc.num_heads, cc.head_dim = E, 1, 0
        cc.mask_config = C.pointer(cfg)
        arena = lib.blt_arena_create(64 << 20, abi.BLT_BACKEND_HIP)
        try:
            lib.blt_hip_profile_begin()
            lib.blt_cross_attention_forward(C.byref(views[0]), C.byref(views[1]), C.byref(wts), C.byref(vo), C.byref(cc), arena)
            assert "cross_block" in api.profile_end()
            lib.blt_backend_pass_sync_hip()
            return to.cpu().numpy()
        finally:
            lib.blt_arena_destroy(arena)

    clean = run(xkv)
    assert np.isfinite(clean).all()
    xkv[at, 0] = 1e30                                # its value's column 5 is infinite now
    out, others = run(xkv), np.arange(P) != patch
    assert np.array_equal(out[others], clean[others])
    assert_close(out[patch], clean[patch], "a faded key's value")
    xkv[at + longest - 1, 0] = 1e30                  # the key that has most of the weight
    out = run(xkv)
    assert not np.isfinite(out[patch]).any() and np.array_equal(out[others], clean[others])


def test_row_ops(oracle, dev):
    """blt_rmsnorm_forward and blt_add bit-identical to the reference loops, blt_swiglu_forward in tolerance."""
    import torch
    lib = api.load()
    rs = np.random.RandomState(61)
    for rows, dim in ((1, 128), (64, 128), (100, 512), (7, 33), (2048, 128), (3, 1000), (5, 20), (118, 132), (33, 4088), (9, 4)):
        x = (rs.randn(rows, dim) * 2).astype(np.float32)
        w = rs.randn(dim).astype(np.float32)
        y = rs.randn(rows, dim).astype(np.float32)
        ref = np.zeros_like(x)
        oracle.orc_rmsnorm_forward(binding.fptr(x.reshape(-1)), binding.fptr(w), binding.fptr(ref.reshape(-1)), rows, dim)
        tx, tw, ty = torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda(), torch.from_numpy(y).cuda()
        to = torch.zeros_like(tx)
        vx, vw, vy, vo = _dev_tensor(tx), _dev_tensor(tw), _dev_tensor(ty), _dev_tensor(to)
        lib.blt_rmsnorm_forward(C.byref(vx), C.byref(vw), C.byref(vo))
        lib.blt_backend_pass_sync_hip()
        assert to.cpu().numpy().tobytes() == ref.tobytes(), (rows, dim)
        oracle.orc_add(binding.fptr(x.reshape(-1)), binding.fptr(y.reshape(-1)), binding.fptr(ref.reshape(-1)), rows * dim)
        lib.blt_add(C.byref(vx), C.byref(vy), C.byref(vo))
        lib.blt_backend_pass_sync_hip()
        assert to.cpu().numpy().tobytes() == ref.tobytes()
        oracle.orc_swiglu_forward(binding.fptr(x.reshape(-1)), binding.fptr(y.reshape(-1)), binding.fptr(ref.reshape(-1)),
                                  rows * dim)
        lib.blt_swiglu_forward(C.byref(vx), C.byref(vy), C.byref(vo))
        lib.blt_backend_pass_sync_hip()
        assert_close(to.cpu().numpy(), ref, "swiglu")


@pytest.mark.parametrize("batch,n,H,hd,hidden,kind", [(3, 1, 2, 32, 96, "causal"), (64, 1, 4, 32, 256, "causal"),
                                                      (5, 6, 2, 64, 200, "causal"), (9, 16, 4, 32, 128, "block"),
                                                      (128, 16, 4, 32, 512, "causal")])
def test_kv_decode_layer(batch, n, H, hd, hidden, kind, oracle, dev):
    """blt_kv_decode_layer_hip for all sequences at once against the restated layer run per sequence."""
    import torch
    lib = api.load()
    rs = np.random.RandomState(batch * 7 + n)
    E, half = H * hd, hd // 2
    max_len = 80 + 2 * n
    lens = rs.randint(1, 70, size=batch).astype(np.uint32)
    ck = rs.randn(batch * max_len, E).astype(np.float32)
    cv = rs.randn(batch * max_len, E).astype(np.float32)
    W = {k: (rs.randn(*shape) / np.sqrt(shape[0])).astype(np.float32)
         for k, shape in dict(qkv=(E, 3 * E), proj=(E, E), up=(E, hidden), gate=(E, hidden), down=(hidden, E)).items()}
    n1, n2 = (1.0 + 0.1 * rs.randn(E)).astype(np.float32), (1.0 + 0.1 * rs.randn(E)).astype(np.float32)
    cos, sin = np.empty(max_len * half, dtype=np.float32), np.empty(max_len * half, dtype=np.float32)
    oracle.orc_rope_precompute(max_len, 500000.0, hd, binding.fptr(cos), binding.fptr(sin))
    x = rs.randn(batch * n, E).astype(np.float32)
    fp = lambda a: binding.fptr(a.reshape(-1))
    # reference: one sequence at a time (block rows: the verify step attends the whole block; the
    # restated layer is causal, so block kind is checked through the device's own causal/block split below)
    ref_k, ref_v = ck.copy(), cv.copy()
    ref_out = np.zeros((batch * n, E), dtype=np.float32)
    if kind == "causal":
        for b in range(batch):
            xb = np.ascontiguousarray(x[b * n:(b + 1) * n])
            ob = np.zeros((n, E), dtype=np.float32)
            assert oracle.orc_kv_decode_layer(fp(ref_k), fp(ref_v), max_len, E, H, b, int(lens[b]), n, 0, fp(n1),
                                              fp(W["qkv"]), fp(W["proj"]), fp(n2), fp(W["up"]), fp(W["gate"]),
                                              fp(W["down"]), hidden, fp(cos), fp(sin), max_len, fp(xb), fp(ob)) == 0
            ref_out[b * n:(b + 1) * n] = ob
    t = {k: torch.from_numpy(v).cuda() for k, v in W.items()}
    tn1, tn2 = torch.from_numpy(n1).cuda(), torch.from_numpy(n2).cuda()
    tck, tcv = torch.from_numpy(ck).cuda(), torch.from_numpy(cv).cuda()
    tlens = torch.from_numpy(lens.astype(np.int32)).cuda()
    tcos, tsin = torch.from_numpy(cos.reshape(max_len, half)).cuda(), torch.from_numpy(sin.reshape(max_len, half)).cuda()
    tx = torch.from_numpy(x).cuda()
    to = torch.zeros_like(tx)
    views = {k: _dev_tensor(v) for k, v in t.items()}
    vn1, vn2 = _dev_tensor(tn1), _dev_tensor(tn2)
    w = abi.BltTransformerWeights()
    w.norm1_weight, w.norm2_weight = C.pointer(vn1), C.pointer(vn2)
    w.attn_qkv_w, w.attn_proj_w = C.pointer(views["qkv"]), C.pointer(views["proj"])
    w.ffn_up_w, w.ffn_gate_w, w.ffn_down_w = C.pointer(views["up"]), C.pointer(views["gate"]), C.pointer(views["down"])
    c = api.BltKvAttnCache()
    c.self_k, c.self_v, c.self_len = tck.data_ptr(), tcv.data_ptr(), tlens.data_ptr()
    c.batch, c.max_seq_len, c.embed_dim, c.num_heads, c.window = batch, max_len, E, H, 0
    arena = lib.blt_arena_create(64 << 20, abi.BLT_BACKEND_HIP)
    try:
        step_kind = api.BLT_KV_STEP_CAUSAL if kind == "causal" else api.BLT_KV_STEP_BLOCK
        lib.blt_kv_decode_layer_hip(C.byref(c), C.byref(w), tx.data_ptr(), to.data_ptr(), tcos.data_ptr(),
                                    tsin.data_ptr(), max_len, n, step_kind, 1 if kind == "causal" else 0,
                                    int(lens.max()) + n, arena)
        lib.blt_backend_pass_sync_hip()
        got = to.cpu().numpy()
        got_k, got_v, got_len = tck.cpu().numpy(), tcv.cpu().numpy(), tlens.cpu().numpy()
    finally:
        lib.blt_arena_destroy(arena)
    if kind == "causal":
        assert (got_len == lens + n).all()
        assert_close(got, ref_out, "decode layer")
        # rows of a batch above 32 come from the matrix-core projection: cache rows in tolerance, not bitwise
        assert_close(got_k, ref_k, "cache k")
        assert_close(got_v, ref_v, "cache v")
    else:
        # block rows: same layer with the block step; check against the device's own pieces
        assert (got_len == lens).all() and np.isfinite(got).all()
        tx2 = torch.from_numpy(x).cuda()
        normed = torch.zeros_like(tx2)
        vx, vnm = _dev_tensor(tx2), _dev_tensor(normed)
        lib.blt_rmsnorm_forward(C.byref(vx), C.byref(vn1), C.byref(vnm))
        qkv = torch.zeros((batch * n, 3 * E), dtype=torch.float32, device="cuda")
        vq = _dev_tensor(qkv)
        lib.blt_matmul(C.byref(vnm), C.byref(views["qkv"]), C.byref(vq))
        tck2, tcv2 = torch.from_numpy(ck).cuda(), torch.from_numpy(cv).cuda()
        c.self_k, c.self_v = tck2.data_ptr(), tcv2.data_ptr()
        comb = torch.zeros_like(tx2)
        lib.blt_kv_rope_attend_step_hip(C.byref(c), qkv.data_ptr(), 3 * E, qkv.data_ptr() + 4 * E, 3 * E,
                                        qkv.data_ptr() + 8 * E, 3 * E, tcos.data_ptr(), tsin.data_ptr(), max_len,
                                        comb.data_ptr(), E, n, step_kind, 0, int(lens.max()) + n)
        lib.blt_backend_pass_sync_hip()
        # the layer folds the norm into the projection (scale applied after the product): tolerance, not bits
        assert_close(got_k, tck2.cpu().numpy(), "cache k (block)")


# ---------------------------------------------------------------------------
# streams and graphs
# ---------------------------------------------------------------------------
# ---------------------------------------------------------------------------
# the whole incremental decoder step on the device (csrc/infer/kv_cache.c:112-416)
# ---------------------------------------------------------------------------
STEP_CASES = [
    dict(E=16, H=2, XH=2, L=2, hidden=24, V=19, max_len=40, k=1, window=0, all_layers=True, placement=0),
    dict(E=24, H=3, XH=2, L=3, hidden=40, V=256, max_len=48, k=2, window=7, all_layers=False, placement=0),
    dict(E=128, H=4, XH=4, L=2, hidden=512, V=256, max_len=64, k=1, window=0, all_layers=True, placement=0),
    dict(E=64, H=2, XH=4, L=2, hidden=96, V=50, max_len=32, k=3, window=5, all_layers=False, placement=4),
    dict(E=64, H=2, XH=2, L=2, hidden=96, V=52, max_len=200, k=1, window=0, all_layers=True, placement=0),
    dict(E=128, H=4, XH=4, L=1, hidden=128, V=64, max_len=160, k=2, window=30, all_layers=True, placement=0),
]


def _decoders(oracle, c, seed):
    """The same seeded decoder twice: over numpy arrays for the checker, over device copies for the library."""
    from fblt_amd import decoder
    hd, half = c["E"] // c["H"], c["E"] // c["H"] // 2
    cos, sin = (np.empty(c["max_len"] * half, dtype=np.float32) for _ in range(2))
    assert oracle.orc_rope_precompute(c["max_len"], 500000.0, hd, binding.fptr(cos), binding.fptr(sin)) == 0
    w = decoder.random_weights(c["E"], c["hidden"], c["L"], c["V"], seed)
    args = (c["E"], c["H"], c["XH"], c["hidden"], c["V"], c["max_len"])
    kw = dict(patch_dim=c["k"] * c["E"], window=c["window"], all_layers=c["all_layers"], placement=c["placement"])
    tables = (cos.reshape(c["max_len"], half), sin.reshape(c["max_len"], half))
    host = decoder.bind(w, *tables, abi.BLT_BACKEND_CPU, decoder.host_place, *args, **kw)
    device = decoder.bind(w, *tables, abi.BLT_BACKEND_HIP, decoder.device_place, *args, **kw)
    return host, device


@pytest.mark.parametrize("case", range(len(STEP_CASES)))
@pytest.mark.parametrize("closed,docs,impl", [(0, [], "public"), (1, [], "twin"), (0, [5, 11], "public"),
                                              (1, [0, 1, 1, 30], "twin")])
def test_local_decoder_forward(case, closed, docs, impl, oracle, dev):
    """The library's own blt_local_decoder_forward_ext (inference form: no loss, D_0 = the encoder's rows) against
    the restated forward (csrc/models/local_decoder.c:233-351): every decoder configuration of the step tests
    (sub-token split, window, placements), trailing_closed, document boundaries in the byte mask; through the
    public name and through the device twin."""
    import torch
    from fblt_amd import decoder
    lib = api.load()
    c = STEP_CASES[case]
    host, device = _decoders(oracle, c, 900 + case)
    rs = np.random.RandomState(900 + case)
    lengths = [3, 4, 2, 5, 1, 6, 9] if c["max_len"] < 64 else [3, 4, 2, 5, 1, 6, 9, 16, 2, 12]
    T, P, E, V = sum(lengths), len(lengths), c["E"], c["V"]
    patches = decoder.patch_table(lengths)
    hidden = rs.randn(T, E).astype(np.float32)
    patch_in = rs.randn(P, E * c["k"]).astype(np.float32)
    bounds = abi.size_array(docs) if docs else None
    num_docs = len(docs) + 1 if docs else 0
    want = np.zeros((T, V), dtype=np.float32)
    assert oracle.orc_local_decoder_forward(host.ptr, binding.fptr(hidden.reshape(-1)), T,
                                            binding.fptr(patch_in.reshape(-1)), patches, P, bounds, num_docs, closed,
                                            binding.fptr(want.reshape(-1))) == 0
    th, tp = torch.from_numpy(hidden).cuda(), torch.from_numpy(patch_in).cuda()
    tl = torch.full((T, V), 7.0, dtype=torch.float32, device="cuda")
    vh, vp, vl = _dev_tensor(th), _dev_tensor(tp), _dev_tensor(tl)
    arena = lib.blt_arena_create(64 << 20, abi.BLT_BACKEND_HIP)
    try:
        if impl == "public":
            lib.blt_local_decoder_forward_ext(device.ptr, C.byref(vh), C.byref(vp), patches, P, None, None, bounds,
                                              num_docs, None, closed, C.byref(vl), None, arena)
        else:
            lib.blt_local_decoder_forward_ext_hip(device.ptr, C.byref(vh), C.byref(vp), patches, P, bounds, num_docs,
                                                  closed, C.byref(vl), arena)
        lib.blt_backend_pass_sync_hip()
    finally:
        lib.blt_arena_destroy(arena)
    assert np.isfinite(want).all() and np.abs(want).max() > 1e-3
    assert_close(tl.cpu().numpy(), want, "decoder forward case %d closed %d docs %s" % (case, closed, docs))


def _tier(lib, cache, name, layer, rows, E):
    out = np.empty((rows, E), dtype=np.float32)
    lib.blt_hip_memcpy_d2h(out.ctypes.data, getattr(cache.contents, name)[layer].data, out.nbytes)
    return out


@pytest.mark.parametrize("impl", IMPLS)
@pytest.mark.parametrize("case", range(len(STEP_CASES)))
def test_kv_decode_step_single_sequence(case, impl, oracle, dev):
    """blt_kv_cache_refresh_cross + blt_kv_decode_step on device memory against the restated step:
    prefill chunk, single rows, re-segmentation; logits and all four cache tiers after every call."""
    import torch
    from fblt_amd import decoder
    lib = api.load()
    entry = _entry(impl, lib)
    c = STEP_CASES[case]
    E, V, k, L = c["E"], c["V"], c["k"], c["L"]
    rs = np.random.RandomState(300 + case)
    host, device = _decoders(oracle, c, 400 + case)
    mine = decoder.HostCache(host, c["max_len"])
    arena = lib.blt_arena_create(64 << 20, abi.BLT_BACKEND_HIP)
    try:
        cache = entry.blt_kv_cache_create(arena, device.ptr, c["max_len"])
        assert cache.contents.k == k and cache.contents.max_subtokens == c["max_len"]
        mark = arena.contents.offset
        d0_all = rs.randn(21, E).astype(np.float32)
        script = [([3, 4], 0, 7, 0), ([3, 4, 1], 2, 1, 0), ([3, 4, 2], 2, 1, 1), ([3, 4, 2, 5], 3, 5, 0),
                  ([3, 4, 2, 5, 1], 4, 1, 0), ([3, 4, 2, 5, 4], 4, 3, 1), ([3, 4, 2, 5, 4, 3], 5, 3, 0)]
        done, prev = 0, None
        for lengths, from_patch, n, closed in script:
            P = len(lengths)
            patches = decoder.patch_table(lengths)
            patch_in = rs.randn(P, k * E).astype(np.float32)
            if from_patch:
                patch_in[:from_patch] = prev[:from_patch]
            prev = patch_in
            same = entry.blt_kv_cache_common_patches(cache, patches, P)
            assert same == from_patch
            entry.blt_kv_cache_truncate(cache, cache.contents.self_len, min(from_patch, cache.contents.cross_num_patches))
            tp = torch.from_numpy(patch_in).cuda()
            vp = _dev_tensor(tp)
            arena.contents.offset = mark
            entry.blt_kv_cache_refresh_cross(cache, C.byref(vp), patches, P, from_patch, arena)
            assert cache.contents.cross_num_patches == P
            assert oracle.orc_kv_cache_refresh_cross(mine.ptr, 0, binding.fptr(patch_in.reshape(-1)), P, from_patch) == 0
            rows = np.ascontiguousarray(d0_all[done:done + n])
            ref = np.zeros((n, V), dtype=np.float32)
            assert oracle.orc_kv_decode_step(mine.ptr, 0, done, patches, P, binding.fptr(rows.reshape(-1)), n, closed,
                                             binding.fptr(ref.reshape(-1))) == 0
            td = torch.from_numpy(rows).cuda()
            tl = torch.full((n, V), 7.0, dtype=torch.float32, device="cuda")
            vd, vl = _dev_tensor(td), _dev_tensor(tl)
            entry.blt_kv_decode_step(cache, C.byref(vp), patches, P, C.byref(vd), closed, C.byref(vl), arena)
            lib.blt_backend_pass_sync_hip()
            done += n
            assert cache.contents.self_len == done
            assert_close(tl.cpu().numpy(), ref, "decode step logits case %d %s" % (case, lengths))
            for name in ("self_k", "self_v", "cross_k", "cross_v"):
                for l in range(L):
                    assert_close(_tier(lib, cache, name, l, c["max_len"], E), mine.tiers[name][l],
                                 "%s[%d] case %d %s" % (name, l, case, lengths))
        entry.blt_kv_cache_reset(cache)
        assert cache.contents.self_len == 0 and cache.contents.cross_num_patches == 0
        entry.blt_kv_cache_destroy(cache)
    finally:
        lib.blt_arena_destroy(arena)


@pytest.mark.parametrize("impl", IMPLS)
@pytest.mark.parametrize("shape", [(2, 8, 2, 12, "causal"), (33, 32, 4, 48, "window"), (70, 48, 3, 64, "docs"),
                                   (40, 64, 2, 96, "docs_window"), (64, 64, 2, 96, "docs_edge"),
                                   (200, 128, 4, 256, "docs_edge_window"),
                                   (512, 128, 4, 512, "docs_window"),    # a byte layer of the local encoder at C1 size
                                   (128, 512, 8, 1024, "docs"),          # a layer of the patch transformer at C2 size
                                   (300, 256, 4, 768, "causal")])
def test_transformer_block(shape, impl, oracle, dev):
    """blt_transformer_forward on device tensors against the restated block (csrc/models/
    transformer.c:97-128); impl = reference_callers runs the reference's transformer.c on this
    library's ops."""
    import torch
    from tests.golden.block_cases import transformer_case
    lib = api.load()
    entry = _entry(impl, lib)
    T, E, H, hidden, mask = shape
    rs = np.random.RandomState(T * 131 + E)
    x, w, cfg, _keep = transformer_case(rs, T, E, H, hidden, mask)
    order = ("norm1", "qkv", "proj", "norm2", "up", "gate", "down")
    ref = np.zeros((T, E), dtype=np.float32)
    assert oracle.orc_transformer_forward(binding.fptr(x.reshape(-1)), *(binding.fptr(w[n].reshape(-1)) for n in order),
                                          binding.fptr(ref.reshape(-1)), T, E, hidden, H, 1, 1, 500000.0, None, None,
                                          C.byref(cfg)) == 0
    tens = {n: torch.from_numpy(w[n]).cuda() for n in order}
    tv = {n: _dev_tensor(t) for n, t in tens.items()}
    wt = abi.BltTransformerWeights()
    wt.norm1_weight, wt.attn_qkv_w, wt.attn_proj_w = C.pointer(tv["norm1"]), C.pointer(tv["qkv"]), C.pointer(tv["proj"])
    wt.norm2_weight, wt.ffn_up_w, wt.ffn_gate_w = C.pointer(tv["norm2"]), C.pointer(tv["up"]), C.pointer(tv["gate"])
    wt.ffn_down_w = C.pointer(tv["down"])
    tc = abi.BltTransformerConfig()
    ac = tc.attn_config
    ac.embed_dim, ac.num_heads, ac.head_dim, ac.is_causal, ac.use_rope, ac.rope_theta = E, H, E // H, True, True, 500000.0
    ac.mask_config = C.pointer(cfg)
    tc.hidden_dim, tc.norm_type, tc.activation_type = hidden, abi.BLT_NORM_RMSNORM, abi.BLT_ACTIVATION_SWIGLU
    tx = torch.from_numpy(x).cuda()
    to = torch.full((T, E), 7.0, dtype=torch.float32, device="cuda")
    vx, vo = _dev_tensor(tx), _dev_tensor(to)
    arena = lib.blt_arena_create(256 << 20, abi.BLT_BACKEND_HIP)
    try:
        entry.blt_transformer_forward(C.byref(vx), C.byref(wt), C.byref(vo), C.byref(tc), arena)
        lib.blt_backend_pass_sync_hip()
        assert_close(to.cpu().numpy(), ref, "transformer block %s" % (shape,))
    finally:
        lib.blt_arena_destroy(arena)


def _transformer_block(T, E, H, hidden, shift=0, change=None):
    """blt_transformer_forward three times (the last one in place), weights `shift` floats off a 16-byte boundary and changed by
    `change`: the outputs, what was launched, and the block in float64."""
    import torch
    from tests.golden.block_cases import transformer_case
    lib = api.load()
    x, w, cfg, _keep = transformer_case(np.random.RandomState(T + E + hidden), T, E, H, hidden, "causal")
    hd = E // H
    pos = torch.arange(T, dtype=torch.float64)[:, None] * 500000.0 ** (-torch.arange(0, hd, 2, dtype=torch.float64) / hd)
    cos, sin = pos.cos().float(), pos.sin().float()
    if change:
        change(w)
    d = {n: torch.from_numpy(t).double() for n, t in w.items()}
    norm = lambda t, s: t / (t.pow(2).mean(1, keepdim=True) + 1e-6).sqrt() * s
    xs = torch.from_numpy(x).double()
    q, k, v = (norm(xs, d["norm1"]) @ d["qkv"]).view(T, 3, H, hd).permute(1, 2, 0, 3)

    def turn(t):
        a, b = t[..., 0::2], t[..., 1::2]
        c, s = cos.double(), sin.double()
        return torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2)
    att = (turn(q) @ turn(k).transpose(1, 2) / hd ** 0.5).masked_fill(torch.ones(T, T).triu(1).bool(), float("-inf")).softmax(-1) @ v
    resid = xs + att.transpose(0, 1).reshape(T, E) @ d["proj"]
    n2 = norm(resid, d["norm2"])
    want = resid + (torch.nn.functional.silu(n2 @ d["gate"]) * (n2 @ d["up"])) @ d["down"]

    order = ("norm1", "qkv", "proj", "norm2", "up", "gate", "down")
    tens = {}
    for n in order:
        room = torch.zeros(w[n].size + 4, device="cuda")
        tens[n] = room[shift:shift + w[n].size].view(w[n].shape)
        tens[n].copy_(torch.from_numpy(w[n]))
    tv = {n: _dev_tensor(t) for n, t in tens.items()}
    wt = abi.BltTransformerWeights()
    wt.norm1_weight, wt.attn_qkv_w, wt.attn_proj_w = C.pointer(tv["norm1"]), C.pointer(tv["qkv"]), C.pointer(tv["proj"])
    wt.norm2_weight, wt.ffn_up_w, wt.ffn_gate_w = C.pointer(tv["norm2"]), C.pointer(tv["up"]), C.pointer(tv["gate"])
    wt.ffn_down_w = C.pointer(tv["down"])
    tc = abi.BltTransformerConfig()
    ac = tc.attn_config
    ac.embed_dim, ac.num_heads, ac.head_dim, ac.is_causal, ac.use_rope, ac.rope_theta = E, H, hd, True, True, 500000.0
    tcos, tsin = cos.cuda(), sin.cuda()
    vc, vs = _dev_tensor(tcos), _dev_tensor(tsin)
    ac.rope_cos_cache, ac.rope_sin_cache, ac.mask_config = C.pointer(vc), C.pointer(vs), C.pointer(cfg)
    tc.hidden_dim, tc.norm_type, tc.activation_type = hidden, abi.BLT_NORM_RMSNORM, abi.BLT_ACTIVATION_SWIGLU
    rows = [torch.from_numpy(x).cuda() for _ in range(3)]
    outs = [torch.full((T, E), 7.0, device="cuda"), torch.full((T, E), 7.0, device="cuda"), rows[2]]   # the last one in place
    arena = lib.blt_arena_create(64 << 20, abi.BLT_BACKEND_HIP)
    try:
        torch.cuda.synchronize()
        lib.blt_hip_profile_begin()
        for r, o in zip(rows, outs):
            arena.contents.offset = 0
            vx, vo = _dev_tensor(r), _dev_tensor(o)
            lib.blt_transformer_forward(C.byref(vx), C.byref(wt), C.byref(vo), C.byref(tc), arena)
        launched = api.profile_end()
    finally:
        lib.blt_arena_destroy(arena)
    return outs, launched, want


@pytest.mark.parametrize("T,E,H,hidden,shift,fused", [(33, 64, 2, 64, 0, True), (48, 64, 2, 320, 0, True), (49, 128, 4, 64, 0, True),
                                                      (65, 128, 4, 576, 0, True), (1024, 128, 4, 512, 0, True),
                                                      (1025, 128, 4, 512, 0, False), (34, 256, 8, 192, 0, True),
                                                      (256, 256, 4, 1024, 0, True), (50, 128, 4, 96, 0, False),
                                                      (50, 128, 4, 512, 1, False), (50, 96, 3, 384, 0, False)])
def test_block_behind_its_attention(T, E, H, hidden, shift, fused, dev):
    """The launch behind the attention of a narrow block, at the edges of its row tiles, hidden slices and of its dispatch
    (shift: weights one float off a 16-byte boundary), in place and again: against float64, and the same bits each time."""
    outs, launched, want = _transformer_block(T, E, H, hidden, shift)
    assert launched.get("block_tail", (0,))[0] == (3 if fused else 0), launched
    got = [o.cpu().numpy() for o in outs]
    # each of the four products rounds a sum of at most 1024 terms: 2^-24 sqrt(1024) of it in the 2-norm, were it one chain of
    # independent roundings, and the four add up as independent errors
    assert _relative(outs[0].cpu(), want) <= 2 * 2 ** -24 * 1024 ** 0.5
    assert got[0].tobytes() == got[1].tobytes() == got[2].tobytes()


@pytest.mark.parametrize("T,E,H,hidden,shift,fused", [(1, 64, 2, 64, 0, True), (15, 128, 4, 512, 0, True), (16, 128, 4, 512, 0, True),
                                                      (17, 256, 4, 1024, 0, True), (32, 128, 4, 512, 0, True), (30, 512, 8, 2048, 0, False),
                                                      (2, 96, 3, 96, 0, False), (31, 128, 4, 512, 1, False), (9, 64, 2, 100, 0, False),
                                                      (25, 40, 2, 72, 0, False)])
def test_block_of_few_rows(T, E, H, hidden, shift, fused, dev):
    """Blocks of up to 32 rows run on the matrix cores like larger ones; widths, hidden layers and weights of every alignment, in place
    and again, against float64."""
    outs, launched, want = _transformer_block(T, E, H, hidden, shift)
    assert launched.get("block_tail", (0,))[0] == (3 if fused else 0) and "matmul_skinny" not in launched, launched
    # four products, each of which rounds a sum of at most max(E, hidden) terms, as above
    assert _relative(outs[0].cpu(), want) <= 2 * 2 ** -24 * max(E, hidden) ** 0.5
    assert outs[0].cpu().numpy().tobytes() == outs[1].cpu().numpy().tobytes() == outs[2].cpu().numpy().tobytes()


def test_block_of_few_rows_in_the_reference_order():
    """BLT_HIP_EXACT_STEP=1 keeps the exact kernel for them (read once a process)."""
    import os
    import subprocess
    import sys
    code = ("from tests.test_gpu_parity import _transformer_block, _relative\n"
            "outs, launched, want = _transformer_block(17, 128, 4, 512)\n"
            "assert 'matmul_skinny' in launched and 'block_tail' not in launched, launched\n"
            "assert _relative(outs[0].cpu(), want) < 1e-5\nprint('OK')\n")
    p = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300, env=dict(os.environ, BLT_HIP_EXACT_STEP="1"),
                       cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    assert p.returncode == 0 and "OK" in p.stdout, p.stdout[-2000:] + p.stderr[-2000:]


@pytest.mark.parametrize("T,E,H,hidden,fused", [(304, 64, 2, 2112, True), (305, 64, 2, 2112, False), (112, 128, 4, 2112, True),
                                                (113, 128, 4, 2112, False), (112, 256, 8, 1088, True), (113, 256, 8, 1088, False)])
def test_block_behind_its_attention_of_many_slices(T, E, H, hidden, fused, dev):
    """Both sides of the line from which the launch's last workgroup would have too many slices of the hidden layer to add up."""
    outs, launched, want = _transformer_block(T, E, H, hidden)
    assert launched.get("block_tail", (0,))[0] == (3 if fused else 0), launched
    # four products, each of which rounds a sum of at most 2112 terms
    assert _relative(outs[0].cpu(), want) <= 2 * 2 ** -24 * 2112 ** 0.5
    assert outs[0].cpu().numpy().tobytes() == outs[1].cpu().numpy().tobytes() == outs[2].cpu().numpy().tobytes()


@pytest.mark.parametrize("T,hidden,shift", [(301, 2048, 0), (301, 2048, 1), (640, 2048, 0), (577, 2050, 0), (1000, 2048, 0), (1000, 2048, 1),
                                            (965, 1100, 2)])
def test_block_whose_down_projection_is_in_slices(T, hidden, shift, dev):
    """A sliced product with a residual, which the last slice's workgroup adds: on parts of either kind, in 16-byte pieces and in
    single values."""
    assert _product_kernel(T, hidden, 512)[0] == "matmul_mfma_slices"
    outs, launched, want = _transformer_block(T, 512, 8, hidden, shift)
    assert launched["matmul_mfma_slices"][0] == 3, launched
    # four products, each of which rounds a sum of at most `hidden` terms
    assert _relative(outs[0].cpu(), want) <= 2 * 2 ** -24 * hidden ** 0.5
    assert outs[0].cpu().numpy().tobytes() == outs[1].cpu().numpy().tobytes() == outs[2].cpu().numpy().tobytes()


@pytest.mark.parametrize("T", [300, 2048])
@pytest.mark.parametrize("what", ["as drawn", "below", "above"])
def test_block_on_halves_out_of_range(T, what, dev):
    """The tile kernel's other ends -- norm and rotation, norm and gate -- with operands that send it from its f16 parts to its bf16
    parts: V columns and an up matrix far below their range, values above it in the last step.  Each column against float64:
    of four products in a row, each rounds a sum of at most 1024 terms like a chain of independent roundings."""
    def change(w):
        E = w["qkv"].shape[0]
        if what == "below":
            w["qkv"][:, 2 * E:] *= np.float32(1e-9)
            w["proj"] *= np.float32(1e9)
            w["up"] *= np.float32(1e-9)
            w["down"] *= np.float32(1e9)
        elif what == "above":
            w["qkv"][E - 1, 2 * E + 5], w["up"][E - 1, 9], w["gate"][E - 1, 7] = 2e3, 3e3, 4e3
    outs, launched, want = _transformer_block(T, 512, 8, 1024, change=change)
    assert launched["matmul_mfma"][0] >= 3 * 2, launched
    off, size = (outs[0].cpu().double() - want).norm(dim=0), want.norm(dim=0)
    assert (off / size).max().item() <= 4 * 2 ** -24 * 1024 ** 0.5
    assert outs[0].cpu().numpy().tobytes() == outs[1].cpu().numpy().tobytes() == outs[2].cpu().numpy().tobytes()


@pytest.mark.parametrize("P,E,H,hidden,L,docs", [(128, 512, 8, 1024, 2, [40, 90]),   # C2's caller: one window of patches
                                                 (50, 64, 2, 96, 3, []), (200, 128, 4, 256, 1, [7, 8, 150])])
def test_global_transformer_on_the_fused_block(P, E, H, hidden, L, docs, oracle, dev):
    """The reference's patch transformer -- csrc/models/global_transformer.c:69-97 over
    transformer_stack.c:228-248, both compiled unmodified -- with this library's
    blt_transformer_forward under it (and blt_build_attention_mask, blt_rope_precompute,
    blt_tensor_create, blt_strided_copy): the model is created in a device arena by the
    reference's own constructor, filled with seeded weights, and compared with the restated
    block applied layer by layer under the document-causal mask."""
    import torch
    lib = api.load()
    stack_lib = binding.load_ref_stack_callers()
    if stack_lib is None:
        pytest.skip("oracle/_ref/libblt_ref_stack_callers.so was not built (needs the reference sources)")
    rs = np.random.RandomState(P * 7 + E)
    arena = lib.blt_arena_create(512 << 20, abi.BLT_BACKEND_HIP)
    try:
        cfg = binding.BltGlobalTransformerConfig(E, L, hidden, H, 500000.0, 256, False, False)
        model = stack_lib.blt_global_transformer_create(arena, C.byref(cfg))
        assert model.contents.stack.num_layers == L and model.contents.stack.head_dim == E // H
        order = ("norm1_weight", "attn_qkv_w", "attn_proj_w", "norm2_weight", "ffn_up_w", "ffn_gate_w", "ffn_down_w")
        layers = []
        for l in range(L):
            w = {"norm1_weight": (1.0 + 0.1 * rs.randn(E)), "attn_qkv_w": rs.randn(E, 3 * E) / np.sqrt(E),
                 "attn_proj_w": rs.randn(E, E) / np.sqrt(E), "norm2_weight": (1.0 + 0.1 * rs.randn(E)),
                 "ffn_up_w": rs.randn(E, hidden) / np.sqrt(E), "ffn_gate_w": rs.randn(E, hidden) / np.sqrt(E),
                 "ffn_down_w": rs.randn(hidden, E) / np.sqrt(hidden)}
            w = {n: np.ascontiguousarray(a, dtype=np.float32) for n, a in w.items()}
            for n in order:
                t = getattr(model.contents.stack.layer_weights[l], n)
                assert tuple(t.contents.shape[:t.contents.ndim]) == w[n].shape
                lib.blt_tensor_upload(t, w[n].ctypes.data, w[n].nbytes)
            layers.append(w)
        x = rs.randn(P, E).astype(np.float32)
        tx = torch.from_numpy(x).cuda()
        to = torch.full((P, E), 7.0, dtype=torch.float32, device="cuda")
        vx, vo = _dev_tensor(tx), _dev_tensor(to)
        bounds = abi.size_array(docs) if docs else None
        stack_lib.blt_global_transformer_forward(model, C.byref(vx), bounds, len(docs) + 1 if docs else 0, C.byref(vo),
                                                 arena)
        lib.blt_backend_pass_sync_hip()
        got = to.cpu().numpy()
    finally:
        lib.blt_arena_destroy(arena)
    mc = abi.BltMaskConfig()
    mc.seq_len_q = mc.seq_len_kv = P
    mc.is_causal = True
    if docs:
        mc.doc_boundaries, mc.num_docs = bounds, len(docs) + 1
    cur = x
    for w in layers:
        nxt = np.zeros((P, E), dtype=np.float32)
        assert oracle.orc_transformer_forward(binding.fptr(cur.reshape(-1)), *(binding.fptr(w[n].reshape(-1)) for n in order),
                                              binding.fptr(nxt.reshape(-1)), P, E, hidden, H, 1, 1, 500000.0, None, None,
                                              C.byref(mc)) == 0
        cur = nxt
    assert_close(got, cur, "global transformer P=%d E=%d L=%d" % (P, E, L))


# (patch lengths of the clean prefix, block rows, trailing_closed, d0 mode, how the block is filled)
DIFFUSION_SCRIPTS = [
    ([3, 4, 2], 4, 1, abi.BLT_D0_ZEROS, "draft"),      # blt_draft_block's batch: all [MASK], positions N + r, o_M
    ([3, 4, 2, 5], 8, 1, abi.BLT_D0_LEARNED, "draft"),
    ([5, 1, 6], 3, 0, abi.BLT_D0_LEARNED, "mixed"),    # some cells unmasked, groups and positions of the caller's
    ([2, 2, 2, 2, 3], 16, 1, abi.BLT_D0_ZEROS, "mixed"),
    ([7], 1, 1, abi.BLT_D0_LEARNED, "draft"),
    ([9, 8, 12, 7, 11, 3], 32, 1, abi.BLT_D0_LEARNED, "draft"),   # 50 clean rows: the prefill kernels
    ([30, 31, 29, 33, 17], 4, 0, abi.BLT_D0_ZEROS, "mixed"),      # 140 clean rows
]


def _diffusion_batch(rs, N, R, P, fill, closed, max_len):
    from fblt_amd import decoder
    if fill == "draft":
        return decoder.BlockBatch(N, R, P, trailing_closed=closed)
    tokens = [int(rs.randint(0, 256)) if rs.rand() < 0.5 else abi.BLT_MASK_TOKEN_ID for _ in range(R)]
    positions = [int(x) for x in np.sort(rs.randint(0, max_len, size=R))]
    groups = [int(rs.randint(0, P)) for _ in range(R)]
    return decoder.BlockBatch(N, R, P, tokens=tokens, positions=positions, groups=groups, trailing_closed=closed)


@pytest.mark.parametrize("impl", IMPLS)
@pytest.mark.parametrize("script", range(len(DIFFUSION_SCRIPTS)))
@pytest.mark.parametrize("case", range(len(STEP_CASES)))
def test_diffusion_infer_forward(case, script, impl, oracle, dev):
    """blt_local_decoder_forward_diffusion_infer on device tensors against the restated dense
    forward (csrc/models/block_diffusion.c:776-795): logits of all N + R rows.  impl =
    reference_callers runs the reference's own block_diffusion.c (S x S attention through one core
    call per head against the dense INFER mask) on this library's ops.  Then the block rows alone
    through blt_kv_block_step_hip over a cache that blt_kv_decode_step filled with the prefix."""
    import torch
    from fblt_amd import decoder
    lib = api.load()
    entry = _entry(impl, lib)
    c = STEP_CASES[case]
    lengths, R, closed, d0_mode, fill = DIFFUSION_SCRIPTS[script]
    E, V, k = c["E"], c["V"], c["k"]
    N, P = sum(lengths), len(lengths)
    if N + R > c["max_len"]:
        pytest.skip("sequence longer than this decoder's tables")
    rs = np.random.RandomState(8000 + 10 * case + script)
    host, device = _decoders(oracle, c, 500 + case)
    patches = decoder.patch_table(lengths)
    hidden = rs.randn(N, E).astype(np.float32)
    patch_in = rs.randn(P, k * E).astype(np.float32)
    batch = _diffusion_batch(rs, N, R, P, fill, closed, c["max_len"])
    ref = np.zeros((N + R, V), dtype=np.float32)
    assert oracle.orc_local_decoder_forward_diffusion_infer(
        host.ptr, binding.fptr(hidden.reshape(-1)), binding.fptr(patch_in.reshape(-1)), patches, P, batch.ptr, d0_mode,
        binding.fptr(ref.reshape(-1))) == 0
    arena = lib.blt_arena_create(256 << 20, abi.BLT_BACKEND_HIP)
    try:
        th, tp = torch.from_numpy(hidden).cuda(), torch.from_numpy(patch_in).cuda()
        tl = torch.full((N + R, V), 7.0, dtype=torch.float32, device="cuda")
        vh, vp, vl = _dev_tensor(th), _dev_tensor(tp), _dev_tensor(tl)
        entry.blt_local_decoder_forward_diffusion_infer(device.ptr, C.byref(vh), C.byref(vp), patches, P, batch.ptr,
                                                        d0_mode, C.byref(vl), arena)
        lib.blt_backend_pass_sync_hip()
        assert_close(tl.cpu().numpy(), ref, "diffusion forward case %d script %d" % (case, script))
        if impl != "library":
            return
        # the draft loop's form: prefix decoded once through the incremental step, block rows per pass
        device.struct.config.local_window = 0      # the diffusion forward has no window
        lib.blt_arena_reset(arena)
        cache = lib.blt_kv_cache_create(arena, device.ptr, c["max_len"])
        lib.blt_kv_cache_refresh_cross(cache, C.byref(vp), patches, P, 0, arena)
        tc = torch.zeros((N, V), dtype=torch.float32, device="cuda")
        vc = _dev_tensor(tc)
        lib.blt_kv_decode_step(cache, C.byref(vp), patches, P, C.byref(vh), closed, C.byref(vc), arena)
        assert cache.contents.self_len == N
        for _ in range(2):                         # a pass changes nothing in the cache
            tb = torch.full((R, V), 7.0, dtype=torch.float32, device="cuda")
            vb = _dev_tensor(tb)
            lib.blt_kv_block_step_hip(cache, P, batch.ptr, d0_mode, C.byref(vb), arena)
            lib.blt_backend_pass_sync_hip()
            assert cache.contents.self_len == N
            assert_close(tb.cpu().numpy(), ref[N:], "block step case %d script %d" % (case, script))
        assert_close(tc.cpu().numpy(), ref[:N], "prefix step case %d script %d" % (case, script))
        lib.blt_kv_cache_destroy(cache)
    finally:
        lib.blt_arena_destroy(arena)


@pytest.mark.parametrize("window", [0, 20])
def test_kv_decode_step_long_prefill(window, oracle, dev):
    """A prompt prefill in one call: more new rows than one step launch takes (45, then 1, then
    50 rows: staged once and attended as one batch of prefill problems), with and without a local
    window, against the restated step; logits and tiers after every call."""
    import torch
    from fblt_amd import decoder
    lib = api.load()
    c = dict(E=128, H=4, XH=4, L=2, hidden=256, V=256, max_len=128, k=1, window=window, all_layers=True, placement=0)
    E, V, L = c["E"], c["V"], c["L"]
    rs = np.random.RandomState(911)
    host, device = _decoders(oracle, c, 912)
    mine = decoder.HostCache(host, c["max_len"])
    arena = lib.blt_arena_create(64 << 20, abi.BLT_BACKEND_HIP)
    try:
        cache = lib.blt_kv_cache_create(arena, device.ptr, c["max_len"])
        mark = arena.contents.offset
        lengths = [5, 7, 3, 9, 6, 8, 4, 10, 2, 9, 7, 11, 15]      # 96 bytes
        P = len(lengths)
        patches = decoder.patch_table(lengths)
        patch_in = rs.randn(P, E).astype(np.float32)
        tp = torch.from_numpy(patch_in).cuda()
        vp = _dev_tensor(tp)
        lib.blt_kv_cache_refresh_cross(cache, C.byref(vp), patches, P, 0, arena)
        assert oracle.orc_kv_cache_refresh_cross(mine.ptr, 0, binding.fptr(patch_in.reshape(-1)), P, 0) == 0
        done = 0
        for n in (45, 1, 50):
            rows = rs.randn(n, E).astype(np.float32)
            ref = np.zeros((n, V), dtype=np.float32)
            assert oracle.orc_kv_decode_step(mine.ptr, 0, done, patches, P, binding.fptr(rows.reshape(-1)), n, 0,
                                             binding.fptr(ref.reshape(-1))) == 0
            td = torch.from_numpy(rows).cuda()
            tl = torch.full((n, V), 7.0, dtype=torch.float32, device="cuda")
            vd, vl = _dev_tensor(td), _dev_tensor(tl)
            arena.contents.offset = mark
            lib.blt_kv_decode_step(cache, C.byref(vp), patches, P, C.byref(vd), 0, C.byref(vl), arena)
            lib.blt_backend_pass_sync_hip()
            done += n
            assert cache.contents.self_len == done
            assert_close(tl.cpu().numpy(), ref, "long prefill logits n=%d" % n)
            for name in ("self_k", "self_v"):
                for l in range(L):
                    assert_close(_tier(lib, cache, name, l, c["max_len"], E), mine.tiers[name][l],
                                 "%s[%d] after %d rows" % (name, l, done))
        lib.blt_kv_cache_destroy(cache)
    finally:
        lib.blt_arena_destroy(arena)


@pytest.mark.parametrize("L,P,launches", [(3, 40, 2), (2, 70, 1), (2, 32, 2)])   # 33 rows and more: two layers a launch
def test_refresh_of_two_layers_in_one_launch(L, P, launches, oracle, dev):
    import torch
    from fblt_amd import decoder
    lib = api.load()
    c = dict(E=128, H=4, XH=4, L=L, hidden=64, V=16, max_len=160, k=1, window=0, all_layers=True, placement=0)
    rs = np.random.RandomState(77 + P)
    host, device = _decoders(oracle, c, 78)
    mine = decoder.HostCache(host, c["max_len"])
    arena = lib.blt_arena_create(64 << 20, abi.BLT_BACKEND_HIP)
    try:
        cache = lib.blt_kv_cache_create(arena, device.ptr, c["max_len"])
        patches = decoder.patch_table([2] * P)
        patch_in = rs.randn(P, c["E"]).astype(np.float32)
        tp = torch.from_numpy(patch_in).cuda()
        vp = _dev_tensor(tp)
        lib.blt_hip_profile_begin()
        lib.blt_kv_cache_refresh_cross(cache, C.byref(vp), patches, P, 0, arena)
        assert sum(e[0] for e in api.profile_end().values()) == launches
        lib.blt_backend_pass_sync_hip()
        assert oracle.orc_kv_cache_refresh_cross(mine.ptr, 0, binding.fptr(patch_in.reshape(-1)), P, 0) == 0
        for name in ("cross_k", "cross_v"):
            for l in range(L):
                assert_close(_tier(lib, cache, name, l, P, c["E"]), mine.tiers[name][l][:P], "%s[%d]" % (name, l))
        lib.blt_kv_cache_destroy(cache)
    finally:
        lib.blt_arena_destroy(arena)


def _decode_steps(batch, n, c, seed, oracle, row_scale=1.0, before_sync=None, cross=None, shifted=()):
    """Two steps of a batched cache against the restated step run sequence by sequence; the kernels each step launched.
    before_sync(logits): called after each step, before the library synchronises.  cross(name, slab): changes the tier-2
    slabs before the first step; sequences whose reference is not finite are then not compared, the others are.  shifted: weights of every layer that lie four bytes off a 16-byte boundary."""
    import torch
    from fblt_amd import decoder
    lib = api.load()
    launched = []
    E, V, k, L, max_len = c["E"], c["V"], c["k"], c["L"], c["max_len"]
    rs = np.random.RandomState(500 + batch + n)
    host, device = _decoders(oracle, c, seed)
    for l in range(L):
        for name in shifted:
            field = getattr(device.layers[l], name)
            values = next(t for t in device.keep if t.data_ptr() == field.data)
            room = torch.zeros(values.numel() + 1, device="cuda")
            room[1:] = values.view(-1)
            device.keep.append(room)
            field.data = room.data_ptr() + 4
    mine = decoder.HostCache(host, max_len, batch)
    arena = lib.blt_arena_create(256 << 20, abi.BLT_BACKEND_HIP)
    try:
        cache = lib.blt_kv_cache_create_batched(arena, device.ptr, max_len, batch)
        mark = arena.contents.offset
        lens = rs.randint(1, max_len - 2 * n, size=batch)
        tables, counts, keep_in = [], [], []
        for b in range(batch):
            # patches tile the decoded bytes plus the rows of both steps
            total = int(lens[b]) + 2 * n
            cuts = np.sort(rs.choice(np.arange(1, total), size=min(total - 1, rs.randint(1, 6)), replace=False))
            lengths = np.diff(np.concatenate([[0], cuts, [total]])).tolist()
            tables.append(decoder.patch_table(lengths))
            counts.append(len(lengths))
            patch_in = rs.randn(len(lengths), k * E).astype(np.float32)
            tp = torch.from_numpy(patch_in).cuda()
            vp = _dev_tensor(tp)
            keep_in.append(tp)
            lib.blt_kv_cache_refresh_cross_seq_hip(cache, b, C.byref(vp), tables[b], counts[b], 0, arena)
            assert oracle.orc_kv_cache_refresh_cross(mine.ptr, b, binding.fptr(patch_in.reshape(-1)), counts[b], 0) == 0
        # valid tier-1 rows: the same random content on both sides
        for name in ("self_k", "self_v"):
            for l in range(L):
                slab = mine.tiers[name][l]
                for b in range(batch):
                    slab[b * max_len:b * max_len + lens[b]] = rs.randn(int(lens[b]), E).astype(np.float32)
                lib.blt_hip_memcpy_h2d(getattr(cache.contents, name)[l].data, slab.ctypes.data, slab.nbytes)
        for name in ("cross_k", "cross_v") if cross else ():
            for l in range(L):
                slab = mine.tiers[name][l]
                cross(name, slab.reshape(batch, -1, E))
                lib.blt_hip_memcpy_h2d(getattr(cache.contents, name)[l].data, slab.ctypes.data, slab.nbytes)
        lib.blt_backend_pass_sync_hip()
        self_len = abi.size_array(lens.tolist())
        table_ptrs = (C.POINTER(abi.BltPatchInfo) * batch)(*(C.cast(t, C.POINTER(abi.BltPatchInfo)) for t in tables))
        num = abi.size_array(counts)
        for step in range(2):
            closed = (C.c_int * batch)(*([0] * batch if step == 0 else rs.randint(0, 2, size=batch).tolist()))
            rows = (rs.randn(batch * n, E) * row_scale).astype(np.float32)
            ref = np.zeros((batch * n, V), dtype=np.float32)
            for b in range(batch):
                r = np.ascontiguousarray(rows[b * n:(b + 1) * n])
                out = np.zeros((n, V), dtype=np.float32)
                assert oracle.orc_kv_decode_step(mine.ptr, b, int(lens[b]) + step * n, tables[b], counts[b],
                                                 binding.fptr(r.reshape(-1)), n, closed[b],
                                                 binding.fptr(out.reshape(-1))) == 0
                ref[b * n:(b + 1) * n] = out
            td = torch.from_numpy(rows).cuda()
            tl = torch.full((batch * n, V), 7.0, dtype=torch.float32, device="cuda")
            vd, vl = _dev_tensor(td), _dev_tensor(tl)
            arena.contents.offset = mark
            lib.blt_hip_profile_begin()
            lib.blt_kv_decode_step_batched_hip(cache, self_len, table_ptrs, num, closed, C.byref(vd), C.byref(vl), arena)
            launched.append(sorted(api.profile_end()))
            if before_sync:
                before_sync(tl)
            lib.blt_backend_pass_sync_hip()
            assert [self_len[b] for b in range(batch)] == (lens + (step + 1) * n).tolist()
            if cross:
                valid = np.isfinite(ref).all(axis=1)
                assert valid.any() and not valid.all()
                assert_close(tl.cpu().numpy()[valid], ref[valid], "batched step %d logits" % step)
                break                                # the cached rows of the others are not finite from here on
            # the absolute term of the tolerance is for rows of order one
            assert_close(tl.cpu().numpy() / np.float32(row_scale), ref / np.float32(row_scale), "batched step %d logits" % step)
            for name in ("self_k", "self_v", "cross_k", "cross_v"):
                for l in range(L):
                    assert_close(_tier(lib, cache, name, l, batch * max_len, E), mine.tiers[name][l],
                                 "%s[%d] batched step %d" % (name, l, step))
        lib.blt_kv_cache_destroy(cache)
    finally:
        lib.blt_arena_destroy(arena)
    return launched


@pytest.mark.parametrize("batch,n,case", [(8, 1, 0), (64, 1, 2), (16, 4, 1), (5, 3, 3), (64, 8, 2),
                                          (3, 40, 4), (5, 33, 5)])   # chunks of more than 32 rows per sequence
def test_kv_decode_step_batched(batch, n, case, oracle, dev):
    """blt_kv_decode_step_batched_hip: every sequence of a batched cache in one pass, against the
    restated step run sequence by sequence; two steps in a row."""
    _decode_steps(batch, n, STEP_CASES[case], 600 + case, oracle)


RESIDENT_CASES = [
    dict(E=64, H=2, XH=2, L=8, hidden=32, V=16, max_len=160, k=1, window=0, all_layers=True, placement=0),
    dict(E=64, H=1, XH=1, L=1, hidden=160, V=48, max_len=300, k=2, window=0, all_layers=True, placement=0),
    dict(E=128, H=4, XH=4, L=2, hidden=1024, V=256, max_len=300, k=1, window=100, all_layers=False, placement=0),
    dict(E=128, H=2, XH=2, L=2, hidden=512, V=64, max_len=300, k=3, window=0, all_layers=True, placement=0),
    dict(E=256, H=8, XH=8, L=2, hidden=1024, V=256, max_len=150, k=2, window=40, all_layers=True, placement=0),
    dict(E=256, H=4, XH=4, L=1, hidden=992, V=272, max_len=300, k=1, window=0, all_layers=True, placement=0),
    dict(E=64, H=2, XH=2, L=1, hidden=96, V=32, max_len=120, k=3, window=0, all_layers=True, placement=0),
]


def in_one_launch(launched):
    """Every step the resident kernel and nothing else (the first one of a stream clears its words)."""
    return all(names in (["kv_step_resident"], ["kv_step_clear", "kv_step_resident"]) for names in launched)


@pytest.mark.parametrize("batch,n,case", [(1, 32, 0), (8, 17, 0), (33, 1, 0), (1, 1, 1), (32, 1, 1),   # rows of a group 1 ... 32 at
                                          (1, 16, 2), (1, 1, 2), (9, 8, 2), (17, 1, 3),               # 64 columns, 1 ... 16 at 128 and
                                          (1, 11, 4), (8, 16, 4), (64, 1, 4), (1, 1, 5), (30, 1, 5),   # 256, heads of 32 and 64;
                                          (9, 9, 0), (9, 16, 0), (17, 8, 0), (33, 5, 0), (58, 3, 0)])  # two row tiles, 3 ... 16 rows
def test_kv_decode_step_in_one_launch(batch, n, case, oracle, dev):
    """The one-launch form of the step at the edges of its shapes, the last group of sequences shorter than the others
    among them, against the restated step."""
    assert in_one_launch(_decode_steps(batch, n, RESIDENT_CASES[case], 600 + case, oracle))


@pytest.mark.parametrize("E,H,batch,n", [(64, 2, 1, 9), (64, 2, 9, 9), (64, 1, 1, 16), (64, 1, 30, 1), (128, 4, 1, 16), (128, 4, 17, 3),
                                         (128, 2, 1, 5), (128, 2, 29, 1)])
@pytest.mark.parametrize("k", [1, 2, 6])
def test_kv_decode_step_in_one_launch_by_sub_tokens(E, H, batch, n, k, oracle, dev):
    """The cross block folded into the QKV tiles (one sub-token a patch) and in stages of its own (more), one and two row tiles,
    heads of 32 and 64, a short last group among them, against the restated step."""
    c = dict(E=E, H=H, XH=H, L=2, hidden=128, V=32, max_len=200, k=k, window=0, all_layers=True, placement=0)
    assert in_one_launch(_decode_steps(batch, n, c, 680 + k, oracle))


@pytest.mark.parametrize("n,case", [(2, 1), (16, 1), (2, 3), (16, 3), (15, 5), (16, 5)])
def test_kv_decode_step_of_one_sequence_with_wide_heads(n, case, oracle, dev):
    """Several rows of one sequence at heads of 64 columns take the one-launch form, up to one row tile."""
    assert in_one_launch(_decode_steps(1, n, RESIDENT_CASES[case], 640 + case, oracle))


def test_kv_decode_step_of_wide_heads_past_one_row_tile(oracle, dev):
    launched = _decode_steps(1, 17, RESIDENT_CASES[1], 641, oracle)
    assert all("kv_step_resident" not in names for names in launched), launched


@pytest.mark.parametrize("batch,n,case", [(1, 17, 2), (1, 32, 4), (9, 2, 3), (40, 1, 5), (9, 17, 0)])
def test_kv_decode_step_past_one_launch(batch, n, case, oracle, dev):
    """One row more than the one-launch form takes: the launches, against the restated step."""
    launched = _decode_steps(batch, n, RESIDENT_CASES[case], 600 + case, oracle)
    assert all("kv_step_resident" not in names for names in launched), launched


@pytest.mark.parametrize("batch,n,case,product", [(2, 33, 2, "matmul_splitk"), (24, 64, 4, "matmul_mfma")])
def test_kv_decode_step_of_chunks_staged_by_their_product(batch, n, case, product, oracle, dev):
    """Chunks of more than 32 rows: the QKV product leaves Q rotated and writes K and V to the slabs, from either kernel."""
    launched = _decode_steps(batch, n, RESIDENT_CASES[case], 660 + case, oracle)
    staged = [sum(name.startswith(("kv_", "rope")) for name in names) for names in launched]
    assert all(product in names for names in launched) and staged == [0, 0], launched


@pytest.mark.parametrize("batch,n,E,H,XH,k,joined", [
    (1, 33, 128, 4, 4, 1, True), (3, 40, 64, 2, 4, 2, True), (4, 12, 128, 2, 8, 1, True), (3, 15, 64, 1, 1, 3, True),   # staged, packed
    (40, 34, 128, 4, 4, 1, True), (42, 33, 128, 4, 4, 1, False), (124, 33, 64, 2, 2, 1, True), (125, 33, 64, 2, 2, 1, False)])
def test_kv_decode_step_whose_cross_blocks_go_with_the_qkv_product(batch, n, E, H, XH, k, joined, oracle, dev):
    """Both products of the rows in one launch, last tiles of 1 ... 16 rows, at the most rows it takes and beyond, against the
    restated step."""
    c = dict(E=E, H=H, XH=XH, L=2, hidden=64, V=32, max_len=160, k=k, window=0, all_layers=True, placement=0)
    launched = _decode_steps(batch, n, c, 670 + batch, oracle)
    assert all(("cross_qkv" in names) == joined and ("cross_block" in names) != joined for names in launched), launched


@pytest.mark.parametrize("batch,n,E,k,every,staged", [
    (1, 33, 128, 2, True, False), (3, 15, 64, 3, True, False), (59, 16, 128, 1, True, False), (130, 10, 64, 1, True, False),
    (1, 1757, 64, 1, True, False), (1, 1758, 64, 1, True, True),           # as many rows as go along, and one more
    (59, 16, 128, 1, False, True), (1, 40, 256, 1, True, True)])             # no cross block in front; none in one launch
def test_kv_decode_step_whose_row_ranges_go_with_the_first_launch(batch, n, E, k, every, staged, oracle, dev):
    """Lengths and row ranges in the arguments of the first layer's cross block, which the later layers find in memory, or by a
    launch of their own, against the restated step."""
    c = dict(E=E, H=E // 32, XH=E // 32, L=2, hidden=64, V=16, max_len=2 * n + 60, k=k, window=0, all_layers=every, placement=0)
    launched = _decode_steps(batch, n, c, 690 + batch, oracle)
    assert all(("upload_words" in names) == staged for names in launched), launched


@pytest.mark.parametrize("batch,n,case", [(1, 1, 2), (9, 8, 2), (33, 1, 0)])
def test_kv_decode_step_of_rows_whose_norm_overflows(batch, n, case, oracle, dev):
    """Input rows of 1e20: their sum of squares is infinite and the normalised row zero, in the one-launch form as in
    the restated step."""
    assert in_one_launch(_decode_steps(batch, n, RESIDENT_CASES[case], 600 + case, oracle, row_scale=1e20))


@pytest.mark.parametrize("batch,n,case", [(16, 1, 1), (33, 1, 6), (136, 1, 6), (24, 1, 3)])   # one and two row tiles at 64 columns; 128
def test_kv_decode_step_in_one_launch_with_faded_keys(batch, n, case, oracle, dev):
    """Sub-tokens of a patch with scores far apart, the first with an infinite value row: where it has no weight against the
    ones behind it, it has no part in the result."""
    c = RESIDENT_CASES[case]
    k, E = c["k"], c["E"]
    up = np.random.RandomState(case).randn(E).astype(np.float32)

    def cross(name, slab):                           # [sequences, sub-tokens, columns]
        for j in range(k):                           # in steps, so that no single step makes the weight zero
            if name == "cross_k":
                slab[:, j::k] = up * (150.0 * j)
            elif j == 0:
                slab[:, j::k, E - 1] = np.inf
    assert in_one_launch(_decode_steps(batch, n, c, 650 + case, oracle, cross=cross))


@pytest.mark.parametrize("case,shifted,one_launch", [
    (0, "attn_proj_w", False), (2, "attn_proj_w", False), (2, "cross_weight_proj", False),   # merged: sixteen bytes at a time
    (4, "attn_proj_w", True), (4, "cross_weight_proj", True), (2, "norm2_weight", True)])    # by the word
def test_kv_decode_step_with_weights_off_their_boundary(case, shifted, one_launch, oracle, dev):
    launched = _decode_steps(8, 1, RESIDENT_CASES[case], 670 + case, oracle, shifted=(shifted,))
    assert in_one_launch(launched) if one_launch else all("kv_step_resident" not in names for names in launched), launched


@pytest.mark.parametrize("mode", ["team", "wrap", "giveup"])
def test_one_launch_step_under_adverse_conditions(mode):
    """Workgroups that are not all resident, tags that run through, waits that run out: see step_pin_case.py."""
    import os
    import subprocess
    import sys
    script = os.path.join(os.path.dirname(os.path.abspath(__file__)), "step_pin_case.py")
    p = subprocess.run([sys.executable, "-u", script, mode], capture_output=True, text=True, timeout=100)
    assert "CHECKED" in p.stdout, (p.stdout[-2000:], p.stderr[-2000:])
    assert "NOT REACHED" not in p.stdout
    if mode == "giveup":
        assert p.returncode == 1 and "gave up waiting" in p.stderr, (p.returncode, p.stderr[-500:])
    else:
        assert p.returncode == 0, (p.returncode, p.stderr[-500:])


class _StepOnStream:
    """A batch of sequences whose next step can be issued over and over, each time from the same lengths."""

    def __init__(self, lib, oracle, c, seed, batch, repeats):
        import torch
        from fblt_amd import decoder
        rs = np.random.RandomState(seed)
        self.lib, self.c, self.batch = lib, c, batch
        self.device = _decoders(oracle, c, seed)[1]
        self.arena = lib.blt_arena_create(256 << 20, abi.BLT_BACKEND_HIP)
        self.cache = lib.blt_kv_cache_create_batched(self.arena, self.device.ptr, c["max_len"], batch)
        self.mark = self.arena.contents.offset
        self.lens = rs.randint(1, c["max_len"] - 2, size=batch).tolist()
        tables = [decoder.patch_table([n + 1]) for n in self.lens]
        pin = torch.from_numpy(rs.randn(1, c["k"] * c["E"]).astype(np.float32)).cuda()
        for b in range(batch):
            vp = _dev_tensor(pin)
            lib.blt_kv_cache_refresh_cross_seq_hip(self.cache, b, C.byref(vp), tables[b], 1, 0, self.arena)
        for name in ("self_k", "self_v"):
            for l in range(c["L"]):
                slab = rs.randn(batch * c["max_len"], c["E"]).astype(np.float32)
                lib.blt_hip_memcpy_h2d(getattr(self.cache.contents, name)[l].data, slab.ctypes.data, slab.nbytes)
        lib.blt_backend_pass_sync_hip()
        self.rows = torch.from_numpy(rs.randn(batch, c["E"]).astype(np.float32)).cuda()
        self.logits = torch.full((repeats, batch, c["V"]), 7.0, device="cuda")
        self.ptrs = (C.POINTER(abi.BltPatchInfo) * batch)(*(C.cast(t, C.POINTER(abi.BltPatchInfo)) for t in tables))
        self.num, self.keep = abi.size_array([1] * batch), (tables, pin)

    def step(self, i):
        self.arena.contents.offset = self.mark
        lens, closed = abi.size_array(self.lens), (C.c_int * self.batch)()
        vd, vl = _dev_tensor(self.rows), _dev_tensor(self.logits[i])
        self.lib.blt_kv_decode_step_batched_hip(self.cache, lens, self.ptrs, self.num, closed, C.byref(vd), C.byref(vl), self.arena)

    def close(self):
        self.lib.blt_kv_cache_destroy(self.cache)
        self.lib.blt_arena_destroy(self.arena)


@pytest.mark.parametrize("threads", [False, True])
def test_one_launch_steps_on_two_streams(threads, oracle, dev):
    """Steps issued on two streams without waiting for each other, from one thread on two streams of its own and from two
    threads on hipStreamPerThread (one handle, two streams): every one gives what the step alone gives, bit for bit."""
    import threading

    import torch
    lib = api.load()
    repeats = 40
    work = [_StepOnStream(lib, oracle, RESIDENT_CASES[i], 900 + i, b, repeats + 1) for i, b in ((2, 16), (4, 64))]
    try:
        for w in work:
            w.step(repeats)
        lib.blt_backend_pass_sync_hip()
        if threads:
            def issue(w):
                lib.blt_hip_set_stream(2)   # hipStreamPerThread
                for i in range(repeats):
                    w.step(i)
                lib.blt_backend_pass_sync_hip()
            pool = [threading.Thread(target=issue, args=(w,)) for w in work]
            for t in pool:
                t.start()
            for t in pool:
                t.join()
        else:
            streams = [torch.cuda.Stream() for _ in work]
            for i in range(repeats):
                for w, s in zip(work, streams):
                    lib.blt_hip_set_stream(s.cuda_stream)
                    w.step(i)
            lib.blt_hip_set_stream(None)
        lib.blt_backend_pass_sync_hip()
        for w in work:
            got = w.logits.cpu().numpy()
            assert np.isfinite(got).all()
            assert all(got[i].tobytes() == got[repeats].tobytes() for i in range(repeats))
    finally:
        lib.blt_hip_set_stream(None)
        for w in work:
            w.close()


def test_step_in_a_capture_of_the_callers_own(oracle, dev):
    """A step recorded by the caller's capture of its stream, which the library does not see begin, goes in launches:
    every replay gives what the step gives."""
    import torch
    lib = api.load()
    w = _StepOnStream(lib, oracle, RESIDENT_CASES[2], 950, 16, 2)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    try:
        lib.blt_hip_set_stream(stream.cuda_stream)
        w.step(0)
        lib.blt_backend_pass_sync_hip()
        want = w.logits[0].cpu().numpy()
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="relaxed"):
            w.step(1)
        for _ in range(3):
            w.logits[1].fill_(7.0)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert_close(w.logits[1].cpu().numpy(), want, "replayed step")
    finally:
        lib.blt_hip_set_stream(None)
        w.close()


class _KernelNode(C.Structure):
    _fields_ = [("block", C.c_uint32 * 3), ("extra", C.c_void_p), ("func", C.c_void_p), ("grid", C.c_uint32 * 3), ("params", C.c_void_p),
                ("lds", C.c_uint32)]


def _grids_of(graph):
    """Grids of a recorded graph's kernels (hipKernelNodeParams), from the runtime that this process has loaded."""
    with open("/proc/self/maps") as maps:
        hip = C.CDLL(next(line.split()[-1] for line in maps if "libamdhip64" in line))
    raw, count = C.c_void_p(graph.raw_cuda_graph()), C.c_size_t(0)
    assert hip.hipGraphGetNodes(raw, None, C.byref(count)) == 0
    nodes, kind, grids = (C.c_void_p * count.value)(), C.c_int(), []
    assert hip.hipGraphGetNodes(raw, nodes, C.byref(count)) == 0
    for node in nodes:
        assert hip.hipGraphNodeGetType(C.c_void_p(node), C.byref(kind)) == 0
        assert kind.value == 0, kind.value          # a kernel
        at = _KernelNode()
        assert hip.hipGraphKernelNodeGetParams(C.c_void_p(node), C.byref(at)) == 0
        grids.append(tuple(at.grid))
    return grids


@pytest.mark.parametrize("m,k,n", [(1000, 1024, 512), (960, 2100, 512), (118, 2048, 512), (64, 4096, 256)])
@pytest.mark.parametrize("warm", [True, False])
def test_long_products_in_a_capture_of_the_callers_own(m, k, n, warm, dev):
    """Products whose K is split over workgroups hand their sums over in memory of the library, which a replay may use beside other
    work: in a capture that the library does not see begin they are recorded whole, one workgroup a tile and nothing else,
    whether or not the stream had that memory before.  Replays between eager products of other shapes give the same bits."""
    import torch
    lib = api.load()
    torch.manual_seed(m + k)
    a, b = torch.randn(m, k, device="cuda"), torch.randn(k, n, device="cuda") / k ** 0.5
    a2, b2 = torch.randn(700, 2048, device="cuda"), torch.randn(2048, 640, device="cuda") / 45.0
    o, o2 = torch.zeros(m, n, device="cuda"), torch.zeros(700, 640, device="cuda")
    va, vb, vo, va2, vb2, vo2 = (_dev_tensor(t) for t in (a, b, o, a2, b2, o2))
    want, want2 = (a.double() @ b.double()).float().cpu().numpy(), (a2.double() @ b2.double()).float().cpu().numpy()
    torch.cuda.synchronize()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph(keep_graph=True)
    try:
        lib.blt_hip_set_stream(stream.cuda_stream)
        if warm:
            lib.blt_matmul(C.byref(va), C.byref(vb), C.byref(vo))
            lib.blt_backend_pass_sync_hip()
            assert_close(o.cpu().numpy(), want, "eager product")
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="relaxed"):
            lib.blt_matmul(C.byref(va), C.byref(vb), C.byref(vo))
        grids = _grids_of(graph)
        assert len(grids) == 1 and grids[0][2] == 1, grids
        graph.instantiate()
        seen = set()
        for _ in range(3):
            o.fill_(7.0)
            o2.fill_(7.0)
            torch.cuda.synchronize()
            lib.blt_matmul(C.byref(va2), C.byref(vb2), C.byref(vo2))
            graph.replay()
            torch.cuda.synchronize()
            assert_close(o.cpu().numpy(), want, "replayed product")
            assert_close(o2.cpu().numpy(), want2, "eager product beside it")
            seen.add(o.cpu().numpy().tobytes())
        assert len(seen) == 1
    finally:
        lib.blt_hip_set_stream(None)


def test_staged_batch_in_a_capture_of_the_callers_own(dev):
    """A batch whose descriptors are staged, recorded by the caller's own capture, still finds them where they were after a larger
    eager batch of that stream has outgrown the buffer."""
    import torch
    lib = api.load()
    qkv, out = torch.randn(3, 40, 32, device="cuda"), torch.zeros(3, 40, 32, device="cuda")
    row = torch.randn(1200, 32, device="cuda")

    def problems(count):
        return [api.problem(api.head_args(qkv.data_ptr(), qkv.data_ptr(), qkv.data_ptr(), (out[i] if count == 3 else row[i]).data_ptr(),
                                          (20 + i * i) if count == 3 else 1, 40 - i % 3, 32, 0.2, 32, 32, 32, 32, 0),
                            api.BLT_ATTN_MASK_CAUSAL) for i in range(count)]
    few, many = api.problem_array(problems(3)), api.problem_array(problems(1200))
    torch.cuda.synchronize()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    try:
        lib.blt_hip_set_stream(stream.cuda_stream)
        lib.blt_attention_batch_hip(few, 3)
        torch.cuda.synchronize()
        want = out.clone()
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="relaxed"):
            lib.blt_attention_batch_hip(few, 3)
        for _ in range(3):
            lib.blt_attention_batch_hip(many, 1200)
            out.fill_(7.0)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            for i in range(3):      # the rows that the batch has
                assert torch.equal(out[i, : 20 + i * i], want[i, : 20 + i * i])
    finally:
        lib.blt_hip_set_stream(None)


def test_long_uploads_in_a_capture_of_the_callers_own_are_refused():
    """Host data past what launch arguments hold goes through pinned buffers that later uploads use again, so a replay would copy
    other data: fatal in a capture of the caller's own too.  What launch arguments hold is part of the recording."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    code = ("import sys\nsys.path.insert(0, %r)\nimport numpy as np, torch\nfrom fblt_amd import api\nlib = api.load()\n"
            "stream, graph, second = torch.cuda.Stream(), torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()\n"
            "words, to = np.arange(1000, dtype=np.uint32), torch.zeros(20000, dtype=torch.int32, device='cuda')\n"
            "many = np.arange(20000, dtype=np.uint32)\ntorch.cuda.synchronize()\nlib.blt_hip_set_stream(stream.cuda_stream)\n"
            "with torch.cuda.graph(graph, stream=stream, capture_error_mode='relaxed'):\n"
            "    lib.blt_hip_memcpy_h2d(to.data_ptr(), words.ctypes.data, words.nbytes)\n"
            "words[:] = 0\ngraph.replay()\ntorch.cuda.synchronize()\n"
            "assert to[:1000].tolist() == list(range(1000))\nprint('SHORT', flush=True)\n"
            "with torch.cuda.graph(second, stream=stream, capture_error_mode='relaxed'):\n"
            "    lib.blt_hip_memcpy_h2d(to.data_ptr(), many.ctypes.data, many.nbytes)\nprint('SURVIVED')\n" % root)
    p = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert "SHORT" in p.stdout and "SURVIVED" not in p.stdout, p.stdout + p.stderr
    assert p.returncode == 1 and "while the stream is captured" in p.stderr, (p.returncode, p.stderr)


def test_profile_holds_every_launch(dev):
    """Uploads that travel in kernel arguments and the small kernels beside the main path are in the kernel-time profile."""
    import torch
    lib = api.load()
    qkv, out = torch.randn(3, 40, 32, device="cuda"), torch.zeros(3, 40, 32, device="cuda")
    probs = [api.problem(api.head_args(qkv.data_ptr(), qkv.data_ptr(), qkv.data_ptr(), out[i].data_ptr(), 20 + i * i, 40, 32, 0.2, 32, 32,
                                       32, 32, 0), api.BLT_ATTN_MASK_CAUSAL) for i in range(3)]   # three sizes: no strided batch
    vd, vs = _dev_tensor(out[0]), _dev_tensor(qkv[0])
    torch.cuda.synchronize()
    lib.blt_hip_profile_begin()
    lib.blt_attention_batch_hip(api.problem_array(probs), 3)
    lib.blt_rows_gather(C.byref(vs), (C.c_size_t * 40)(*range(40)), C.byref(vd))
    launched = api.profile_end()
    assert launched["upload_words"][0] >= 1 and launched["rows_gather"][0] == 1, launched


def test_graph_replay_of_a_plan_and_a_decode_layer(oracle, dev):
    """Library launches recorded into a HIP graph: every replay, with eager work and
    synchronisations in between, gives the eager result."""
    import torch
    lib = api.load()
    # 1. a resident attention plan
    w = workloads.config2(batch=2, P=48, H=2, hd=64, T_bytes=192)
    d = dev.DeviceWorkload(w)
    try:
        plan = d.make_plan("descriptor")
        d.zero_outputs()
        lib.blt_attention_plan_run_hip(plan)
        lib.blt_backend_pass_sync_hip()
        eager = d.output("out").copy()
        lib.blt_hip_capture_begin()
        lib.blt_attention_plan_run_hip(plan)
        graph = lib.blt_hip_capture_end()
        for _ in range(3):
            d.zero_outputs()                      # eager work between the replays
            lib.blt_hip_graph_launch(graph)
            lib.blt_backend_pass_sync_hip()
            assert d.output("out").tobytes() == eager.tobytes()
        lib.blt_hip_graph_destroy(graph)
        lib.blt_attention_plan_destroy_hip(plan)
    finally:
        d.close()
    # 2. a KV step (rotation fused) recorded without commit, so that a replay repeats the same step
    kw = workloads.config4(batch=16, steps=1, len_hi=200, rope=True)
    kw.commit = False
    dk = dev.DeviceKvWorkload(kw)
    dk.step(0)                                    # eager warm-up: scratch gets allocated here
    lib.blt_backend_pass_sync_hip()
    out0, ck0, cv0, _ = dk.results()
    lib.blt_hip_capture_begin()
    dk.step(0)
    graph = lib.blt_hip_capture_end()
    for _ in range(3):
        dk.out.zero_()
        torch.cuda.synchronize()
        lib.blt_hip_graph_launch(graph)
        lib.blt_backend_pass_sync_hip()
        out, ck, cv, _ = dk.results()
        assert out.tobytes() == out0.tobytes() and ck.tobytes() == ck0.tobytes() and cv.tobytes() == cv0.tobytes()
    lib.blt_hip_graph_destroy(graph)


def test_sliced_product_replays_in_a_graph(dev):
    """A product whose K is split over workgroups, recorded into a graph after an eager run has sized its sums and
    tickets: three replays, each with an eager sliced product of another shape in between (same tickets), give the
    eager bits."""
    import torch
    lib = api.load()
    torch.manual_seed(9)
    a, b = torch.randn(118, 2048, device="cuda"), torch.randn(2048, 512, device="cuda") / 45.0
    a2, b2 = torch.randn(64, 4096, device="cuda"), torch.randn(4096, 256, device="cuda") / 64.0
    o, o2 = torch.zeros(118, 512, device="cuda"), torch.zeros(64, 256, device="cuda")
    va, vb, vo, va2, vb2, vo2 = (_dev_tensor(t) for t in (a, b, o, a2, b2, o2))
    lib.blt_matmul(C.byref(va), C.byref(vb), C.byref(vo))          # eager: scratch gets allocated here
    lib.blt_matmul(C.byref(va2), C.byref(vb2), C.byref(vo2))
    lib.blt_backend_pass_sync_hip()
    want, want2 = o.cpu().numpy().copy(), o2.cpu().numpy().copy()
    assert_close(want, (a.double() @ b.double()).float().cpu().numpy(), "sliced product")
    lib.blt_hip_capture_begin()
    lib.blt_matmul(C.byref(va), C.byref(vb), C.byref(vo))
    graph = lib.blt_hip_capture_end()
    for _ in range(3):
        o.zero_()
        o2.zero_()
        torch.cuda.synchronize()
        lib.blt_hip_graph_launch(graph)
        lib.blt_matmul(C.byref(va2), C.byref(vb2), C.byref(vo2))
        lib.blt_backend_pass_sync_hip()
        assert o.cpu().numpy().tobytes() == want.tobytes() and o2.cpu().numpy().tobytes() == want2.tobytes()
    lib.blt_hip_graph_destroy(graph)


def test_library_follows_the_chosen_stream(oracle, dev):
    """blt_hip_set_stream: launches go to the caller's stream; results are the null-stream results."""
    import torch
    lib = api.load()
    w = workloads.config1(batch=1, T=96, H=2, hd=32)
    ref = _oracle_out(w, oracle)
    d = dev.DeviceWorkload(w)
    side = torch.cuda.Stream()
    try:
        d.zero_outputs()
        lib.blt_hip_set_stream(side.cuda_stream)
        assert lib.blt_hip_get_stream() == side.cuda_stream
        d.run_batch("descriptor")                 # ends with a device-wide sync
        got = d.output("out")
    finally:
        lib.blt_hip_set_stream(None)
        d.close()
    assert_close(got, ref["out"], "side stream")


@pytest.mark.gpu
def test_decoder_step_with_exact_projections():
    """The decoder step takes its projections on the matrix cores by default; BLT_HIP_EXACT_STEP=1
    keeps the thread-per-column kernel (sums in the reference's order) for steps of up to 32 rows.
    The switch is read once per process, so the step, layer and diffusion tests run again in a
    process of their own with it set."""
    import os
    import subprocess
    import sys
    here = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, BLT_HIP_EXACT_STEP="1")
    p = subprocess.run([sys.executable, "-u", "-m", "pytest", os.path.join(here, "test_gpu_parity.py"), "-x", "-q", "-m",
                        "gpu", "-k", "kv_decode_step_single_sequence or kv_decode_layer or diffusion_infer_forward "
                        "or kv_decode_step_batched", "-p", "no:cacheprovider"],
                       capture_output=True, text=True, timeout=900, env=env, cwd=os.path.dirname(here))
    assert p.returncode == 0, p.stdout[-3000:] + p.stderr[-2000:]


@pytest.mark.parametrize("T,E,H,ngrams,vocab,lengths,pool,on_device", [
    (61, 64, 2, (3, 4, 5, 6, 7, 8), 1000, [1, 7, 8, 9, 16, 17, 3], "mean", True),   # one to three rounds of rows
    (61, 64, 2, (3, 4, 5, 6, 7, 8), 1000, [1, 7, 8, 9, 16, 17, 3], "max", False),
    (513, 18, 3, (2,), 50, [1, 2] * 171, "mean", False),                             # single columns; two launches of patches
    (40, 640, 10, (3, 8), 31, [30, 10], "max", True), (19, 1032, 2, (), 7, [9, 10], "mean", False),   # columns in two, three groups
    (2560, 4, 1, (1, 8), 5000011, [10] * 256, "mean", False),                        # hashes past 32 bits; as many bytes as travel along
    (2561, 8, 1, (3,), 97, [10] * 256 + [1], "mean", False), (300, 16, 1, (3,), 97, [257, 43], "max", True)])   # a byte more; too long
def test_encoder_embeds_and_pools_in_one_launch(T, E, H, ngrams, vocab, lengths, pool, on_device, oracle, dev):
    """Bytes, hashed n-grams and pooled patches at the edges of the launch, against the restated forward."""
    from tests import encoder_runs
    from tests.golden import block_cases
    lib = api.load()
    c = dict(T=T, E=E, H=H, XH=H, L=1, hidden=16, ngrams=ngrams, vocab=vocab, k=1, window=0, placement=0, all_layers=True,
             pool=pool, docs=None, normalize=True, mean_patch=4)
    assert sum(lengths) == T
    data, _, weights = block_cases.encoder_case(np.random.RandomState(T), c)
    want_p, want_h = encoder_runs.run_oracle(oracle, c, data, lengths, weights)
    lib.blt_hip_profile_begin()
    got_p, got_h = encoder_runs.run_device(lib.blt_local_encoder_forward, lib, oracle, c, data, lengths, weights, bytes_on_device=on_device)
    names = set(api.profile_end())
    assert "embed_pool" in names and ("patch_pool" in names) == (max(lengths) > 256), names
    assert_close(got_h, want_h, "byte_hidden_out")
    assert_close(got_p, want_p, "patch_out")


ENCODER_CAPTURE = """
import sys
import numpy as np, torch
from fblt_amd import abi, api
from oracle import binding
from tests import encoder_runs
from tests.golden import block_cases

def run(T, lengths, on_device):
    lib, orc = api.load(), binding.load_oracle()
    c = dict(T=T, E=64, H=2, XH=2, L=2, hidden=64, ngrams=(3, 4), vocab=1000, k=1, window=0, placement=0, all_layers=True, pool="mean",
             docs=None, normalize=True, mean_patch=4)
    data, _, weights = block_cases.encoder_case(np.random.RandomState(T), c)
    want = encoder_runs.run_oracle(orc, c, data, lengths, weights)
    stream, graph, outs = torch.cuda.Stream(), torch.cuda.CUDAGraph(), []

    def entry(*args):
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="relaxed"):
            lib.blt_local_encoder_forward(*args)
        data[:] = 0
        for _ in range(3):
            graph.replay()
            torch.cuda.synchronize()

    lib.blt_hip_set_stream(stream.cuda_stream)
    got = encoder_runs.run_device(entry, lib, orc, c, data, lengths, weights, bytes_on_device=on_device)
    lib.blt_hip_set_stream(None)
    for a, b in zip(got, want):
        assert (np.abs(a - b) <= 1e-5 + 1e-4 * np.abs(b)).all()
"""


@pytest.mark.parametrize("T", [61, 2560])
def test_encoder_in_a_capture_of_the_callers_own(T):
    """Bytes on the host, patches and documents are those of the recording in every replay.  Bytes on the device, which a replay would
    read anew under the patches of the recording, and more text than launch arguments hold are fatal."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    lengths = [1, 7, 8, 9, 16, 17, 3] if T == 61 else [10] * 256
    code = "import sys\nsys.path.insert(0, %r)\n" % root + ENCODER_CAPTURE + (
        "run(%d, %r, False)\nprint('REPLAYED', flush=True)\n" % (T, lengths) +
        ("run(61, %r, True)\n" % lengths if T == 61 else "run(2561, [10] * 256 + [1], False)\n") + "print('SURVIVED')\n")
    p = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert "REPLAYED" in p.stdout and "SURVIVED" not in p.stdout, p.stdout + p.stderr
    assert p.returncode == 1 and ("record it with the bytes" if T == 61 else "while the stream is captured") in p.stderr, p.stderr


def test_encoder_ops(oracle, dev):
    """blt_indexed_row_accumulate / blt_scale / blt_patch_pool_forward on device tensors against the
    restated ops: bit for bit (the kernels keep the reference's order of additions).  Index lists
    longer than one launch carries, sentinel entries, both pools, patches of 1 ... 300 rows."""
    import torch
    from fblt_amd import decoder
    lib = api.load()
    rs = np.random.RandomState(5)
    T, E, V = 1300, 48, 97
    table = rs.randn(V, E).astype(np.float32)
    idx = rs.randint(0, V, size=T).astype(np.uint32)
    idx[rs.randint(0, T, size=150)] = abi.BLT_IDX_SENTINEL
    io = rs.randn(T, E).astype(np.float32)
    want = io.copy()
    u32 = C.POINTER(C.c_uint32)
    assert oracle.orc_indexed_row_accumulate(binding.fptr(table.reshape(-1)), V, idx.ctypes.data_as(u32),
                                             binding.fptr(want.reshape(-1)), T, E) == 0
    oracle.orc_scale(binding.fptr(want.reshape(-1)), want.size, 0.25)
    tt, ti = torch.from_numpy(table).cuda(), torch.from_numpy(io).cuda()
    vt, vi = _dev_tensor(tt), _dev_tensor(ti)
    lib.blt_indexed_row_accumulate(C.byref(vt), idx.ctypes.data_as(u32), C.byref(vi))
    lib.blt_scale(C.byref(vi), 0.25)
    lib.blt_backend_pass_sync_hip()
    assert ti.cpu().numpy().tobytes() == want.tobytes()

    lengths = [1, 300, 2, 7, 1, 13] + [3] * 290   # more patches than one launch carries
    patches = decoder.patch_table(lengths)
    h = rs.randn(sum(lengths), E).astype(np.float32)
    th = torch.from_numpy(h).cuda()
    vh = _dev_tensor(th)
    for pool in (abi.BLT_POOL_MEAN, abi.BLT_POOL_MAX):
        want = np.zeros((len(lengths), E), dtype=np.float32)
        assert oracle.orc_patch_pool_forward(binding.fptr(h.reshape(-1)), h.shape[0], E, patches, len(lengths), pool,
                                             binding.fptr(want.reshape(-1))) == 0
        to = torch.full((len(lengths), E), 9.0, dtype=torch.float32, device="cuda")
        vo = _dev_tensor(to)
        lib.blt_patch_pool_forward(C.byref(vh), patches, len(lengths), pool, C.byref(vo))
        lib.blt_backend_pass_sync_hip()
        assert to.cpu().numpy().tobytes() == want.tobytes(), pool


ENCODER_GPU_SHAPES = {
    "small_k1": dict(T=37, E=32, H=2, XH=2, L=1, hidden=48, ngrams=(3,), vocab=101, k=1, window=0, placement=0,
                     all_layers=True, pool="mean", docs=None, normalize=True, mean_patch=3),
    "k3_docs_first": dict(T=90, E=64, H=2, XH=1, L=3, hidden=96, ngrams=(0, 4, 200), vocab=64, k=3, window=0,
                          placement=4, all_layers=False, pool="mean", docs=[25], normalize=True, mean_patch=2),
    "no_cross_window": dict(T=130, E=32, H=1, XH=2, L=2, hidden=32, ngrams=(), vocab=8, k=1, window=17, placement=1,
                            all_layers=True, pool="max", docs=None, normalize=True, mean_patch=7),
    "six_tables_all": dict(T=300, E=128, H=4, XH=4, L=2, hidden=256, ngrams=(3, 4, 5, 6, 7, 8), vocab=509, k=1, window=0,
                           placement=3, all_layers=False, pool="max", docs=[100, 101], normalize=True, mean_patch=4),
}


@pytest.mark.parametrize("impl", ["library", "reference_callers"])
@pytest.mark.parametrize("name", list(ENCODER_GPU_SHAPES) + ["enc_T512_L2", "enc_T150_k2_window_docs_max"])
def test_local_encoder_forward(name, impl, oracle, dev):
    """blt_local_encoder_forward on device tensors against the restated forward: patch_out and
    byte_hidden_out within the fp32 tolerance.  `library` = this library's entry point (bytes given
    on the device and, for one case, on the host); `reference_callers` = the reference's own
    local_encoder.c / hash_ngram.c / byte_embedding.c, compiled unmodified, with this library's
    ops and fused blocks under them -- for configurations without a sub-token split only: with
    k > 1 the reference writes its expanded group ids through a host pointer into arena memory
    (csrc/models/local_encoder.c:100-103), which a device arena does not allow."""
    from tests import encoder_runs
    from tests.golden import block_cases
    lib = api.load()
    if name in ENCODER_GPU_SHAPES:
        c = ENCODER_GPU_SHAPES[name]
        data, lengths, weights = block_cases.encoder_case(np.random.RandomState(len(name) * 31 + c["T"]), c)
    else:
        c, data, lengths, weights = block_cases.encoder_inputs(name)
    if impl == "library":
        entry = lib.blt_local_encoder_forward
    else:
        if c["k"] > 1:
            pytest.skip("the reference's encoder body cannot split patches on a device arena")
        stack_lib = binding.load_ref_stack_callers()
        if stack_lib is None or not hasattr(stack_lib, "blt_local_encoder_forward"):
            pytest.skip("oracle/_ref/libblt_ref_stack_callers.so was not built (needs the reference sources)")
        entry = stack_lib.blt_local_encoder_forward
    want_p, want_h = encoder_runs.run_oracle(oracle, c, data, lengths, weights)
    got_p, got_h = encoder_runs.run_device(entry, lib, oracle, c, data, lengths, weights,
                                           bytes_on_device=name != "small_k1")
    assert_close(got_h, want_h, name + " byte_hidden_out")
    assert_close(got_p, want_p, name + " patch_out")



@pytest.mark.parametrize("T,E,L,k,mean_patch,all_layers,placement", [
    (300, 128, 3, 1, 4, True, 0), (170, 64, 4, 1, 5, True, 0),      # a cross block behind every layer, all but the last beside the next one
    (133, 64, 2, 2, 8, True, 0), (1040, 128, 2, 1, 3, True, 0),     # sub-tokens; more workgroups than go along
    (260, 128, 3, 1, 4, False, 4), (90, 64, 3, 1, 30, True, 0),     # behind the first layer only; too few patches for the launch
    (230, 256, 2, 1, 5, True, 0), (2300, 64, 2, 1, 64, True, 0)])   # wide; patches of more bytes
def test_cross_blocks_beside_the_next_layer(T, E, L, k, mean_patch, all_layers, placement, oracle, dev):
    """The encoder leaves a layer's cross block to the next layer's launches, the decoder makes two layers' keys and values in one:
    every layer's block against the restated forwards, for shapes that share the launches and shapes that cannot."""
    import torch
    from fblt_amd import decoder
    from tests import encoder_runs
    from tests.golden import block_cases
    lib = api.load()
    c = dict(T=T, E=E, H=E // 32, XH=E // 32, L=L, hidden=2 * E, ngrams=(3,), vocab=64, k=k, window=0, placement=placement,
             all_layers=all_layers, pool="mean", docs=None, normalize=True, mean_patch=mean_patch)
    data, lengths, weights = block_cases.encoder_case(np.random.RandomState(T), c)
    want_p, want_h = encoder_runs.run_oracle(oracle, c, data, lengths, weights)
    got_p, got_h = encoder_runs.run_device(lib.blt_local_encoder_forward, lib, oracle, c, data, lengths, weights)
    assert_close(got_h, want_h, "byte_hidden_out")
    assert_close(got_p, want_p, "patch_out")

    host, device = _decoders(oracle, dict(E=E, H=E // 32, XH=E // 32, L=L, hidden=2 * E, V=64, k=k, window=0, placement=placement,
                                          all_layers=all_layers, max_len=T), T)
    P, patches = len(lengths), decoder.patch_table(lengths)
    want = np.zeros((T, 64), dtype=np.float32)
    assert oracle.orc_local_decoder_forward(host.ptr, binding.fptr(want_h.reshape(-1)), T, binding.fptr(want_p.reshape(-1)), patches,
                                            P, None, 0, 0, binding.fptr(want.reshape(-1))) == 0
    th, tp = torch.from_numpy(want_h).cuda(), torch.from_numpy(want_p).cuda()
    tl = torch.full((T, 64), 7.0, dtype=torch.float32, device="cuda")
    vh, vp, vl = _dev_tensor(th), _dev_tensor(tp), _dev_tensor(tl)
    arena = lib.blt_arena_create(256 << 20, abi.BLT_BACKEND_HIP)
    try:
        lib.blt_local_decoder_forward_ext(device.ptr, C.byref(vh), C.byref(vp), patches, P, None, None, None, 0, None, 0,
                                          C.byref(vl), None, arena)
        lib.blt_backend_pass_sync_hip()
    finally:
        lib.blt_arena_destroy(arena)
    assert_close(tl.cpu().numpy(), want, "logits")


@pytest.mark.parametrize("driver", ["reference_encoder", "library_encoder", "library_stages"])
@pytest.mark.parametrize("name", ["model_T96", "model_T200_docs_window"])
def test_model_forward_on_the_library(name, driver, oracle, dev):
    """The reference's whole-model inference forward -- blt_model_encode + blt_model_decode of
    csrc/models/model.c:68-131 over its local_encoder.c, global_transformer.c / transformer_stack.c
    and local_decoder.c, all compiled unmodified -- on device tensors, with this library's ops and
    fused blocks under them (blt_transformer_forward, blt_cross_attention_forward, the embedding,
    n-gram, pooling, norm, add and product twins, the mask builders and the memory shim): logits
    against the composition of the restated stages, which tests/test_oracle_vs_ref.py pins bit for
    bit against the reference's CPU build.  `library_encoder`: the same driver built without the
    reference's encoder sources, so that blt_model_encode runs this library's own
    blt_local_encoder_forward; `library_stages`: without its decoder sources either
    (blt_local_decoder_forward_ext is the library's too)."""
    from fblt_amd import decoder
    from tests import model_runs
    lib = api.load()
    stack_lib = {"reference_encoder": binding.load_ref_stack_callers, "library_encoder": binding.load_ref_model_callers,
                 "library_stages": binding.load_ref_model_driver}[driver]()
    if stack_lib is None or not hasattr(stack_lib, "blt_model_encode"):
        pytest.skip("oracle/_ref does not hold the model driver build (needs the reference sources)")
    args = model_runs.inputs(name)

    def fill(t, arr):
        assert tuple(t.contents.shape[:t.contents.ndim]) == arr.shape
        lib.blt_tensor_upload(t, arr.ctypes.data, arr.nbytes)

    got = model_runs.run(stack_lib, lib, oracle, abi.BLT_BACKEND_HIP, decoder.device_place, fill,
                         lib.blt_backend_pass_sync_hip, *args)
    want = model_runs.run_oracle(oracle, *args)
    assert np.abs(want).max() > 1e-3
    assert_close(got, want, name + " logits")
