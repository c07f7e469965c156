"""On-GPU prefill: the batched prefill (sinter_model_prefill_batched, each
layer once per ubatch of tokens) and the decode program over the prompt
(sinter_model_prefill_tokenwise, each pass's next token forced to the
prompt's) leave the KV rows, the recurrent and conv states and the logits of
decoding the prompt one token at a time -- checked bit for bit against
single-pass decodes, against each other (ragged ubatches, both KV cache
types, split-K geometries whose chunk length changes inside a block of
queries) and against the CPU oracle."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_model import compare_logits, small_config

pytestmark = pytest.mark.gpu


def device_bytes(m, d, nb):
    a = np.empty(nb, np.uint8)
    m.d2h(a, d, nb)
    return a


def same_state(a, b, cfg):
    for il in range(cfg.n_layer):
        for s in range(2):
            da, na = a.state(il, s)
            db, nb = b.state(il, s)
            assert na == nb
            assert np.array_equal(device_bytes(a, da, na), device_bytes(b, db, nb)), (il, s)


@pytest.mark.parametrize("mode", ["tokenwise", "batched"])
def test_prefill_equals_single_pass_decodes(sn, torch_gpu, mode):
    """1100 tokens: more passes than one decode-program launch runs (1024),
    five ubatches of the batched prefill (the last one ragged)."""
    cfg = small_config(sn, n_layer=8, n_ctx=1280)
    n = 1100
    toks = [int(t) for t in np.random.default_rng(3).integers(0, cfg.n_vocab, n)]
    a, b = sn.Model(cfg, seed=41), sn.Model(cfg, seed=41)
    try:
        print(f"prefill {mode}: {n} tokens", flush=True)
        nxt_a = a.prefill(toks, 0, mode=mode)
        print("prefill: the same tokens one pass per call", flush=True)
        nxt_b = None
        for i, t in enumerate(toks):
            nxt_b = b.decode(t, i)
        assert nxt_a == nxt_b
        assert np.array_equal(a.logits(), b.logits())
        same_state(a, b, cfg)
        assert a.greedy(nxt_a, n, 8) == b.greedy(nxt_b, n, 8)
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("mode", ["tokenwise", "batched"])
def test_prefill_matches_oracle_from_a_context(sn, orc, torch_gpu, mode):
    cfg = small_config(sn, n_layer=4, n_ctx=256)
    m = sn.Model(cfg, seed=43)
    try:
        m.synth_context(40, seed=44)
        mirror = orc.ModelMirror(m)
        prompt = [17, 2999, 0, 1234, 77, 5]
        print(f"prefill {mode}: {len(prompt)} tokens after a 40-token context", flush=True)
        nxt = m.prefill(prompt, 40, mode=mode)
        rtok, rlog = None, None
        for i, t in enumerate(prompt):
            rtok, rlog = mirror.step(t, 40 + i)
        print(f"prefill next: gpu {nxt} oracle {rtok}", flush=True)
        assert nxt == rtok
        compare_logits(m.logits(), rlog)
        # decoding continues from the prefilled state
        gpu = m.greedy(nxt, 46, 3)
        ref, t = [], nxt
        for p in (46, 47, 48):
            t = mirror.step(t, p)[0]
            ref.append(t)
        assert gpu == ref
    finally:
        m.close()


def test_prefill_refuses_bad_arguments(sn, torch_gpu):
    cfg = small_config(sn, n_layer=4, n_ctx=64)
    m = sn.Model(cfg, seed=45)
    try:
        L = sn.lib()
        arr = (C.c_int32 * 8)(*range(8))
        nxt = C.c_int32()
        assert L.sinter_model_prefill(m.h, arr, 8, 60, C.byref(nxt)) == sn.ERR_ARG      # past n_ctx
        assert L.sinter_model_prefill(m.h, arr, 0, 0, C.byref(nxt)) == sn.ERR_ARG
        bad = (C.c_int32 * 2)(1, cfg.n_vocab)
        assert L.sinter_model_prefill(m.h, bad, 2, 0, C.byref(nxt)) == sn.ERR_ARG      # token out of range
        assert 0 <= m.prefill([1, 2, 3], 0) < cfg.n_vocab      # the refusals left the model usable
    finally:
        m.close()


# (ubatch, KV type, attn_chunks, attn_chunk_min, context, prompt): one-token
# ubatches; a ragged 7; chunks of 2 and 3 per kv head, where a query's chunk
# length (tiles per chunk) changes every few positions, so the 16 queries of a
# block split differently; a Q8_0 cache
BATCH_CASES = [
    (1, "f16", 0, 0, 0, 40),
    (7, "f16", 0, 0, 30, 150),
    (64, "f16", 2, 128, 0, 300),
    (33, "q8_0", 3, 32, 17, 260),
    (256, "q8_0", 0, 0, 100, 380),
]


@pytest.mark.parametrize("ub,kv,chunks,cmin,ctx,n", BATCH_CASES)
def test_batched_prefill_equals_tokenwise(sn, torch_gpu, ub, kv, chunks, cmin, ctx, n):
    cfg = small_config(sn, n_layer=4, n_ctx=512)
    cfg.t_kv = {"f16": sn.F16, "q8_0": sn.Q8_0}[kv]
    cfg.attn_chunks, cfg.attn_chunk_min = chunks, cmin
    rng = np.random.default_rng(ub * 1000 + n)
    toks = [int(t) for t in rng.integers(0, cfg.n_vocab, n)]
    a, b = sn.Model(cfg, seed=47), sn.Model(cfg, seed=47)
    try:
        if ctx:
            a.synth_context(ctx, seed=48)
            b.synth_context(ctx, seed=48)
        print(f"batched prefill ubatch={ub} kv={kv} chunks={chunks} cmin={cmin} ctx={ctx} n={n}", flush=True)
        nxt_a = a.prefill(toks, ctx, mode="batched", ubatch=ub)
        print("tokenwise prefill of the same prompt", flush=True)
        nxt_b = b.prefill(toks, ctx, mode="tokenwise")
        assert nxt_a == nxt_b
        assert np.array_equal(a.logits(), b.logits())
        same_state(a, b, cfg)
        # a second prefill continues from the first (its positions follow)
        more = [int(t) for t in rng.integers(0, cfg.n_vocab, 20)]
        print("a second batched prefill after the first", flush=True)
        assert a.prefill(more, ctx + n, mode="batched", ubatch=ub) == b.prefill(more, ctx + n, mode="tokenwise")
        assert np.array_equal(a.logits(), b.logits())
        same_state(a, b, cfg)
    finally:
        a.close()
        b.close()


def test_batched_prefill_refuses_other_weight_types(sn, torch_gpu):
    """A bf16 model has no batched path: sinter_model_prefill_batched refuses
    it, sinter_model_prefill runs the decode passes instead."""
    cfg = small_config(sn, n_layer=4, n_ctx=64, quant="bf16")
    m = sn.Model(cfg, seed=49)
    try:
        L = sn.lib()
        arr = (C.c_int32 * 4)(5, 6, 7, 8)
        nxt = C.c_int32()
        assert L.sinter_model_prefill_batched(m.h, arr, 4, 0, 16, C.byref(nxt)) == sn.ERR_ARG
        assert L.sinter_model_prefill(m.h, arr, 4, 0, C.byref(nxt)) == sn.OK
    finally:
        m.close()
    cfg = small_config(sn, n_layer=4, n_ctx=64)
    m = sn.Model(cfg, seed=49)
    try:
        L = sn.lib()
        arr = (C.c_int32 * 4)(5, 6, 7, 8)
        nxt = C.c_int32()
        assert L.sinter_model_prefill_batched(m.h, arr, 4, 0, 0, C.byref(nxt)) == sn.ERR_ARG      # ubatch 0
        assert L.sinter_model_prefill_batched(m.h, arr, 4, 0, 4096, C.byref(nxt)) == sn.ERR_ARG   # over the max
        assert L.sinter_model_prefill_batched(m.h, arr, 4, 62, 16, C.byref(nxt)) == sn.ERR_ARG   # past n_ctx
    finally:
        m.close()


@pytest.mark.parametrize("d,hk,hv", [(64, 2, 4), (256, 1, 2)])
def test_batched_prefill_gdn_head_sizes(sn, torch_gpu, d, hk, hv):
    """The GDN scan's other layouts (head size 64: 16 columns per item, 4 rows
    per thread; 256: 32 rows per thread) against the decode program."""
    cfg = small_config(sn, n_layer=4, n_ctx=256)
    cfg.gdn_d, cfg.gdn_hk, cfg.gdn_hv = d, hk, hv
    toks = [int(t) for t in np.random.default_rng(d).integers(0, cfg.n_vocab, 70)]
    a, b = sn.Model(cfg, seed=51), sn.Model(cfg, seed=51)
    try:
        print(f"batched prefill gdn_d={d} hk={hk} hv={hv}", flush=True)
        nxt_a = a.prefill(toks, 0, mode="batched", ubatch=32)
        nxt_b = b.prefill(toks, 0, mode="tokenwise")
        assert nxt_a == nxt_b
        assert np.array_equal(a.logits(), b.logits())
        same_state(a, b, cfg)
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("d,hk,hv", [(64, 2, 4), (128, 2, 4), (256, 1, 2)])
def test_batched_prefill_gdn_stage_edges(sn, torch_gpu, d, hk, hv):
    """The GDN scan takes 8 tokens per stage: ubatches of 1, 7, 8, 9, 15, 16
    and 17 tokens (whole and partial last stages) against one pass per token."""
    cfg = small_config(sn, n_layer=2, n_ctx=128)
    cfg.gdn_d, cfg.gdn_hk, cfg.gdn_hv = d, hk, hv
    toks = [int(t) for t in np.random.default_rng(d + 1).integers(0, cfg.n_vocab, 73)]
    a, b = sn.Model(cfg, seed=53), sn.Model(cfg, seed=53)
    try:
        pos = 0
        for n in (1, 7, 8, 9, 15, 16, 17):
            print(f"gdn stages d={d}: {n} tokens at {pos}", flush=True)
            nxt_a = a.prefill(toks[pos:pos + n], pos, mode="batched")
            nxt_b = b.prefill(toks[pos:pos + n], pos, mode="tokenwise")
            pos += n
            assert nxt_a == nxt_b
            assert np.array_equal(a.logits(), b.logits())
            same_state(a, b, cfg)
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("past,n,chunks,cmin", [(78, 33, 3, 32), (8180, 40, 64, 128)])
def test_batched_prefill_across_a_change_of_tiles_per_chunk(sn, torch_gpu, past, n, chunks, cmin):
    """Where the tiles per chunk grow inside a ubatch, its shallower queries
    are split into more chunks than its deepest one (8192 positions: 64
    chunks, 8193: 52): every chunk of every query is computed."""
    cfg = small_config(sn, n_layer=2, n_ctx=past + n + 8)
    cfg.attn_every, cfg.attn_chunks, cfg.attn_chunk_min = 1, chunks, cmin
    toks = [int(t) for t in np.random.default_rng(past).integers(0, cfg.n_vocab, n)]
    a, b = sn.Model(cfg, seed=61), sn.Model(cfg, seed=61)
    try:
        a.synth_context(past, seed=62)
        b.synth_context(past, seed=62)
        print(f"prefill of {n} tokens at {past}, {chunks} chunks", flush=True)
        assert a.prefill(toks, past, mode="batched") == b.prefill(toks, past, mode="tokenwise")
        assert np.array_equal(a.logits(), b.logits())
        same_state(a, b, cfg)
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("kv", ["f16", "q8_0"])
@pytest.mark.parametrize("past,chunks,cmin", [(0, 64, 32), (30, 3, 32), (250, 5, 64), (508, 64, 128)])
def test_batched_prefill_attention_query_blocks(sn, torch_gpu, kv, past, chunks, cmin):
    """The prefill attention takes 16 queries per item: 1, 15, 16, 17 and 33
    of them behind a context, at depths where the split's tiles per chunk and
    chunk count change inside a block, against one pass per token."""
    cfg = small_config(sn, n_layer=2, n_ctx=past + 96)
    cfg.attn_every, cfg.attn_chunks, cfg.attn_chunk_min = 1, chunks, cmin
    cfg.t_kv = sn.Q8_0 if kv == "q8_0" else sn.F16
    toks = [int(t) for t in np.random.default_rng(past + chunks).integers(0, cfg.n_vocab, 82)]
    a, b = sn.Model(cfg, seed=57), sn.Model(cfg, seed=57)
    try:
        a.synth_context(past, seed=58)
        b.synth_context(past, seed=58)
        pos, i = past, 0
        for n in (1, 15, 16, 17, 33):
            print(f"attention blocks kv={kv} past={past} chunks={chunks}: {n} tokens at {pos}", flush=True)
            nxt_a = a.prefill(toks[i:i + n], pos, mode="batched")
            nxt_b = b.prefill(toks[i:i + n], pos, mode="tokenwise")
            pos, i = pos + n, i + n
            assert nxt_a == nxt_b
            assert np.array_equal(a.logits(), b.logits())
            same_state(a, b, cfg)
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("kv", ["f16", "q8_0"])
@pytest.mark.parametrize("at", [0, 5, 15, 16, 30, 39])
def test_batched_prefill_keeps_an_overflowing_value_to_its_rows(sn, torch_gpu, kv, at):
    """A token whose values overflow the cache (an infinite f16, or Q8_0 block
    scale) reaches only the queries that attend to it: the tokens before it in
    the same blocks of queries are as one pass per token leaves them, and so
    are those after it."""
    cfg = small_config(sn, n_layer=2, n_ctx=64)
    cfg.attn_every, cfg.t_kv = 1, sn.Q8_0 if kv == "q8_0" else sn.F16
    rng = np.random.default_rng(7)
    toks = [int(t) for t in rng.choice(cfg.n_vocab, 40, replace=False)]
    SLOT_V = 7
    a, b, probe = (sn.Model(cfg, seed=71) for _ in range(3))
    try:
        # each token's largest value in the first layer, where it depends on the token alone
        probe.prefill(toks, 0, mode="tokenwise")
        d, nb = probe.state(0, 1)
        row = nb // cfg.n_ctx
        rows = device_bytes(probe, d, nb).reshape(cfg.n_ctx, row)[:40]
        if kv == "f16":
            v = np.abs(rows.view(np.float16).astype(np.float32))
        else:
            v = rows.reshape(40, -1, 34)[:, :, :2].copy().view(np.float16).astype(np.float32)
        big = v.reshape(40, -1).max(1)
        order = np.argsort(big)
        top, lim = order[-1], np.sqrt(big[order[-1]] * big[order[-2]])
        toks[at], toks[top] = toks[top], toks[at]
        # the value matrix scaled so that this token alone passes the f16 range
        d, nb, t = a.tensor(0, SLOT_V)
        w = device_bytes(a, d, nb).reshape(-1, sn.BLOCK_BYTES[t])
        at_d = {sn.Q4_K: slice(0, 4), sn.Q6_K: slice(208, 210)}[t]
        w[:, at_d] = (w[:, at_d].copy().view(np.float16).astype(np.float32) * (65520.0 / lim)).astype(np.float16).view(np.uint8)
        for m in (a, b):
            m.h2d(m.tensor(0, SLOT_V)[0], w.reshape(-1), nb)
        print(f"overflowing value kv={kv} at {at} (largest {big[order[-1]]}, next {big[order[-2]]})", flush=True)
        a.prefill(toks, 0, mode="batched")
        b.prefill(toks, 0, mode="tokenwise")
        for il in range(2):
            for s in range(2):
                da, n = a.state(il, s)
                ga, gb = (device_bytes(m, m.state(il, s)[0], n).reshape(cfg.n_ctx, -1) for m in (a, b))
                if kv == "f16":
                    ga, gb = ga.view(np.float16), gb.view(np.float16)
                    if (il, s) == (0, 1):
                        assert np.isinf(ga).any(1).nonzero()[0].tolist() == [at]
                    assert np.array_equal(ga, gb, equal_nan=True), (il, s)
                else:
                    assert np.array_equal(ga, gb), (il, s)
        assert np.array_equal(a.logits(), b.logits(), equal_nan=True)
    finally:
        for m in (a, b, probe):
            m.close()


def test_prefill_attention_keeps_subnormals(sn, orc, torch_gpu):
    """The prefill attention's matrix instructions flush no subnormal: V sums of
    weights around exp(-90) and values down to the smallest f16, in tiles whose
    largest scores have V = 0, bit for bit the oracle's fmaf chains (the
    launcher is internal to the library and found by its C++ name)."""
    torch = torch_gpu
    NQ, NKV, HD, T, pos0 = 8, 2, 256, 17, 190
    rows = pos0 + T
    rng = np.random.default_rng(5)
    K = np.zeros((rows, NKV, HD), np.float16)
    V = (rng.standard_normal((rows, NKV, HD)) * 10.0 ** rng.uniform(-7, 0, (rows, NKV, HD))).astype(np.float16)
    high = np.arange(rows) // 8 % 4 == 0               # in every tile and row group
    K[:, :, 0] = np.where(high[:, None], 0.0, rng.uniform(-103, -78, (rows, NKV)))
    V[high] = 0
    qr = np.zeros((T, NQ, HD), np.float32)
    qr[:, :, 0] = rng.uniform(15.9, 16.1, (T, NQ))
    qg = np.zeros((T, NQ, 2 * HD), np.float32)         # gate: sigmoid(0) = 1/2
    dev = [torch.from_numpy(a).cuda() for a in (qr, qg, K.view(np.int16), V.view(np.int16))]
    part = torch.zeros(T * NQ * 64 * (HD + 4), device="cuda")
    out = torch.zeros(T, NQ, HD, device="cuda")
    launch = sn.lib()["_ZN6sinter19launch_attn_prefillEPKfS1_PKvS3_jijjjjjjfPfS4_P12ihipStream_t"]
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    print("prefill attention of subnormal sums", flush=True)
    u32 = C.c_uint32
    assert launch(*(C.c_void_p(t.data_ptr()) for t in dev), u32(sn.F16), C.c_int32(pos0), u32(T), u32(NQ), u32(NKV), u32(HD),
                  u32(64), u32(128), C.c_float(0.0625), C.c_void_p(part.data_ptr()), C.c_void_p(out.data_ptr()),
                  C.c_void_p(s.cuda_stream)) == 0
    torch.cuda.synchronize()
    got, want = out.cpu().numpy(), np.zeros((T, NQ, HD), np.float32)
    for t in range(T):
        orc.lib().or_attn_split(qr[t].ctypes.data, K.ctypes.data, V.ctypes.data, orc.F16, pos0 + t + 1, NQ, NKV, HD, 0.0625,
                                64, 128, want[t].ctypes.data)
    want *= np.float32(0.5)
    tiny = np.finfo(np.float32).tiny
    assert ((want != 0) & (np.abs(want) < tiny)).mean() > 0.02 and (np.abs(want) >= tiny).mean() > 0.02
    assert np.array_equal(got, want)
