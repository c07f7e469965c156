"""Performance cases: the work a user of the library has it do, through its
public entry points, over the sizes it is used at.

Kinds of case:
  decode       one pass of sinter_model_decode: token and position in, logits
               and the greedy token back (one token of a chat reply)
  prefill      sinter_model_prefill of a prompt, or of a later turn's tokens
               behind a context of `past` positions
  ffn          the feed-forward sub-layer of a ubatch through the batched
               entry points: norm + Q8_K, gate and up, SwiGLU + Q8_K, down
               added to the residual
  gdn_in       the input side of a gated-DeltaNet layer over a ubatch: norm +
               Q8_K, the four projections, conv + silu
  gemv_ubatch  one matrix over a ubatch of Q8_K activations
  op_gemv      one GEMV instruction (activation quantiser included)
  op_attn      one decode-attention instruction over a KV cache

Layer shapes are the 27B hybrid's (sinter.qwen36_27b_config); models with
fewer layers and a short vocabulary stand for single layers.  Weights,
contexts and inputs are synthetic, made on the device from the seed.
"""
import ctypes as C
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "sinter-qwen36-nomtp-tu102_amd"))
import sinter  # noqa: E402

F16, Q8_0, Q4_K, Q6_K, BF16 = sinter.F16, sinter.Q8_0, sinter.Q4_K, sinter.Q6_K, sinter.BF16
TYPES = {"q4_k": Q4_K, "q6_k": Q6_K, "q8_0": Q8_0, "bf16": BF16}
# the 27B hybrid's layer shapes
E, F, HK, HV, D, DCONV = 5120, 17408, 16, 32, 128, 4
CH, VD = (2 * HK + HV) * D, HV * D                  # conv channels, value width
NQ, NKV, HD, ROPE = 24, 4, 256, 64
RW = NKV * HD                                        # a position's K (or V) row
VOCAB, EPS, THETA = 151936, 1e-6, 1e7
Q8K_BYTES = 292


def listed():
    return [
        # one token of a reply: the whole 27B model, 4096 positions behind it
        {"name": "decode_27b_4k", "kind": "decode", "layers": 64, "vocab": VOCAB, "quant": "q4_k_m", "kv": "f16",
         "ctx": 4096},
        # the same at the end of a very long document, one period of the
        # hybrid (3 gated-DeltaNet layers, 1 attention layer), Q8_0 KV cache
        {"name": "decode_period_128k", "kind": "decode", "layers": 4, "vocab": 4096, "quant": "q4_k_m",
         "kv": "q8_0", "ctx": 131000},
        # a long prompt through the whole model
        {"name": "prefill_27b_2k", "kind": "prefill", "layers": 64, "every": 4, "vocab": VOCAB, "kv": "f16",
         "past": 0, "tokens": 2048},
        # a one-line question: latency of a short prompt
        {"name": "prefill_27b_24", "kind": "prefill", "layers": 64, "every": 4, "vocab": VOCAB, "kv": "f16",
         "past": 0, "tokens": 24},
        # a later turn of a long chat in an attention layer: 500 tokens behind 8192
        {"name": "prefill_attn_8k", "kind": "prefill", "layers": 1, "every": 1, "vocab": 512, "kv": "f16",
         "past": 8192, "tokens": 500},
        # a prompt in a gated-DeltaNet layer
        {"name": "prefill_gdn_1k", "kind": "prefill", "layers": 1, "every": 0, "vocab": 512, "kv": "f16",
         "past": 0, "tokens": 1000},
        # the feed-forward sub-layer: a full ubatch, and the last few tokens of a prompt
        {"name": "ffn_256", "kind": "ffn", "tokens": 256},
        {"name": "ffn_13", "kind": "ffn", "tokens": 13},
        # a gated-DeltaNet layer's projections and conv, a ragged ubatch
        {"name": "gdn_in_77", "kind": "gdn_in", "tokens": 77},
        # the head on a prompt's last token
        {"name": "head_1", "kind": "gemv_ubatch", "type": "q6_k", "rows": VOCAB, "k": E, "tokens": 1},
        # one GEMV and one decode attention as single ops, as a host that
        # schedules its own layers calls them
        {"name": "op_gemv_q8_0", "kind": "op_gemv", "type": "q8_0", "rows": F, "k": E, "norm": False},
        {"name": "op_attn_4k", "kind": "op_attn", "kv": "f16", "pos": 4095},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "prefill", "prefill", "prefill", "ffn", "gdn_in", "gemv_ubatch", "op_gemv", "op_attn"])
    kv = rng.choice(["f16", "f16", "q8_0"])
    if kind == "decode":
        return {"kind": kind, "layers": rng.choice([4, 8, 16]), "vocab": rng.randrange(2000, 40000),
                "quant": rng.choice(["q4_k_m", "q4_k_m", "bf16"]), "kv": kv, "ctx": _log(rng, 16, 131000)}
    if kind == "prefill":
        every = rng.choice([0, 1, 4])
        layers = rng.choice([4, 8]) if every == 4 else rng.choice([1, 2, 3])
        past = rng.choice([0, _log(rng, 64, 32768)])
        tokens = min(_log(rng, 1, 4096), 40000 // layers // (1 + past // 8192))
        return {"kind": kind, "layers": layers, "every": every, "vocab": rng.randrange(500, 5000), "kv": kv,
                "past": past, "tokens": tokens}
    if kind in ("ffn", "gdn_in"):
        return {"kind": kind, "tokens": _log(rng, 1, 1024)}
    if kind == "gemv_ubatch":
        return {"kind": kind, "type": rng.choice(["q4_k", "q6_k"]), "rows": _log(rng, 32, 40000),
                "k": 256 * _log(rng, 2, 68), "tokens": _log(rng, 1, 1024)}
    if kind == "op_gemv":
        return {"kind": kind, "type": rng.choice(["q4_k", "q6_k", "q8_0", "bf16"]), "rows": _log(rng, 256, 40000),
                "k": rng.choice([1024, 2048, 4096, 5120, 6144]), "norm": rng.random() < 0.5}
    return {"kind": kind, "kv": kv, "pos": _log(rng, 16, 131071)}


# ------------------------------------------------------------------ inputs

_stream = None


def _s():
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return C.c_void_p(_stream.cuda_stream)


class _Raw:
    """Device memory of the library as an array torch can view."""

    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False), "version": 2}


def _view(ptr, shape, typestr, owner):
    """A view of the model's memory, which lives as long as the view."""
    t = torch.as_tensor(_Raw(ptr, tuple(shape), typestr), device="cuda")
    t.owner = owner
    return t


def _weights(t, rows, k, seed):
    w = torch.empty(sinter.row_bytes(t, k) * rows, dtype=torch.uint8, device="cuda")
    sinter.check(sinter.lib().sinter_synth(1, C.c_void_p(w.data_ptr()), sinter.SYN_WEIGHT, t, rows, k, seed, 0, 0, _s()),
                 "synth")
    return w


def _normal(gen, *shape, mean=0.0, std=1.0):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32) * std + mean


def _config(case):
    n = case["ctx"] + 8 if case["kind"] == "decode" else case["past"] + case["tokens"] + 8
    cfg = sinter.qwen36_27b_config(n_ctx=n, quant=case.get("quant", "q4_k_m"), n_layer=case["layers"], kv=case["kv"])
    cfg.n_vocab = case["vocab"]
    cfg.attn_every = case.get("every", 4)
    return cfg


def _is_attn(case, il):
    every = case.get("every", 4)
    return every > 0 and il % every == every - 1


def _views(case, m):
    """Per layer: the K and V rows this case appends (attention), or the conv and recurrent state."""
    first, n = (case["ctx"], 1) if case["kind"] == "decode" else (case["past"], case["tokens"])
    out = []
    for il in range(case["layers"]):
        (a, _), (b, _) = m.state(il, 0), m.state(il, 1)
        if not _is_attn(case, il):
            out += [_view(a, (CH, DCONV - 1), "<f4", m), _view(b, (HV, D, D), "<f4", m)]
        elif case["kv"] == "q8_0":
            row = RW // 32 * 34
            out += [_view(p + first * row, (n, row), "|u1", m) for p in (a, b)]
        else:
            out += [_view(p + first * RW * 2, (n, RW), "<f2", m) for p in (a, b)]
    return out


def prepare(case, seed):
    kind = case["kind"]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    L = sinter.lib()
    if kind in ("decode", "prefill"):
        m = sinter.Model(_config(case), seed=seed)
        m.synth_context(case["ctx"] if kind == "decode" else case["past"], seed=seed + 1)
        st = {"case": case, "m": m}
        if kind == "decode":
            st["token"] = seed * 7919 % case["vocab"]
        else:
            toks = torch.randint(0, case["vocab"], (case["tokens"],), generator=gen, device="cuda")
            st["tokens"] = [int(t) for t in toks.cpu()]
        # (a full model's 128 state buffers stay with it)
        st["views"] = _views(case, m) if case["layers"] <= 16 else []
        return st
    st = {"case": case}
    if kind in ("ffn", "gdn_in"):
        T = case["tokens"]
        st["x"] = _normal(gen, T, E)
        st["norm"] = _normal(gen, E, mean=1.0, std=0.02)
        st["xq"] = torch.empty(T * (F // 256) * Q8K_BYTES, dtype=torch.uint8, device="cuda")
        names = [("gate", Q4_K, F, E), ("up", Q4_K, F, E), ("down", Q6_K, E, F)] if kind == "ffn" else \
            [("qkv", Q4_K, CH, E), ("z", Q4_K, VD, E), ("alpha", Q4_K, HV, E), ("beta", Q4_K, HV, E)]
        for i, (name, t, rows, k) in enumerate(names):
            st[name] = (t, rows, k, _weights(t, rows, k, seed * 31 + i))
            st["y_" + name] = torch.empty(T, rows, device="cuda")
        if kind == "ffn":
            st["y_down"] = _normal(gen, T, E)      # the residual the sub-layer is added to
        else:
            st["conv_w"] = _normal(gen, CH, DCONV, std=0.3)
            st["conv_state"] = _normal(gen, CH, DCONV - 1)
            st["conv"] = torch.empty(T, CH, device="cuda")
    elif kind == "gemv_ubatch":
        t, T, k = TYPES[case["type"]], case["tokens"], case["k"]
        st["w"] = (t, case["rows"], k, _weights(t, case["rows"], k, seed))
        x = _normal(gen, T, k)
        st["x"] = x
        st["xq"] = torch.empty(T * (k // 256) * Q8K_BYTES, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        sinter.check(L.sinter_quant_q8k_ubatch(C.c_void_p(x.data_ptr()), k, T, C.c_void_p(st["xq"].data_ptr()), _s()),
                     "quant")
        st["y_w"] = torch.empty(T, case["rows"], device="cuda")
    elif kind == "op_gemv":
        t, rows, k = TYPES[case["type"]], case["rows"], case["k"]
        st["w"] = (t, rows, k, _weights(t, rows, k, seed))
        st["x"], st["norm"], st["y"] = _normal(gen, k), _normal(gen, k, mean=1.0, std=0.02), torch.empty(rows, device="cuda")
        a = sinter.GemvArgs(K=k, pro=sinter.PRO_RMSNORM if case["norm"] else sinter.PRO_PLAIN, n_seg=1, eps=EPS)
        a.x, a.norm_w = st["x"].data_ptr(), st["norm"].data_ptr()
        a.seg[0] = sinter.GemvSeg(w=st["w"][3].data_ptr(), y=st["y"].data_ptr(), rows=rows, type=t, epi=sinter.EPI_STORE)
        st["args"] = a
    else:
        pos, chunks = case["pos"], 64
        n = pos + 1
        q8 = case["kv"] == "q8_0"
        for i, name in enumerate(("kc", "vc")):
            # zeroed past the context, then N(0, 1) rows (Q8_0 blocks of them)
            c = torch.zeros(n * (RW // 32 * 34 if q8 else RW * 2), dtype=torch.uint8, device="cuda")
            torch.cuda.synchronize()
            sinter.check(L.sinter_synth(1, C.c_void_p(c.data_ptr()), sinter.SYN_NORMAL_Q8_0 if q8 else
                                        sinter.SYN_NORMAL_F16, 0, n, RW, seed * 31 + i, 0.0, 1.0, _s()), "synth")
            st[name] = c
        st["qg"], st["k"], st["v"] = _normal(gen, NQ, 2, HD), _normal(gen, RW), _normal(gen, RW)
        st["qn"], st["kn"] = _normal(gen, HD, mean=1.0, std=0.02), _normal(gen, HD, mean=1.0, std=0.02)
        st["part"] = torch.zeros(L.sinter_attn_part_len(NQ, NKV, HD, chunks), device="cuda")
        st["count"] = torch.zeros(L.sinter_attn_count_len(NKV, chunks), dtype=torch.int32, device="cuda")
        st["out"] = torch.empty(NQ * HD, device="cuda")
        st["cell"] = torch.tensor([0, pos, 0, 0], dtype=torch.int32, device="cuda")
        a = sinter.AttnArgs(nq=NQ, nkv=NKV, hd=HD, rope_dims=ROPE, n_ctx=n, n_chunks=chunks,
                            theta_scale=THETA ** (-2.0 / ROPE), eps=EPS, scale=HD ** -0.5,
                            kv_type=Q8_0 if q8 else F16, chunk_min=sinter.ATTN_CHUNK_MIN)
        a.qg, a.k, a.v, a.q_norm, a.k_norm = (st[x].data_ptr() for x in ("qg", "k", "v", "qn", "kn"))
        a.kc, a.vc, a.part, a.count, a.out, a.pass_cell = (st[x].data_ptr() for x in
                                                           ("kc", "vc", "part", "count", "out", "cell"))
        st["args"] = a
        row = RW // 32 * 34 if q8 else RW * 2
        rows = [st[x][pos * row:] for x in ("kc", "vc")]
        st["rows"] = rows if q8 else [r.view(torch.float16) for r in rows]
    torch.cuda.synchronize()   # (inputs are made on torch's stream, used on the library call's)
    return st


# ------------------------------------------------------------------ one pass

def _p(t):
    return C.c_void_p(t.data_ptr())


def _ubatch(st, name, T, y, accumulate=0):
    t, rows, k, w = st[name]
    sinter.check(sinter.lib().sinter_op_gemv_ubatch(t, _p(w), rows, k, _p(st["xq"]), T, _p(y), accumulate, _s()),
                 "gemv_ubatch")


def run(st):
    case, L = st["case"], sinter.lib()
    kind = case["kind"]
    if kind == "decode":
        logits = torch.empty(case["vocab"], dtype=torch.float32).numpy()
        token = st["m"].decode(st["token"], case["ctx"], logits)
        return {"token": token, "logits": logits, "state": st["views"]}
    if kind == "prefill":
        token = st["m"].prefill(st["tokens"], case["past"])
        return {"token": token, "logits": st["m"].logits(), "state": st["views"]}
    if kind in ("ffn", "gdn_in"):
        T = case["tokens"]
        sinter.check(L.sinter_rmsnorm_quant_q8k_ubatch(_p(st["x"]), _p(st["norm"]), EPS, E, T, _p(st["xq"]), _s()), "norm")
        if kind == "ffn":
            _ubatch(st, "gate", T, st["y_gate"])
            _ubatch(st, "up", T, st["y_up"])
            sinter.check(L.sinter_swiglu_quant_q8k_ubatch(_p(st["y_gate"]), _p(st["y_up"]), F, T, _p(st["xq"]), _s()), "swiglu")
            _ubatch(st, "down", T, st["y_down"], 1)
            return {"gate": st["y_gate"], "up": st["y_up"], "out": st["y_down"]}
        for name in ("qkv", "z", "alpha", "beta"):
            _ubatch(st, name, T, st["y_" + name])
        sinter.check(L.sinter_conv_silu_ubatch(_p(st["y_qkv"]), _p(st["conv_state"]), _p(st["conv_w"]), _p(st["conv"]),
                                               CH, DCONV, T, _s()), "conv")
        return {"qkv": st["y_qkv"], "z": st["y_z"], "alpha": st["y_alpha"], "beta": st["y_beta"], "conv": st["conv"],
                "state": st["conv_state"]}
    if kind == "gemv_ubatch":
        _ubatch(st, "w", case["tokens"], st["y_w"])
        return st["y_w"]
    if kind == "op_gemv":
        sinter.check(L.sinter_op_gemv(C.byref(st["args"]), 256, _s()), "op_gemv")
        return st["y"]
    sinter.check(L.sinter_op_attn_decode(C.byref(st["args"]), 256, _s()), "op_attn_decode")
    return {"out": st["out"], "rows": st["rows"]}


# ------------------------------------------------------------------ what a pass cannot do without

def _mats(case):
    """(type, rows, k) of a model case's matrices, the head last."""
    q4 = case.get("quant", "q4_k_m") == "q4_k_m"
    a, b = (Q4_K, Q6_K) if q4 else (BF16, BF16)
    out = []
    for il in range(case["layers"]):
        if _is_attn(case, il):
            out += [(a, NQ * 2 * HD, E), (a, RW, E), (b, RW, E), (a, E, NQ * HD)]
        else:
            out += [(a, CH, E), (a, VD, E), (a, HV, E), (a, HV, E), (a, E, VD)]
        out += [(a, F, E), (a, F, E), (b, E, F)]
    return out + [(b, case["vocab"], E)]


def _ops(mats, T):
    return (sum(sinter.row_bytes(t, k) * r for t, r, k in mats), 2.0 * T * sum(r * k for t, r, k in mats))


def work(case):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        T = 1 if kind == "decode" else case["tokens"]
        past = case["ctx"] if kind == "decode" else case["past"]
        mats = _mats(case)
        by, fl = _ops(mats[:-1], T)
        hb, hf = _ops(mats[-1:], 1)              # the head runs on the last token
        by += hb + case["vocab"] * 4 + T * E * 4
        fl += hf
        row = RW // 32 * 34 if case["kv"] == "q8_0" else RW * 2
        for il in range(case["layers"]):
            if _is_attn(case, il):
                by += 2 * row * (past + 2 * T)
                fl += 4.0 * NQ * HD * (T * past + T * (T + 1) / 2)
            else:
                by += 2 * 4 * (HV * D * D + CH * (DCONV - 1))
                fl += 8.0 * T * HV * D * D
        return {"bytes": by, "flops": fl}
    if kind in ("ffn", "gdn_in"):
        T = case["tokens"]
        mats = [(Q4_K, F, E), (Q4_K, F, E), (Q6_K, E, F)] if kind == "ffn" else \
            [(Q4_K, CH, E), (Q4_K, VD, E), (Q4_K, HV, E), (Q4_K, HV, E)]
        by, fl = _ops(mats, T)
        outs = 2 * F + 2 * E if kind == "ffn" else 2 * CH + VD + 2 * HV
        return {"bytes": by + 4 * T * (E + outs), "flops": fl}
    if kind == "gemv_ubatch":
        by, fl = _ops([(TYPES[case["type"]], case["rows"], case["k"])], case["tokens"])
        return {"bytes": by + case["tokens"] * (case["k"] // 256 * Q8K_BYTES + 4 * case["rows"]), "flops": fl}
    if kind == "op_gemv":
        by, fl = _ops([(TYPES[case["type"]], case["rows"], case["k"])], 1)
        return {"bytes": by + 4 * (case["k"] + case["rows"]), "flops": fl}
    row = RW // 32 * 34 if case["kv"] == "q8_0" else RW * 2
    return {"bytes": 2 * row * (case["pos"] + 2) + 4 * (3 * NQ * HD + 2 * RW), "flops": 4.0 * NQ * HD * (case["pos"] + 1)}


def tolerance(case):
    """Four times the difference from exact(), rounded: fp32 sums alone where
    the inputs of the products are given, and what an activation code that
    rounds the other way moves where the pass quantises its own activations."""
    kind = case["kind"]
    if kind == "gemv_ubatch":
        return {"rel": 2e-6, "max": 1e-4}
    if kind == "op_gemv":
        return {"rel": 2e-5, "max": 2e-3} if case["type"] == "bf16" else {"rel": 5e-4, "max": 2e-2}
    if kind == "op_attn":
        return {"rel": 2e-4, "max": 1e-2}
    if kind == "ffn":
        return {"rel": 4e-3, "max": 0.2}
    if kind == "gdn_in":
        return {"rel": 5e-4, "max": 5e-2}
    # layers and models: rounding travels through every later layer (one
    # attention layer's logits are 1e-2 from exact(), its angles in 32 bits)
    if case.get("every", 4) == 0:
        return {"rel": 5e-3, "max": 0.5, "differ": 0.01}
    return {"rel": 3e-2, "max": 0.9, "differ": 0.01}


# ------------------------------------------------------------------ the same in 64 bits

def _dequant(t, raw, rows, k):
    """float64 [rows, k] of ggml weight rows."""
    dev = raw.device
    if t == BF16:
        return raw.view(torch.bfloat16).double().view(rows, k)
    if t == sinter.F32:
        return raw.view(torch.float32).double().view(rows, k)
    if t == Q8_0:
        b = raw.view(-1, 34)
        return (b[:, :2].contiguous().view(torch.float16).double() * b[:, 2:].contiguous().view(torch.int8).double()).view(rows, k)
    if t == Q4_K:
        b = raw.view(-1, 144)
        d = b[:, :4].contiguous().view(torch.float16).double()
        s = b[:, 4:16].long()
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        qs = b[:, 16:].view(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(-1, 8, 32).double()
        return (q * (d[:, :1] * sc)[:, :, None] - (d[:, 1:] * mn)[:, :, None]).view(rows, k)
    b = raw.view(-1, 210)
    d = b[:, 208:].contiguous().view(torch.float16).double()
    sc = b[:, 192:208].contiguous().view(torch.int8).double()
    ql, qh = b[:, :128].view(-1, 2, 64), b[:, 128:192].view(-1, 2, 32)
    sh = torch.tensor([0, 2, 4, 6], dtype=torch.uint8, device=dev).view(1, 1, 4, 1)
    lo = torch.cat([ql & 15, ql >> 4], 2).view(-1, 2, 4, 32)
    q = (lo | (((qh.unsqueeze(2) >> sh) & 3) << 4)).double() - 32.0
    return (q.view(-1, 16, 16) * (d * sc)[:, :, None]).view(rows, k)


def _q8k(x):
    """x through ggml's Q8_K quantiser: codes of 256-element blocks scaled by -127 / (first element of largest |x|)."""
    b = x.reshape(-1, 256)
    mx = b.gather(1, b.abs().argmax(1, keepdim=True))
    isc = torch.where(mx != 0, -127.0 / mx, torch.zeros_like(mx))
    q = torch.clamp(torch.round(b * isc), max=127.0)
    return torch.where(isc != 0, q / isc, torch.zeros_like(q)).view(x.shape)


def _act(t, x):
    """x as the weights' dot product sees it."""
    if t == BF16:
        return x.float().bfloat16().double()
    if t == Q8_0:
        b = x.reshape(-1, 32)
        am = b.abs().amax(1, keepdim=True)
        q = torch.where(am != 0, torch.round(b * (127.0 / am)), torch.zeros_like(b))
        return (q * (am / 127.0).half().double()).view(x.shape)
    return _q8k(x)


def _mm(x, t, raw, rows, k):
    """x [T, k] (f64, not yet quantised) by the rows of raw, in slices of rows."""
    xa, out, n = _act(t, x), [], sinter.row_bytes(t, k)
    for r in range(0, rows, 16384):
        m = min(16384, rows - r)
        out.append(xa @ _dequant(t, raw[r * n:(r + m) * n].contiguous(), m, k).t())
    return torch.cat(out, 1)


def _norm(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _silu(x):
    return x / (1.0 + torch.exp(-x))


def _rope(x, pos):
    """NEOX rotation of the first ROPE dims of x [T, heads, HD] at positions pos [T]."""
    h = ROPE // 2
    th = pos.double()[:, None] * (THETA ** (-2.0 / ROPE)) ** torch.arange(h, device=x.device, dtype=torch.float64)
    c, s = torch.cos(th)[:, None], torch.sin(th)[:, None]
    a, b = x[..., :h], x[..., h:2 * h]
    return torch.cat([a * c - b * s, a * s + b * c, x[..., 2 * h:]], -1)


def _q8_rows(x):
    """x through ggml's reference Q8_0 quantiser (the KV cache's)."""
    b = x.reshape(-1, 32)
    d = b.abs().amax(1, keepdim=True) / 127.0
    q = torch.where(d != 0, b / d, torch.zeros_like(b))
    q = torch.sign(q) * torch.floor(q.abs() + 0.5)
    return (q * d.half().double()).view(x.shape)


def _attention(qg, k, v, qn, kn, kc, vc, q8):
    """Gated causal attention of T new tokens behind kc / vc (f64 [past, RW]): (output [T, NQ * HD], K rows, V rows)."""
    T, past = qg.shape[0], kc.shape[0]
    pos = torch.arange(past, past + T, device=qg.device)
    qg = qg.view(T, NQ, 2, HD)
    q = _rope(_norm(qg[:, :, 0], qn), pos)
    kr = _rope(_norm(k.view(T, NKV, HD), kn), pos).reshape(T, RW)
    rnd = _q8_rows if q8 else (lambda x: x.half().double())
    kk, vv = rnd(kr), rnd(v)
    K, V = torch.cat([kc, kk]).view(-1, NKV, HD), torch.cat([vc, vv]).view(-1, NKV, HD)
    out = torch.empty(T, NQ, HD, dtype=torch.float64, device=qg.device)
    dead = torch.arange(past + T, device=qg.device)[None, :] > pos[:, None]
    for h in range(NQ):
        g = h // (NQ // NKV)
        s = (q[:, h] @ K[:, g].t().contiguous()) * HD ** -0.5
        out[:, h] = torch.softmax(s.masked_fill(dead, -math.inf), 1) @ V[:, g].contiguous()
    return (out / (1.0 + torch.exp(-qg[:, :, 1]))).view(T, NQ * HD), kk, vv


def _conv(x, st, w):
    """Causal conv + silu over tokens: x [T, CH], st [CH, 3], w [CH, 4] -> (y, new state)."""
    win = torch.cat([st.t(), x])
    y = sum(win[j:j + x.shape[0]] * w[:, j] for j in range(DCONV))
    return _silu(y), win[-(DCONV - 1):].t().contiguous()


def _delta_rule(cv, alpha, beta, dt, a, S):
    """The gated-DeltaNet recurrence over tokens: cv [T, CH], S [HV, D(col), D(row)] -> (o [T, VD], S)."""
    T = cv.shape[0]
    q, k = cv[:, :HK * D].view(T, HK, D), cv[:, HK * D:2 * HK * D].view(T, HK, D)
    v = cv[:, 2 * HK * D:].view(T, HV, D)

    def unit(x):
        return (x / torch.clamp(torch.sqrt((x * x).sum(-1, keepdim=True)), min=EPS)).repeat(1, HV // HK, 1)
    q, k = unit(q), unit(k)
    sp = torch.where(alpha + dt > 20.0, alpha + dt, torch.log1p(torch.exp(alpha + dt)))
    g, b = torch.exp(sp * a)[:, :, None], (1.0 / (1.0 + torch.exp(-beta)))[:, :, None]
    o = torch.empty_like(v)
    for t in range(T):
        S = S * g[t][:, :, None]
        delta = (v[t] - (S * k[t][:, None, :]).sum(-1)) * b[t]
        S = S + delta[:, :, None] * k[t][:, None, :]
        o[t] = (S * q[t][:, None, :]).sum(-1) * D ** -0.5
    return o.view(T, VD), S


def _exact_model(case, st):
    m = st["m"]
    q8 = case["kv"] == "q8_0"

    def raw(il, slot):
        p, nb, t = m.tensor(il, slot)
        return t, _view(p, (nb,), "|u1", m)

    def mat(x, il, slot, rows):
        t, w = raw(il, slot)
        return _mm(x, t, w, rows, x.shape[1])

    def vec(il, slot):
        return raw(il, slot)[1].view(torch.float32).double()

    def cache(p, n):
        if n == 0:
            return torch.zeros(0, RW, dtype=torch.float64, device="cuda")
        if q8:
            return _dequant(Q8_0, _view(p, (n * RW // 32 * 34,), "|u1", m), n, RW)
        return _view(p, (n, RW), "<f2", m).double()

    toks = [st["token"]] if case["kind"] == "decode" else st["tokens"]
    past = case["ctx"] if case["kind"] == "decode" else case["past"]
    te, emb = raw(case["layers"], 0)
    n = sinter.row_bytes(te, E)
    x = torch.cat([_dequant(te, emb[t * n:(t + 1) * n].contiguous(), 1, E) for t in toks])
    states = []
    for il in range(case["layers"]):
        xn = _norm(x, vec(il, 0))
        (p0, _), (p1, _) = m.state(il, 0), m.state(il, 1)
        if _is_attn(case, il):
            qg, k, v = mat(xn, il, 5, NQ * 2 * HD), mat(xn, il, 6, RW), mat(xn, il, 7, RW)
            att, kk, vv = _attention(qg, k, v, vec(il, 9), vec(il, 10), cache(p0, past), cache(p1, past), q8)
            x = x + mat(att, il, 8, E)
            states += [None, None] if q8 else [kk, vv]
        else:
            qkv, z = mat(xn, il, 5, CH), mat(xn, il, 6, VD)
            al, be = mat(xn, il, 7, HV), mat(xn, il, 8, HV)
            cv, cs = _conv(qkv, _view(p0, (CH, DCONV - 1), "<f4", m).double(), vec(il, 10).view(CH, DCONV))
            o, S = _delta_rule(cv, al, be, vec(il, 11), vec(il, 12), _view(p1, (HV, D, D), "<f4", m).double())
            on = _norm(o.view(-1, HV, D), vec(il, 13)) * _silu(z.view(-1, HV, D))
            x = x + mat(on.reshape(-1, VD), il, 9, E)
            states += [cs, S]
        xn = _norm(x, vec(il, 1))
        f = _silu(mat(xn, il, 2, F)) * mat(xn, il, 3, F)
        x = x + mat(f, il, 4, E)
    logits = mat(_norm(x[-1:], vec(case["layers"], 1)), case["layers"], 2, case["vocab"])[0]
    return {"token": None, "logits": logits, "state": states}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        T = 1 if kind == "decode" else case["tokens"]
        past = case["ctx"] if kind == "decode" else case["past"]
        # (whole models and the longest attention: over 20 seconds)
        if case["layers"] > 16 or T * case["layers"] > 4000 or T * past * case["layers"] > 20e6:
            return None
        st = prepare(case, seed)
        out = _exact_model(case, st)
        torch.cuda.synchronize()   # (the model goes with st)
        return out
    st = prepare(case, seed)
    if kind in ("ffn", "gdn_in"):
        xn = _norm(st["x"].double(), st["norm"].double())
        if kind == "ffn":
            g, u = _mm(xn, *_w(st["gate"])), _mm(xn, *_w(st["up"]))
            return {"gate": g, "up": u, "out": st["y_down"].double() + _mm(_silu(g) * u, *_w(st["down"]))}
        y = {n: _mm(xn, *_w(st[n])) for n in ("qkv", "z", "alpha", "beta")}
        y["conv"], y["state"] = _conv(y["qkv"], st["conv_state"].double(), st["conv_w"].double())
        return y
    if kind == "gemv_ubatch":
        t, rows, k, raw = st["w"]
        b = st["xq"].view(-1, Q8K_BYTES)
        x = (b[:, :4].contiguous().view(torch.float32).double() * b[:, 4:260].contiguous().view(torch.int8).double()).view(-1, k)
        n = sinter.row_bytes(t, k)
        return torch.cat([x @ _dequant(t, raw[r * n:(r + 16384) * n].contiguous(), min(16384, rows - r), k).t()
                          for r in range(0, rows, 16384)], 1)
    if kind == "op_gemv":
        x = st["x"].double()[None]
        return _mm(_norm(x, st["norm"].double()) if case["norm"] else x, *_w(st["w"]))[0]
    q8, pos = case["kv"] == "q8_0", case["pos"]
    caches = [_dequant(Q8_0, st[c], pos + 1, RW) if q8 else st[c].view(torch.float16).double().view(-1, RW)
              for c in ("kc", "vc")]
    out, kk, vv = _attention(st["qg"].double().view(1, -1), st["k"].double()[None], st["v"].double()[None],
                             st["qn"].double(), st["kn"].double(), caches[0][:pos], caches[1][:pos], q8)
    return {"out": out[0], "rows": [None, None] if q8 else [kk[0], vv[0]]}


def _w(m):
    t, rows, k, raw = m
    return t, raw, rows, k
