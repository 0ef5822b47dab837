"""The measured work of this framework: one entry per operator call that a serving engine makes, through the public
entry points of qwengine_amd.ops.

The model is a hybrid of 16 attention layers (24 query / 4 KV heads, head_dim 256, quantized KV cache) and 48 Gated
DeltaNet layers; an engine decodes one token at a time or verifies a few drafted ones, and prefills prompts in chunks
of up to 1024 tokens whose last chunk is ragged.  A decode-side pass goes over several layers, each with its own cache,
state or weights, as a model does, so the 256 MB last-level cache does not hold a pass's data; a prefill-side pass is
one layer's call.  Cache contents, weights and activations are synthetic: K / V ~N(0,1) with 1% of the key rows scaled
by 8, quantized as the append does it; weights are random codes with small normal fp16 block scales.
"""
import math
import os
import re

import torch

import qwengine_amd.ops as ops

DEV = "cuda"
NH, NKV, HD, QD = 24, 4, 256, 6144          # query heads, KV heads, head_dim, floats of one token's q / gate / out
POS_BYTES = {"f16": 4096, "q8_0": 2176, "q4_0": 1152}  # K + V values and scales of one position, all KV heads
CH, DQK, VD, VH, KH, DH = 10240, 2048, 6144, 48, 16, 128  # Gated DeltaNet: channels, q / k width, value dim, heads
EPS, THETA = 1e-6, 1e7
WEIGHTS = {"q2_k": (10, 84, (80, 82)), "q4_k": (12, 144, (0, 2)), "q6_k": (14, 210, (208,)), "iq2_xxs": (16, 66, (0,)),
           "iq2_xs": (17, 74, (0,)), "iq3_xxs": (18, 98, (0,)), "iq3_s": (21, 110, (0,)), "iq2_s": (22, 82, (0,)),
           "iq4_xs": (23, 136, (0,))}  # format id, bytes of a 256-weight block, offsets of its fp16 scale fields
OUT_PROJ = "iq3_s iq2_xs iq2_xxs iq2_s"     # the model's formats of the attention output projection, layer after layer


# ---- the cases ------------------------------------------------------------------------------------------------------
def listed():
    return [
        # one token's decode over the longest context in use: the headline, bound by the cache's bytes
        {"name": "decode_q4_0_150000", "kind": "decode", "kv": "q4_0", "n": 150000, "nq": 1, "layers": 4},
        # speculative verify of 6 drafted tokens at a long context, the most queries a step of the engine has
        {"name": "verify7_q4_0_32775", "kind": "decode", "kv": "q4_0", "n": 32775, "nq": 7, "layers": 8},
        # a short verify over the higher-precision quantized cache, at a length that is no multiple of anything
        {"name": "verify4_q8_0_60013", "kind": "decode", "kv": "q8_0", "n": 60013, "nq": 4, "layers": 3},
        # decode early in a conversation over an unquantized cache: launches and latency
        {"name": "decode_f16_4096", "kind": "decode", "kv": "f16", "n": 4096, "nq": 1, "layers": 16},
        # a full prefill chunk deep in a long prompt: bound by the matrix cores
        {"name": "prefill_1024_q8_0_at_32768", "kind": "prefill", "kv": "q8_0", "B": 1024, "p0": 32768},
        # the ragged last chunk of a prompt, or a short follow-up message on a long conversation
        {"name": "prefill_77_q4_0_at_20011", "kind": "prefill", "kv": "q4_0", "B": 77, "p0": 20011},
        # a prompt that fits one chunk: the first thing that every request does
        {"name": "prefill_509_f16_at_0", "kind": "prefill", "kv": "f16", "B": 509, "p0": 0},
        # norm, rotary embedding and quantize-on-append of a chunk's rows, before its attention
        {"name": "prep_1024_q8_0", "kind": "prep", "kv": "q8_0", "B": 1024, "p0": 32768},
        # one token through the 48 recurrent layers
        {"name": "dn_decode", "kind": "dn", "commit": 0, "new": 1, "layers": 48},
        # a full prefill chunk of one recurrent layer
        {"name": "dn_prefill_1024", "kind": "dn_rows", "B": 1024},
        # the output projection of one decoded token in the model's 16 attention layers
        {"name": "out_proj_decode", "kind": "gemv", "fmts": OUT_PROJ, "K": 6144, "N": 5120, "nb": 1, "layers": 16},
        # the output projection of a prefill chunk: weights to fp16, then the matrix product, for four layers
        {"name": "out_proj_prefill_1024", "kind": "gemm", "fmts": OUT_PROJ, "K": 6144, "N": 5120, "B": 1024},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["decode"] * 4 + ["prefill"] * 3 + ["prep", "dn", "dn_rows", "gemv", "gemm"])
    kv = rng.choice(list(POS_BYTES))
    if kind == "decode":
        nq = rng.choice([1, 1, 1, 2, 3, 4, 5, 6, 7, 8])
        n = _log(rng, 64, 150000)
        return {"kind": kind, "kv": kv, "n": n, "nq": nq,
                "layers": max(1, min(16, 300_000_000 // (n * POS_BYTES[kv])))}
    if kind == "prefill":
        B = _log(rng, 1, 1024)
        p0 = _log(rng, 1, min(100000, int(8.3e11 / (4 * QD * B)) - B)) - 1
        return {"kind": kind, "kv": kv, "B": B, "p0": p0}
    if kind == "prep":
        return {"kind": kind, "kv": kv, "B": _log(rng, 1, 1024), "p0": _log(rng, 1, 60000) - 1}
    if kind == "dn":
        new = rng.choice([1, 2, 3, 4, 5, 6, 7])
        return {"kind": kind, "commit": rng.randrange(0, 7) if new > 1 else 0, "new": new, "layers": rng.randint(16, 48)}
    if kind == "dn_rows":
        return {"kind": kind, "B": _log(rng, 1, 1024)}
    fmts, K = rng.choice(list(WEIGHTS)), rng.choice([5120, 6144, 17408])
    if kind == "gemv":
        N = _log(rng, 1000, 8000)
        return {"kind": kind, "fmts": fmts, "K": K, "N": N, "nb": rng.choice([1, 1, 2, 3, 4]),
                "layers": max(1, min(16, 300_000_000 // (N * K * WEIGHTS[fmts][1] // 256)))}
    return {"kind": kind, "fmts": fmts, "K": K if K < 17408 else 6144, "N": rng.choice([1024, 5120, 6144]),
            "B": _log(rng, 9, 1024)}


# ---- inputs ---------------------------------------------------------------------------------------------------------
def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed((seed * 1000003 + salt) % (1 << 62))


def _rn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV)


def _quantize(x, kv):
    """Rows x [4][n][256] as the cache stores them: (value bytes [4][n][vb], fp16 scale bits [4][n][8] or None)."""
    if kv == "f16":
        return x.half().view(torch.uint8), None
    b = x.view(*x.shape[:2], 8, 32)
    if kv == "q8_0":
        d = b.abs().amax(-1) / 127.0
        y = b * torch.where(d > 0, 1.0 / d, torch.zeros_like(d))[..., None]
        q = (torch.sign(y) * torch.floor(y.abs() + 0.5)).to(torch.int8).view(torch.uint8)
        return q.view(*x.shape), d.half().view(torch.int16)
    big = b.gather(-1, b.abs().argmax(-1, keepdim=True))[..., 0]
    d = big / -8.0
    y = b * torch.where(d != 0, 1.0 / d, torch.zeros_like(d))[..., None]
    q = (y + 8.5).to(torch.int32).clamp_(0, 15).to(torch.uint8)
    return (q[..., 0::2] | (q[..., 1::2] << 4)).view(*x.shape[:2], 128), d.half().view(torch.int16)


def _dequantize(vals, scales, kv):
    """Cache rows [n] of one KV head in 64 bits, [n][256]."""
    if kv == "f16":
        return vals.view(torch.float16).double()
    d = scales.view(torch.float16).double()[..., None]
    if kv == "q8_0":
        return (vals.view(torch.int8).double().view(-1, 8, 32) * d).view(-1, 256)
    q = torch.stack([vals & 15, vals >> 4], -1).view(-1, 8, 32).double() - 8.0
    return (q * d).view(-1, 256)


def _cache(kv, n, capacity, g):
    """A layer's cache with n positions filled."""
    c = ops.KVLayer.allocate(kv, capacity, device=DEV)
    for vals, scales, key in ((c.k, c.ks, True), (c.v, c.vs, False)):
        for p in range(0, n, 32768):
            m = min(32768, n - p)
            x = _rn(g, NKV, m, HD)
            if key:
                x[torch.rand((NKV, m), generator=g, device=DEV) < 0.01] *= 8.0
            q, s = _quantize(x, kv)
            vals[:, p:p + m] = q
            if s is not None:
                scales[:, p:p + m] = s
    return c


def _act(x):
    """Rows x [n][K] as ActQ8."""
    b = x.view(-1, 32)
    d = b.abs().amax(-1) / 127.0
    q = torch.where(d[:, None] > 0, torch.round(b / d[:, None]), torch.zeros_like(b))
    return ops.ActQ8(q.to(torch.int8).view(-1), d, d * q.sum(-1))


def _weights(fmt, N, K, g):
    _, size, offsets = WEIGHTS[fmt]
    w = torch.randint(0, 256, (N, K // 256, size), generator=g, device=DEV, dtype=torch.uint8)
    for o in offsets:
        w[:, :, o:o + 2] = (0.01 * _rn(g, N, K // 256, 1)).half().view(torch.uint8)
    return w.view(N, -1)


def _dn_params(g, L):
    """L recurrent layers, and their conv windows [L][2][3][CH] and states [L][48][128][128]."""
    window, state = 0.5 * _rn(g, L, 2, 3, CH), 0.1 * _rn(g, L, VH, DH, DH)
    return [ops.DNParams(0.5 * _rn(g, CH, 4), _rn(g, VH), -torch.exp(0.5 * _rn(g, VH)), 1.0 + 0.1 * _rn(g, DH),
                         window[i], state[i]) for i in range(L)], window, state


def _captured(warm, call):
    """call() as a HIP graph, the way an engine issues the fixed part of its decode step."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        warm()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    return graph


def _inputs(c, seed):
    """What the call reads, from the seed alone."""
    g = _gen(seed)
    kind = c["kind"]
    if kind == "decode":
        return {"q": _rn(g, c["nq"], NH, HD), "gate": _rn(g, c["nq"], NH, HD),
                "kv": [_cache(c["kv"], c["n"], c["n"] + 64, _gen(seed, 1 + i)) for i in range(c["layers"])]}
    if kind == "prefill":
        n = c["p0"] + c["B"]
        return {"q": _rn(g, c["B"], NH, HD), "gate": _rn(g, c["B"], NH, HD), "kv": _cache(c["kv"], n, n + 64, g)}
    if kind == "prep":
        B = c["B"]
        return {"qg": _rn(g, B, NH, 512), "k": _rn(g, B, NKV, HD), "v": _rn(g, B, NKV, HD),
                "qn": 0.5 + torch.rand(HD, generator=g, device=DEV),
                "kn": 0.5 + torch.rand(HD, generator=g, device=DEV)}
    if kind == "dn":
        m, n = c["commit"], c["new"]
        p, window, state = _dn_params(g, c["layers"])
        return {"p": p, "window": window, "state": state, "qkv": 0.5 * _rn(g, n, CH), "z": _rn(g, n, VD),
                "b": _rn(g, n, 64), "a": 2.0 * _rn(g, n, 64), "sqkv": 0.5 * _rn(g, max(m, 1), CH),
                "sb": _rn(g, max(m, 1), 64), "sa": 2.0 * _rn(g, max(m, 1), 64)}
    if kind == "dn_rows":
        B = c["B"]
        p, window, state = _dn_params(g, 1)
        return {"p": p, "window": window, "state": state, "qkv": 0.5 * _rn(g, B, CH), "z": _rn(g, B, VD), "b": _rn(g, B, VH),
                "a": 2.0 * _rn(g, B, VH)}
    fmts = c["fmts"].split()
    W = [(fmts[i % len(fmts)], _weights(fmts[i % len(fmts)], c["N"], c["K"], g))
         for i in range(c["layers"] if kind == "gemv" else len(fmts))]
    if kind == "gemv":
        return {"W": W, "act": _act(_rn(g, c["nb"], c["K"]))}
    return {"W": W, "X": _rn(g, c["B"], c["K"]).half()}


def prepare(case, seed):
    c = case
    s = dict(_inputs(c, seed), case=c)
    new = lambda *shape, **kw: torch.empty(shape, device=DEV, **kw)
    kind = c["kind"]
    if kind == "decode":
        L, nq = c["layers"], c["nq"]
        s["out"] = new(L, nq, NH, HD)
        s["act"] = [new(L, nq * QD, dtype=torch.int8), new(L, nq * QD // 32), new(L, nq * QD // 32)]
        s["oq"] = [ops.ActQ8(*(t[i] for t in s["act"])) for i in range(L)]
        s["work"] = new(ops.attn_work_bytes(c["n"]) // 4 + 1)
    elif kind == "prefill":
        s["out"] = new(c["B"], NH, HD, dtype=torch.float16)
        ops.attn_prefill_reserve(c["B"], c["p0"] + c["B"])
    elif kind == "prep":
        B, n = c["B"], c["p0"] + c["B"]
        s["kv"] = ops.KVLayer.allocate(c["kv"], n + 64, device=DEV)
        s["rope"], s["q"], s["gate"] = new(B, 64), new(B, NH, HD), new(B, NH, HD)
        s["src"] = [ops.RowSrc.device(s["qg"], NH * 512), ops.RowSrc.device(s["k"], NKV * HD),
                    ops.RowSrc.device(s["v"], NKV * HD)]
    elif kind == "dn":
        L, m, n = c["layers"], c["commit"], c["new"]
        s["o"] = new(L, n, VD)
        s["act"] = [new(L, n * VD, dtype=torch.int8), new(L, n * VD // 32), new(L, n * VD // 32)]
        oq = [ops.ActQ8(*(t[i] for t in s["act"])) for i in range(L)]
        # a verified block is only committed by the next step, which learns how many of its tokens were accepted:
        # this step applies the pending ones and saves the new ones; a single decoded token is applied at once
        s["saved"] = [torch.zeros((L, n, w), device=DEV) for w in (CH, 64, 64)] if n > 1 else []
        tok = [ops.DNTokens(sqkv=s["sqkv"] if m else None, sbeta=s["sb"] if m else None, salpha=s["sa"] if m else None,
                            qkv=s["qkv"], z=s["z"], beta=s["b"], alpha=s["a"],
                            **dict(zip(("oqkv", "obeta", "oalpha"), (t[i] for t in s["saved"])))) for i in range(L)]
        call = lambda l, after: ops.deltanet_multi(s["p"][l], 0, tok[l], m, n, after, EPS, s["o"][l], oq[l])
        s["graph"] = _captured(lambda: call(0, 0), lambda: [call(l, m if n > 1 else 1) for l in range(L)])
    elif kind == "dn_rows":
        B = c["B"]
        s["work"], s["core"] = new(ops.dn_work_bytes(B) // 4 + 1), new(B, VD)
        s["o16"] = new(B, VD, dtype=torch.float16)
    elif kind == "gemv":
        s["y"] = new(c["layers"], c["nb"], c["N"])

        def call(l):
            fmt, w = s["W"][l]
            args = (WEIGHTS[fmt][0], w, w.shape[1], c["K"], c["N"], s["act"])
            if c["nb"] == 1:
                ops.gemv_q8(*args, s["y"][l])
            else:
                ops.gemv_q8n(*args, c["nb"], c["K"], s["y"][l], c["N"])
        s["graph"] = _captured(lambda: [call(l) for l in range(min(4, c["layers"]))],
                               lambda: [call(l) for l in range(c["layers"])])
    else:
        s["gemm"] = ops.Gemm()
        s["w16"] = new(len(s["W"]), c["N"], c["K"], dtype=torch.float16)
        s["y"] = new(len(s["W"]), c["B"], c["N"])
    return s


# ---- one pass -------------------------------------------------------------------------------------------------------
def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "decode":
        for i, kv in enumerate(s["kv"]):
            ops.attn_decode_multi(s["q"], s["gate"], kv, kv.kvt, c["n"] - c["nq"], c["nq"], s["work"], s["out"][i],
                                  s["oq"][i])
        return {"out": s["out"], "act_q": s["act"][0], "act_d": s["act"][1], "act_s": s["act"][2]}
    if kind == "prefill":
        ops.attn_prefill(s["q"], s["gate"], s["kv"], s["kv"].kvt, c["B"], c["p0"], s["out"])
        return {"out": s["out"]}
    if kind == "prep":
        kv, B, p0 = s["kv"], c["B"], c["p0"]
        if B <= 8:  # a decode step's tokens
            ops.attn_prep_multi(*s["src"], s["qn"], s["kn"], p0, p0, B, THETA, EPS, kv.kvt, kv, s["q"], s["gate"])
        else:
            ops.rope_table(p0, B, THETA, s["rope"])
            ops.attn_prep_rows(s["qg"], s["k"], s["v"], s["qn"], s["kn"], B, p0, s["rope"], EPS, kv.kvt, kv, s["q"],
                               s["gate"])
        rows = lambda t: None if t is None else t[:, p0:p0 + B]
        return {"q": s["q"], "gate": s["gate"], "k": rows(kv.k), "v": rows(kv.v), "ks": rows(kv.ks), "vs": rows(kv.vs)}
    if kind == "dn":
        s["graph"].replay()
        return {"o": s["o"], "act_q": s["act"][0], "act_d": s["act"][1], "act_s": s["act"][2],
                "state": s["state"], "window": s["window"],
                "saved": s["saved"]}
    if kind == "dn_rows":
        ops.deltanet_rows(s["p"][0], s["qkv"], s["z"], s["b"], s["a"], c["B"], 0, EPS, s["work"], s["core"], s["o16"])
        return {"o": s["o16"], "state": s["state"], "window": s["window"]}
    if kind == "gemv":
        s["graph"].replay()
        return {"y": s["y"]}
    for i, (fmt, w) in enumerate(s["W"]):
        ops.dequant_rows_f16(WEIGHTS[fmt][0], w, w.shape[1], c["K"], c["N"], s["w16"][i])
        s["gemm"].f16(s["w16"][i], c["N"], c["K"], s["X"], c["K"], c["B"], s["y"][i], c["N"])
    return {"y": s["y"], "w16": s["w16"]}


# ---- what a pass cannot do without ----------------------------------------------------------------------------------
def work(case):
    c = case
    kind = c["kind"]
    keys = lambda n, b: sum(n - b + t + 1 for t in range(b))
    if kind == "decode":
        return {"bytes": c["layers"] * (c["n"] * POS_BYTES[c["kv"]] + c["nq"] * QD * (4 * 3 + 1 + 0.25)),
                "flops": c["layers"] * 4.0 * QD * keys(c["n"], c["nq"])}
    if kind == "prefill":
        n = c["p0"] + c["B"]
        return {"bytes": n * POS_BYTES[c["kv"]] + c["B"] * QD * (4 + 4 + 2), "flops": 4.0 * QD * keys(n, c["B"])}
    if kind == "prep":
        return {"bytes": c["B"] * (2 * 4 * QD * 2 + 2 * 4 * NKV * HD + POS_BYTES[c["kv"]]), "flops": c["B"] * QD * 8.0}
    if kind == "dn":
        m, n = c["commit"], c["new"]
        state = VH * DH * DH * 4
        writes = n == 1 or m > 0
        rows = (m + n) * (CH + 128) * 4 + n * VD * (4 + 4 + 1.25) + (n * (CH + 128) * 4 if n > 1 else 0)
        return {"bytes": c["layers"] * (state * (1 + writes) + CH * 4 * (4 + 3 + 3 * writes) + rows),
                "flops": c["layers"] * (m + n) * VH * 6.0 * DH * DH}
    if kind == "dn_rows":
        return {"bytes": c["B"] * (CH * 4 + VD * 4 + 2 * VH * 4 + VD * 2) + 2 * VH * DH * DH * 4 + CH * 4 * 10,
                "flops": c["B"] * VH * 6.0 * DH * DH}
    size = sum(c["N"] * c["K"] // 256 * WEIGHTS[f][1] for f in c["fmts"].split()) / len(c["fmts"].split())
    if kind == "gemv":
        return {"bytes": c["layers"] * (size + c["nb"] * (c["K"] * 1.25 + c["N"] * 4)),
                "flops": c["layers"] * 2.0 * c["N"] * c["K"] * c["nb"]}
    L = len(c["fmts"].split())
    return {"bytes": L * (size + c["N"] * c["K"] * 2 + c["B"] * (c["K"] * 2 + c["N"] * 4)),
            "flops": L * 2.0 * c["N"] * c["K"] * c["B"]}


def tolerance(case):
    """About four times the distance of the path from 64 bits, over its formats and sizes.  "differ": ActQ8 codes and
    cache bytes that sit on a rounding edge move with the last bits of their input."""
    kind = case["kind"]
    if kind == "decode":   # fp16 probabilities, 32-bit sums: 2e-4
        return {"rel": 8e-4, "max": 0.02, "differ": 0.01}
    if kind == "prefill":  # fp16 keys, queries, probabilities and output: 9e-4
        return {"rel": 3e-3, "max": 0.1}
    if kind == "prep":     # 32-bit sums of 256 squares: 6e-8
        return {"rel": 3e-7, "max": 1e-5, "differ": 1e-4}
    if kind == "dn":       # 32-bit sums over a head's 128 x 128 state: 1.5e-7
        return {"rel": 1e-6, "max": 1e-4, "differ": 1e-3}
    if kind == "dn_rows":  # the same over the chunk's tokens; fp16 output: 2e-4
        return {"rel": 8e-4, "max": 2e-3}
    if kind == "gemv":     # exact integer dots, 32-bit sums over the blocks: 1e-7
        return {"rel": 5e-7, "max": 1e-5}
    return {"rel": 2e-6, "max": 1e-4}  # fp16 operands, 32-bit sums: 5e-7


# ---- the same in 64 bits --------------------------------------------------------------------------------------------
def _attention(q, gate, kv, fmt, n, p0, B):
    """q, gate [B][24][256] over cache positions [0, p0 + t] for token t."""
    out = torch.empty((B, NH, HD), dtype=torch.float64, device=DEV)
    G = NH // NKV
    seen = torch.arange(n, device=DEV)[None, :] <= p0 + torch.arange(B, device=DEV)[:, None]
    for h in range(NKV):
        K = _dequantize(kv.k[h, :n], None if kv.ks is None else kv.ks[h, :n], fmt)
        V = _dequantize(kv.v[h, :n], None if kv.vs is None else kv.vs[h, :n], fmt)
        for t in range(0, B, 256):
            e = min(B, t + 256)
            x = q[t:e, h * G:(h + 1) * G].double()
            sc = (x.reshape(-1, HD) @ K.T / 16.0).view(e - t, G, n)
            sc = sc.masked_fill_(~seen[t:e, None, :], -math.inf)
            out[t:e, h * G:(h + 1) * G] = (torch.softmax(sc, -1).view(-1, n) @ V).view(e - t, G, HD)
    return out * torch.sigmoid(gate.double())


def _silu(x):
    return x * torch.sigmoid(x)


def _delta(params, window, qkv, z, b, a, S, emit):
    """Tokens qkv [T][CH] through layers batched in front, window [L][3][CH], S [L][48][128 j][128 i]: the outputs
    [L][T - emit][VD] of the tokens from `emit` on, the states (after each of up to 16 tokens, else the last one) and
    the conv's inputs with the window in front."""
    w = torch.stack([p.conv_w for p in params]).double()
    dt = torch.stack([p.dt_bias for p in params]).double()
    A = torch.stack([p.ssm_a for p in params]).double()
    norm = torch.stack([p.ssm_norm for p in params]).double()
    L, T = len(params), qkv.shape[0]
    x = torch.cat([window.double(), qkv.double()[None].expand(L, T, CH)], 1)
    outs, states = [], [S]
    for t in range(T):
        conv = _silu((x[:, t:t + 4] * w.transpose(1, 2)).sum(1))
        q = conv[:, :DQK].view(L, KH, DH)
        k = conv[:, DQK:2 * DQK].view(L, KH, DH)
        q = (q / q.norm(dim=-1, keepdim=True).clamp_min(EPS)).repeat(1, VH // KH, 1)
        k = (k / k.norm(dim=-1, keepdim=True).clamp_min(EPS)).repeat(1, VH // KH, 1)
        v = conv[:, 2 * DQK:].view(L, VH, DH)
        beta = torch.sigmoid(b[t, :VH].double())[None, :, None]
        decay = torch.exp(torch.nn.functional.softplus(a[t, :VH].double() + dt) * A)
        S = S * decay[..., None, None]
        u = (v - (S @ k[..., None])[..., 0]) * beta
        S = S + u[..., None] * k[..., None, :]
        states = states + [S] if T <= 16 else [S]
        if t >= emit:
            o = (S @ q[..., None])[..., 0] / math.sqrt(DH)
            o = o / torch.sqrt((o * o).mean(-1, keepdim=True) + EPS) * norm[:, None, :]
            outs.append((o.reshape(L, VD) * _silu(z[t - emit].double())))
    return torch.stack(outs, 1), states, x


def _codebook(name):
    """A grid format's codebook, from the tables of the format in the source tree: uint8 [entries][bytes]."""
    src = open(os.path.join(os.path.dirname(ops.__file__), "csrc", "iq_grids.inc")).read()
    nums = lambda what: [int(v, 0) for v in re.search(what + r"\[\d+\] = \{([^}]*)\}", src).group(1).replace(
        "\n", " ").split(",") if v.strip()]
    bits, size = (int(re.search(name + what + r" = (\d+)", src).group(1)) for what in ("_BITS", "_BYTES"))
    levels, codes = torch.tensor(nums(name + "_LEVELS")), torch.tensor(nums(name + "_CODES"))
    at = (codes[:, None] >> (bits * torch.arange(size))) & ((1 << bits) - 1)
    return levels[at].to(DEV)


IQ4_LEVELS = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)


def _weight_values(fmt, w, K):
    """Rows of weights in 64 bits, [N][K], from the formats' block layouts."""
    N = w.shape[0]
    b = w.view(N * (K // 256), WEIGHTS[fmt][1])
    nb = b.shape[0]
    at = lambda *v: torch.tensor(v, device=DEV)
    half = lambda o: b[:, o:o + 2].contiguous().view(torch.float16).double()
    i64 = lambda lo, hi: b[:, lo:hi].long()
    u16 = lambda lo, hi: i64(lo, hi)[:, 0::2] | (i64(lo, hi)[:, 1::2] << 8)
    u32 = lambda lo, hi: u16(lo, hi)[:, 0::2] | (u16(lo, hi)[:, 1::2] << 16)
    bits8 = lambda x: (x[..., None] >> torch.arange(8, device=DEV)) & 1
    if fmt == "q4_k":
        s = i64(4, 16)
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        q = i64(16, 144).view(nb, 4, 32)
        q = torch.stack([q & 15, q >> 4], 2).view(nb, 8, 32)
        return (half(0)[..., None] * sc[..., None] * q - half(2)[..., None] * mn[..., None]).view(N, K)
    if fmt == "q2_k":
        s, q = i64(0, 16), i64(16, 80).view(nb, 2, 1, 2, 16)
        q = ((q >> at(0, 2, 4, 6).view(1, 1, 4, 1, 1)) & 3).reshape(nb, 16, 16)
        return (half(80)[..., None] * (s & 15)[..., None] * q - half(82)[..., None] * (s >> 4)[..., None]).view(N, K)
    if fmt == "q6_k":
        lo, hi = i64(0, 128).view(nb, 2, 2, 32), i64(128, 192).view(nb, 2, 1, 32)
        q = torch.cat([lo & 15, lo >> 4], 2) | (((hi >> at(0, 2, 4, 6).view(1, 1, 4, 1)) & 3) << 4)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        return (half(208)[..., None] * sc[..., None] * (q.view(nb, 16, 16) - 32)).view(N, K)
    if fmt == "iq4_xs":
        j = torch.arange(8, device=DEV)
        ls = ((i64(4, 8)[:, j // 2] >> (4 * (j % 2))) & 15) | (((u16(2, 4) >> (2 * j)) & 3) << 4)
        q = i64(8, 136).view(nb, 8, 16)
        lev = at(*IQ4_LEVELS)[torch.cat([q & 15, q >> 4], 2)]
        return (half(0)[..., None] * (ls - 32)[..., None] * lev).view(N, K)
    parity = torch.arange(128, device=DEV)
    parity = parity | ((bits8(parity).sum(-1) & 1) << 7)  # 7 sign bits and the one that makes the negatives even
    if fmt in ("iq2_xxs", "iq3_xxs"):
        if fmt == "iq2_xxs":
            blk = i64(2, 66).view(nb, 8, 8)
            aux = (blk[..., 4:] << at(0, 8, 16, 24)).sum(-1)
            g = _codebook("IQ2XXS")[blk[..., :4]].view(nb, 8, 4, 8)
        else:
            aux = u32(66, 98)
            g = _codebook("IQ3XXS")[i64(2, 66)].view(nb, 8, 4, 8)
        sign = bits8(parity[(aux[..., None] >> at(0, 7, 14, 21)) & 127])
        scale = (0.5 + (aux >> 28).double()) * (0.25 if fmt == "iq2_xxs" else 0.5)
        scale = scale[:, :, None, None]
    elif fmt in ("iq2_xs", "iq2_s"):
        if fmt == "iq2_xs":
            q = u16(2, 66).view(nb, 8, 4)
            g, sign, sc = _codebook("IQ2XS")[q & 511], bits8(parity[q >> 9]), i64(66, 74)
        else:
            idx = i64(2, 34).view(nb, 8, 4) | (((i64(66, 74)[..., None] >> at(0, 2, 4, 6)) & 3) << 8)
            g, sign, sc = _codebook("IQ2S")[idx], bits8(i64(34, 66).view(nb, 8, 4)), i64(74, 82)
        scale = 0.25 * (0.5 + torch.stack([sc & 15, sc >> 4], -1).double())
        scale = scale.repeat_interleave(2, -1)[..., None]
    else:
        idx = i64(2, 66).view(nb, 8, 8) | (bits8(i64(66, 74)) << 8)
        g, sign = _codebook("IQ3S")[idx].view(nb, 8, 4, 8), bits8(i64(74, 106).view(nb, 8, 4))
        sc = i64(106, 110)
        scale = (1.0 + 2.0 * torch.stack([sc & 15, sc >> 4], -1).view(nb, 8).double())[:, :, None, None]
    return (half(0)[..., None, None] * scale * g * (1 - 2 * sign)).view(N, K)


def exact(case, seed):
    c, s = case, _inputs(case, seed)
    kind = c["kind"]
    amax = lambda x: x.view(*x.shape[:1], -1, 32).abs().amax(-1) / 127.0
    if kind == "decode":
        out = torch.stack([_attention(s["q"], s["gate"], kv, c["kv"], c["n"], c["n"] - c["nq"], c["nq"])
                           for kv in s["kv"]])
        return {"out": out, "act_q": None, "act_d": amax(out), "act_s": None}
    if kind == "prefill":
        return {"out": _attention(s["q"], s["gate"], s["kv"], c["kv"], c["p0"] + c["B"], c["p0"], c["B"])}
    if kind == "prep":
        i = torch.arange(32, device=DEV, dtype=torch.float64)
        ang = (c["p0"] + torch.arange(c["B"], device=DEV))[:, None].double() * THETA ** (-2.0 * i / 64.0)
        cos, sin = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
        x = s["qg"].double()[..., :HD]
        x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * s["qn"].double()
        lo, hi = x[..., :32], x[..., 32:64]
        q = torch.cat([lo * cos - hi * sin, hi * cos + lo * sin, x[..., 64:]], -1)
        return {"q": q, "gate": s["qg"].double()[..., HD:], "k": None, "v": None, "ks": None, "vs": None}
    if kind == "dn":
        m, n = c["commit"], c["new"]
        cat = lambda x, y: torch.cat([x[:m], y])
        window = s["window"].double()
        o, states, x = _delta(s["p"], window[:, 0], cat(s["sqkv"], s["qkv"]), s["z"], cat(s["sb"], s["b"]),
                              cat(s["sa"], s["a"]), s["state"].double(), m)
        after = m if n > 1 else 1
        if after:
            window[:, 1] = x[:, after:after + 3]
        saved = [t[None].expand(len(s["p"]), *t.shape).double() for t in (s["qkv"], s["b"], s["a"])] if n > 1 else []
        saved = [t if i == 0 else None for i, t in enumerate(saved)]
        return {"o": o, "act_q": None, "act_d": amax(o), "act_s": None, "state": states[after],
                "window": window, "saved": saved}
    if kind == "dn_rows":
        window = s["window"].double()
        o, states, x = _delta(s["p"], window[:, 0], s["qkv"], s["z"], s["b"], s["a"], s["state"].double(), 0)
        window[:, 1] = x[:, c["B"]:]
        return {"o": o[0], "state": states[-1], "window": window}
    W = [_weight_values(fmt, w, c["K"]) for fmt, w in s["W"]]
    if kind == "gemv":
        x = (s["act"].q.view(-1, 32).double() * s["act"].d.double()[:, None]).view(c["nb"], c["K"])
        return {"y": torch.stack([x @ w.T for w in W])}
    W = [w.half() for w in W]  # the product's operands are fp16
    return {"y": torch.stack([s["X"].double() @ w.double().T for w in W]), "w16": torch.stack(W).double()}
