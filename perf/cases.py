"""The measured work of this framework: single kernels and whole calls through
the public entry points of ``arcllm_amd``, as a program that serves a packed
Q4_K/Q6_K model calls them.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges,
``prepare(case, seed)`` makes the device inputs, ``run(state)`` is one pass,
``exact(case, seed)`` the same outputs in float64 from plain torch.

Sizes are the 7B shape of the benchmark (hidden 3584, 28/4 heads of 128, ffn
18944, vocabulary 152064, 28 layers) and generic smaller ones.  Weights are
random super-blocks with the scales of the synthetic model (zero-mean rows,
standard deviation about 0.03); activations are N(0, 1), or N(0, 1) with a few
large channels as a residual stream has them.
"""
import math

import numpy as np
import torch

import arcllm_amd as arc

QK = 256
HEAD = 128
DEV = "cuda"
BLOCK = {arc.Q4_K: 144, arc.Q6_K: 210, arc.Q6_K_PADDED: 212, arc.EXEC148: 148}
EPS = 1e-6
THETA = 1e6

# 7B shape
HIDDEN, KV_HEADS, HPK, FFN, VOCAB, LAYERS = 3584, 4, 7, 18944, 152064, 28


# ------------------------------------------------------------------- cases
def listed():
    return [
        # the smallest call: one k or v projection of a token (latency and launch)
        dict(name="gemv k 512x3584", kind="gemv", qtype=arc.Q4_K, rows=512, K=3584, bias=1),
        # the FFN of one token, eight layers in turn, so the weights come from HBM as
        # they do in a model (gate/up + SwiGLU, then the split-K down + residual)
        dict(name="ffn 7B 8 layers", kind="ffn", hidden=HIDDEN, ffn=FFN, down=arc.Q6_K_PADDED, layers=8),
        # the LM head of one token: output norm, logits and argmax
        dict(name="lm head 152064", kind="lmhead", qtype=arc.Q6_K_PADDED, rows=VOCAB, K=HIDDEN),
        # cached attention of one token, a short and a long odd context
        dict(name="attention T=500", kind="attn", kv_heads=KV_HEADS, hpk=HPK, T=500),
        dict(name="attention T=4001", kind="attn", kv_heads=KV_HEADS, hpk=HPK, T=4001),
        # prompt pass, single products: the narrow q|k|v of a short ragged prompt, the
        # gate/up of a medium ragged one, gate/up and down of a full pass
        dict(name="prompt qkv M=23", kind="pf_qkv", hidden=HIDDEN, kvd=KV_HEADS * HEAD, v=arc.Q6_K_PADDED, M=23),
        dict(name="prompt gateup M=100", kind="pf_gateup", N=FFN, K=HIDDEN, M=100),
        dict(name="prompt gateup M=256", kind="pf_gateup", N=FFN, K=HIDDEN, M=256),
        dict(name="prompt down M=256", kind="pf_gemm", qtype=arc.Q6_K_PADDED, N=HIDDEN, K=FFN, M=256),
        # prompt-pass attention of a later pass of a long prompt
        dict(name="prompt attention 256@768", kind="pf_attn", kv_heads=KV_HEADS, hpk=HPK, pos0=768, M=256),
        # whole calls: greedy decode of 8 tokens, and a full 256-token prompt
        dict(name="decode 7B 8 steps @512", kind="decode", hidden=HIDDEN, kv_heads=KV_HEADS, hpk=HPK, ffn=FFN,
             vocab=VOCAB, layers=LAYERS, mixed=1, ctx=512, steps=8),
        dict(name="prompt 7B 256 tokens", kind="prompt", hidden=HIDDEN, kv_heads=KV_HEADS, hpk=HPK, ffn=FFN,
             vocab=VOCAB, layers=LAYERS, mixed=1, M=256),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _blocks(rng, lo, hi):
    """A multiple of 256 between lo and hi super-blocks, spread over the logarithm."""
    return QK * _log(rng, lo, hi)


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "ffn", "lmhead", "attn", "pf_qkv", "pf_gateup", "pf_gemm", "pf_attn", "decode",
                       "prompt"])
    if kind == "gemv":
        return dict(kind=kind, qtype=rng.choice([arc.Q4_K, arc.Q4_K, arc.Q6_K, arc.Q6_K_PADDED, arc.EXEC148]),
                    rows=_log(rng, 128, 24000), K=_blocks(rng, 2, 74), bias=rng.randint(0, 1))
    if kind == "ffn":
        return dict(kind=kind, hidden=_blocks(rng, 2, 16), ffn=_blocks(rng, 4, 74),
                    down=rng.choice([arc.Q4_K, arc.Q6_K_PADDED, arc.EXEC148]), layers=rng.randint(1, 8))
    if kind == "lmhead":
        return dict(kind=kind, qtype=rng.choice([arc.Q6_K, arc.Q6_K_PADDED]), rows=_log(rng, 4000, VOCAB),
                    K=_blocks(rng, 2, 16))
    if kind == "attn":
        return dict(kind=kind, kv_heads=rng.randint(1, 8), hpk=rng.randint(1, 8), T=_log(rng, 1, 8192))
    if kind == "pf_qkv":
        kvd = HEAD * rng.randint(1, 8)
        return dict(kind=kind, hidden=kvd * 2 * rng.randint(1, 3), kvd=kvd, v=rng.choice([arc.Q4_K, arc.Q6_K_PADDED]),
                    M=_log(rng, 2, 256))
    if kind == "pf_gateup":
        return dict(kind=kind, N=_log(rng, 1000, FFN), K=_blocks(rng, 2, 16), M=_log(rng, 2, 256))
    if kind == "pf_gemm":
        return dict(kind=kind, qtype=rng.choice([arc.Q4_K, arc.Q6_K_PADDED]), N=_log(rng, 512, 4096),
                    K=_blocks(rng, 2, 74), M=_log(rng, 2, 256))
    if kind == "pf_attn":
        return dict(kind=kind, kv_heads=rng.randint(1, 8), hpk=rng.randint(1, 8), pos0=rng.choice([0, _log(rng, 1, 3000)]),
                    M=_log(rng, 2, 256))
    kv, hpk = rng.choice([(1, 2), (2, 2), (2, 4), (2, 7), (4, 4), (4, 7), (8, 3)])
    model = dict(kind=kind, hidden=kv * hpk * HEAD, kv_heads=kv, hpk=hpk, ffn=_blocks(rng, 4, 48),
                 vocab=_log(rng, 4000, 64000), layers=rng.randint(1, 4), mixed=rng.randint(0, 1))
    if kind == "decode":
        return dict(model, ctx=_log(rng, 1, 4096), steps=rng.randint(1, 8))
    return dict(model, M=_log(rng, 2, 700))


# ------------------------------------------------------- random super-blocks
def _gen(seed, stream):
    return torch.Generator(device=DEV).manual_seed((int(seed) * 1000003 + stream * 7919 + 12345) & 0x7FFFFFFFFFFF)


def _halves(g, n, sigma):
    return (torch.randn(n, 1, generator=g, device=DEV) * sigma).abs().half().view(torch.uint8)


def _weights(g, qtype, rows, K):
    """rows x K random super-blocks, uint8 [rows * K / 256, block bytes]."""
    n = rows * (K // QK)
    w = torch.randint(0, 256, (n, BLOCK[qtype]), dtype=torch.uint8, generator=g, device=DEV)
    if qtype in (arc.Q4_K, arc.EXEC148):
        if qtype == arc.EXEC148:
            w[:, 4:20] &= 63  # unpacked 6-bit scales and mins
        w[:, 0:2] = _halves(g, n, 1e-4)
        w[:, 2:4] = _halves(g, n, 7.5e-4)
    else:
        w[:, 192:208] = torch.randint(-32, 32, (n, 16), dtype=torch.int8, generator=g, device=DEV).view(torch.uint8)
        w[:, 208:210] = _halves(g, n, 1e-4)
        w[:, 210:] = 0
    return w


def _floats(g, *shape, mean=0.0, sigma=1.0):
    return torch.randn(*shape, generator=g, device=DEV) * sigma + mean


def _residual(g, n):
    """N(0, 1) with a few channels some ten times as large, as residual streams have."""
    x = _floats(g, n)
    x[torch.randint(0, n, (max(1, n // 500),), generator=g, device=DEV)] *= 12.0
    return x


def _f64(w, qtype, rows, K):
    """The tensor's weights in float64 [rows, K]."""
    n = w.shape[0]
    half = lambda a: w[:, a:a + 2].contiguous().view(torch.float16).double()  # noqa: E731
    if qtype == arc.Q4_K:
        s = w[:, 4:16].to(torch.int32)
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        q = w[:, 16:144].reshape(n, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(n, 8, 32)
    elif qtype == arc.EXEC148:
        sc, mn = w[:, 4:20:2], w[:, 5:20:2]
        q = w[:, 20:148].reshape(n, 128, 1)
        q = torch.cat([q & 15, q >> 4], 2).reshape(n, 8, 32)
    else:
        ql, qh = w[:, 0:128].reshape(n, 2, 1, 64), w[:, 128:192].reshape(n, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2).reshape(n, 2, 4, 32)
        hi = torch.cat([(qh >> 2 * i) & 3 for i in range(4)], 2)
        q = (lo | (hi << 4)).reshape(n, 16, 16).double() - 32.0
        sc = w[:, 192:208].contiguous().view(torch.int8).double()
        return ((half(208) * sc).unsqueeze(2) * q).reshape(rows, K)
    return ((half(0) * sc.double()).unsqueeze(2) * q.double() - (half(2) * mn.double()).unsqueeze(2)).reshape(rows, K)


# ------------------------------------------------------------------- models
def _dims(c):
    d = arc.ModelDims()
    d.hidden, d.q_heads, d.kv_heads, d.head_dim = c["hidden"], c["kv_heads"] * c["hpk"], c["kv_heads"], HEAD
    d.ffn, d.vocab, d.layers, d.rms_eps, d.rope_theta = c["ffn"], c["vocab"], c["layers"], EPS, THETA
    for i in range(c["layers"]):  # Q4_K_M mixes Q6_K and Q4_K over attn_v and ffn_down
        d.v_type[i] = d.down_type[i] = arc.Q4_K if c["mixed"] and i % 2 else arc.Q6_K
    return d


def _slot(c, seed, layer, which, info):
    """One tensor of the model, on the GPU."""
    qtype, rows, K, nbytes = info
    g = _gen(seed, 100 + 16 * layer + which if layer >= 0 else which)
    if qtype:
        return _weights(g, qtype, rows, K)
    norm = which in (arc.T_ATTN_NORM, arc.T_FFN_NORM) if layer >= 0 else True
    return _floats(g, nbytes // 4, mean=1.0, sigma=0.05) if norm else _floats(g, nbytes // 4, sigma=0.1)


class _Cache:
    """A session's K or V cache as the buffer [layers, max_ctx, kv_dim] that it is.  Tensors made
    from it hold it, and it holds the session, so the memory lives as long as they do."""

    def __init__(self, session, base, stride, layers, max_ctx, kvd):
        self.session = session
        self.__cuda_array_interface__ = dict(shape=(layers, max_ctx, kvd), typestr="<f2", data=(base, False), version=2,
                                             strides=(stride, kvd * 2, 2))


def _model(c, seed, max_ctx):
    d = _dims(c)
    host = []
    for layer, which in arc.model_slots(d):
        t = _slot(c, seed, layer, which, arc.tensor_info(d, layer, which))
        host.append(t.cpu().numpy().reshape(-1))
    model = arc.Model(d, host)
    session = arc.Session(model, max_ctx)
    kvd, (k0, v0) = c["kv_heads"] * HEAD, session.kv(0)
    stride = session.kv(1)[0] - k0 if c["layers"] > 1 else max_ctx * kvd * 2
    views = [torch.as_tensor(_Cache(session, p, stride, c["layers"], max_ctx, kvd), device=DEV) for p in (k0, v0)]
    return model, session, views


def _context(c, seed):
    """The cached K and V of the positions before the first decoded one."""
    shape = (c["layers"], c["ctx"], c["kv_heads"] * HEAD)
    return [_floats(_gen(seed, 50 + i), *shape).half() for i in (0, 1)]


def _tokens(c, seed):
    n = c.get("M", 1)
    return torch.randint(0, c["vocab"], (n,), generator=_gen(seed, 60), device=DEV).cpu().numpy().astype(np.uint32)


# ------------------------------------------------------------------ prepare
def prepare(case, seed):
    c, g, e = case, _gen(seed, 0), {}
    kind = c["kind"]
    if kind == "gemv":
        e = dict(w=_weights(g, c["qtype"], c["rows"], c["K"]), x=_floats(g, c["K"]),
                 bias=_floats(g, c["rows"], sigma=0.1) if c["bias"] else None, y=torch.empty(c["rows"], device=DEV))
    elif kind == "ffn":
        H, F = c["hidden"], c["ffn"]
        e = dict(layers=[dict(gate=_weights(g, arc.Q4_K, F, H), up=_weights(g, arc.Q4_K, F, H),
                              down=_weights(g, c["down"], H, F), h=_residual(g, H), s=torch.empty(F, device=DEV),
                              y=torch.empty(H, device=DEV)) for _ in range(c["layers"])],
                 x=_floats(g, H), part=torch.empty(H * (F // QK), device=DEV))
    elif kind == "lmhead":
        e = dict(w=_weights(g, c["qtype"], c["rows"], c["K"]), h=_residual(g, c["K"]),
                 norm=_floats(g, c["K"], mean=1.0, sigma=0.05), logits=torch.empty(c["rows"], device=DEV),
                 ws=torch.empty(arc.lmhead_workspace_bytes(c["qtype"], c["rows"], c["K"]), dtype=torch.uint8, device=DEV),
                 out=torch.empty(2, dtype=torch.int32, device=DEV))
    elif kind in ("attn", "pf_attn"):
        kvh, hpk = c["kv_heads"], c["hpk"]
        rows, ctx = c.get("M", 1), c["T"] if kind == "attn" else c["pos0"] + c["M"]
        e = dict(ctx=ctx, q=_floats(g, rows, kvh * hpk * HEAD), k=_floats(g, ctx, kvh * HEAD).half(),
                 v=_floats(g, ctx, kvh * HEAD).half())
        if kind == "attn":
            e.update(out=torch.empty(kvh * hpk * HEAD, device=DEV),
                     ws=torch.empty(arc.attention_workspace_bytes(kvh, hpk), dtype=torch.uint8, device=DEV))
        else:
            e.update(out=torch.empty(rows, kvh * hpk * HEAD, dtype=torch.float16, device=DEV))
    elif kind == "pf_gemm":
        e = dict(w=_weights(g, c["qtype"], c["N"], c["K"]), x=_floats(g, c["M"], c["K"]).half(),
                 y=torch.empty(c["M"], c["N"], device=DEV),
                 ws=torch.empty(arc.prefill_gemm_workspace_bytes(c["N"], c["K"]), dtype=torch.uint8, device=DEV))
    elif kind == "pf_gateup":
        e = dict(gate=_weights(g, arc.Q4_K, c["N"], c["K"]), up=_weights(g, arc.Q4_K, c["N"], c["K"]),
                 x=_floats(g, c["M"], c["K"]).half(), s=torch.empty(c["M"], c["N"], dtype=torch.float16, device=DEV),
                 ws=torch.empty(arc.prefill_gemm_workspace_bytes(c["N"], c["K"]), dtype=torch.uint8, device=DEV))
    elif kind == "pf_qkv":
        H, kvd = c["hidden"], c["kvd"]
        e = dict(q=_weights(g, arc.Q4_K, H, H), k=_weights(g, arc.Q4_K, kvd, H), v=_weights(g, c["v"], kvd, H),
                 x=_floats(g, c["M"], H).half(), y=torch.empty(c["M"], H + 2 * kvd, device=DEV),
                 ws=torch.empty(arc.prefill_gemm_workspace_bytes(H + 2 * kvd, H), dtype=torch.uint8, device=DEV))
    elif kind == "decode":
        max_ctx = c["ctx"] + c["steps"]
        model, session, views = _model(c, seed, max_ctx)
        for view, past in zip(views, _context(c, seed)):
            view[:, : c["ctx"]] = past
        e = dict(model=model, session=session, views=views, token=int(_tokens(c, seed)[0]))
    else:
        model, session, views = _model(c, seed, c["M"])
        e = dict(model=model, session=session, views=views, tokens=_tokens(c, seed))
    return dict(e, c=c)


# ---------------------------------------------------------------------- run
def run(state):
    e, c = state, state["c"]
    kind = c["kind"]
    p = torch.Tensor.data_ptr
    if kind == "gemv":
        arc.gemv(c["qtype"], p(e["w"]), c["rows"], c["K"], p(e["x"]), p(e["y"]),
                 bias=None if e["bias"] is None else p(e["bias"]))
        return e["y"]
    if kind == "ffn":
        H, F = c["hidden"], c["ffn"]
        for la in e["layers"]:
            arc.gateup_swiglu(arc.Q4_K, p(la["gate"]), p(la["up"]), F, H, p(e["x"]), p(la["s"]))
            arc.gemv_splitk(c["down"], p(la["down"]), H, F, F // QK, p(la["s"]), p(e["part"]), p(la["y"]),
                            residual=p(la["h"]))
        return [t for la in e["layers"] for t in (la["s"], la["y"])]
    if kind == "lmhead":
        arc.lmhead_argmax(c["qtype"], p(e["w"]), c["rows"], c["K"], p(e["h"]), p(e["norm"]), EPS, p(e["logits"]),
                          p(e["ws"]), p(e["out"]))
        return dict(logits=e["logits"], token=e["out"])
    if kind == "attn":
        arc.attention_decode(p(e["q"]), p(e["k"]), p(e["v"]), c["kv_heads"], c["hpk"], e["ctx"], c["T"], p(e["out"]),
                             p(e["ws"]))
        return e["out"]
    if kind == "pf_attn":
        arc.prefill_attention(p(e["q"]), p(e["k"]), p(e["v"]), c["kv_heads"], c["hpk"], e["ctx"], c["pos0"], c["M"],
                              p(e["out"]), c["kv_heads"] * c["hpk"] * HEAD)
        return e["out"]
    if kind == "pf_gemm":
        arc.prefill_gemm(c["qtype"], p(e["w"]), c["N"], c["K"], p(e["x"]), c["M"], p(e["y"]), p(e["ws"]))
        return e["y"]
    if kind == "pf_gateup":
        arc.prefill_gateup(p(e["gate"]), p(e["up"]), c["N"], c["K"], p(e["x"]), c["M"], p(e["s"]), p(e["ws"]))
        return e["s"]
    if kind == "pf_qkv":
        arc.prefill_qkv(p(e["q"]), p(e["k"]), p(e["v"]), c["v"], c["hidden"], c["kvd"], c["hidden"], p(e["x"]), c["M"],
                        p(e["y"]), p(e["ws"]))
        return e["y"]
    # the calls of a session are synchronous and hand tokens and logits to the host
    if kind == "decode":
        tokens, _ = e["session"].decode(e["token"], c["ctx"], c["steps"], logits=True)
        rows = slice(c["ctx"], c["ctx"] + c["steps"])
        return dict(logits=e["session"].logits(), tokens=tokens.astype(np.int64), k=e["views"][0][:, rows],
                    v=e["views"][1][:, rows])
    token, _ = e["session"].prefill(e["tokens"], 0, logits=True)
    return dict(logits=e["session"].logits(), k=e["views"][0], v=e["views"][1])


# --------------------------------------------------------------------- work
def _bytes(qtype, rows, K):
    """Packed bytes as GGUF holds them (a padded Q6_K block counts its 210)."""
    return rows * (K // QK) * {arc.Q6_K_PADDED: 210}.get(qtype, BLOCK[qtype])


def work(case):
    c, kind = case, case["kind"]
    if kind == "gemv":
        return dict(bytes=_bytes(c["qtype"], c["rows"], c["K"]) + 4 * (c["K"] + c["rows"] * (1 + c["bias"])),
                    flops=2.0 * c["rows"] * c["K"])
    if kind == "ffn":
        H, F = c["hidden"], c["ffn"]
        return dict(bytes=c["layers"] * (2 * _bytes(arc.Q4_K, F, H) + _bytes(c["down"], H, F) + 8 * F + 12 * H),
                    flops=c["layers"] * 6.0 * H * F)
    if kind == "lmhead":
        return dict(bytes=_bytes(c["qtype"], c["rows"], c["K"]) + 8 * c["K"] + 4 * c["rows"],
                    flops=2.0 * c["rows"] * c["K"])
    if kind == "attn":
        return dict(bytes=c["kv_heads"] * HEAD * (4 * c["T"] + 8 * c["hpk"]),
                    flops=4.0 * c["kv_heads"] * c["hpk"] * HEAD * c["T"])
    if kind == "pf_attn":
        keys = c["M"] * c["pos0"] + c["M"] * (c["M"] + 1) // 2
        return dict(bytes=c["kv_heads"] * HEAD * (4 * (c["pos0"] + c["M"]) + 6 * c["hpk"] * c["M"]),
                    flops=4.0 * c["kv_heads"] * c["hpk"] * HEAD * keys)
    if kind == "pf_gemm":
        return dict(bytes=_bytes(c["qtype"], c["N"], c["K"]) + c["M"] * (2 * c["K"] + 4 * c["N"]),
                    flops=2.0 * c["M"] * c["N"] * c["K"])
    if kind == "pf_gateup":
        return dict(bytes=2 * _bytes(arc.Q4_K, c["N"], c["K"]) + 2 * c["M"] * (c["K"] + c["N"]),
                    flops=4.0 * c["M"] * c["N"] * c["K"])
    if kind == "pf_qkv":
        H, kvd = c["hidden"], c["kvd"]
        return dict(bytes=_bytes(arc.Q4_K, H + kvd, H) + _bytes(c["v"], kvd, H) + c["M"] * (2 * H + 4 * (H + 2 * kvd)),
                    flops=2.0 * c["M"] * H * (H + 2 * kvd))
    H, F, kvd, L = c["hidden"], c["ffn"], c["kv_heads"] * HEAD, c["layers"]
    d = _dims(c)
    layer = sum(2 * _bytes(arc.Q4_K, H, H) + _bytes(arc.Q4_K, kvd, H) + _bytes(d.v_type[i], kvd, H)
                + 2 * _bytes(arc.Q4_K, F, H) + _bytes(d.down_type[i], H, F) for i in range(L))
    head = _bytes(arc.Q6_K, c["vocab"], H)
    per = L * (2 * H * H + 2 * H * kvd + 3 * H * F)  # weights multiplied for one position
    if kind == "decode":
        past = sum(c["ctx"] + i + 1 for i in range(c["steps"]))
        return dict(bytes=c["steps"] * (layer + head) + 4 * L * kvd * past + 4 * c["vocab"],
                    flops=2.0 * c["steps"] * (per + c["vocab"] * H) + 4.0 * L * H * past)
    return dict(bytes=layer + head + 4 * L * kvd * c["M"] + 4 * c["vocab"],
                flops=2.0 * (c["M"] * per + c["vocab"] * H) + 4.0 * L * H * (c["M"] * (c["M"] + 1) // 2))


# ---------------------------------------------------------------- tolerance
def tolerance(case):
    kind = case["kind"]
    # About four times the error against exact() (in brackets, 2-norm).
    # fp32 sums of exact products (2e-7 .. 3.4e-7)
    if kind in ("gemv", "ffn", "lmhead", "attn"):
        return dict(rel=1.5e-6, max=2e-5, differ=0.0)
    # fp16 results of fp32 arithmetic (2.1e-4); fp16 operands, each weight rounded
    # once (2.1e-4), and a product of two such with an fp16 result (3.6e-4)
    if kind in ("pf_attn", "pf_gemm", "pf_qkv"):
        return dict(rel=8e-4, max=1e-2)
    if kind == "pf_gateup":
        return dict(rel=1.5e-3, max=2e-2)
    # whole calls: one layer's rounding (fp16 cache rows; fp16 operands in the prompt
    # pass) travels through the layers that follow (28 layers: 2.3e-3, 3.8e-2)
    if kind == "decode":
        return dict(rel=8e-3, max=0.1)
    return dict(rel=0.03, max=0.5)


# -------------------------------------------------------------------- exact
def _silu(x):
    return x / (1.0 + torch.exp(-x))


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, pos0):
    """Adjacent pairs of each head of x [M, heads, 128], rows at pos0, pos0 + 1, ..."""
    f = THETA ** (-torch.arange(0, HEAD, 2, dtype=torch.float64, device=DEV) / HEAD)
    a = (pos0 + torch.arange(x.shape[0], dtype=torch.float64, device=DEV))[:, None] * f
    co, si = torch.cos(a)[:, None], torch.sin(a)[:, None]
    return torch.stack([x[..., ::2] * co - x[..., 1::2] * si, x[..., ::2] * si + x[..., 1::2] * co], -1).flatten(-2)


def _attention(q, k, v, kv_heads, hpk, pos0):
    """q [M, heads*128] at positions pos0.. over k, v [ctx, kv*128], causal; one kv head at a time."""
    M, ctx = q.shape[0], k.shape[0]
    q, out = q.double().reshape(M, kv_heads, hpk, HEAD), []
    mask = torch.arange(ctx, device=DEV) > pos0 + torch.arange(M, device=DEV)[:, None]
    for j in range(kv_heads):
        kj, vj = (t.double()[:, j * HEAD:(j + 1) * HEAD] for t in (k, v))
        s = (q[:, j].reshape(M * hpk, HEAD) @ kj.t().contiguous() / math.sqrt(HEAD)).reshape(M, hpk, ctx)
        s = torch.softmax(s.masked_fill(mask[:, None], -math.inf), -1)
        out.append((s.reshape(M * hpk, ctx) @ vj.contiguous()).reshape(M, hpk * HEAD))
    return torch.cat(out, 1)


def _mul(x, w, qtype, rows, K):
    """x [M, K] times the tensor's transpose in float64, some rows at a time."""
    out, step, nb = [], max(1, (1 << 26) // K), K // QK
    for r in range(0, rows, step):
        n = min(step, rows - r)
        out.append((_f64(w[r * nb:(r + n) * nb], qtype, n, K) @ x.t().contiguous()).t())
    return torch.cat(out, 1)


def _forward(c, seed, h, pos0, past):
    """Rows h [M, hidden] through the layers at positions pos0..; past holds (k, v) per layer and grows."""
    d, H, kvd = _dims(c), c["hidden"], c["kv_heads"] * HEAD
    for i in range(c["layers"]):
        t = {w: _slot(c, seed, i, w, arc.tensor_info(d, i, w)) for w in range(arc.T_LAYER_COUNT)}

        def mul(x, w):
            qtype, rows, K, _ = arc.tensor_info(d, i, w)
            return _mul(x, t[w], qtype, rows, K)

        x, m = _rms(h, t[arc.T_ATTN_NORM]), h.shape[0]
        q = _rope((mul(x, arc.T_ATTN_Q) + t[arc.T_ATTN_Q_BIAS].double()).reshape(m, -1, HEAD), pos0).reshape(m, H)
        k = _rope((mul(x, arc.T_ATTN_K) + t[arc.T_ATTN_K_BIAS].double()).reshape(m, -1, HEAD), pos0).reshape(m, kvd)
        v = mul(x, arc.T_ATTN_V) + t[arc.T_ATTN_V_BIAS].double()
        past[i] = [torch.cat([a.double(), b]) for a, b in zip(past[i], (k, v))]
        h = h + mul(_attention(q, past[i][0], past[i][1], c["kv_heads"], c["hpk"], pos0), arc.T_ATTN_O)
        x = _rms(h, t[arc.T_FFN_NORM])
        h = h + mul(_silu(mul(x, arc.T_FFN_GATE)) * mul(x, arc.T_FFN_UP), arc.T_FFN_DOWN)
    return h


def _exact_model(c, seed):
    d, H, V = _dims(c), c["hidden"], c["vocab"]
    emb, out, norm = (_slot(c, seed, -1, w, arc.tensor_info(d, -1, w))
                      for w in (arc.T_TOKEN_EMBD, arc.T_OUTPUT, arc.T_OUTPUT_NORM))
    nb = H // QK

    def embed(tokens):
        return torch.cat([_f64(emb[int(t) * nb:(int(t) + 1) * nb], arc.Q4_K, 1, H) for t in tokens])

    def logits(h):
        return _mul(_rms(h[-1:], norm), out, arc.Q6_K, V, H)[0]

    if c["kind"] == "prompt":
        none = torch.empty(0, c["kv_heads"] * HEAD, device=DEV)
        past = [[none, none] for _ in range(c["layers"])]
        lg = logits(_forward(c, seed, embed(_tokens(c, seed)), 0, past))
        return dict(logits=lg.cpu().numpy(), k=torch.stack([a for a, _ in past]), v=torch.stack([b for _, b in past]))
    ks, vs = _context(c, seed)
    past = [[ks[i], vs[i]] for i in range(c["layers"])]
    tokens = [int(_tokens(c, seed)[0])]
    for i in range(c["steps"]):
        lg = logits(_forward(c, seed, embed(tokens[-1:]), c["ctx"] + i, past))
        tokens.append(int(lg.argmax()))
    return dict(logits=lg.cpu().numpy(), tokens=np.array(tokens[1:], np.int64),
                k=torch.stack([a[c["ctx"]:] for a, _ in past]), v=torch.stack([b[c["ctx"]:] for _, b in past]))


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("decode", "prompt"):
        return _exact_model(c, seed)
    e = prepare(case, seed)
    if kind == "gemv":
        y = _mul(e["x"].double()[None], e["w"], c["qtype"], c["rows"], c["K"])[0]
        return y if e["bias"] is None else y + e["bias"].double()
    if kind == "ffn":
        H, F, got = c["hidden"], c["ffn"], []
        for la in e["layers"]:
            x = e["x"].double()[None]
            s = _silu(_mul(x, la["gate"], arc.Q4_K, F, H)) * _mul(x, la["up"], arc.Q4_K, F, H)
            got += [s[0], _mul(s, la["down"], c["down"], H, F)[0] + la["h"].double()]
        return got
    if kind == "lmhead":
        lg = _mul(_rms(e["h"].double(), e["norm"])[None], e["w"], c["qtype"], c["rows"], c["K"])[0]
        return dict(logits=lg, token=None)
    if kind in ("attn", "pf_attn"):
        o = _attention(e["q"], e["k"], e["v"], c["kv_heads"], c["hpk"], c["T"] - 1 if kind == "attn" else c["pos0"])
        return o[0] if kind == "attn" else o
    x = e["x"].double()
    if kind == "pf_gemm":
        return _mul(x, e["w"], c["qtype"], c["N"], c["K"])
    if kind == "pf_gateup":
        return _silu(_mul(x, e["gate"], arc.Q4_K, c["N"], c["K"])) * _mul(x, e["up"], arc.Q4_K, c["N"], c["K"])
    H, kvd = c["hidden"], c["kvd"]
    return torch.cat([_mul(x, e["q"], arc.Q4_K, H, H), _mul(x, e["k"], arc.Q4_K, kvd, H),
                      _mul(x, e["v"], c["v"], kvd, H)], 1)
