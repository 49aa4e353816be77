"""Performance cases of the framework, through its public entry points.

Each case is one call (or one short session) that a program using the
framework makes: the attention operators of one layer (prefill, chunked
prefill, decode, the fused norm/RoPE/KV write), the decode GEMV blocks over
f16 and GGUF-block weights, and engine sessions (prompt, further prompt
chunks, decode steps).  Sizes are those of the Qwen3 models that the tests and
the benchmark run; drawn cases spread over the same ranges.

A case is a dict of plain values; ``kind`` selects how it is prepared and run.
``exact`` restates each kind in float64 torch without the framework's code.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from grout_amd import ops
from grout_amd._lib import call, lib
from grout_amd.model import Engine, QuantWeights, Qwen3Config, Qwen3Weights

D = 128
EPS = 1e-6
THETA = 1e6
F16, Q8_0, Q4_K, Q5_K, Q6_K = 0, 8, 12, 13, 14
BLOCK = {Q8_0: (32, 34), Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210)}  # weights, bytes
# bytes of one weight as stored
WBYTES = {F16: 2.0, Q8_0: 34 / 32, Q4_K: 144 / 256, Q5_K: 176 / 256, Q6_K: 210 / 256}

# Qwen3 layer shapes: hidden, intermediate, query heads, kv heads, layers
MODELS = {
    "0.6b": (1024, 3072, 16, 8, 28),
    "1.7b": (2048, 6144, 16, 8, 28),
    "4b": (2560, 9728, 32, 8, 36),
    "8b": (4096, 12288, 32, 8, 36),
    "14b": (5120, 17408, 40, 8, 40),
    "32b": (5120, 25600, 64, 8, 64),
}
VOCAB = 151936
SMALL_VOCAB = 32000  # sessions over a few layers: the head stays a small part


def listed():
    return [
        # one layer's decode attention of a chat at ~640 positions: raw QKV
        # row to attention output, the smallest call of the decode loop
        dict(name="decode_layer_4b_641", kind="decode_layer", model="4b", ctx=641, max_ctx=4096),
        # one layer's decode attention at a long context (split pass + merge)
        dict(name="decode_attn_32b_32k", kind="decode_attn", model="32b", ctx=32768,
             max_ctx=32768),
        # norm + RoPE + cache write of a 2048-token prompt
        dict(name="kv_write_4b_2048", kind="kv_write", model="4b", seq=2048, pos0=0,
             max_ctx=4096),
        # causal attention of a 2048-token prompt, and of a long one at the
        # largest head count
        dict(name="prefill_attn_4b_2048", kind="prefill_attn", model="4b", seq=2048, pos0=0,
             max_ctx=4096),
        dict(name="prefill_attn_32b_8192", kind="prefill_attn", model="32b", seq=8192, pos0=0,
             max_ctx=8192),
        # the next user turn of a long chat: a short ragged chunk whose rows
        # attend to 8k cached positions
        dict(name="extend_attn_4b_61_at_8131", kind="prefill_attn", model="4b", seq=61,
             pos0=8131, max_ctx=16384),
        # MLP block of one decode step, f16 weights and the Q4_K_M mix
        dict(name="mlp_step_4b_f16", kind="mlp_step", model="4b", gate_up=F16, down=F16),
        dict(name="mlp_step_4b_q4km", kind="mlp_step", model="4b", gate_up=Q4_K, down=Q6_K),
        # final norm + vocabulary projection of one decode step (Q6_K head)
        dict(name="head_step_4b_q6k", kind="head_step", model="4b", vocab=VOCAB, fmt=Q6_K),
        # a few layers over a 512-token prompt: projections, norms, attention
        dict(name="prompt_layers_4b_512", kind="session", model="4b", layers=4, vocab=SMALL_VOCAB,
             mix="f16", prompt=512, extend=0, decode=0, max_ctx=1024),
        # whole requests: a short question (18 prompt tokens) in f16, and a
        # chat over Q4_K_M weights: prompt, a second turn, decode steps
        dict(name="request_4b_f16", kind="session", model="4b", layers=36, vocab=VOCAB, mix="f16",
             prompt=18, extend=0, decode=8, max_ctx=1024),
        dict(name="request_4b_q4km", kind="session", model="4b", layers=36, vocab=VOCAB,
             mix="q4km", prompt=131, extend=23, decode=8, max_ctx=1024),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _ctx_for(n):
    return next(c for c in (1024, 4096, 8192, 16384, 32768, 40960) if c >= n)


def draw(rng):
    kind = rng.choice(["decode_layer", "decode_attn", "kv_write", "prefill_attn", "prefill_attn",
                       "mlp_step", "mlp_step", "head_step", "session", "session", "session"])
    model = rng.choice(list(MODELS))
    if kind in ("decode_layer", "decode_attn"):
        ctx = _log_int(rng, 1, 32768)
        return dict(kind=kind, model=model, ctx=ctx, max_ctx=_ctx_for(rng.choice([ctx, 4 * ctx])
                                                                      if ctx < 8192 else ctx))
    if kind in ("kv_write", "prefill_attn"):
        seq = _log_int(rng, 1, 6000)
        pos0 = rng.choice([0, 0, _log_int(rng, 1, 16000)])
        return dict(kind=kind, model=model, seq=seq, pos0=pos0, max_ctx=_ctx_for(seq + pos0))
    fmts = [F16, Q8_0, Q4_K, Q5_K, Q6_K]
    if kind == "mlp_step":
        return dict(kind=kind, model=model, gate_up=rng.choice(fmts), down=rng.choice(fmts))
    if kind == "head_step":
        return dict(kind=kind, model=model, vocab=rng.choice([SMALL_VOCAB, VOCAB]),
                    fmt=rng.choice(fmts))
    mix = rng.choice(["f16", "f16", "q4km", "q5km", "q8"])
    prompt, extend = _log_int(rng, 1, 1500), rng.choice([0, _log_int(rng, 1, 200)])
    return dict(kind=kind, model=model, layers=2, vocab=SMALL_VOCAB, mix=mix, prompt=prompt,
                extend=extend, decode=rng.choice([0, 2]), max_ctx=4096)


# ---------------------------------------------------------------- inputs


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, *shape, std=1.0):
    return torch.empty(shape, dtype=torch.float16, device="cuda").normal_(0.0, std, generator=g)


def _gamma(g, n):
    return torch.empty(n, dtype=torch.float16, device="cuda").uniform_(0.8, 1.2, generator=g)


def _blocks(g, fmt, rows, k, std=0.02):
    """Random ggml blocks whose weights spread about std (payload bytes and
    6-bit scales uniform, dmin centring the Q4_K / Q5_K weights); f16 rows for
    F16."""
    if fmt == F16:
        return _normal(g, rows, k, std=std)
    be, bb = BLOCK[fmt]
    b = torch.randint(0, 256, (rows * (k // be), bb), dtype=torch.uint8, device="cuda",
                      generator=g)

    def put(col, v):
        b[:, col:col + 2] = torch.tensor([v], dtype=torch.float16).view(torch.uint8).cuda()

    if fmt == Q8_0:
        put(0, std / 74.0)
    elif fmt == Q4_K:
        put(0, std / (32.0 * 4.6))
        put(2, 7.5 * std / (32.0 * 4.6))
    elif fmt == Q5_K:
        put(0, std / (32.0 * 9.2))
        put(2, 15.5 * std / (32.0 * 9.2))
    else:
        put(208, std / (74.0 * 18.5))
    return b.reshape(rows, -1)


def _attn_inputs(case, seed):
    """Caches of one layer and what its kind of call takes beside them."""
    _, _, hq, hkv, _ = MODELS[case["model"]]
    g = _gen(seed)
    kc, vc = _normal(g, hkv, case["max_ctx"], D), _normal(g, hkv, case["max_ctx"], D)
    kind = case["kind"]
    if kind == "decode_attn":
        return dict(q=_normal(g, hq, D), k_cache=kc, v_cache=vc)
    if kind == "prefill_attn":
        return dict(q=_normal(g, case["seq"], hq, D), k_cache=kc, v_cache=vc)
    norms = dict(q_norm=_gamma(g, D), k_norm=_gamma(g, D), k_cache=kc, v_cache=vc)
    if kind == "decode_layer":
        return dict(qkv=_normal(g, (hq + 2 * hkv) * D), **norms)
    s = case["seq"]
    return dict(q=_normal(g, s, hq, D), k=_normal(g, s, hkv, D), v=_normal(g, s, hkv, D), **norms)


def _gemv_inputs(case, seed):
    h, inter = MODELS[case["model"]][:2]
    g = _gen(seed)
    d = dict(x=_normal(g, h), residual=_normal(g, h), gamma=_gamma(g, h))
    if case["kind"] == "mlp_step":
        d["gate_up"] = _blocks(g, case["gate_up"], 2 * inter, h)
        d["down"] = _blocks(g, case["down"], h, inter)
    else:
        d["head"] = _blocks(g, case["fmt"], case["vocab"], h)
    return d


def _mix(case, layer):
    """(q, k, o, gate, up | v, down) formats of a layer: one format, or the
    Q4_K_M / Q5_K_M mixes (v and down in Q6_K for some layers)."""
    n, mix = case["layers"], case["mix"]
    if mix in ("f16", "q8"):
        return (F16, F16) if mix == "f16" else (Q8_0, Q8_0)
    base = Q4_K if mix == "q4km" else Q5_K
    more = layer < n // 8 or layer >= 7 * n // 8 or (layer - n // 8) % 3 == 2
    return base, (Q6_K if more else base)


def _embed_fmt(case):
    return {"f16": F16, "q8": Q8_0}.get(case["mix"], Q6_K)


def _session_layer(case, g, layer):
    """One layer's weights as ggml blocks or f16, in the checkpoint's matrices."""
    h, inter, hq, hkv, _ = MODELS[case["model"]]
    base, hi = _mix(case, layer)
    return {
        "input_layernorm": _gamma(g, h), "q_norm": _gamma(g, D), "k_norm": _gamma(g, D),
        "post_attention_layernorm": _gamma(g, h),
        "q_proj": (base, _blocks(g, base, hq * D, h)),
        "k_proj": (base, _blocks(g, base, hkv * D, h)),
        "v_proj": (hi, _blocks(g, hi, hkv * D, h)),
        "o_proj": (base, _blocks(g, base, h, hq * D)),
        "gate_proj": (base, _blocks(g, base, inter, h)),
        "up_proj": (base, _blocks(g, base, inter, h)),
        "down_proj": (hi, _blocks(g, hi, h, inter)),
    }


def _session_ends(case, g):
    h = MODELS[case["model"]][0]
    f = _embed_fmt(case)
    return (f, _blocks(g, f, case["vocab"], h)), _gamma(g, h)


def _session_tokens(case, seed):
    rng = np.random.default_rng(seed)
    n = case["prompt"] + case["extend"] + case["decode"]
    return rng.integers(0, case["vocab"], n).astype(np.int64)


def _session_config(case):
    h, inter, hq, hkv, _ = MODELS[case["model"]]
    return Qwen3Config(case["layers"], h, inter, hq, hkv, case["vocab"], rms_norm_eps=EPS,
                       rope_theta=THETA, tie_word_embeddings=True)


# ---------------------------------------------------------------- prepare


def _p(t):
    return C.c_void_p(t.data_ptr())


def _repacked(fmt, blocks, rows, k):
    """The weights as a program keeps them: f16 rows, or the decode layout."""
    if fmt == F16:
        return blocks
    out = torch.empty(lib().grout_qweight_bytes(fmt, rows, k), dtype=torch.uint8, device="cuda")
    call("grout_qweight_repack", fmt, _p(blocks), rows, k, _p(out),
         C.c_void_p(torch.cuda.current_stream().cuda_stream))
    return out


def _step_calls(st):
    """The step's calls (name, arguments before the stream), as a program that
    keeps its buffers would hold them."""
    case, h, inter = st["case"], st["h"], st["inter"]
    x, res, gam, ro, y = (_p(st[k]) for k in ("x", "residual", "gamma", "residual_out", "y"))
    if case["kind"] == "mlp_step":
        gu, dn, ff = _p(st["gate_up"]), _p(st["down"]), _p(st["ff"])
        f, d = case["gate_up"], case["down"]
        first = (("grout_gemv_rms_norm_silu_mul",) if f == F16 else
                 ("grout_gemv_q_rms_norm_silu_mul", f)) + (gu, res, x, gam, ro, ff, inter, h, EPS)
        second = (("grout_gemv",) if d == F16 else ("grout_gemv_q", d)) + (dn, ff, y, h, inter)
    else:
        nx, f = _p(st["normed"]), case["fmt"]
        first = ("grout_add_rms_norm", res, x, gam, nx, ro, 1, h, EPS)
        second = (("grout_gemv",) if f == F16 else ("grout_gemv_q", f)) + (
            _p(st["head"]), nx, y, case["vocab"], h)
    return first, second


def prepare(case, seed):
    kind = case["kind"]
    h, inter, hq, hkv, _ = MODELS[case["model"]]
    if kind in ("decode_layer", "decode_attn", "kv_write", "prefill_attn"):
        st = dict(case=case, hq=hq, **_attn_inputs(case, seed))
        if kind in ("decode_layer", "kv_write"):
            st["rope"] = ops.rope_tables(case["max_ctx"], D, THETA, "cuda")
        if kind in ("decode_layer", "decode_attn"):
            st["position"] = torch.tensor([case["ctx"] - 1], dtype=torch.int32, device="cuda")
            st["splits"] = ops.default_splits(case["max_ctx"], hq, hkv)
            st["workspace"] = ops.decode_workspace(hq, hkv, st["splits"], "cuda")
            st["out"] = torch.empty((hq, D), dtype=torch.float16, device="cuda")
        else:
            st["out"] = torch.empty_like(st["q"])
        return st
    if kind in ("mlp_step", "head_step"):
        st = dict(case=case, h=h, inter=inter, **_gemv_inputs(case, seed))
        if kind == "mlp_step":
            st["gate_up"] = _repacked(case["gate_up"], st["gate_up"], 2 * inter, h)
            st["down"] = _repacked(case["down"], st["down"], h, inter)
            st["ff"] = torch.empty(inter, dtype=torch.float16, device="cuda")
            st["y"] = torch.empty(h, dtype=torch.float16, device="cuda")
        else:
            st["head"] = _repacked(case["fmt"], st["head"], case["vocab"], h)
            st["normed"] = torch.empty(h, dtype=torch.float16, device="cuda")
            st["y"] = torch.empty(case["vocab"], dtype=torch.float16, device="cuda")
        st["residual_out"] = torch.empty(h, dtype=torch.float16, device="cuda")
        st["calls"] = _step_calls(st)
        return st
    # session
    cfg, g = _session_config(case), _gen(seed)
    layers = [_session_layer(case, g, l) for l in range(case["layers"])]
    (ef, embed), norm = _session_ends(case, g)
    if case["mix"] == "f16":
        fused = [{
            "input_layernorm": L["input_layernorm"], "q_norm": L["q_norm"],
            "k_norm": L["k_norm"],
            "post_attention_layernorm": L["post_attention_layernorm"],
            "qkv_proj": torch.cat([L[k][1] for k in ("q_proj", "k_proj", "v_proj")]),
            "o_proj": L["o_proj"][1],
            "gate_up_proj": torch.cat([L[k][1] for k in ("gate_proj", "up_proj")]),
            "down_proj": L["down_proj"][1],
        } for L in layers]
        del layers
        torch.cuda.synchronize()
        eng = Engine(cfg, Qwen3Weights(embed, norm, fused), max_ctx=case["max_ctx"])
    else:
        qw = QuantWeights(cfg, (ef, embed), norm, layers)
        torch.cuda.synchronize()
        eng = Engine.from_quantized(cfg, qw, max_ctx=case["max_ctx"])
    return dict(case=case, engine=eng, tokens=_session_tokens(case, seed))


# ---------------------------------------------------------------- run


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "decode_layer":
        out = ops.attn_decode_fused(state["qkv"], state["q_norm"], state["k_norm"], state["rope"],
                                    state["k_cache"], state["v_cache"], state["position"],
                                    state["hq"], num_splits=state["splits"], out=state["out"],
                                    workspace=state["workspace"], eps=EPS)
        return dict(out=out, k_cache=state["k_cache"], v_cache=state["v_cache"])
    if kind == "decode_attn":
        return ops.attn_decode(state["q"], state["k_cache"], state["v_cache"], state["position"],
                               num_splits=state["splits"], out=state["out"],
                               workspace=state["workspace"])
    if kind == "kv_write":
        out = ops.qk_norm_rope_kv_prefill(state["q"], state["k"], state["v"], state["q_norm"],
                                          state["k_norm"], state["rope"], state["k_cache"],
                                          state["v_cache"], case["pos0"], EPS, out=state["out"])
        return dict(out=out, k_cache=state["k_cache"], v_cache=state["v_cache"])
    if kind == "prefill_attn":
        return ops.fmha_prefill(state["q"], state["k_cache"], state["v_cache"], case["pos0"],
                                out=state["out"])
    if kind in ("mlp_step", "head_step"):
        s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        for args in state["calls"]:
            call(*args, s)
        return dict(y=state["y"], residual_out=state["residual_out"])
    eng, t = state["engine"], state["tokens"]
    n, m = case["prompt"], case["extend"]
    logits = [eng.prefill(t[:n]).values]
    if m:
        logits.append(eng.extend(t[n:n + m]).values)
    for i in range(case["decode"]):
        logits.append(eng.decode(int(t[n + m + i])).values)
    return logits


# ---------------------------------------------------------------- work, tolerance


def _pairs(seq, pos0):
    return seq * pos0 + seq * (seq + 1) // 2


def work(case):
    kind = case["kind"]
    h, inter, hq, hkv, _ = MODELS[case["model"]]
    row = 2 * hkv * D * 2  # one position's K and V rows
    if kind == "decode_attn":
        return dict(bytes=case["ctx"] * row + 4 * hq * D, flops=4 * hq * D * case["ctx"])
    if kind == "decode_layer":
        return dict(bytes=case["ctx"] * row + 2 * (hq + 2 * hkv) * D + 2 * hq * D,
                    flops=4 * hq * D * case["ctx"])
    if kind == "kv_write":
        n = case["seq"] * (hq + 2 * hkv) * D
        return dict(bytes=4 * n + case["seq"] * D * 4, flops=8 * n)
    if kind == "prefill_attn":
        s, p = case["seq"], case["pos0"]
        return dict(bytes=(s + p) * row + 4 * s * hq * D, flops=4 * hq * D * _pairs(s, p))
    if kind == "mlp_step":
        return dict(bytes=int(2 * inter * h * WBYTES[case["gate_up"]] +
                              inter * h * WBYTES[case["down"]] + 10 * h),
                    flops=6 * inter * h)
    if kind == "head_step":
        v = case["vocab"]
        return dict(bytes=int(v * h * WBYTES[case["fmt"]] + 2 * v + 8 * h), flops=2 * v * h)
    # session: every call reads the weights once; logits of each call's last token
    per = layer_bytes = 0
    for l in range(case["layers"]):
        base, hi = _mix(case, l)
        nb = h * D * (hq + hkv) + h * hq * D + 2 * inter * h
        nh = h * D * hkv + inter * h
        per += nb + nh
        layer_bytes += nb * WBYTES[base] + nh * WBYTES[hi]
    head = case["vocab"] * h
    calls = 1 + (1 if case["extend"] else 0) + case["decode"]
    n = case["prompt"] + case["extend"] + case["decode"]
    kv = n * row * case["layers"]
    attn = 4 * hq * D * _pairs(n, 0) * case["layers"]
    reread = sum(range(n - case["decode"], n)) * row * case["layers"]
    if case["extend"]:
        reread += case["prompt"] * row * case["layers"]
    return dict(bytes=int(calls * (layer_bytes + head * WBYTES[_embed_fmt(case)] +
                                   4 * case["vocab"]) + kv + reread),
                flops=2 * per * n + 2 * head * calls + attn)


def tolerance(case):
    """About four times the distance from float64 that the path shows (f16
    results, fp32 accumulation); bits of the norm/RoPE/KV write are defined.
    A session's rounding differences travel through its layers, and further
    with weights that the prompt rounds to f16 and the decode step does not."""
    kind = case["kind"]
    if kind == "kv_write":
        return "exact"
    if kind in ("decode_layer", "decode_attn"):
        return dict(rel=1.2e-3, max=1e-2)
    if kind == "prefill_attn":
        return dict(rel=1.2e-3, max=3e-2)
    if kind in ("mlp_step", "head_step"):
        return dict(rel=2e-3, max=8e-3)
    if case["layers"] <= 4:
        return dict(rel=8e-3, max=3e-2)
    return dict(rel=1.5e-2, max=7e-2) if case["mix"] == "f16" else dict(rel=3.5e-2, max=1.7e-1)


# ---------------------------------------------------------------- exact


def _rope_rows(x, pos):
    """NeoX rotation of [..., D] float64 rows; pos broadcasts over the leading
    dimensions.  The angle is the float32 product that the tables are built
    from."""
    i = torch.arange(0, D, 2, dtype=torch.float64, device=x.device)
    inv = (1.0 / THETA ** (i / D)).to(torch.float32)
    ang = (pos.to(torch.float32)[..., None] * inv).to(torch.float64)
    c, s = torch.cos(ang), torch.sin(ang)
    lo, hi = x[..., :D // 2], x[..., D // 2:]
    return torch.cat([lo * c - hi * s, hi * c + lo * s], -1)


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _attend(q, k, v, pos0):
    """q [S, Hq, D], k/v [Hkv, >= pos0 + S, D] in float64 -> [S, Hq, D]."""
    s, hq, _ = q.shape
    hkv = k.shape[0]
    grp = hq // hkv
    n = pos0 + s
    out = torch.empty_like(q)
    rows = torch.arange(s, device=q.device) + pos0
    mask = torch.arange(n, device=q.device)[None, :] > rows[:, None]
    for h in range(hq):
        sc = (q[:, h] @ k[h // grp, :n].T) / math.sqrt(D)
        sc.masked_fill_(mask, -math.inf)
        out[:, h] = torch.softmax(sc, -1) @ v[h // grp, :n]
    return out


def _dequant(fmt, blocks, decode):
    """float64 weights of ggml blocks [rows, bytes]; decode: Q4_K's effective
    scale and min rounded to f16, as the decode layout defines them."""
    if fmt == F16:
        return blocks.double()
    rows = blocks.shape[0]
    be, bb = BLOCK[fmt]
    b = blocks.reshape(-1, bb)

    def half(col):
        return b[:, col:col + 2].contiguous().view(torch.float16).double()

    if fmt == Q8_0:
        return (b[:, 2:].contiguous().view(torch.int8).double() * half(0)).reshape(rows, -1)
    if fmt in (Q4_K, Q5_K):
        s = b[:, 4:16].to(torch.int32)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        sc, mn = half(0) * sc, half(2) * mn
        if decode and fmt == Q4_K:
            sc, mn = sc.half().double(), mn.half().double()
        qs = b[:, 16:144] if fmt == Q4_K else b[:, 48:176]
        qs = qs.reshape(-1, 4, 1, 32).to(torch.int32)
        q = torch.cat([qs & 15, qs >> 4], 2)  # [blocks, 4, 2, 32]
        if fmt == Q5_K:
            qh = b[:, 16:48].to(torch.int32)[:, None, None, :]
            bit = torch.arange(8, device=b.device, dtype=torch.int32).reshape(1, 4, 2, 1)
            q = q + (((qh >> bit) & 1) << 4)
        w = q.double().reshape(-1, 8, 32) * sc[..., None] - mn[..., None]
        return w.reshape(rows, -1)
    ql = b[:, :128].reshape(-1, 2, 2, 32).to(torch.int32)
    qh = b[:, 128:192].reshape(-1, 2, 1, 32).to(torch.int32)
    lo, hi = ql & 15, ql >> 4  # [blocks, half, 32-run of ql, 32]
    q = torch.cat([lo, hi], 2)  # runs i = 0..3 of each half
    bit = 2 * torch.arange(4, device=b.device, dtype=torch.int32).reshape(1, 1, 4, 1)
    q = (q | (((qh >> bit) & 3) << 4)) - 32
    sc = b[:, 192:208].contiguous().view(torch.int8).double() * half(208)
    w = q.double().reshape(-1, 16, 16) * sc[..., None]
    return w.reshape(rows, -1)


def _silu_mul(g, u):
    return g * torch.sigmoid(g) * u


def _exact_session(case, seed):
    h, inter, hq, hkv, _ = MODELS[case["model"]]
    g = _gen(seed)
    # layers are drawn before the embedding: keep the generator's order
    state = g.get_state()
    for l in range(case["layers"]):
        _session_layer(case, g, l)
    (ef, embed), norm = _session_ends(case, g)
    t = torch.from_numpy(_session_tokens(case, seed)).cuda()
    x = _dequant(ef, embed[t], False)
    n = x.shape[0]
    pos = torch.arange(n, device="cuda")[:, None]
    g.set_state(state)
    for l in range(case["layers"]):
        w = _session_layer(case, g, l)

        def lin(name, y):
            return y @ _dequant(w[name][0], w[name][1], True).T

        y = _rms(x, w["input_layernorm"])
        q = _rope_rows(_rms(lin("q_proj", y).reshape(n, hq, D), w["q_norm"]), pos)
        k = _rope_rows(_rms(lin("k_proj", y).reshape(n, hkv, D), w["k_norm"]), pos)
        v = lin("v_proj", y).reshape(n, hkv, D)
        a = _attend(q, k.transpose(0, 1).contiguous(), v.transpose(0, 1).contiguous(), 0)
        x = x + lin("o_proj", a.reshape(n, hq * D))
        y = _rms(x, w["post_attention_layernorm"])
        x = x + lin("down_proj", _silu_mul(lin("gate_proj", y), lin("up_proj", y)))
    last = [case["prompt"] - 1]
    if case["extend"]:
        last.append(last[-1] + case["extend"])
    last += [last[-1] + 1 + i for i in range(case["decode"])]
    y = _rms(x[last], norm)
    logits = torch.empty((len(last), case["vocab"]), dtype=torch.float64, device="cuda")
    for r in range(0, case["vocab"], 16384):
        logits[:, r:r + 16384] = y @ _dequant(ef, embed[r:r + 16384], True).T
    return [row for row in logits.cpu().numpy()]


def exact(case, seed):
    kind = case["kind"]
    hq, hkv = MODELS[case["model"]][2:4]
    if kind == "session":
        return _exact_session(case, seed)
    if kind in ("mlp_step", "head_step"):
        d = _gemv_inputs(case, seed)
        c = d["residual"].double() + d["x"].double()
        y = _rms(c, d["gamma"])
        if kind == "mlp_step":
            gu = _dequant(case["gate_up"], d["gate_up"], True) @ y
            inter = gu.shape[0] // 2
            y = _dequant(case["down"], d["down"], True) @ _silu_mul(gu[:inter], gu[inter:])
        else:
            y = torch.cat([_dequant(case["fmt"], d["head"][r:r + 16384], True) @ y
                           for r in range(0, case["vocab"], 16384)])
        return dict(y=y, residual_out=c)
    d = _attn_inputs(case, seed)
    if kind in ("decode_attn", "prefill_attn"):
        pos0 = case["ctx"] - 1 if kind == "decode_attn" else case["pos0"]
        q = d["q"].double().reshape(-1, hq, D)
        out = _attend(q, d["k_cache"].double(), d["v_cache"].double(), pos0)
        return out.reshape(d["q"].shape)
    if kind == "kv_write":
        s = case["seq"]
        pos0, q, k, v = case["pos0"], d["q"].double(), d["k"].double(), d["v"]
    else:
        s, pos0 = 1, case["ctx"] - 1
        qkv = d["qkv"].reshape(1, hq + 2 * hkv, D)
        q, k, v = qkv[:, :hq].double(), qkv[:, hq:hq + hkv].double(), qkv[:, hq + hkv:]
    pos = (torch.arange(s, device="cuda") + pos0)[:, None]
    q, k = _rope_rows(_rms(q, d["q_norm"]), pos), _rope_rows(_rms(k, d["k_norm"]), pos)
    kc, vc = d["k_cache"].double(), d["v_cache"].double()
    kc[:, pos0:pos0 + s] = k.transpose(0, 1)
    vc[:, pos0:pos0 + s] = v.double().transpose(0, 1)
    out = q if kind == "kv_write" else _attend(q, kc, vc, pos0)[0]
    return dict(out=out, k_cache=kc, v_cache=vc)
