"""The work whose speed is kept: calls of this framework as a serving program
makes them, from one fp32 decode attention of a few microseconds to a whole
prompt through a 1B-parameter decoder.

Each case is a family ("kind") with its sizes and options:

  attn_decode   gpu_attention_decode: one sequence over the reference's fp32
                caches (the reference's call contract)
  step          decode_step: qkNorm, RoPE, KV write and attention of the new
                token of B sequences (fp16 / bf16 / fp8 caches)
  prefill_attn  attn_prefill: RoPE, KV write and causal attention of a prompt
  proj_prefill  gpu_linear_col: the Q, K, V and O projections of a prompt
  ffn_prefill   gpu_linear_col + gpu_silu_mul: the feed-forward block of a
                prompt
  proj_decode   the Q, K, V and O projections of one token, GGUF weights
  ffn_decode    the feed-forward block of one token, GGUF weights
  head          final norm, output projection and greedy token
  model_decode  DenseModel.decode: one token through a dense decoder
  model_prefill DenseModel.prefill: a prompt through a dense decoder

Sizes are those of the benchmark's and tests' shapes (TinyLlama, Llama-3.2-1B,
Llama-3-8B, Qwen3-30B-A3B attention) and of generic ones between them.
"""
import math

import numpy as np
import torch

from hippo_leap_amd import _lib as L
from hippo_leap_amd import attention as A

F16, Q8_0, Q4_K, Q5_K, Q6_K = L.HL_GGML_F16, L.HL_GGML_Q8_0, L.HL_GGML_Q4_K, L.HL_GGML_Q5_K, L.HL_GGML_Q6_K
WTYPES = {"f32": 0, "f16": F16, "q8_0": Q8_0, "q4_k": Q4_K, "q5_k": Q5_K, "q6_k": Q6_K}
BLOCK = {F16: (1, 2), Q8_0: (32, 34), Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210)}  # weights, bytes
KV = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "fp8": torch.float8_e4m3fn}
KV_BYTES = {"f32": 4, "f16": 2, "bf16": 2, "fp8": 1}
EPS = 1e-5


def listed():
    return [
        # The smallest call there is: one token of TinyLlama against 512
        # cached positions, fp32 caches (the reference's own decode).
        {"name": "attn_decode_f32_512", "kind": "attn_decode", "hq": 32, "hkv": 4, "d": 64, "len": 512},
        # A serving batch of 8 at 2K context, Llama-3.2-1B attention, caches in
        # the reference's column-major layout.
        {"name": "step_f16_b8_2k", "kind": "step", "b": 8, "hq": 32, "hkv": 8, "d": 64, "len": 2049, "kv": "f16",
         "layout": "col", "qknorm": False, "base": 5e5},
        # Long context: 16 sequences at 32K, Qwen3-30B-A3B attention with
        # qkNorm, caches in the layout the library prefers (tiled).
        {"name": "step_bf16_b16_32k", "kind": "step", "b": 16, "hq": 32, "hkv": 4, "d": 128, "len": 32769,
         "kv": "bf16", "layout": "tiled", "qknorm": True, "base": 1e6},
        # A 4K prompt's attention, Llama-3-8B shape, bf16 activations.
        {"name": "prefill_attn_bf16_4k", "kind": "prefill_attn", "hq": 32, "hkv": 8, "d": 128, "t": 4096, "io": "bf16",
         "kv": "bf16", "layout": "tiled", "base": 5e5},
        # A 512-token prompt's attention, TinyLlama shape, fp32 (the
        # reference's own prefill).
        {"name": "prefill_attn_f32_512", "kind": "prefill_attn", "hq": 32, "hkv": 4, "d": 64, "t": 512, "io": "f32",
         "kv": "f32", "layout": "col", "base": 1e4},
        # The projections of a short chat turn (an odd number of tokens),
        # Llama-3-8B shape: 37 columns against 168 MB of weights.
        {"name": "proj_prefill_t37", "kind": "proj_prefill", "e": 4096, "q": 4096, "kv_rows": 1024, "t": 37},
        # The feed-forward block of a 1000-token prompt, Llama-3-8B shape.
        {"name": "ffn_prefill_t1000", "kind": "ffn_prefill", "e": 4096, "ff": 14336, "t": 1000},
        # One token's projections in a Q8_0 file of the Llama-3.2-1B shape:
        # small matrices, where each launch's latency counts.
        {"name": "proj_decode_q8_1b", "kind": "proj_decode", "e": 2048, "q": 2048, "kv_rows": 512, "w": "q8_0"},
        # One token's feed-forward block in a Q4_K_M file of the Llama-3-8B
        # shape (its down projections are Q6_K in half of the layers).
        {"name": "ffn_decode_q4_q6_8b", "kind": "ffn_decode", "e": 4096, "ff": 14336, "w": "q4_k", "down": "q6_k"},
        # The end of a decode step: norm, a Q6_K output head of 128256 rows,
        # the greedy token.
        {"name": "head_q6_8b", "kind": "head", "e": 4096, "vocab": 128256, "w": "q6_k"},
        # A whole decode step: Llama-3.2-1B shape, Q4_K layers, Q6_K head, bf16
        # cache at 2000 positions.
        {"name": "model_decode_1b_q4", "kind": "model_decode", "layers": 16, "e": 2048, "hq": 32, "hkv": 8, "d": 64,
         "ff": 8192, "vocab": 128256, "w": "q4_k", "head": "q6_k", "kv": "bf16", "pos": 2000, "qknorm": False},
        # A whole prompt of 301 tokens through the same decoder with fp32
        # weights (prefill takes fp32 weights, as the reference's does).
        {"name": "model_prefill_1b_t301", "kind": "model_prefill", "layers": 16, "e": 2048, "hq": 32, "hkv": 8,
         "d": 64, "ff": 8192, "vocab": 128256, "t": 301, "kv": "bf16", "qknorm": False},
    ]


def _log(rng, lo, hi, step=1):
    """An integer of [lo, hi], even over the logarithm, a multiple of step."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, min(hi, v // step * step if step > 1 else v))


def draw(rng):
    kind = rng.choice(["attn_decode", "step", "prefill_attn", "proj_prefill", "ffn_prefill", "proj_decode",
                       "ffn_decode", "head", "model_decode", "model_prefill"])
    d = rng.choice([64, 128])
    hkv = rng.choice([4, 8])
    hq = hkv * rng.choice([1, 4, 8])
    layout = lambda kv: "col" if kv == "f32" else "tiled" if kv == "fp8" else rng.choice(["col", "tiled"])  # noqa: E731
    if kind == "attn_decode":
        return {"kind": kind, "hq": hq, "hkv": hkv, "d": d, "len": _log(rng, 16, 8192)}
    if kind == "step":
        b, kv = rng.choice([1, 2, 3, 8, 16]), rng.choice(["f16", "bf16", "fp8"])
        return {"kind": kind, "b": b, "hq": hq, "hkv": hkv, "d": d, "len": _log(rng, 16, 32768 if b <= 4 else 8192),
                "kv": kv, "layout": layout(kv), "qknorm": rng.random() < 0.5, "base": 5e5}
    if kind == "prefill_attn":
        io = rng.choice(["bf16", "f16", "f32"])
        kv = "f32" if io == "f32" and rng.random() < 0.5 else rng.choice(["f16", "bf16"])
        return {"kind": kind, "hq": hq, "hkv": hkv, "d": d, "t": _log(rng, 5, 4096 if io != "f32" else 2048),
                "io": io, "kv": kv, "layout": layout(kv), "base": 5e5}
    if kind == "proj_prefill":
        e = _log(rng, 512, 4096, 64)
        return {"kind": kind, "e": e, "q": hq * d, "kv_rows": hkv * d, "t": _log(rng, 2, 2048)}
    if kind == "ffn_prefill":
        return {"kind": kind, "e": _log(rng, 512, 4096, 64), "ff": _log(rng, 1024, 14336, 32), "t": _log(rng, 2, 1000)}
    w = rng.choice(["f32", "f16", "q8_0", "q4_k", "q4_k", "q5_k", "q6_k"])
    if kind == "proj_decode":
        return {"kind": kind, "e": _log(rng, 512, 8192, 256), "q": hq * d, "kv_rows": hkv * d, "w": w}
    if kind == "ffn_decode":
        down = "q6_k" if w in ("q4_k", "q5_k") and rng.random() < 0.5 else w
        return {"kind": kind, "e": _log(rng, 512, 8192, 256), "ff": _log(rng, 1024, 14336, 256), "w": w, "down": down}
    if kind == "head":
        return {"kind": kind, "e": _log(rng, 512, 4096, 256), "vocab": _log(rng, 8000, 128256),
                "w": rng.choice(["f32", "f16", "q8_0", "q6_k"])}
    shape = {"kind": kind, "layers": rng.choice([1, 2, 3]), "e": _log(rng, 512, 4096, 256), "hq": hq, "hkv": hkv,
             "d": d, "ff": _log(rng, 1024, 14336, 256), "vocab": _log(rng, 4000, 32000)}
    if kind == "model_decode":
        shape.update(w=w, head=w if w in ("f32", "f16", "q8_0") else "q6_k", kv=rng.choice(["bf16", "f16", "fp8", "f32"]),
                     pos=_log(rng, 1, 4000), qknorm=rng.random() < 0.5)
        return shape
    shape.update(t=_log(rng, 2, 512), kv=rng.choice(["bf16", "f16", "f32"]), qknorm=rng.random() < 0.5)
    return shape


# --- inputs -----------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed * 7919 + 17)


def _acts(g, *shape):
    """Hidden-state values after a norm: unit normal, one channel (row) in 256
    an outlier some 20 times larger, as trained decoders have."""
    x = torch.randn(*shape, device="cuda", generator=g)
    x[torch.rand(shape[0], device="cuda", generator=g) < 1 / 256] *= 20.0
    return x


def _weight(g, rows, cols, wtype):
    """A [rows, cols] weight of standard deviation ~ 1/sqrt(cols): fp32, or
    GGUF rows of random quants (block scales vary by half around their mean)."""
    sd = 1.0 / math.sqrt(cols)
    if wtype in (0, F16):
        w = torch.randn(rows, cols, device="cuda", generator=g) * sd
        return w if wtype == 0 else w.to(torch.float16).view(torch.uint8).reshape(rows, -1)
    qk, nbytes = BLOCK[wtype]
    n = rows * cols // qk
    b = torch.randint(0, 256, (n, nbytes), device="cuda", generator=g, dtype=torch.uint8)
    spread = 0.5 + torch.rand(n, device="cuda", generator=g)
    half = lambda v: v.to(torch.float16).view(torch.uint8).reshape(n, 2)  # noqa: E731
    if wtype == Q8_0:  # d, 32 int8 (standard deviation 74)
        b[:, 0:2] = half(spread * (sd / 74))
    elif wtype in (Q4_K, Q5_K):
        # d, dmin, 12 bytes of 6-bit scales and mins: mins equal to the scales
        # and dmin half the quants' range times d, so that weights are centred.
        mid = 7.5 if wtype == Q4_K else 15.5
        d = half(spread * (sd / (37 * mid * 0.6)))
        b[:, 0:2] = d
        b[:, 2:4] = half(d.contiguous().view(torch.float16).reshape(n).float() * mid)
        b[:, 8:12] = b[:, 4:8]
        lo = b[:, 12:16] & 15
        b[:, 12:16] = lo | (lo << 4)
    else:  # Q6_K: 128 + 64 bytes of 6-bit quants, 16 int8 scales, d
        b[:, 208:210] = half(spread * (sd / (74 * 18.5)))
    return b.reshape(rows, -1)


def _dequant(w, rows, cols, wtype):
    """The weight's values in 64 bits, from the GGUF block definitions."""
    if wtype == 0:
        return w.double()
    if wtype == F16:
        return w.reshape(-1).view(torch.float16).reshape(rows, cols).double()
    b = w.reshape(-1, BLOCK[wtype][1])
    n = b.shape[0]
    half = lambda at: b[:, at:at + 2].contiguous().view(torch.float16).double()  # noqa: E731  [n, 1]
    if wtype == Q8_0:
        return (half(0) * b[:, 2:].contiguous().view(torch.int8).double()).reshape(rows, cols)
    if wtype == Q6_K:
        ql, qh = b[:, :128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 1, 32)
        sc = b[:, 192:208].contiguous().view(torch.int8).double().reshape(n, 2, 4, 2, 1)
        q = torch.stack([(ql[:, :, t & 1] >> (4 * (t >> 1))) & 15 | ((qh[:, :, 0] >> (2 * t)) & 3) << 4
                         for t in range(4)], 2)  # [n, 2, 4, 32]
        q = (q.double() - 32).reshape(n, 2, 4, 2, 16)
        return (half(208).reshape(n, 1, 1, 1, 1) * sc * q).reshape(rows, cols)
    s = b[:, 4:16].to(torch.int32)
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
    qs = (b[:, 16:] if wtype == Q4_K else b[:, 48:]).reshape(n, 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], 2).reshape(n, 8, 32).to(torch.int32)
    if wtype == Q5_K:
        bit = torch.arange(8, device=b.device, dtype=torch.int32).reshape(1, 8, 1)
        q = q | ((b[:, 16:48].reshape(n, 1, 32).to(torch.int32) >> bit) & 1) << 4
    return ((half(0) * sc).unsqueeze(2) * q.double() - (half(2) * mn).unsqueeze(2)).reshape(rows, cols)


def _cache(g, shape, kv):
    x = torch.randn(*shape, device="cuda", generator=g) * 0.5
    return x.to(KV[kv])


def _pad(n, to):
    return (n + to - 1) // to * to


def _cache_len(case):
    n = case["pos"] + 1 if "pos" in case else case.get("len") or case["t"]
    return _pad(n, 64)


def _columns(cache, hkv, d, max_len, layout):
    """[B, hkv, d, max_len] view or copy of caches in either layout."""
    if layout == "tiled":
        return cache.reshape(-1, hkv, max_len // 32, d, 32).permute(0, 1, 3, 2, 4).reshape(-1, hkv, d, max_len)
    return cache.reshape(-1, hkv, d, max_len)


LAYOUT = {"col": L.HL_KV_COLMAJOR, "tiled": L.HL_KV_TILED32}


def _linear(y, x, w, cols, rows, wtype):
    if wtype == 0:
        A.gpu_linear_col(y, x, w, cols, rows, 1)
    else:
        A.gpu_linear_col_quant(y, x, w, cols, rows, wtype)


def _model(case, seed):
    """A dense decoder's weights and handle."""
    from hippo_leap_amd.model import DenseModel
    g = _gen(seed)
    e, d, ff, vocab = case["e"], case["d"], case["ff"], case["vocab"]
    q, kv, wt, ht = case["hq"] * d, case["hkv"] * d, WTYPES[case.get("w", "f32")], WTYPES[case.get("head", "f32")]
    shapes = {"wq": (q, e), "wk": (kv, e), "wv": (kv, e), "wo": (e, q), "w_gate": (ff, e), "w_up": (ff, e),
              "w_down": (e, ff)}
    gain = lambda n: torch.rand(n, device="cuda", generator=g) + 0.5  # noqa: E731
    layers = []
    for _ in range(case["layers"]):
        one = {n: _weight(g, r, c, wt) for n, (r, c) in shapes.items()}
        one.update({n + "_type": wt for n in shapes})
        one.update(attn_norm=gain(e), ffn_norm=gain(e))
        if case["qknorm"]:
            one.update(q_norm=gain(d), k_norm=gain(d))
        layers.append(one)
    emb, onorm, head = torch.randn(vocab, e, device="cuda", generator=g), gain(e), _weight(g, vocab, e, ht)
    cfg = dict(n_layer=case["layers"], n_emb=e, n_head=case["hq"], n_head_kv=case["hkv"], head_dim=d, rope_dim=d,
               n_ff=ff, n_vocab=vocab, max_len=_cache_len(case), rms_eps=EPS, rope_base=5e5)
    m = DenseModel(torch, cfg, emb, onorm, head, ht, layers, max_tokens=case.get("t", 1),
                   kv_dtype={"f32": L.HL_F32, "f16": L.HL_F16, "bf16": L.HL_BF16, "fp8": L.HL_FP8}[case["kv"]])
    for t in m.cache.k + m.cache.v:
        t.copy_(_cache(g, (t.numel() // KV_BYTES[case["kv"]],), case["kv"]).view(torch.uint8))
    caches = {"k": [t.view(KV[case["kv"]]) for t in m.cache.k], "v": [t.view(KV[case["kv"]]) for t in m.cache.v]}
    return {"m": m, "caches": caches, "emb": emb, "onorm": onorm, "head": head, "layers": layers, "g": g}


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("model_decode", "model_prefill"):
        s = _model(case, seed)
        n = case["t"] if kind == "model_prefill" else 1
        s.update(kind=kind, pos=case.get("pos", 0),
                 tokens=torch.randint(0, case["vocab"], (n,), device="cuda", generator=s["g"], dtype=torch.int32))
        s["next"] = torch.zeros(1, device="cuda", dtype=torch.int32)
        return s
    g = _gen(seed)
    s = {"kind": kind, "case": case}
    empty = lambda *n: torch.empty(*n, device="cuda")  # noqa: E731
    if kind == "attn_decode":
        hq, hkv, d, m = case["hq"], case["hkv"], case["d"], _cache_len(case)
        s.update(q=torch.randn(hq * d, device="cuda", generator=g), k=_cache(g, (hkv * d, m), "f32"),
                 v=_cache(g, (hkv * d, m), "f32"), out=empty(hq * d), max_len=m)
    elif kind == "step":
        b, hq, hkv, d, m = case["b"], case["hq"], case["hkv"], case["d"], _cache_len(case)
        s.update(q=torch.randn(b * hq * d, device="cuda", generator=g), k=torch.randn(b * hkv * d, device="cuda", generator=g),
                 v=torch.randn(b * hkv * d, device="cuda", generator=g) * 0.5, kc=_cache(g, (b, hkv * d, m), case["kv"]),
                 vc=_cache(g, (b, hkv * d, m), case["kv"]), out=empty(b * hq * d))
        if case["qknorm"]:
            s.update(qn=torch.rand(d, device="cuda", generator=g) + 0.5, kn=torch.rand(d, device="cuda", generator=g) + 0.5)
        lay = LAYOUT[case["layout"]]
        s["rs"] = A.rope_store_args(s["q"], s["k"], s["v"], s["kc"], s["vc"], hq, hkv, d, m, case["len"] - 1,
                                    case["base"], q_norm_w=s.get("qn"), k_norm_w=s.get("kn"), eps=EPS, kv_layout=lay)
        s["at"] = A.decode_args(s["q"], s["kc"], s["vc"], s["out"], hq, hkv, d, m, case["len"], kv_layout=lay)
        s["ws"] = A.decode_step_workspace(s["rs"], s["at"])
    elif kind == "prefill_attn":
        hq, hkv, d, t, m, io = case["hq"], case["hkv"], case["d"], case["t"], _cache_len(case), KV[case["io"]]
        for n, h in (("q", hq), ("k", hkv), ("v", hkv)):
            s[n] = torch.randn(h * d, t, device="cuda", generator=g).to(io)
        s.update(kc=torch.zeros(hkv * d, m, device="cuda", dtype=KV[case["kv"]]),
                 vc=torch.zeros(hkv * d, m, device="cuda", dtype=KV[case["kv"]]), out=empty(hq * d, t))
        s["args"] = A.prefill_args(s["q"], s["k"], s["v"], s["out"], hq, hkv, d, t, rope_base=case["base"],
                                   apply_rope=True, k_cache=s["kc"], v_cache=s["vc"], max_len=m,
                                   kv_layout=LAYOUT[case["layout"]])
        s["ws"] = A.workspace(A.prefill_workspace_bytes(s["args"]))
    elif kind in ("proj_prefill", "proj_decode"):
        e, q, kv, t, wt = case["e"], case["q"], case["kv_rows"], case.get("t", 1), WTYPES[case.get("w", "f32")]
        s.update(x=_acts(g, e, t), a=torch.randn(q, t, device="cuda", generator=g), wq=_weight(g, q, e, wt),
                 wk=_weight(g, kv, e, wt), wv=_weight(g, kv, e, wt), wo=_weight(g, e, q, wt), yq=empty(q, t),
                 yk=empty(kv, t), yv=empty(kv, t), yo=empty(e, t), wt=wt)
    elif kind in ("ffn_prefill", "ffn_decode"):
        e, ff, t = case["e"], case["ff"], case.get("t", 1)
        wt, dt = WTYPES[case.get("w", "f32")], WTYPES[case.get("down", "f32")]
        s.update(x=_acts(g, e, t), wg=_weight(g, ff, e, wt), wu=_weight(g, ff, e, wt), wd=_weight(g, e, ff, dt),
                 gate=empty(ff, t), up=empty(ff, t), h=empty(ff, t), y=empty(e, t), wt=wt, dt=dt)
    elif kind == "head":
        e, vocab, wt = case["e"], case["vocab"], WTYPES[case["w"]]
        s.update(x=_acts(g, e, 1), gain=torch.rand(e, device="cuda", generator=g) + 0.5, w=_weight(g, vocab, e, wt), wt=wt,
                 xn=empty(e), logits=empty(vocab), token=torch.zeros(1, device="cuda", dtype=torch.int32))
    return s


# --- one pass ---------------------------------------------------------------
def run(s):
    kind = s["kind"]
    if kind == "model_decode":
        m = s["m"]
        m.cache.desc.cur_len = s["pos"]  # the sequence's length: the same token again
        m.decode(s["tokens"], s["next"])
        return {"logits": m.logits, **s["caches"]}
    if kind == "model_prefill":
        return {"logits": s["m"].prefill(s["tokens"]), **s["caches"]}
    c = s["case"]
    if kind == "attn_decode":
        A.gpu_attention_decode(s["out"], s["q"], s["k"], s["v"], c["hq"], c["hkv"], c["d"], c["len"], s["max_len"])
        return {"out": s["out"]}
    if kind == "step":
        A.decode_step(s["rs"], s["at"], s["ws"])
        return {"out": s["out"], "k": s["kc"], "v": s["vc"]}
    if kind == "prefill_attn":
        A.attn_prefill(s["args"], s["ws"])
        return {"out": s["out"], "k": s["kc"], "v": s["vc"]}
    if kind == "proj_prefill":
        e, q, kv, t = c["e"], c["q"], c["kv_rows"], c["t"]
        A.gpu_linear_col(s["yq"], s["x"], s["wq"], e, q, t)
        A.gpu_linear_col(s["yk"], s["x"], s["wk"], e, kv, t)
        A.gpu_linear_col(s["yv"], s["x"], s["wv"], e, kv, t)
        A.gpu_linear_col(s["yo"], s["a"], s["wo"], q, e, t)
        return {"q": s["yq"], "k": s["yk"], "v": s["yv"], "o": s["yo"]}
    if kind == "proj_decode":
        e, q, kv, wt = c["e"], c["q"], c["kv_rows"], s["wt"]
        _linear(s["yq"], s["x"], s["wq"], e, q, wt)
        if wt:
            A.gpu_fused_kv_linear_quant(s["yk"], s["yv"], s["x"], s["wk"], s["wv"], e, kv, wt, wt)
        else:
            _linear(s["yk"], s["x"], s["wk"], e, kv, wt)
            _linear(s["yv"], s["x"], s["wv"], e, kv, wt)
        _linear(s["yo"], s["a"], s["wo"], q, e, wt)
        return {"q": s["yq"], "k": s["yk"], "v": s["yv"], "o": s["yo"]}
    if kind == "ffn_prefill":
        e, ff, t = c["e"], c["ff"], c["t"]
        A.gpu_linear_col(s["gate"], s["x"], s["wg"], e, ff, t)
        A.gpu_linear_col(s["up"], s["x"], s["wu"], e, ff, t)
        A.gpu_silu_mul(s["h"], s["gate"], s["up"], ff * t)
        A.gpu_linear_col(s["y"], s["h"], s["wd"], ff, e, t)
        return {"h": s["h"], "y": s["y"]}
    if kind == "ffn_decode":
        e, ff = c["e"], c["ff"]
        if s["wt"]:
            A.gpu_fused_gate_up_silu_quant(s["h"], s["x"], s["wg"], s["wu"], e, ff, s["wt"])
        else:
            A.gpu_linear_col(s["gate"], s["x"], s["wg"], e, ff, 1)
            A.gpu_linear_col(s["up"], s["x"], s["wu"], e, ff, 1)
            A.gpu_silu_mul(s["h"], s["gate"], s["up"], ff)
        _linear(s["y"], s["h"], s["wd"], ff, e, s["dt"])
        return {"h": s["h"], "y": s["y"]}
    A.gpu_rmsnorm_cols(s["xn"], s["x"], s["gain"], c["e"], 1, EPS)
    _linear(s["logits"], s["xn"], s["w"], c["e"], c["vocab"], s["wt"])
    A.argmax_async(s["logits"], c["vocab"], s["token"])
    return {"logits": s["logits"], "token": s["token"]}


# --- what a pass cannot do without --------------------------------------------
def _wbytes(rows, cols, wtype):
    if wtype == 0:
        return 4 * rows * cols
    qk, nbytes = BLOCK[wtype]
    return rows * cols // qk * nbytes


def work(case):
    kind, t = case["kind"], case.get("t", 1)
    if kind == "attn_decode":
        hq, hkv, d, n = case["hq"], case["hkv"], case["d"], case["len"]
        return {"bytes": 8 * hkv * d * n + 8 * hq * d, "flops": 4 * hq * d * n}
    if kind == "step":
        b, hq, hkv, d, n, eb = case["b"], case["hq"], case["hkv"], case["d"], case["len"], KV_BYTES[case["kv"]]
        return {"bytes": b * (2 * hkv * d * n * eb + 8 * (hq + hkv) * d), "flops": 4 * b * hq * d * n}
    if kind == "prefill_attn":
        hq, hkv, d, io, eb = case["hq"], case["hkv"], case["d"], KV_BYTES[case["io"]], KV_BYTES[case["kv"]]
        return {"bytes": t * d * ((hq + 2 * hkv) * io + 4 * hq + 2 * hkv * eb), "flops": 2 * hq * d * t * (t + 1)}
    if kind in ("proj_prefill", "proj_decode"):
        e, q, kv, wt = case["e"], case["q"], case["kv_rows"], WTYPES[case.get("w", "f32")]
        return {"bytes": _wbytes(2 * q + 2 * kv, e, wt) + 4 * t * (2 * e + 2 * q + 2 * kv), "flops": 4 * t * e * (q + kv)}
    if kind in ("ffn_prefill", "ffn_decode"):
        e, ff = case["e"], case["ff"]
        w = 2 * _wbytes(ff, e, WTYPES[case.get("w", "f32")]) + _wbytes(e, ff, WTYPES[case.get("down", "f32")])
        return {"bytes": w + 4 * t * (2 * e + ff), "flops": 6 * t * e * ff}
    if kind == "head":
        return {"bytes": _wbytes(case["vocab"], case["e"], WTYPES[case["w"]]) + 4 * (case["e"] + case["vocab"]),
                "flops": 2 * case["e"] * case["vocab"]}
    e, d, ff, n, vocab = case["e"], case["d"], case["ff"], case["layers"], case["vocab"]
    q, kv, wt, ht = case["hq"] * d, case["hkv"] * d, WTYPES[case.get("w", "f32")], WTYPES[case.get("head", "f32")]
    eb = KV_BYTES[case["kv"]]
    w = n * (_wbytes(2 * q + 2 * kv + 2 * ff, e, wt) + _wbytes(e, ff, wt)) + _wbytes(vocab, e, ht)
    flops = 2 * t * (n * e * (2 * q + 2 * kv + 3 * ff) + vocab * e)
    if kind == "model_decode":
        return {"bytes": w + n * 2 * kv * (case["pos"] + 1) * eb + 4 * (e + vocab),
                "flops": flops + n * 4 * q * (case["pos"] + 1)}
    return {"bytes": w + n * 2 * kv * t * eb + 4 * t * (e + vocab), "flops": flops + n * 2 * q * t * (t + 1)}


# --- how far correct results may be apart -------------------------------------
def tolerance(case):
    """About four times the largest distance from exact() that 100 draws of
    these ranges showed (2-norm / largest value): linear layers 8e-7 / 5e-6,
    the prompt's feed-forward block 2.1e-6 / 2.4e-5, fp32 attention 2.9e-7 /
    2.4e-6, decode steps 2.8e-6 / 1.1e-5, 16-bit prefill attention 3.1e-4 /
    1.2e-2, whole decoders 2.1e-6 / 1.2e-5.  A new key or value that rounds
    to the other side in a 16-bit or 8-bit cache adds up to one unit there
    ("max" of the caches) and 3.4e-5 to the logits at a few cached positions."""
    kind, kv = case["kind"], case.get("kv")
    ulp = {"bf16": 2.0 ** -7, "f16": 2.0 ** -10, "fp8": 2.0 ** -3}.get(kv, 0.0)
    if kind == "ffn_prefill":
        return {"rel": 8e-6, "max": 1e-4}
    if kind in ("proj_prefill", "proj_decode", "ffn_decode", "head"):
        return {"rel": 3e-6, "max": 2e-5}
    if kind == "attn_decode":
        return {"rel": 1e-6, "max": 5e-6}
    if kind == "step":
        return {"rel": 1.2e-5, "max": max(5e-5, ulp)}
    if kind == "prefill_attn":
        if case["io"] == "f32":
            return {"rel": 1.2e-6 if kv == "f32" else 1e-5, "max": max(2e-5, ulp)}
        return {"rel": 1.2e-3, "max": max(0.05, ulp)}
    if kv == "f32":
        return {"rel": 8e-6, "max": 5e-5}
    return {"rel": 1e-3 if kv == "fp8" else 1.4e-4, "max": max(1e-3, ulp)}


# --- the same in 64 bits -------------------------------------------------------
def _angles(d, base, first, n):
    """cos and sin [d/2, n] of RoPE: the frequency and the angle are 32-bit
    values by definition of the path, the rest is 64 bits."""
    i = (np.arange(d // 2, dtype=np.float32) * 2 / np.float32(d)).astype(np.float64)
    theta = np.power(np.float64(np.float32(1) / np.float32(base)), i).astype(np.float32)
    a = (theta[:, None] * np.arange(first, first + n, dtype=np.float32)[None, :]).astype(np.float64)
    return torch.from_numpy(np.cos(a)).cuda(), torch.from_numpy(np.sin(a)).cuda()


def _norm(x, w, dim):
    """RMSNorm over dimension `dim` (w along it)."""
    shape = [1] * x.dim()
    shape[dim] = -1
    return x / torch.sqrt((x * x).mean(dim, keepdim=True) + EPS) * w.double().reshape(shape)


def _rope(x, cs):
    """Half-split rotation of x [..., d, n]."""
    a, b = x.chunk(2, -2)
    return torch.cat([a * cs[0] - b * cs[1], a * cs[1] + b * cs[0]], -2)


def _attend(q, k, v):
    """q [hq, d, 1], k / v [hkv, d, n] of one sequence: [hq, d]."""
    hq, d = q.shape[0], q.shape[1]
    hkv = k.shape[0]
    p = torch.matmul(q.reshape(hkv, hq // hkv, d), k) / math.sqrt(d)
    return torch.matmul(torch.softmax(p, -1), v.transpose(1, 2).contiguous()).reshape(hq, d)


def _causal(q, k, v):
    """q [hq, d, t], k / v [hkv, d, t]: [hq, d, t], a head at a time."""
    hq, d, t = q.shape
    per = hq // k.shape[0]
    mask = torch.ones(t, t, device=q.device, dtype=torch.bool).tril()
    out = torch.empty_like(q)
    for h in range(hq):
        p = torch.matmul(q[h].t().contiguous(), k[h // per]) / math.sqrt(d)
        p = torch.softmax(p.masked_fill(~mask, float("-inf")), -1)
        out[h] = torch.matmul(p, v[h // per].t().contiguous()).t()
    return out


def _silu(x):
    return x / (1 + torch.exp(-x))


def _exact_model(case, seed):
    s = prepare(case, seed)
    e, d, hq, hkv = case["e"], case["d"], case["hq"], case["hkv"]
    kind, t, m = case["kind"], case.get("t", 1), _cache_len(case)
    ff, wt, ht = case["ff"], WTYPES[case.get("w", "f32")], WTYPES[case.get("head", "f32")]
    layout = "tiled" if case["kv"] != "f32" else "col"
    first = case.get("pos", 0)
    cs = _angles(d, 5e5, first, t)
    x = s["emb"].double()[s["tokens"].long()].t().contiguous()  # [e, t]
    shapes = {"wq": (hq * d, e), "wk": (hkv * d, e), "wv": (hkv * d, e), "wo": (e, hq * d), "w_gate": (ff, e),
              "w_up": (ff, e), "w_down": (e, ff)}
    to_cache = lambda v: v.float().to(KV[case["kv"]]).double()  # noqa: E731
    for i, lw in enumerate(s["layers"]):
        mul = lambda n, v: _dequant(lw[n], *shapes[n], wt) @ v  # noqa: E731,B023
        xn = _norm(x, lw["attn_norm"], 0)
        q, k, v = (mul(n, xn).reshape(-1, d, t) for n in ("wq", "wk", "wv"))
        if "q_norm" in lw:
            q, k = _norm(q, lw["q_norm"], 1), _norm(k, lw["k_norm"], 1)
        q, k = _rope(q, cs), _rope(k, cs)
        if kind == "model_decode":
            kc = _columns(s["caches"]["k"][i], hkv, d, m, layout)[0, :, :, :first].double()
            vc = _columns(s["caches"]["v"][i], hkv, d, m, layout)[0, :, :, :first].double()
            a = _attend(q, torch.cat([kc, to_cache(k)], -1), torch.cat([vc, to_cache(v)], -1)).reshape(-1, 1)
        else:
            a = _causal(q, k, v).reshape(-1, t)
        x = x + mul("wo", a)
        xn = _norm(x, lw["ffn_norm"], 0)
        x = x + mul("w_down", _silu(mul("w_gate", xn)) * mul("w_up", xn))
    logits = _dequant(s["head"], case["vocab"], e, ht) @ _norm(x, s["onorm"], 0)
    n = case["layers"]
    return {"logits": logits.reshape(-1) if kind == "model_decode" else logits, "k": [None] * n, "v": [None] * n}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("model_decode", "model_prefill"):
        return _exact_model(case, seed)
    s = prepare(case, seed)
    if kind == "attn_decode":
        hq, hkv, d, n = case["hq"], case["hkv"], case["d"], case["len"]
        k, v = (s[c].reshape(hkv, d, -1)[:, :, :n].double() for c in ("k", "v"))
        return {"out": _attend(s["q"].double().reshape(hq, d, 1), k, v).reshape(-1)}
    if kind == "step":
        b, hq, hkv, d, n, m = case["b"], case["hq"], case["hkv"], case["d"], case["len"], _cache_len(case)
        q, k, v = (s[c].double().reshape(b, -1, d, 1) for c in ("q", "k", "v"))
        if case["qknorm"]:
            q, k = _norm(q, s["qn"], 2), _norm(k, s["kn"], 2)
        cs = _angles(d, case["base"], n - 1, 1)
        q, k = _rope(q, cs), _rope(k, cs)
        new = [c.float().to(KV[case["kv"]]).double() for c in (k, v)]  # as the cache holds them
        out = []
        for i in range(b):
            old = [_columns(s[c][i], hkv, d, m, case["layout"])[0, :, :, :n - 1].double() for c in ("kc", "vc")]
            out.append(_attend(q[i], *(torch.cat([o, c[i]], -1) for o, c in zip(old, new))).reshape(-1))
        return {"out": torch.cat(out), "k": None, "v": None}
    if kind == "prefill_attn":
        d, t = case["d"], case["t"]
        q, k, v = (s[c].double().reshape(-1, d, t) for c in ("q", "k", "v"))
        cs = _angles(d, case["base"], 0, t)
        return {"out": _causal(_rope(q, cs), _rope(k, cs), v).reshape(-1, t), "k": None, "v": None}
    if kind in ("proj_prefill", "proj_decode"):
        e, q, kv, wt = case["e"], case["q"], case["kv_rows"], s["wt"]
        x, a = s["x"].double(), s["a"].double()
        return {"q": _dequant(s["wq"], q, e, wt) @ x, "k": _dequant(s["wk"], kv, e, wt) @ x,
                "v": _dequant(s["wv"], kv, e, wt) @ x, "o": _dequant(s["wo"], e, q, wt) @ a}
    if kind in ("ffn_prefill", "ffn_decode"):
        e, ff, x = case["e"], case["ff"], s["x"].double()
        h = _silu(_dequant(s["wg"], ff, e, s["wt"]) @ x) * (_dequant(s["wu"], ff, e, s["wt"]) @ x)
        return {"h": h, "y": _dequant(s["wd"], e, ff, s["dt"]) @ h}
    logits = _dequant(s["w"], case["vocab"], case["e"], s["wt"]) @ _norm(s["x"].double(), s["gain"], 0)
    return {"logits": logits.reshape(-1), "token": None}
