"""End-to-end greedy decode of small dense decoders through
hl_forward_decode_token (the reference's forwardDecodeToken for
lkAttentionFfn layers, backends/naive.nim:4592-4760, 5520-5545) against an
oracle step composed from the pinned oracle pieces in the reference's order:
embedding, rmsnorm, projections (tensor.nim matmul; GGUF rows through the
quant.nim dequantisers), qk-norm, RoPE, K/V store, attention, residual +
rmsnorm, SiLU * up, down, residual, final norm, output projection, argmax.
Several steps chain on the device; the oracle follows the same tokens.
Bar: logits within 1e-4 (fp32) at every step, and the next token equal to
the reference argmax of the GPU's logits."""
import numpy as np
import pytest
import torch

from gguf_pack import random_rows
from hippo_leap_amd import _lib
from util import TOL_F32, rel_err

pytestmark = pytest.mark.gpu


def _weights(rng, orc, rows, cols, qtype, seed):
    """(device tensor, dense fp32 [rows, cols] the oracle multiplies by)."""
    if qtype == 0:
        w = (orc.normal(rows * cols, seed) / np.float32(np.sqrt(cols))).astype(np.float32)
        w = w.reshape(rows, cols)
        return torch.from_numpy(w).cuda(), w
    raw = random_rows(rng, qtype, rows, cols)
    return torch.from_numpy(raw).cuda(), orc.dequant_rows(qtype, raw, rows, cols)


def _build(orc, cfg, types, qk_norm, seed):
    rng = np.random.default_rng(seed)
    E, D, ff, V = cfg["n_emb"], cfg["head_dim"], cfg["n_ff"], cfg["n_vocab"]
    q, kv = cfg["n_head"] * D, cfg["n_head_kv"] * D
    shapes = {"wq": (q, E), "wk": (kv, E), "wv": (kv, E), "wo": (E, q), "w_gate": (ff, E),
              "w_up": (ff, E), "w_down": (E, ff)}
    dev_layers, ref_layers = [], []
    s = seed * 100
    for _ in range(cfg["n_layer"]):
        dl, rl = {}, {}
        for n, (r, c) in shapes.items():
            s += 1
            dl[n], rl[n] = _weights(rng, orc, r, c, types.get(n, 0), s)
            dl[n + "_type"] = types.get(n, 0)
        for n, size in (("attn_norm", E), ("ffn_norm", E)) + ((("q_norm", D), ("k_norm", D)) if qk_norm else ()):
            s += 1
            rl[n] = orc.uniform(size, s, 0.5, 1.5)
            dl[n] = torch.from_numpy(rl[n]).cuda()
        for n in ("k_cache", "v_cache"):
            rl[n] = np.zeros((kv, cfg["max_len"]), np.float32)
            dl[n] = torch.zeros(kv, cfg["max_len"], device="cuda")
        dev_layers.append(dl)
        ref_layers.append(rl)
    emb = orc.normal(V * E, seed + 1).reshape(V, E)
    onorm = orc.uniform(E, seed + 2, 0.5, 1.5)
    out_d, out_r = _weights(rng, orc, V, E, types.get("output", 0), seed + 3)
    dev = dict(tok_emb=torch.from_numpy(emb).cuda(), output_norm=torch.from_numpy(onorm).cuda(),
               output=out_d, output_type=types.get("output", 0), layers=dev_layers)
    ref = dict(tok_emb=emb, output_norm=onorm, output=out_r, layers=ref_layers)
    return dev, ref


def _oracle_step(orc, cfg, ref, tok, pos):
    E, D, eps = cfg["n_emb"], cfg["head_dim"], cfg["rms_eps"]
    H, Hkv, ff = cfg["n_head"], cfg["n_head_kv"], cfg["n_ff"]
    q_dim, kv_dim, L = H * D, Hkv * D, cfg["max_len"]
    theta = orc.theta_table(cfg["rope_dim"], cfg["rope_base"])
    mv = lambda w, v: orc.matmul(w, v.reshape(-1, 1)).reshape(-1)
    norm = lambda v, w: orc.rmsnorm_cols(v.reshape(-1, 1), w, eps).reshape(-1)
    x = orc.embedding(ref["tok_emb"], [tok], E).reshape(-1)
    xn = norm(x, ref["layers"][0]["attn_norm"])
    for li, lw in enumerate(ref["layers"]):
        q, k, v = mv(lw["wq"], xn), mv(lw["wk"], xn), mv(lw["wv"], xn)
        if "q_norm" in lw:
            q = orc.qk_norm(q, lw["q_norm"], H, D, eps)
            k = orc.qk_norm(k, lw["k_norm"], Hkv, D, eps)
        q = orc.rope_heads(q, H, D, cfg["rope_dim"], theta, pos)
        k = orc.rope_heads(k, Hkv, D, cfg["rope_dim"], theta, pos)
        orc.store_kv(lw["k_cache"], orc.F32, k.reshape(kv_dim, 1), kv_dim, 1, L, pos)
        orc.store_kv(lw["v_cache"], orc.F32, v.reshape(kv_dim, 1), kv_dim, 1, L, pos)
        a = orc.attention_decode(q, lw["k_cache"], lw["v_cache"], H, Hkv, D, pos + 1, L)
        x = (x + mv(lw["wo"], a)).astype(np.float32)
        xn = norm(x, lw["ffn_norm"])
        g, u = mv(lw["w_gate"], xn), mv(lw["w_up"], xn)
        with np.errstate(over="ignore"):  # exp(-g) -> inf gives silu's limit 0
            h = (g * (np.float32(1) / (np.float32(1) + np.exp(-g))) * u).astype(np.float32)
        x = (x + mv(lw["w_down"], h)).astype(np.float32)
        if li + 1 < len(ref["layers"]):
            xn = norm(x, ref["layers"][li + 1]["attn_norm"])
    return mv(ref["output"], norm(x, ref["output_norm"]))


CFG = dict(n_layer=2, n_emb=256, n_head=4, n_head_kv=2, head_dim=64, rope_dim=64, n_ff=512,
           n_vocab=300, max_len=16, rms_eps=1e-6, rope_base=1e4)
CASES = [
    ("fp32", {}, False),
    ("fp32_qknorm", {}, True),  # Qwen3-style per-head q/k norm
    ("gguf", {"wq": 12, "wk": 8, "wv": 14, "wo": 13, "w_gate": 12, "w_up": 11, "w_down": 14,
              "output": 14}, True),
    # gate/up and K/V of one type: the fused launches
    ("gguf_fused", {"wq": 12, "wk": 12, "wv": 12, "wo": 12, "w_gate": 12, "w_up": 12, "w_down": 14,
                    "output": 14}, False),
    ("gguf_fused_q8", {"wq": 8, "wk": 8, "wv": 8, "wo": 8, "w_gate": 8, "w_up": 8, "w_down": 8,
                       "output": 8}, True),
]


@pytest.mark.parametrize("name,types,qk_norm", CASES, ids=[c[0] for c in CASES])
def test_forward_decode_token_matches_oracle(hl, orc, name, types, qk_norm):
    from hippo_leap_amd.model import DenseDecoder
    print(f"decode model case {name}", flush=True)
    dev, ref = _build(orc, CFG, types, qk_norm, 31 + len(name))
    m = DenseDecoder(torch, CFG, dev["tok_emb"], dev["output_norm"], dev["output"],
                     dev["output_type"], dev["layers"])
    tok = 7
    m.tokens[0] = tok
    for pos in range(6):
        m.step(pos, m.tokens[0:1], m.tokens[1:2])
        torch.cuda.synchronize()
        logits = m.logits.cpu().numpy()
        nxt = int(m.tokens[1].item())
        ref_logits = _oracle_step(orc, CFG, ref, tok, pos)
        assert rel_err(logits, ref_logits) < TOL_F32, f"step {pos}"
        assert nxt == orc.argmax(logits)
        m.tokens[0] = nxt
        tok = nxt


# Width 2048: the direct kernels split each row's blocks over four waves
# (the three-matrix Q/K/V launch included), F16 and Q8_0 weights.
CFG_WIDE = dict(CFG, n_emb=2048, n_head=32, n_head_kv=8, n_ff=1024)


@pytest.mark.parametrize("types", [{"wq": 1, "wk": 1, "wv": 1, "wo": 8, "w_gate": 8, "w_up": 8, "w_down": 8},
                                   {"wq": 8, "wk": 8, "wv": 8, "wo": 8, "w_gate": 8, "w_up": 8, "w_down": 8}],
                         ids=["qkv_f16", "qkv_q8_0"])
def test_forward_decode_token_wide_fused_projections(hl, orc, types):
    from hippo_leap_amd.model import DenseDecoder
    print(f"decode model wide {types['wq']}", flush=True)
    dev, ref = _build(orc, CFG_WIDE, types, False, 97)
    m = DenseDecoder(torch, CFG_WIDE, dev["tok_emb"], dev["output_norm"], dev["output"],
                     dev["output_type"], dev["layers"])
    tok = 5
    m.tokens[0] = tok
    for pos in range(3):
        m.step(pos, m.tokens[0:1], m.tokens[1:2])
        torch.cuda.synchronize()
        logits = m.logits.cpu().numpy()
        ref_logits = _oracle_step(orc, CFG_WIDE, ref, tok, pos)
        assert rel_err(logits, ref_logits) < TOL_F32, f"step {pos}"
        tok = int(m.tokens[1].item())
        m.tokens[0] = tok


# Q4_K gate/up of 2^25 weights each: the matrix-core pair kernel with the
# residual + FFN norm folded into its x prologue (the sum parked in the norm
# buffer until the next residual moves it back).
# n_ff 8192: 2^24 weights per matrix, 2^25 for the pair.
CFG_FFN = dict(CFG, n_emb=2048, n_head=32, n_head_kv=8, n_ff=16384)


# The fold at other widths: on the int8 kernel K = 4096 (one step of sixteen
# waves, the Llama-3-8B width), 8192 (two steps) and 2560 (ten waves); on the
# fp16 kernel K = 1792 (seven blocks of a group of eight: threads past K/8 load
# zeros and write no sum).
@pytest.mark.parametrize("n_emb,n_ff", [(2048, 16384), (2048, 8192), (4096, 4096), (8192, 2048), (2560, 6656),
                                        (1792, 9472)])
def test_forward_decode_token_norm_folded_into_gate_up(hl, orc, launches, n_emb, n_ff):
    from hippo_leap_amd.model import DenseDecoder
    types = {"wq": 12, "wk": 12, "wv": 12, "wo": 12, "w_gate": 12, "w_up": 12, "w_down": 12}
    print(f"decode model: norm folded into the Q4_K gate/up, n_emb {n_emb} n_ff {n_ff}", flush=True)
    cfg = dict(CFG_FFN, n_emb=n_emb, n_ff=n_ff)
    dev, ref = _build(orc, cfg, types, False, 131)
    m = DenseDecoder(torch, cfg, dev["tok_emb"], dev["output_norm"], dev["output"],
                     dev["output_type"], dev["layers"])
    tok = 9
    m.tokens[0] = tok
    for pos in range(3):
        m.step(pos, m.tokens[0:1], m.tokens[1:2])
        torch.cuda.synchronize()
        logits = m.logits.cpu().numpy()
        ref_logits = _oracle_step(orc, cfg, ref, tok, pos)
        assert rel_err(logits, ref_logits) < TOL_F32, f"step {pos}"
        tok = int(m.tokens[1].item())
        m.tokens[0] = tok
    fp16 = n_emb == 1792
    assert launches(_lib.HL_LK_Q4K_MFMA_NORM) == (3 * cfg["n_layer"] if fp16 else 0)
    assert (launches(_lib.HL_LK_I8_NORM) >= 3 * cfg["n_layer"]) == (not fp16)


# The folds of the Q/K/V and gate/up launches at the Llama-3-8B width: K = 4096
# is one step of sixteen waves, for Q8_0 two steps of eight.
@pytest.mark.parametrize("qtype", [8, 12, 13, 14])
def test_forward_decode_folds_at_width_4096(hl, orc, launches, qtype):
    from hippo_leap_amd.model import DenseModel
    print(f"decode model: folds at width 4096, type {qtype}", flush=True)
    cfg = dict(CFG_WIDE, n_emb=4096, n_ff=6144)
    types = {n: qtype for n in ("wq", "wk", "wv", "wo", "w_gate", "w_up", "w_down", "output")}
    dev, ref = _build(orc, cfg, types, False, 211)
    m = DenseModel(torch, cfg, dev["tok_emb"], dev["output_norm"], dev["output"], dev["output_type"], dev["layers"])
    tok = 9
    for pos in range(2):
        m.tokens[0] = tok
        m.decode()
        torch.cuda.synchronize()
        logits = m.logits.cpu().numpy()
        assert rel_err(logits, _oracle_step(orc, cfg, ref, tok, pos)) < TOL_F32, f"step {pos}"
        _check_hidden(m.fbufs, cfg, ref, logits)
        tok = int(m.tokens[1].item())
    # gate/up of both layers, Q/K/V of the second
    assert launches(_lib.HL_LK_I8_NORM) == 2 * (2 * cfg["n_layer"] - 1)


# Residual + norm folded into the Q/K/V launch (3072 x 2048), of one type;
# scratch wide enough for q behind the residual (n_ff >= 2 n_emb), at 4032 it
# is not.  The head does not fold: it leaves the residual stream in x and the
# final norm in x_norm.  logits may lie in tmp0, which it is done with.
def _check_hidden(bufs, cfg, ref, logits):
    """x and x_norm after a step: the residual stream (its norm times the
    output weights gives the logits) and its final norm."""
    x, xn = (b[:cfg["n_emb"]].cpu().numpy().astype(np.float64) for b in bufs[:2])
    want = x / np.sqrt((x * x).mean() + cfg["rms_eps"]) * ref["output_norm"]
    assert rel_err(xn, want) < TOL_F32
    assert rel_err(logits, ref["output"].reshape(-1, len(xn)).astype(np.float64) @ xn) < TOL_F32


@pytest.mark.parametrize("qtype,n_ff,logits_in_tmp0", [(8, 4096, False), (12, 4352, False), (13, 4096, False),
                                                       (14, 4096, False), (8, 4032, False), (8, 4096, True)])
def test_forward_decode_norm_folded_into_qkv_and_head(hl, orc, qtype, n_ff, logits_in_tmp0):
    from hippo_leap_amd.model import DenseModel
    print(f"decode model: norm folded into Q/K/V and head, type {qtype} n_ff {n_ff}", flush=True)
    cfg = dict(CFG_WIDE, n_layer=3, n_ff=n_ff, n_vocab=2100)
    types = {"wq": qtype, "wk": qtype, "wv": qtype, "wo": 8, "w_gate": 8, "w_up": 8, "w_down": 8, "output": qtype}
    dev, ref = _build(orc, cfg, types, False, 173)
    m = DenseModel(torch, cfg, dev["tok_emb"], dev["output_norm"], dev["output"], dev["output_type"], dev["layers"])
    if logits_in_tmp0:
        m.logits = m.fbufs[2][:cfg["n_vocab"]]
    tok = 9
    for pos in range(3):
        m.tokens[0] = tok
        m.decode()
        torch.cuda.synchronize()
        logits, nxt = m.logits.cpu().numpy(), int(m.tokens[1].item())
        ref_logits = _oracle_step(orc, cfg, ref, tok, pos)
        assert rel_err(logits, ref_logits) < TOL_F32, f"step {pos}"
        assert nxt == orc.argmax(logits)
        _check_hidden(m.fbufs, cfg, ref, logits)
        if not logits_in_tmp0:  # the descriptor's own caches, same step
            m.step(pos)
            torch.cuda.synchronize()
            assert rel_err(m.logits.cpu().numpy(), ref_logits) < TOL_F32, f"step {pos}"
            _check_hidden(m.bufs, cfg, ref, m.logits.cpu().numpy())
        tok = nxt


def test_forward_decode_token_rope_dim_zero(hl, orc):
    """rope_dim 0 means the whole head, as the reference's ropeDim =
    headDim when the model file has no rope dimension (naive.nim:3979)."""
    from hippo_leap_amd.model import DenseDecoder
    cfg = dict(CFG, rope_dim=0)
    dev, ref = _build(orc, cfg, {}, False, 71)
    m = DenseDecoder(torch, cfg, dev["tok_emb"], dev["output_norm"], dev["output"], 0, dev["layers"])
    tok = 11
    for pos in range(3):
        m.tokens[0] = tok
        m.step(pos)
        torch.cuda.synchronize()
        logits = m.logits.cpu().numpy()
        assert rel_err(logits, _oracle_step(orc, dict(cfg, rope_dim=cfg["head_dim"]), ref, tok, pos)) < TOL_F32
        tok = int(m.tokens[1].item())


def test_generate_chains_on_device(hl, orc):
    """generate() chains the steps on the device (the next token of one step
    is the next step's input, no host read in between) and gives the tokens
    of step-by-step decoding."""
    from hippo_leap_amd.model import DenseDecoder
    dev, _ = _build(orc, CFG, {}, False, 90)
    m = DenseDecoder(torch, CFG, dev["tok_emb"], dev["output_norm"], dev["output"], 0, dev["layers"])
    toks = m.generate(5, 8)
    for L in dev["layers"]:
        L["k_cache"].zero_()
        L["v_cache"].zero_()
    seq, tok = [], 5
    for pos in range(8):
        m.tokens[0] = tok
        m.step(pos)
        tok = int(m.tokens[1].item())
        seq.append(tok)
    assert toks == seq


def test_elementwise_dropins(hl, orc):
    from hippo_leap_amd import attention as A
    n = 1000
    g = torch.from_numpy(orc.normal(n, 1)).cuda()
    u = torch.from_numpy(orc.normal(n, 2)).cuda()
    out = torch.empty(n, device="cuda")
    A.gpu_silu_mul(out, g, u, n)
    gn, un = g.cpu().numpy(), u.cpu().numpy()
    assert rel_err(out.cpu().numpy(), gn * (1 / (1 + np.exp(-gn.astype(np.float64)))) * un) < 1e-6
    A.gpu_add(out, g, u, n)
    assert np.array_equal(out.cpu().numpy(), gn + un)
    A.gpu_silu_mul(g, g, u, n)  # in place, as the reference's MoE path calls it
    assert rel_err(g.cpu().numpy(), gn * (1 / (1 + np.exp(-gn.astype(np.float64)))) * un) < 1e-6
