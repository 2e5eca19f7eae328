"""End-to-end forwardPrefill followed by forwardDecodeToken on the same KV
cache (backends/naive.nim:3967-4590, 4592-4760; lkAttentionFfn layers),
through hl_forward_prefill / hl_forward_decode over an hl_kv_cache_desc,
against an oracle composed from the pinned oracle pieces in the
reference's order: embedding; per layer rmsnorm, Q/K/V (tensor.nim
matmul), qk-norm, RoPE at positions 0 .. T-1, K/V into the cache, causal
attention, O projection + residual (add), rmsnorm, SiLU(gate) * up, down +
residual; final norm, output projection -> logits [n_vocab, T].  Then
decode steps continue at position T on the cache the prefill left.

The cache may hold fp32 (the reference's), bf16 or fp8 values in the
column-major or tiled layout; the oracle stores the same rounded values
(round to nearest even), so the GPU and the oracle read identical caches.
Bars: 1e-4 for fp32 caches, 2e-3 for bf16/fp8 caches (north star), on the
logits of every column and every decode step; the greedy token of each
step equals the reference argmax of the GPU's logits."""
import numpy as np
import pytest
import torch

from test_gpu_model import _build
from util import TOL_F32, TOL_LOWP, rel_err

pytestmark = pytest.mark.gpu

CFG = dict(n_layer=2, n_emb=256, n_head=4, n_head_kv=2, head_dim=64, rope_dim=0, n_ff=512,
           n_vocab=300, max_len=32, rms_eps=1e-6, rope_base=1e4)


def _stored(orc, x, dt):
    """The values a cache of dtype dt holds for fp32 x (RNE), as fp32."""
    return x if dt == orc.F32 else orc.upcast(orc.to_storage(x, dt), dt).reshape(x.shape)


def _oracle_prefill(orc, cfg, ref, tokens, dt):
    E, D, eps, T = cfg["n_emb"], cfg["head_dim"], cfg["rms_eps"], len(tokens)
    H, Hkv = cfg["n_head"], cfg["n_head_kv"]
    rd = cfg["rope_dim"] or D
    theta = orc.theta_table(rd, cfg["rope_base"])
    x = orc.embedding(ref["tok_emb"], tokens, E)
    for lw in ref["layers"]:
        xn = orc.rmsnorm_cols(x, lw["attn_norm"], eps)
        q, k, v = orc.matmul(lw["wq"], xn), orc.matmul(lw["wk"], xn), orc.matmul(lw["wv"], xn)
        if "q_norm" in lw:
            q = orc.qk_norm_cols(q, lw["q_norm"], H, D, T, eps)
            k = orc.qk_norm_cols(k, lw["k_norm"], Hkv, D, T, eps)
        q = orc.rope_cols(q, H, D, T, rd, theta, 0)
        k = orc.rope_cols(k, Hkv, D, T, rd, theta, 0)
        lw["k_cache"][:, :T] = _stored(orc, k, dt)  # gpuStoreKV at columns 0 .. T-1
        lw["v_cache"][:, :T] = _stored(orc, v, dt)
        a = orc.attention_prefill(q, k, v, H, Hkv, D, T)
        x = orc.add(x, orc.matmul(lw["wo"], a))
        xn = orc.rmsnorm_cols(x, lw["ffn_norm"], eps)
        h = orc.silu_mul(orc.matmul(lw["w_gate"], xn), orc.matmul(lw["w_up"], xn))
        x = orc.add(x, orc.matmul(lw["w_down"], h))
    return orc.matmul(ref["output"], orc.rmsnorm_cols(x, ref["output_norm"], eps))


def _oracle_decode(orc, cfg, ref, tok, pos, dt):
    E, D, eps = cfg["n_emb"], cfg["head_dim"], cfg["rms_eps"]
    H, Hkv, L = cfg["n_head"], cfg["n_head_kv"], cfg["max_len"]
    rd = cfg["rope_dim"] or D
    theta = orc.theta_table(rd, cfg["rope_base"])
    mv = lambda w, v: orc.matmul(w, v.reshape(-1, 1)).reshape(-1)
    norm = lambda v, w: orc.rmsnorm_cols(v.reshape(-1, 1), w, eps).reshape(-1)
    x = orc.embedding(ref["tok_emb"], [tok], E).reshape(-1)
    for lw in ref["layers"]:
        xn = norm(x, lw["attn_norm"])
        q, k, v = mv(lw["wq"], xn), mv(lw["wk"], xn), mv(lw["wv"], xn)
        if "q_norm" in lw:
            q = orc.qk_norm(q, lw["q_norm"], H, D, eps)
            k = orc.qk_norm(k, lw["k_norm"], Hkv, D, eps)
        q = orc.rope_heads(q, H, D, rd, theta, pos)
        k = orc.rope_heads(k, Hkv, D, rd, theta, pos)
        lw["k_cache"][:, pos] = _stored(orc, k, dt)
        lw["v_cache"][:, pos] = _stored(orc, v, dt)
        a = orc.attention_decode(q, lw["k_cache"], lw["v_cache"], H, Hkv, D, pos + 1, L)
        x = orc.add(x, mv(lw["wo"], a))
        xn = norm(x, lw["ffn_norm"])
        h = orc.silu_mul(mv(lw["w_gate"], xn), mv(lw["w_up"], xn))
        x = orc.add(x, mv(lw["w_down"], h))
    return mv(ref["output"], norm(x, ref["output_norm"]))


CASES = [  # (name, kv dtype, layout, qk-norm)
    ("fp32_colmajor", 0, 0, False),
    ("fp32_colmajor_qknorm", 0, 0, True),
    ("bf16_colmajor", 2, 0, False),
    ("f16_tiled_qknorm", 1, 1, True),
    ("fp8_tiled", 3, 1, False),
]


# head dim 128 (the Llama-3-8B / Qwen3 head) with fp32 activations and caches:
# the split-operand prefill kernel at 128 (q dim 512 != n_emb 256)
CFG128 = dict(CFG, head_dim=128)
CASES128 = [("fp32_colmajor_d128", 0, 0, False), ("fp32_colmajor_qknorm_d128", 0, 0, True)]


@pytest.mark.parametrize("name,dt,lay,qk", CASES + CASES128, ids=[c[0] for c in CASES + CASES128])
def test_prefill_then_decode_matches_oracle(hl, orc, name, dt, lay, qk):
    from hippo_leap_amd.model import DenseModel
    print(f"prefill+decode case {name}", flush=True)
    CFG = CFG128 if name.endswith("_d128") else globals()["CFG"]
    dev, ref = _build(orc, CFG, {}, qk, 77 + len(name))
    T = 12
    m = DenseModel(torch, CFG, dev["tok_emb"], dev["output_norm"], dev["output"], 0, dev["layers"],
                   max_tokens=T, kv_dtype=dt, kv_layout=lay)
    for lw in ref["layers"]:
        lw["k_cache"] = np.zeros((CFG["n_head_kv"] * CFG["head_dim"], CFG["max_len"]), np.float32)
        lw["v_cache"] = np.zeros_like(lw["k_cache"])
    tokens = [int(t) for t in np.random.default_rng(5).integers(0, CFG["n_vocab"], T)]
    logits = m.prefill(tokens)
    torch.cuda.synchronize()
    assert m.cache.cur_len == T
    tol = TOL_F32 if dt == 0 else TOL_LOWP
    ref_logits = _oracle_prefill(orc, CFG, ref, tokens, dt)
    got = logits.cpu().numpy()
    for t in range(T):  # every column (token) against the oracle's
        assert rel_err(got[:, t], ref_logits[:, t]) < tol, f"prefill column {t}"
    # the reference's generate: first token = argmax of the last column
    tok = orc.argmax(got[:, T - 1])
    m.tokens[0] = tok
    for step in range(5):
        pos = T + step
        m.decode()
        torch.cuda.synchronize()
        assert m.cache.cur_len == pos + 1
        lg = m.logits.cpu().numpy()
        assert rel_err(lg, _oracle_decode(orc, CFG, ref, tok, pos, dt)) < tol, f"decode step {step}"
        nxt = int(m.tokens[1].item())
        assert nxt == orc.argmax(lg)
        m.tokens[0] = nxt
        tok = nxt


def test_decode_full_cache_is_refused(hl, orc):
    """A decode step at cur_len == max_len returns "KV cache full" (the
    reference's ValueError, naive.nim:4598-4599) and changes nothing."""
    from hippo_leap_amd import _lib
    from hippo_leap_amd.model import DenseModel
    dev, _ = _build(orc, CFG, {}, False, 99)
    m = DenseModel(torch, CFG, dev["tok_emb"], dev["output_norm"], dev["output"], 0, dev["layers"],
                   max_tokens=CFG["max_len"])
    m.prefill(list(range(CFG["max_len"])))
    torch.cuda.synchronize()
    with pytest.raises(_lib.HLError, match="KV cache full"):
        m.decode()
    assert m.cache.cur_len == CFG["max_len"]


def test_decode_only_with_gguf_weights(hl, orc):
    """hl_forward_decode with quantized weights (the reference's decode
    takes GGUF rows through gpuLinearColQuant) and a bf16 cache, from an
    empty cache: every step writes its column and attends over the columns
    before it."""
    from hippo_leap_amd.model import DenseModel
    types = {"wq": 12, "wk": 12, "wv": 12, "wo": 8, "w_gate": 14, "w_up": 14, "w_down": 13, "output": 14}
    dev, ref = _build(orc, CFG, types, True, 123)
    m = DenseModel(torch, CFG, dev["tok_emb"], dev["output_norm"], dev["output"], 14, dev["layers"],
                   kv_dtype=2)
    for lw in ref["layers"]:
        lw["k_cache"] = np.zeros((CFG["n_head_kv"] * CFG["head_dim"], CFG["max_len"]), np.float32)
        lw["v_cache"] = np.zeros_like(lw["k_cache"])
    tok = 3
    m.tokens[0] = tok
    for pos in range(6):
        m.decode()
        torch.cuda.synchronize()
        lg = m.logits.cpu().numpy()
        assert rel_err(lg, _oracle_decode(orc, CFG, ref, tok, pos, 2)) < TOL_LOWP, f"step {pos}"
        tok = int(m.tokens[1].item())
        assert tok == orc.argmax(lg)
        m.tokens[0] = tok


def test_decode_timed_matches_decode(hl, orc):
    """hl_forward_decode_timed (forwardDecodeTokenTimed, megakernel.nim:
    2514-2529): the same tokens and logits as hl_forward_decode on a twin
    model, a positive GPU time below the host's wall time of the call, and
    HL_ECAPTURE under stream capture."""
    import time
    from hippo_leap_amd import _lib
    from hippo_leap_amd.model import DenseModel
    dev, ref = _build(orc, CFG, {}, True, 321)
    twins = [DenseModel(torch, CFG, dev["tok_emb"], dev["output_norm"], dev["output"], 0, dev["layers"],
                        max_tokens=4, kv_dtype=2) for _ in range(2)]
    for m in twins:
        m.prefill([1, 2, 3, 4])
        m.tokens[0] = 7
    torch.cuda.synchronize()
    for step in range(4):
        twins[0].decode()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        tok, ms = twins[1].decode_timed()
        wall_ms = (time.perf_counter() - t0) * 1e3
        assert 0.0 < ms < wall_ms, (ms, wall_ms)
        assert tok == int(twins[0].tokens[1].item()) == int(twins[1].tokens[1].item())
        assert np.array_equal(twins[0].logits.cpu().numpy(), twins[1].logits.cpu().numpy())
        assert twins[1].cache.cur_len == twins[0].cache.cur_len == 5 + step
        for m in twins:
            m.tokens[0] = tok
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with pytest.raises(_lib.HLError, match="capture"):
        with torch.cuda.graph(g, stream=s):
            twins[1].decode_timed(stream=s)


# The merged prefill launches (Q/K/V as one row list, gate/up with SiLU * up
# on the sums, the residual added on the way out) at ragged rows of each
# matrix and every tile size of either, against float64.  wide: gate and up
# rows with one element far above the rest, whose tiles leave the split's
# range and are computed a second time (w_down takes the size out again).
# Bound: the fp32 model bar, on logits and on the cached K and V.
@pytest.mark.parametrize("E,H,Hkv,ff,T,wide", [(72, 2, 1, 100, 3, False), (160, 4, 2, 331, 37, True),
                                               (512, 8, 2, 1003, 301, True), (512, 16, 4, 4003, 301, False),
                                               (512, 8, 2, 4003, 1000, True), (256, 32, 16, 2057, 303, False),
                                               (1024, 16, 4, 2500, 300, True)])
def test_prefill_merged_launches(hl, E, H, Hkv, ff, T, wide):
    from hippo_leap_amd.model import DenseModel
    print(f"prefill merged launches E={E} H={H}/{Hkv} ff={ff} T={T} wide={wide}", flush=True)
    D, V = 64, 70
    cfg = dict(n_layer=2, n_emb=E, n_head=H, n_head_kv=Hkv, head_dim=D, rope_dim=D, n_ff=ff, n_vocab=V,
               max_len=T + 5, rms_eps=1e-6, rope_base=1e4)
    g = torch.Generator(device="cuda").manual_seed(E + ff + T)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)
    shapes = {"wq": (H * D, E), "wk": (Hkv * D, E), "wv": (Hkv * D, E), "wo": (E, H * D), "w_gate": (ff, E),
              "w_up": (ff, E), "w_down": (E, ff)}
    layers = []
    for _ in range(2):
        L = {n: rnd(*s) / s[1] ** 0.5 for n, s in shapes.items()}
        if wide:
            for n, r in (("w_up", 7), ("w_gate", ff - 1)):
                L[n][r, -1] += 3e5
                L["w_down"][:, r] *= 3e-6
        L["attn_norm"], L["ffn_norm"] = 1 + 0.1 * rnd(E), 1 + 0.1 * rnd(E)
        L["k_cache"], L["v_cache"] = (torch.zeros(Hkv * D, T + 5, device="cuda") for _ in range(2))
        layers.append(L)
    emb, onorm, out = rnd(V, E), 1 + 0.1 * rnd(E), rnd(V, E) / E ** 0.5
    m = DenseModel(torch, cfg, emb, onorm, out, 0, layers, max_tokens=T)
    tokens = torch.randint(V, (T,), device="cuda", generator=g, dtype=torch.int32)
    logits = m.prefill(tokens)
    torch.cuda.synchronize()

    norm = lambda x, w: x / (x.pow(2).mean(0, True) + 1e-6).sqrt() * w.double()[:, None]
    ang = torch.arange(T, device="cuda").double() * (1e4 ** (-torch.arange(D // 2, device="cuda").double() * 2 / D))[:, None]
    c, s = ang.cos(), ang.sin()

    def rope(x):
        a, b = x.view(-1, D, T).split(D // 2, 1)
        return torch.cat([a * c - b * s, a * s + b * c], 1)

    x = emb.double()[tokens.long()].T
    for i, L in enumerate(layers):
        w = {n: L[n].double() for n in shapes}
        xn = norm(x, L["attn_norm"])
        q, k, v = rope(w["wq"] @ xn), rope(w["wk"] @ xn), (w["wv"] @ xn).view(-1, D, T)
        for cache, ref in ((m.cache.k[i], k), (m.cache.v[i], v)):
            got = cache.view(torch.float32).view(Hkv * D, T + 5)[:, :T]
            assert rel_err(got.cpu(), ref.reshape(Hkv * D, T).cpu()) < TOL_F32
        heads = []
        for h in range(H):
            p = (q[h].T @ k[h * Hkv // H] / D ** 0.5).masked_fill(
                torch.ones(T, T, device="cuda", dtype=torch.bool).triu(1), float("-inf")).softmax(1)
            heads.append(v[h * Hkv // H] @ p.T)
        x = x + w["wo"] @ torch.cat(heads)
        xn = norm(x, L["ffn_norm"])
        x = x + w["w_down"] @ (torch.nn.functional.silu(w["w_gate"] @ xn) * (w["w_up"] @ xn))
    ref = out.double() @ norm(x, onorm)
    assert rel_err(logits.cpu(), ref.cpu()) < TOL_F32


# Scratch buffers that overlap are refused as the projections' own entry
# points refuse them, also where one launch covers several of those calls.
@pytest.mark.parametrize("T", [1, 5])
@pytest.mark.parametrize("buf,onto", [("tmp0", "x_norm"), ("tmp1", "x_norm"), ("tmp2", "x_norm"), ("tmp2", "tmp0")])
def test_prefill_refuses_overlapping_scratch(hl, orc, T, buf, onto):
    from hippo_leap_amd import _lib
    from hippo_leap_amd.model import DenseModel
    print(f"prefill overlapping scratch {buf} -> {onto} T={T}", flush=True)
    dev, _ = _build(orc, CFG, {}, False, 7)
    m = DenseModel(torch, CFG, dev["tok_emb"], dev["output_norm"], dev["output"], 0, dev["layers"], max_tokens=8)
    setattr(m.fscratch, buf, getattr(m.fscratch, onto))
    with pytest.raises(_lib.HLError, match="overlap|alias"):
        m.prefill(list(range(T)))
    torch.cuda.synchronize()


# tmp0 (tmp1) of n_ff columns reaching into x_norm behind the n_emb and
# n_head * head_dim columns that the projections before gate / up write there.
@pytest.mark.parametrize("T", [1, 5])
@pytest.mark.parametrize("buf", ["tmp0", "tmp1"])
def test_prefill_refuses_gate_and_up_reaching_into_x_norm(hl, orc, T, buf):
    from hippo_leap_amd import _lib
    from hippo_leap_amd.model import DenseModel
    print(f"prefill {buf} reaching into x_norm T={T}", flush=True)
    cfg = dict(CFG, n_ff=4 * max(CFG["n_emb"], CFG["n_head"] * CFG["head_dim"]))
    dev, _ = _build(orc, cfg, {}, False, 7)
    m = DenseModel(torch, cfg, dev["tok_emb"], dev["output_norm"], dev["output"], 0, dev["layers"], max_tokens=8)
    n = cfg["n_ff"] // 4 * T
    both = torch.zeros(8 * cfg["n_ff"], device="cuda")
    setattr(m.fscratch, buf, both.data_ptr())
    m.fscratch.x_norm = both[n:].data_ptr()
    with pytest.raises(_lib.HLError, match="overlap"):
        m.prefill(list(range(T)))
    torch.cuda.synchronize()


def test_decode_refuses_overlapping_norm_buffer(hl):
    """x_norm on x: the residual norm refuses it, also at a size whose Q/K/V
    and gate/up launches could take the norm in."""
    from hippo_leap_amd import _lib
    from hippo_leap_amd.model import DenseModel
    E, ff, V = 2048, 2048, 64
    cfg = dict(n_layer=2, n_emb=E, n_head=32, n_head_kv=8, head_dim=64, rope_dim=64, n_ff=ff, n_vocab=V, max_len=32,
               rms_eps=1e-6, rope_base=1e4)
    rows = {"wq": 2048, "wk": 512, "wv": 512, "wo": E, "w_gate": ff, "w_up": ff, "w_down": E}
    layers = []
    for _ in range(2):
        L = {n: torch.zeros(r, E // 256 * 144, dtype=torch.uint8, device="cuda") for n, r in rows.items()}
        L.update({n + "_type": _lib.HL_GGML_Q4_K for n in rows})
        L["attn_norm"], L["ffn_norm"] = (torch.ones(E, device="cuda") for _ in range(2))
        L["k_cache"], L["v_cache"] = (torch.zeros(512, 32, device="cuda") for _ in range(2))
        layers.append(L)
    m = DenseModel(torch, cfg, torch.randn(V, E, device="cuda"), torch.ones(E, device="cuda"),
                   torch.zeros(V, E, device="cuda"), 0, layers)
    m.fscratch.x_norm = m.fscratch.x
    with pytest.raises(_lib.HLError, match="norm_out overlaps x"):
        m.decode()
    torch.cuda.synchronize()
