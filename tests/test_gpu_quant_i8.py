"""GPU: the int8 matrix-core GEMV (Q4_K, Q5_K, Q6_K, Q8_0 matrices of 2^25
weights and more through hl_gpu_linear_col_quant, the fused gate/up and K/V
entry points) against the oracle's dequantisers and float64 products, at row
counts off the 16-row groups and widths of one and several steps.

Bound: products and group sums are exact; what rounds in fp32 is each group's
scaling and the sum over at most 64 of them per lane, 4 lanes and 16 waves:
100 roundings of partial sums, each at most about twice the largest output:
200 2^-24 = 1.2e-5 of it."""
import numpy as np
import pytest
import torch

from gguf_pack import random_rows
from hippo_leap_amd import _lib

pytestmark = pytest.mark.gpu
BOUND = 1.2e-5
Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14


def _weights(orc, qtype, rows, cols, seed):
    """GGUF rows (a block of 256 rows tiled, shifted by seed) and their float64 values."""
    n = min(rows, 256)
    raw = random_rows(np.random.default_rng(seed), qtype, n, cols)
    dense = orc.dequant_rows(qtype, raw, n, cols)
    reps = -(-rows // n)
    w = torch.from_numpy(raw.reshape(n, -1)).cuda().repeat(reps, 1)[:rows].contiguous()
    d = torch.from_numpy(np.asarray(dense, np.float64).reshape(n, cols)).cuda()
    return w, lambda v: (d @ v.double()).repeat(reps)[:rows]


def _x(K, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(K, device="cuda", generator=g)
    x[::97] *= 50.0
    x[256:512] = 0.0        # a superblock of zeros
    x[512:768] *= 1e-20
    x[768:1024] *= 1e-42    # subnormal
    return x


def _close(got, ref):
    err = (got.double() - ref).abs().max().item() / max(ref.abs().max().item(), 1e-30)
    assert err < BOUND, err


SHAPES = [(20471, 2048), (20200, 2304), (16375, 3840), (12279, 4096), (12200, 4352), (8187, 4864), (4087, 8704),
          (4081, 14336), (4090, 16384)]
# Q6_K takes multiples of eight superblocks and 40 million weights, Q8_0 below
# K = 4096 1.5 2^25 weights; the others of these run on the vector ALUs.
SHAPES_OF = {Q4_K: SHAPES, Q5_K: SHAPES,
             Q6_K: SHAPES + [(8180, 6144), (8187, 8192)],
             Q8_0: SHAPES + [(24583, 2048), (23000, 2304), (27999, 2304)]}
ON_ALUS = [(Q6_K, M, K) for M, K in SHAPES if K in (2304, 3840, 4352, 4864, 8704)] + [
    (Q8_0, 20471, 2048), (Q8_0, 20200, 2304), (Q8_0, 12283, 2048), (Q6_K, 6100, 4352)]


def _took(launches, qtype, M, K, n):
    alus = (qtype, M, K) in ON_ALUS
    assert (launches(_lib.HL_LK_QUANT), launches(_lib.HL_LK_I8)) == ((n, 0) if alus else (0, n))


@pytest.mark.parametrize("qtype,M,K", [(q, *s) for q, shapes in SHAPES_OF.items() for s in shapes])
def test_one(hl, orc, launches, qtype, M, K):
    from hippo_leap_amd import attention as A
    print(f"int8 gemv type {qtype} M={M} K={K}", flush=True)
    w, times = _weights(orc, qtype, M, K, M + qtype)
    x = _x(K, K)
    y = torch.full((M + 32,), 3.25, device="cuda")
    A.gpu_linear_col_quant(y, x, w, K, M, qtype)
    _close(y[:M], times(x))
    assert bool((y[M:] == 3.25).all())
    again = torch.empty(M, device="cuda")
    A.gpu_linear_col_quant(again, x, w, K, M, qtype)
    assert torch.equal(again, y[:M])
    _took(launches, qtype, M, K, 2)


PAIRS = [(12283, 2048), (6139, 4096), (6100, 4352), (4093, 8192), (4083, 14336)]
PAIRS_OF = {Q4_K: PAIRS, Q5_K: PAIRS, Q6_K: PAIRS + [(8190, 6144)], Q8_0: PAIRS + [(12300, 2048), (14331, 2304)]}


@pytest.mark.parametrize("qtype,M,K", [(q, *s) for q, shapes in PAIRS_OF.items() for s in shapes])
def test_pairs(hl, orc, launches, qtype, M, K):
    from hippo_leap_amd import attention as A
    print(f"int8 pair type {qtype} M={M} K={K}", flush=True)
    wa, ta = _weights(orc, qtype, M, K, M)
    wb, tb = _weights(orc, qtype, M, K, M + 1)
    x = _x(K, K + 1)
    a, b = ta(x), tb(x)
    s = 4.0 / a.abs().max().item()  # keep silu's exponential in range
    x, a, b = (x * s).contiguous(), None, None
    a, b = ta(x), tb(x)
    h = torch.full((M + 8,), 3.25, device="cuda")
    A.gpu_fused_gate_up_silu_quant(h, x, wa, wb, K, M, qtype)
    _close(h[:M], a / (1 + torch.exp(-a)) * b)
    assert bool((h[M:] == 3.25).all())
    k, v = torch.empty(M, device="cuda"), torch.empty(M, device="cuda")
    A.gpu_fused_kv_linear_quant(k, v, x, wa, wb, K, M, qtype, qtype)
    _close(k, a)
    _close(v, b)
    _took(launches, qtype, M, K, 2)


@pytest.mark.parametrize("qtype,M", [(Q4_K, 20480), (Q5_K, 20480), (Q6_K, 20480), (Q8_0, 20480), (Q8_0, 24583)])
def test_large_and_non_finite_x(hl, orc, launches, qtype, M):
    """x up to the fp32 range is held to 2^-31 of its superblock's largest; an
    inf or NaN in x makes every row NaN (q x summed with its offset or min, as
    in fp32)."""
    from hippo_leap_amd import attention as A
    K = 2048
    w, times = _weights(orc, qtype, M, K, 77)
    x = _x(K, 5) * 1e33
    y = torch.empty(M, device="cuda")
    A.gpu_linear_col_quant(y, x, w, K, M, qtype)
    _close(y, times(x))
    for bad in (float("inf"), float("nan")):
        x[700] = bad
        A.gpu_linear_col_quant(y, x, w, K, M, qtype)
        assert bool(torch.isnan(y).all())
    alus = (qtype, M) == (Q8_0, 20480)
    assert launches(_lib.HL_LK_QUANT if alus else _lib.HL_LK_I8) == 3
