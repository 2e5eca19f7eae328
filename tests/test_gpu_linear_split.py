"""GPU: the split-operand GEMM of hl_gpu_linear_col (seq_len > 1) at the edges
of its tiles, chunks and column vectors, and with operands that leave the
range of its split (zero runs, values far above a row's first ones,
subnormal rows, inf and NaN), against float64 products of the same inputs.

Bound: each operand is held to 2^-23 of itself and 2^-31 of the largest of a
16-element run of its row (column), three of the four partial products are
kept (the fourth is below 2^-22), and every 16-long sum is added to an fp32
accumulator.  So |error| <= (2^-20 + (K / 16 + 32) 2^-24) |W| |X| + 2^-30
(max|w| sum|x| + max|x| sum|w|) per output; a tile that falls back to fp32
MFMAs accumulates K terms, K 2^-24 more."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _run(w, x):
    from hippo_leap_amd import attention as A
    M, K = w.shape
    T = x.shape[1]
    y = torch.full((M * T + 64,), 7.25, device="cuda")  # 64 guard values behind
    A.gpu_linear_col(y, x, w, K, M, T)
    torch.cuda.synchronize()
    assert bool((y[M * T:] == 7.25).all()), "written past the output"
    return y[:M * T].reshape(M, T)


def _check(w, x, fp32=False):
    K = w.shape[1]
    y = _run(w, x)
    ref = w.double() @ x.double()
    mag = w.double().abs() @ x.double().abs()
    bound = (2.0 ** -20 + ((K if fp32 else 0) + K / 16 + 32) * 2.0 ** -24) * mag
    wa, xa = w.double().abs(), x.double().abs()
    bound += 2.0 ** -30 * (wa.amax(1, True) * xa.sum(0, True) + xa.amax(0, True) * wa.sum(1, True))
    worst = ((y.double() - ref).abs() / bound.clamp_min(1e-300)).max().item()
    assert worst <= 1.0, worst


def _operands(M, K, T, seed, offset=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    w = torch.randn(M * K + offset, device="cuda", generator=g)[offset:].reshape(M, K)
    x = torch.randn(K * T + offset, device="cuda", generator=g)[offset:].reshape(K, T)
    return w, x


SHAPES = [(1, 1, 2), (33, 15, 2), (31, 16, 3), (32, 17, 31), (65, 63, 32), (64, 64, 33), (130, 65, 63), (70, 511, 65),
          (96, 513, 127), (5, 1003, 129), (257, 4099, 7),             # 32 x 32 tiles
          (2048, 512, 301), (2081, 545, 257), (2111, 97, 303),        # 64 x 64
          (8192, 256, 301), (8225, 129, 333),                         # 64 x 64, four waves
          (4096, 256, 1000), (4133, 161, 1027), (3001, 191, 2049)]    # 64 x 128


@pytest.mark.parametrize("M,K,T", SHAPES)
def test_edges(hl, M, K, T):
    print(f"split gemm M={M} K={K} T={T}", flush=True)
    for offset in (0, 1):  # addresses on 16 and on 4 bytes
        _check(*_operands(M, K, T, 17 * M + K + T, offset))


@pytest.mark.parametrize("M,K,T", [(96, 700, 45), (2048, 600, 301), (4096, 300, 1000)])
def test_zero_runs(hl, M, K, T):
    """Rows and columns that start with (or are) zeros: their scale comes from
    their largest element, also where that is far from 1."""
    print(f"split gemm zero runs M={M} K={K} T={T}", flush=True)
    w, x = _operands(M, K, T, 5)
    w[3, :K // 2] = 0.0
    w[3, K // 2:] *= 1e-12
    w[7] = 0.0
    w[9, :-1] = 0.0
    x[:K - 5, 1] = 0.0
    x[:, 1] *= 3e9
    x[:, T - 1] = 0.0
    _check(w, x)


@pytest.mark.parametrize("M,K,T", [(96, 700, 45), (2048, 600, 301), (4096, 300, 1000)])
def test_out_of_split_range(hl, M, K, T):
    """Elements more than 2^9 above the first ones of their row or column,
    and rows below 2^-100: the tile's fp32 MFMAs."""
    print(f"split gemm out of range M={M} K={K} T={T}", flush=True)
    w, x = _operands(M, K, T, 6)
    w[40, K - 1] = 1e9
    x[K - 2, T - 3] = -3e12
    w[65] *= 1e-33
    _check(w, x, fp32=True)


@pytest.mark.parametrize("M,K,T", [(96, 700, 45), (2048, 600, 301), (4096, 300, 1000)])
def test_inf_nan(hl, M, K, T):
    print(f"split gemm inf / nan M={M} K={K} T={T}", flush=True)
    w, x = _operands(M, K, T, 7)
    w[2, K - 1] = float("inf")
    x[K - 1, 4] = 0.0
    w[70, 0] = float("nan")
    x[5, T - 1] = float("-inf")
    w[71, 5] = 0.0
    y = _run(w, x).cpu()
    ref = (w.double() @ x.double()).cpu()
    assert bool((torch.isnan(y) == torch.isnan(ref)).all())
    inf = torch.isinf(ref)
    assert bool((y[inf].double() == ref[inf]).all()) and bool((torch.isinf(y) == inf).all())
    fin = torch.isfinite(ref)
    err = (y.double() - ref)[fin].abs().max().item() / np.sqrt(K)
    assert err < 1e-4  # the bar of the fp32 entry points


def test_graph_replays(hl):
    """The GEMM keeps nothing between calls: replays with a fallback input in
    between give the eager results."""
    from hippo_leap_amd import attention as A
    M, K, T = 300, 520, 77
    w, x = _operands(M, K, T, 8)
    y = torch.empty(M, T, device="cuda")
    A.gpu_linear_col(y, x, w, K, M, T)
    torch.cuda.synchronize()
    first = y.clone()
    st, gr = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(st), torch.cuda.graph(gr, stream=st):
        A.gpu_linear_col(y, x, w, K, M, T)
    keep = x[3, 5].item()
    for i in range(4):
        x[3, 5] = 1e30 if i % 2 else keep
        torch.cuda.synchronize()
        gr.replay()
        torch.cuda.synchronize()
        if i % 2 == 0:
            assert torch.equal(y, first)
        else:
            got = y.clone()
            A.gpu_linear_col(y, x, w, K, M, T)
            torch.cuda.synchronize()
            assert torch.equal(y, got)
