"""GPU: the split-operand GEMM of hl_gpu_linear_col (seq_len > 1) at the edges
of its tiles, chunks and column vectors, and with operands of every fp32 range
(zero runs, elements far above and far below the others of their row, subnormal
parts, inf and NaN), against float64 products of the same inputs.

Bound, per output and without a term in a row's or column's largest element:
the three bf16 parts hold an element whole, the products of parts that are left
out are at most 2^-24 of the element's product, and the six kept ones of 16 k
are each added to an fp32 accumulator with one rounding, K split over at least
four waves, whose sums meet in eight more.  So |error| <= (6 / 4 K / 16 + 8 +
16 + 1) 2^-24 |W| |X|, here (K / 10 + 48) 2^-24; results below the normal range
add 2^-149 per rounding.  A tile that goes to fp32 MFMAs accumulates K terms,
K 2^-24 more."""
import numpy as np
import pytest
import torch

from hippo_leap_amd import _lib

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
    bound = ((K if fp32 else 0) + K / 10 + 48) * 2.0 ** -24 * mag + (K + 48) * 2.0 ** -149
    worst = ((y.double() - ref).abs() / bound).max().item()
    assert worst <= 1.0, worst


def _operands(M, K, T, seed, offset=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    w = torch.randn(M * K + offset, device="cuda", generator=g)[offset:].reshape(M, K)
    x = torch.randn(K * T + offset, device="cuda", generator=g)[offset:].reshape(K, T)
    return w, x


# M, K, T and the tile that takes them.
SHAPES = [(*s, kind) for kind, shapes in {
    _lib.HL_LK_SPLIT_32X32: [(1, 1, 2), (33, 15, 2), (31, 16, 3), (32, 17, 31), (65, 63, 32), (64, 64, 33),
                             (130, 65, 63), (70, 511, 65), (96, 513, 127), (5, 1003, 129), (257, 4099, 7)],
    _lib.HL_LK_SPLIT_64X64_W8: [(2048, 512, 301), (2081, 545, 257), (2111, 97, 303)],
    _lib.HL_LK_SPLIT_64X64_W4: [(8192, 256, 301), (8225, 129, 333), (4096, 256, 1000), (4133, 161, 1027),
                                (3001, 191, 2049)],
    _lib.HL_LK_SPLIT_64X128: [(4096, 1600, 1000), (4033, 1603, 1021), (3969, 1611, 1024), (3905, 2001, 901)],
}.items() for s in shapes]


@pytest.mark.parametrize("M,K,T,kind", SHAPES)
def test_edges(hl, launches, M, K, T, kind):
    print(f"split gemm M={M} K={K} T={T}", flush=True)
    for offset in (0, 1):  # addresses on 16 and on 4 bytes
        _check(*_operands(M, K, T, 17 * M + K + T, offset))
    assert launches(kind) == 2


# One shape for each tile (two for the 64 x 64 one of four waves).
TILES = [(96, 700, 45), (2048, 600, 301), (8225, 270, 333), (4096, 300, 1000), (4033, 1603, 1021)]


@pytest.mark.parametrize("M,K,T", TILES)
def test_zero_runs(hl, M, K, T):
    """Rows and columns that start with (or are) zeros, also far from 1."""
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


@pytest.mark.parametrize("R", [2.0 ** 12, 2.0 ** 20, 2.0 ** 31, 2.0 ** 60, 2.0 ** 100])
@pytest.mark.parametrize("M,K,T", TILES)
def test_large_beside_small(hl, M, K, T, R):
    """Elements R times the others of their row (column), first in every
    64-k chunk, at k = 5 alone, or among any wave's first 16 k, whose partners
    are zero or 1 / R: the small elements' products are the result."""
    print(f"split gemm large beside small M={M} K={K} T={T} R=2^{np.log2(R):.0f}", flush=True)
    for every, partner in ((64, 0.0), (K, 0.0), (64, 1.0 / R), (32, 0.0)):
        at = torch.arange(5 if every == K else 0, K, every, device="cuda")
        for large_in_w in (True, False):
            w, x = _operands(M, K, T, 9)
            a, b = (w, x.t()) if large_in_w else (x.t(), w)
            a[:, at] *= R
            b[:, at] *= partner
            _check(w, x)


@pytest.mark.parametrize("M,K,T", TILES)
def test_far_from_the_first(hl, M, K, T):
    """Single elements far above the first ones of their row or column, and a
    row far below the others."""
    print(f"split gemm far from the first M={M} K={K} T={T}", flush=True)
    w, x = _operands(M, K, T, 6)
    w[40, K - 1] = 1e9
    x[K - 2, T - 3] = -3e12
    w[65] *= 1e-33
    _check(w, x)


@pytest.mark.parametrize("M,K,T", TILES)
def test_small_parts(hl, M, K, T):
    """Rows whose second and third bf16 parts are bf16 subnormals (held, and
    multiplied as they are), and rows with bits below those, which send their
    tiles to fp32 MFMAs; products down to 2^-140."""
    print(f"split gemm small parts M={M} K={K} T={T}", flush=True)
    w, x = _operands(M, K, T, 10)
    w[4] = 2.0 ** -115 * (1.0 + 2.0 ** -16)
    w[20, ::2] = 2.0 ** -109 * (1.0 + 2.0 ** -9 + 2.0 ** -17)
    w[20, 1::2] = 0.0
    _check(w, x)
    w[36] *= 2.0 ** -120
    w[68, :] = 0.0
    w[68, K - 1] = 2.0 ** -140
    x[:, 3] *= 2.0 ** 90
    _check(w, x, fp32=True)


@pytest.mark.parametrize("M,K,T", TILES)
def test_lost_bits(hl, M, K, T):
    """Elements with bits below the parts' range among ordinary ones, and one
    that a partner of 2^100 brings up."""
    print(f"split gemm lost bits M={M} K={K} T={T}", flush=True)
    w, x = _operands(M, K, T, 11)
    x[::3, ::2] *= 2.0 ** -125
    w[1::5, ::7] = 2.0 ** -140
    _check(w, x, fp32=True)
    x[:, 5] = 0.0
    x[7, 5] = 2.0 ** -120 * (1.0 + 2.0 ** -20)
    w[:, 7] = 2.0 ** 100
    _check(w, x, fp32=True)


def test_longest_rows(hl):
    """Rows so long that an element's offset inside a tile needs more than 32
    bits (138.6 million columns: row 31 starts behind 2^32)."""
    from hippo_leap_amd import attention as A
    M, K, T = 32, 138_600_000, 2
    print(f"split gemm longest rows M={M} K={K} T={T}", flush=True)
    w = torch.empty(M, K, device="cuda")
    for r in range(M):
        w[r].fill_(float(r + 1))
    x = torch.zeros(K, T, device="cuda")
    x[::100_003] = torch.tensor([1.0, 3.0], device="cuda")
    x[K - 1] = torch.tensor([2.0, 5.0], device="cuda")
    y = torch.empty(M, T, device="cuda")
    A.gpu_linear_col(y, x, w, K, M, T)
    want = torch.arange(1, M + 1, device="cuda", dtype=torch.float64)[:, None] * x.double().sum(0)
    assert torch.equal(y.double(), want)


@pytest.mark.parametrize("M,K,T", TILES)
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
