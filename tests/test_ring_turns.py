"""Strips of the transfer ring that start at steps of their own: fewer steps than strips, one step,
runs of columns of unequal length, and which forms the products take."""

import pytest
import torch

from opsagent_amd import ops


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,splits", [(3, 4104, 64, 1), (40, 2056, 192, 1), (17, 3000, 704, 3),
                                          (77, 5000, 512, 1), (128, 2304, 1088, 5)])
@pytest.mark.parametrize("narrow", [False, True])
def test_turned(M, N, K, splits, narrow):
    """Whole numbers: every product and sum is exact in whatever order."""
    torch.manual_seed(M + N + K)
    x, w = (torch.randint(-2, 3, (r, K), device="cuda").bfloat16() for r in (M, 2 * N))
    tile = min(32 * -(-M // 32), 64 if narrow else 128)
    want = x.double() @ w.double().T
    got = ops._ring(x, w[:N], (tile, splits, narrow))
    assert torch.equal(got, want[:, :N].to(torch.bfloat16))
    both = ops._ring(x, w, (tile, splits, narrow), act=1).double()
    f = torch.nn.functional.silu(want[:, :N]) * want[:, N:]
    # one rounding to bf16, and float32 roundings of exp of up to |g| / ln 2 scaled bits
    bound = 2.0 ** -8 * f.abs() + 2.0 ** -20 * (1 + want[:, :N].abs()) * (want[:, :N] * want[:, N:]).abs()
    assert ((both - f).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(3, 20288, 1664), (24, 12288, 4096), (40, 12584, 3520), (112, 32000, 2048)])
def test_products(M, N, K):
    torch.manual_seed(M)
    x = torch.randn(M, K, device="cuda").bfloat16()
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    assert ops._ring_form(M, N, K)
    want = x.double() @ w.double().T
    assert (ops.linear(x, w).double() - want).norm() <= 2.0 ** -8 * want.norm()     # one rounding


def test_forms():
    form = ops._ring_form
    assert form(47, 14336, 4096, True) == (64, 1, False) and form(128, 14336, 4096, True) == (128, 1, False)
    assert form(16, 20288, 1664) == (32, 1, False) and form(40, 12584, 3520) == (64, 2, False)
    assert form(3, 25088, 1024, True) is None and form(3, 2048, 2048) is None       # short rows, light weights
    assert form(24, 14336, 768) is None and form(8, 4096, 14336) == ops._ring_choice(8, 4096, 14336)
    for gateup in (False, True):
        for K in (64, 640, 1408, 2048, 4096, 14336):
            for N in (7, 8, 1024, 3072, 32000, 128256):
                assert form(2, N, K, gateup) == ops._ring_choice(2, N, K, gateup)
                for M in range(3, 129):
                    plan = form(M, N, K, gateup)
                    if plan:
                        assert plan[0] in (32, 64, 96, 128) and 1 <= plan[1] <= K // 64
                        assert not plan[2] or plan[0] <= 64


def test_full_rounds():
    """Gate-up in two tiles of 64 rows that fill the CUs: only where the estimate is far ahead of the
    splits of 128-row tiles, which answer sooner than it knows."""
    for M, N, K in ((103, 7552, 3648), (128, 8128, 4160), (112, 8192, 4032)):
        assert ops._ring_form(M, N, K, True) == ops._ring_choice(M, N, K, True) == (128, 2, False)
    for M, N, K in ((128, 6720, 3264), (128, 7040, 3264), (128, 8192, 2048)):
        assert ops._ring_form(M, N, K, True) == (64, 1, False)


def test_short_rows():
    """Gate-up of 33 to 64 short rows stays in splits of 64-row strips."""
    for M, N, K in ((47, 2816, 2048), (33, 2816, 2048), (46, 2816, 1664), (34, 3008, 1344)):
        assert ops._ring_form(M, N, K, True) == ops._ring_choice(M, N, K, True) == (64, 2, True)
    assert ops._ring_form(38, 3008, 3136, True) == (64, 5, False)
