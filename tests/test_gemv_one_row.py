"""The one-row GEMV of long rows (K a multiple of 2048) against float64: rows that
do not divide among waves, short and long K, norm prologue, residual, gate-up."""

import pytest
import torch

from opsagent_amd import ops


@pytest.mark.gpu
@pytest.mark.parametrize("N", [8, 16, 4097, 6144, 9001])
@pytest.mark.parametrize("K", [2048, 4096, 6144, 14336])
def test_one_row(N, K):
    gen = torch.Generator(device="cuda").manual_seed(N + K)
    rn = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    x, res = rn(1, K).bfloat16(), rn(1, N).bfloat16()
    w = (rn(N, K) * K ** -0.5).bfloat16()
    nw = (1.0 + 0.1 * rn(K)).bfloat16()
    xd, wd = x.double(), w.double()
    normed = xd / torch.sqrt((xd * xd).mean() + 1e-5) * nw.double()

    def check(got, want):
        # one bf16 rounding of a float32 sum: at most 2^-8 of a value, 0.0016 in the mean
        # over many (a second one would make it 0.0023)
        tol = 2e-3 if want.numel() >= 1024 else 2.0 ** -8 + 1e-5
        assert float((got.double() - want).norm() / want.norm()) < tol

    check(ops.linear(x, w), xd @ wd.T)
    check(ops.linear_norm(x, nw, 1e-5, w), normed @ wd.T)
    # the sum is rounded once, after the residual
    check(ops.linear_addres(x, w, res), xd @ wd.T + res.double())
    if N % 2 == 0:
        h = N // 2
        g, u = (normed @ wd.T).chunk(2, -1)
        check(ops.gateup_silu_norm(x, nw, 1e-5, w, h), g * torch.sigmoid(g) * u)
        g, u = (xd @ wd.T).chunk(2, -1)
        check(ops.gateup_act(x, w, h, "silu"), g * torch.sigmoid(g) * u)
        check(ops.gateup_act(x, w, h, "gelu_tanh"),
              torch.nn.functional.gelu(g, approximate="tanh") * u)


@pytest.mark.gpu
@pytest.mark.parametrize("N,K", [(8, 2048), (4097, 4096), (6144, 2048), (9001, 14336)])
def test_one_row_whole_numbers(N, K):
    """Whole numbers: every float32 sum is exact, the result its one rounding to bf16."""
    gen = torch.Generator(device="cuda").manual_seed(N + K)
    x = torch.randint(-8, 9, (1, K), generator=gen, device="cuda").bfloat16()
    w = torch.randint(-8, 9, (N, K), generator=gen, device="cuda").bfloat16()
    res = torch.randint(-99, 100, (1, N), generator=gen, device="cuda").bfloat16()
    want = x.double() @ w.double().T
    assert torch.equal(ops.linear(x, w), want.bfloat16())
    assert torch.equal(ops.linear_addres(x, w, res), (want + res.double()).bfloat16())


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 4])
@pytest.mark.parametrize("N,K", [(96, 512), (96, 2048)])
def test_weights_with_gaps(M, N, K):
    """Weight rows that lie further apart than they are long, in every entry point."""
    gen = torch.Generator(device="cuda").manual_seed(M + K)
    rn = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    x, res = rn(M, K).bfloat16(), rn(M, N).bfloat16()
    w = (rn(N, K + 64) * K ** -0.5).bfloat16()[:, :K]
    nw = (1.0 + 0.1 * rn(K)).bfloat16()
    xd, wd = x.double(), w.double()
    normed = xd / torch.sqrt((xd * xd).mean(-1, keepdim=True) + 1e-5) * nw.double()

    def check(got, want):
        # roundings of the normed row, of both halves (twofold in silu) and of the result
        assert float((got.double() - want).norm() / want.norm()) < 8e-3

    def silu_halves(y):
        g, u = y.chunk(2, -1)
        return g * torch.sigmoid(g) * u

    check(ops.linear(x, w), xd @ wd.T)
    check(ops.linear_norm(x, nw, 1e-5, w), normed @ wd.T)
    check(ops.linear_addres(x, w, res), xd @ wd.T + res.double())
    check(ops.gateup_silu(x, w, N // 2), silu_halves(xd @ wd.T))
    check(ops.gateup_silu_norm(x, nw, 1e-5, w, N // 2), silu_halves(normed @ wd.T))


@pytest.mark.gpu
def test_three_rows_a_wave():
    """More rows than 32 blocks of four waves per CU take two at a time, some waves with
    one row less: every row once, with its own residual and scale."""
    N, K = 65536 + 70, 2048
    gen = torch.Generator(device="cuda").manual_seed(5)
    rn = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    x, res = rn(1, K).bfloat16(), (10 * rn(1, N)).bfloat16()
    w = (rn(N, K) * K ** -0.5).bfloat16()
    wq, ws = ops.quant_fp8(w)
    want = (x.float() @ w.float().T + res.float())
    want8 = x.float() @ (wq.view(torch.float8_e4m3fn).float() * ws[:, None]).T + res.float()
    # one bf16 rounding of the value and float32 sums of 2048 products of about 1 / sqrt(K)
    for got, ref in ((ops.linear_addres(x, w, res), want),
                     (ops.linear_addres_fp8(x, wq, ws, res), want8)):
        assert ((got.float() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-4).all()


@pytest.mark.gpu
def test_blocks_of_four_and_eight_waves_agree():
    """Both sides of the lines between them: the same sums in the same order."""
    K, gen = 4096, torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(1, K, generator=gen, device="cuda").bfloat16()
    nw = (1.0 + 0.1 * torch.randn(K, generator=gen, device="cuda")).bfloat16()
    w = (torch.randn(16400, K, generator=gen, device="cuda") * K ** -0.5).bfloat16()
    few = torch.cat([w[:8192], w[8200:16392]])
    assert torch.equal(ops.gateup_silu_norm(x, nw, 1e-5, w, 8200)[:, :8192],
                       ops.gateup_silu_norm(x, nw, 1e-5, few, 8192))
    assert torch.equal(ops.linear_norm(x, nw, 1e-5, w[:1025])[:, :1024],
                       ops.linear_norm(x, nw, 1e-5, w[:1024]))
