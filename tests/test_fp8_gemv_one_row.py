"""The one-row fp8 product against its operands in float64: plain, normalised, with a
residual, gate-up; rows that do not fill the last wave, one unit and many per wave."""

import pytest
import torch

from opsagent_amd import ops

pytestmark = pytest.mark.gpu


def _case(N, K):
    g = torch.Generator(device="cuda").manual_seed(N + K)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    x = (r(1, K) * 2).bfloat16()
    wq, ws = ops.quant_fp8((r(N, K) * K ** -0.5).bfloat16())
    wd = wq.view(torch.float8_e4m3fn).double() * ws.double()[:, None]
    return x, wq, ws, wd, (1 + 0.2 * r(K)).bfloat16(), r(1, N).bfloat16()


# one unit, a block and one more, several units a wave, rows of 2 to 7 groups
@pytest.mark.parametrize("N,K", [(2, 2048), (16, 4096), (18, 6144), (4096, 14336), (6144, 4096),
                                 (8194, 2048), (20002, 2048), (14, 16384)])
def test_plain_forms(N, K):
    x, wq, ws, wd, nw, res = _case(N, K)
    xd = x.double()
    xn = xd * torch.rsqrt((xd * xd).mean() + 1e-5) * nw.double()
    for got, row, add in ((ops.linear_fp8(x, wq, ws), xd, 0.0),
                          (ops.linear_norm_fp8(x, nw, 1e-5, wq, ws), xn, 0.0),
                          (ops.linear_addres_fp8(x, wq, ws, res), xd, res.double())):
        ref = row @ wd.T + add
        # float32 sums over K, a few roundings of each term, one rounding to bf16
        bound = (K + 8) * 2.0 ** -24 * (row.abs() @ wd.abs().T) + 2.0 ** -8 * ref.abs() + 1e-30
        assert ((got.double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("I,K", [(1, 2048), (9, 4096), (1408, 2048), (14336, 4096), (8200, 6144)])
def test_gateup(I, K, norm):
    x, wq, ws, wd, nw, _ = _case(2 * I, K)
    row = x.double()
    if norm:
        row = row * torch.rsqrt((row * row).mean() + 1e-5) * nw.double()
    got = ops.gateup_silu_fp8(x, wq, ws, I, nw if norm else None, 1e-5).double()
    g, u = (row @ wd.T).split(I, 1)
    eg, eu = ((K + 8) * 2.0 ** -24 * (row.abs() @ wd.abs().T)).split(I, 1)
    ref = torch.nn.functional.silu(g) * u
    # the halves' errors through silu (slope at most 1.1), float32 exp, one rounding to bf16
    bound = 1.1 * eg * u.abs() + (g.abs() + eg) * eu + 2.0 ** -20 * (g * u).abs() + 2.0 ** -8 * ref.abs()
    assert ((got - ref).abs() <= bound + 1e-30).all()
