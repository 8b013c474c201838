"""A sum over pairs whose shared expert is still its product's float32 parts, against that product added up
first; and products of more than 128 rows that are split for the norm behind them."""

import pytest
import torch

from opsagent_amd import ops
from opsagent_amd.engine.model import _product_parts


def added(planes):
    total = planes[0].clone()
    for plane in planes[1:]:
        total += plane
    return total.bfloat16()


@pytest.mark.gpu
@pytest.mark.parametrize("T,top,D,n", [(1, 1, 8, 1), (3, 6, 2048, 2), (130, 2, 1000, 5), (17, 8, 8192, 8)])
def test_pairs(T, top, D, n):
    g = torch.Generator(device="cuda").manual_seed(D + n)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    y, residual, w = rn(T * top, D).bfloat16(), rn(T, D).bfloat16(), (1 + 0.1 * rn(D)).bfloat16()
    planes = rn(n, T, D)
    want, want_r = ops.fused_add_rms_norm(ops.moe_combine(y, top, added(planes), parts=True), residual.clone(), w)
    x = ops.moe_combine(y, top, ops.PlaneSum(planes), parts=True)
    assert isinstance(x, ops.PairSum) and isinstance(x.more, ops.PlaneSum)
    assert torch.equal(ops._added_up(x), ops.moe_combine(y, top, added(planes)))
    got, got_r = ops.fused_add_rms_norm(x, residual, w)
    assert got_r.data_ptr() == residual.data_ptr() and torch.equal(got_r, want_r) and torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("T,N,K", [(129, 4096, 4096), (200, 4096, 4096), (300, 4096, 4096), (512, 2048, 2048),
                                   (512, 2048, 2816), (2000, 4096, 4096)])
def test_shallow_products(T, N, K):
    g = torch.Generator(device="cuda").manual_seed(T + K)
    x = torch.randn(T, K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    y = ops.shallow_parts(x, w)
    assert (y is not None) == (T < 2000)
    got = added(y.planes) if y is not None else ops.linear_parts(x, w)
    want = x.double() @ w.double().T
    # one rounding of sums of K products, whose own float32 error is far below it
    assert torch.allclose(got.double(), want, rtol=2.0 ** -8, atol=2.0 ** -12)
    one = ops.linear_parts(x, w, shallow=True)
    assert isinstance(one, ops.PlaneSum) == (y is not None)
    assert torch.equal(one.planes, y.planes) if y is not None else torch.equal(one, got)


def test_asked_once(monkeypatch):
    """A product for a norm looks its operands over once, as the plain one does."""
    x, w, asked = torch.randn(130, 64), torch.randn(32, 64), []
    look = ops._skinny_ok
    monkeypatch.setattr(ops, "_skinny_ok", lambda x, w: asked.append(1) or look(x, w))
    want = ops.linear(x, w)
    plain = len(asked)
    assert torch.equal(_product_parts(x, w), want) and len(asked) == 2 * plain == 2
