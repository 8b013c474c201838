"""One-row product with the add and the dynamic-tanh norm behind it in its epilogue, against the
two launches that it stands for: several rows a wave and none, rows of every length that it takes,
with and without a next norm; and who gets it."""

import pytest
import torch

from opsagent_amd import ops
from opsagent_amd.ops import mixer_ops as mx


def _norm(g, n):
    r = lambda m: torch.randn(m, generator=g, device="cuda")  # noqa: E731
    return 1 + 0.1 * r(n), 0.1 * r(n), 0.5 + 0.1 * r(1)


def _counted(monkeypatch):
    """The fused launches, as they are made."""
    calls, lib = [], ops._lib()[0]
    inner = lib.oa_gemv_dyt
    monkeypatch.setattr(lib, "oa_gemv_dyt", lambda *a: calls.append(a) or inner(*a))
    return calls


@pytest.mark.gpu
@pytest.mark.parametrize("last", [False, True])
@pytest.mark.parametrize("N,K", [(2048, 2048), (2048, 8192), (4096, 14336), (1, 2048), (37, 4096),
                                 (5001, 6144), (20000, 2048), (33000, 4096), (7, 16384)])
def test_against_two_launches(monkeypatch, N, K, last):
    g = torch.Generator(device="cuda").manual_seed(N + K)
    x = torch.randn(1, K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(N, K, generator=g, device="cuda") * 2 * K ** -0.5).bfloat16()
    r = torch.randn(1, N, generator=g, device="cuda")
    post, nxt = _norm(g, N), None if last else _norm(g, N)
    want_r, got_r = r.clone(), r.clone()
    want = mx.dyt_norm(want_r, nxt, torch.bfloat16, y=ops.linear(x, w), post=post)
    calls = _counted(monkeypatch)
    got = mx.linear_dyt_norm(x, w, got_r, nxt, torch.bfloat16, post)
    assert len(calls) == 1
    # the same operations in float32: a contraction apart, 4 roundings of numbers up to 4
    assert (got_r - want_r).abs().max() <= 4 * 4 * 2.0 ** -24
    if last:
        assert got is None and want is None
    else:
        assert torch.allclose(got.float(), want.float(), rtol=2.0 ** -7, atol=2.0 ** -20)
        assert (got != want).float().mean() < 0.01


@pytest.mark.gpu
def test_norms_of_another_width():
    """A weight or bias of one number, or a slope of many, is refused and not read past its end."""
    g = torch.Generator(device="cuda").manual_seed(0)
    x, w = (torch.randn(n, 2048, generator=g, device="cuda").bfloat16() for n in (1, 64))
    r, good = torch.zeros(1, 64, device="cuda"), _norm(g, 64)
    for i in range(3):
        bad = tuple(t.new_ones(1 if n < 2 else 64) if n == i else t for n, t in enumerate(good))
        for post, nxt in ((bad, good), (good, bad), (bad, None)):
            with pytest.raises(AssertionError):
                mx.linear_dyt_norm(x, w, r, nxt, torch.bfloat16, post)
    assert not r.any()


@pytest.mark.gpu
def test_others_go_the_old_way(monkeypatch):
    """Two rows, short rows, float32 and operands off the 16-byte grid."""
    g = torch.Generator(device="cuda").manual_seed(0)
    N, calls = 64, _counted(monkeypatch)
    for T, K, dtype, off in ((2, 2048, torch.bfloat16, 0), (1, 1024, torch.bfloat16, 0),
                             (1, 2048, torch.float32, 0), (1, 2048, torch.bfloat16, 1)):
        x = torch.randn(T * K + off, generator=g, device="cuda").to(dtype)[off:].view(T, K)
        w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(dtype)
        post, nxt = _norm(g, N), _norm(g, N)
        r = torch.randn(T, N, generator=g, device="cuda")
        want_r, got_r = r.clone(), r.clone()
        want = mx.dyt_norm(want_r, nxt, dtype, y=ops.linear(x, w), post=post)
        got = mx.linear_dyt_norm(x, w, got_r, nxt, dtype, post)
        assert torch.equal(got, want) and torch.equal(got_r, want_r)
    assert not calls


def test_cpu():
    g = torch.Generator().manual_seed(0)
    r = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    x, w, res, post, nxt = r(1, 32), r(8, 32), r(1, 8), (r(8), r(8), r(1)), (r(8), r(8), r(1))
    a, b = res.clone(), res.clone()
    assert torch.equal(mx.linear_dyt_norm(x, w, a, nxt, torch.float32, post),
                       mx.dyt_norm(b, nxt, torch.float32, y=x @ w.T, post=post))
    assert torch.equal(a, b)
