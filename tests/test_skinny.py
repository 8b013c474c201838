"""Skinny products (skinny.hip) against float64 at the edges of strips, fragments
and steps, in both forms, and what the rule sends where."""

import pytest
import torch

from opsagent_amd import ops


def _err(got, want):
    return float((got.double() - want).norm() / want.norm())


# one bf16 rounding of a float32 sum: half a unit in the last of 8 bits, at most 2^-8
# of a value and 0.0016 in the mean over many (a second rounding would make it 0.0023),
# and float32 sums far below that
TOL = 2.0 ** -8 + 1e-5


def _tol(out):
    return 2e-3 if out.numel() >= 1024 else TOL


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 3, 8, 16, 17, 32])
@pytest.mark.parametrize("N,K,form", [
    (16, 32, 1),              # one strip, one step: most waves have none
    (40, 96, 1),              # a strip of eight rows
    (100, 1408, 1),           # 44 steps over eight waves
    (2048, 2816, 1),          # 88 steps: rounds and a remainder
    (48, 14336, 1),           # deep K on four waves
    (16, 4096, 2),            # one strip for one block
    (4104, 4096, 2),          # one strip more than there are blocks, half empty
    (24592, 4096, 2),         # blocks with unequal numbers of strips
])
def test_skinny(M, N, K, form):
    gen = torch.Generator(device="cuda").manual_seed(M * 131 + N)
    rn = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    wide = rn(M, K + 24).bfloat16()
    w = (rn(N, K) * K ** -0.5).bfloat16()
    for x in (wide[:, :K].contiguous(), wide[:, 8 : 8 + K]):
        assert ops._skinny_ok(x, w)
        got = ops._skinny(x, w, form)
        assert _err(got, x.double() @ w.double().T) < _tol(got)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(2, 4104, 192), (8, 14344, 128), (31, 16384, 96), (17, 32000, 288),
                                   (24, 14336, 768)])
@pytest.mark.parametrize("far", [0, 64])
def test_short_rows(M, N, K, far):
    gen = torch.Generator(device="cuda").manual_seed(N + M)
    x = torch.randn(M, K + far, generator=gen, device="cuda").bfloat16()[:, :K]
    w = (torch.randn(N, K, generator=gen, device="cuda") * K ** -0.5).bfloat16()
    got = ops.linear(x, w)
    assert torch.equal(got, ops._skinny(x, w, 1))
    assert _err(got, x.double() @ w.double().T) < _tol(got)
    assert not ops._skinny_ok(wide[:, 3 : 3 + K], w)          # rows start off 16 bytes
    if form == 2 and M > 16:
        return
    x = wide[:, :K].contiguous()
    up = (rn(N, K) * K ** -0.5).bfloat16()
    g, u = x.double() @ w.double().T, x.double() @ up.double().T
    both = torch.cat([w, up])
    assert _err(ops._skinny(x, both, form, gateup=True), g * torch.sigmoid(g) * u) < _tol(g)
    want = torch.nn.functional.gelu(g, approximate="tanh") * u
    assert _err(ops._skinny(x, both, form, gateup=True, act=1), want) < _tol(g)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 3, 16, 17, 32])
@pytest.mark.parametrize("N,K,form", [(40, 96, 1), (100, 1408, 1), (48, 14336, 1), (4104, 4096, 2)])
def test_skinny_whole_numbers(M, N, K, form):
    """Whole numbers: every float32 sum is exact, the result its one rounding to bf16."""
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randint(-8, 9, (M, K), generator=gen, device="cuda").bfloat16()
    w = torch.randint(-8, 9, (N, K), generator=gen, device="cuda").bfloat16()
    assert torch.equal(ops._skinny(x, w, form), (x.double() @ w.double().T).bfloat16())


@pytest.mark.gpu
@pytest.mark.parametrize("M", [2, 3, 13, 16, 31, 33])
@pytest.mark.parametrize("N,K", [(6144, 4096), (4096, 4096), (4096, 14336), (1008, 264)])
def test_linear_routes_agree(M, N, K):
    """Whatever the rule says, linear and gateup_silu give the product."""
    gen = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K, generator=gen, device="cuda").bfloat16()
    w = (torch.randn(N, K, generator=gen, device="cuda") * K ** -0.5).bfloat16()
    want = x.double() @ w.double().T
    assert _err(ops.linear(x, w), want) < _tol(want)
    assert _err(ops.linear(x.view(M, 1, K), w).view(M, N), want) < _tol(want)
    g, u = want.chunk(2, -1)
    # the unfused form rounds gate and up to bf16 before their product (the gate's
    # error grows up to twofold in silu): 0.0016 * sqrt(1 + 2^2 + 1) in the mean
    assert _err(ops.gateup_silu(x, w, N // 2), g * torch.sigmoid(g) * u) < 6e-3


def test_rule():
    """The lines as stated at _skinny_form."""
    form = ops._skinny_form
    assert form(8, 14336, 4096, gateup=True) == 2 and form(17, 14336, 4096, gateup=True) == 0
    assert form(8, 6144, 4096) == 2 and form(17, 6144, 4096) == 0
    assert form(32, 32000, 4096) == 2 and form(33, 32000, 4096) == 0
    assert form(13, 4096, 4096) == 1 and form(32, 4096, 4096) == 0
    assert form(3, 4096, 14336) == 1 and form(16, 4096, 14336) == 0
    assert form(13, 2816, 2048, gateup=True) == 1
    assert form(8, 64, 1000) == 0                             # K not a multiple of 32
    x, w = torch.zeros(4, 64, dtype=torch.bfloat16), torch.zeros(8, 64, dtype=torch.bfloat16)
    assert not ops._skinny_ok(x, w)                           # CPU tensors: the general path


@pytest.mark.gpu
def test_switches(monkeypatch):
    """The two switches choose between the staged GEMVs and the library, whatever the
    newer forms would take."""
    from opsagent_amd.ops import hip_lib

    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(8, 4096, generator=gen, device="cuda").bfloat16()
    w = (torch.randn(6144, 4096, generator=gen, device="cuda") * 2.0 ** -6).bfloat16()
    assert ops._ring_plan(8, 6144, 4096) and ops._skinny_ok(x, w)
    staged = torch.empty(8, 6144, dtype=x.dtype, device="cuda")
    hip_lib.check(hip_lib.get_lib().oa_gemv_ex(hip_lib.current_stream_ptr(), x.data_ptr(), w.data_ptr(),
                                               staged.data_ptr(), None, None, 8, 6144, 4096, 0.0, 0), "")
    library = torch.nn.functional.linear(x, w)
    monkeypatch.setenv("OPSAGENT_BF16_GEMV_MFMA", "m2")
    assert not ops._skinny_ok(x, w) and torch.equal(ops.linear(x, w), staged)
    assert ops.gateup_fused(x, w, 3072)
    monkeypatch.setenv("OPSAGENT_BF16_GEMV_MFMA", "0")
    assert torch.equal(ops.linear(x, w), library) and not ops.gateup_fused(x, w, 3072)
    monkeypatch.delenv("OPSAGENT_BF16_GEMV_MFMA")
    monkeypatch.setenv("OPSAGENT_GEMV_MAX_M", "1")
    assert torch.equal(ops.linear(x[:2], w), torch.nn.functional.linear(x[:2], w))


@pytest.mark.gpu
@pytest.mark.parametrize("M", [24, 64])
def test_mismatches_are_refused(M):
    """A weight on another device, of other columns or with other than 2 I rows is an error of
    the general path, not an address that a kernel reads."""
    x = torch.zeros(M, 4096, dtype=torch.bfloat16, device="cuda")
    w = torch.zeros(8192, 4096, dtype=torch.bfloat16, device="cuda")
    assert ops._skinny_form(M, 8192, 4096) or ops._ring_plan(M, 8192, 4096)
    for other in (w.cpu(), w[:, :2048].contiguous()):
        with pytest.raises(RuntimeError):
            ops.linear(x, other)
    for rows in (8064, 8192 + 128):
        other = torch.zeros(rows, 4096, dtype=torch.bfloat16, device="cuda")
        assert not ops.gateup_fused(x, other, 4096)
        with pytest.raises(RuntimeError):
            ops.gateup_silu(x, other, 4096)
    assert ops.gateup_fused(x, w, 4096)


def test_plain_calls():
    x, w = torch.zeros(3, 8), torch.zeros(5, 8)
    seen = []

    def look(a, b=w):
        seen.append(ops._plain_call(a, b))
        return a @ b.T

    look(x)
    assert seen.pop()
    torch.vmap(look)(x[None])
    torch.func.jvp(look, (x,), (x,))
    torch.jit.trace(look, (x, w), check_trace=False)
    with torch._subclasses.FakeTensorMode(allow_non_fake_inputs=True):
        look(torch.empty(3, 8))
    look(x.clone().requires_grad_())
    look(x, torch.nn.Parameter(w))
    with torch.autograd.forward_ad.dual_level():
        look(torch.autograd.forward_ad.make_dual(x, x))
    assert len(seen) == 7 and not any(seen)
    with torch.no_grad():
        look(x, torch.nn.Parameter(w))
    assert seen.pop()


@pytest.mark.gpu
@pytest.mark.parametrize("M", [24, 64])
def test_gradients_and_transforms(M):
    """Rows that the library took before keep its gradients, transforms and traces."""
    gen = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, 4096, generator=gen, device="cuda").bfloat16()
    w = (torch.randn(8192, 4096, generator=gen, device="cuda") * 2.0 ** -6).bfloat16()
    plain = ops.linear(x, w)
    assert ops._skinny_ok(x, w)
    library = torch.nn.functional.linear(x, w)
    assert _err(plain, library.double()) < 4e-3              # one rounding each
    p, v = torch.nn.Parameter(w), x.clone().requires_grad_()
    out = ops.linear(v, p)
    assert torch.equal(out, library)
    grad = torch.autograd.grad(out.float().sum(), [v, p])
    want = [w.float().sum(0).expand(M, -1), x.float().sum(0).expand(8192, -1)]
    for got, ref in zip(grad, want):
        assert _err(got, ref.double()) < 4e-3
    each = torch.vmap(lambda a: ops.linear(a, w))(torch.stack([x, x]))
    assert _err(each[1], library.double()) < 4e-3
    with torch.no_grad():
        assert torch.equal(ops.linear(v, p), plain)


@pytest.mark.gpu
@pytest.mark.parametrize("N,K", [(2048, 128), (2040, 288), (4096, 4096), (1000, 4096)])
def test_two_rows_that_lie_apart(N, K):
    gen = torch.Generator(device="cuda").manual_seed(N)
    x = torch.randn(2, K + 64, generator=gen, device="cuda").bfloat16()[:, 32 : 32 + K]
    w = (torch.randn(N, K, generator=gen, device="cuda") * K ** -0.5).bfloat16()
    assert ops._skinny_form(2, N, K, strided=True) == 1
    got = ops.linear(x, w)
    assert torch.equal(got, ops._skinny(x, w, 1))
    assert _err(got, x.double() @ w.double().T) < _tol(got)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(2, 4104, 192), (8, 14344, 128), (31, 16384, 96), (17, 32000, 288),
                                   (24, 14336, 768)])
@pytest.mark.parametrize("far", [0, 64])
def test_short_rows(M, N, K, far):
    gen = torch.Generator(device="cuda").manual_seed(N + M)
    x = torch.randn(M, K + far, generator=gen, device="cuda").bfloat16()[:, :K]
    w = (torch.randn(N, K, generator=gen, device="cuda") * K ** -0.5).bfloat16()
    got = ops.linear(x, w)
    assert torch.equal(got, ops._skinny(x, w, 1))
    assert _err(got, x.double() @ w.double().T) < _tol(got)
