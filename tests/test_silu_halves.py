"""The activation read from the two halves of a product, plain and quantized, and the
row quantization: bit for bit what the separate steps give."""

import pytest
import torch

from opsagent_amd import ops

pytestmark = pytest.mark.gpu


def _rows(M, K, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(M, K, generator=g, device="cuda") * 2).to(torch.bfloat16)


# one vector, a part of a block, one block, one more; registers' last column (16384) and past
SIZES = [(1, 8), (3, 248), (77, 2048), (2, 2056), (9, 14336), (2, 16384), (2, 16392), (3, 28672)]


@pytest.mark.parametrize("M,I", SIZES)
def test_silu_halves(M, I):
    gu = _rows(M, 2 * I, M + I)
    want = ops.silu_mul(gu[:, :I].contiguous(), gu[:, I:].contiguous())
    assert torch.equal(ops.silu_halves(gu, I), want)


def _quantized(x):
    amax = x.float().abs().amax(1).clamp_min(1e-8)
    scale = amax / torch.full_like(amax, 448.0)
    q = (x.float() * (448.0 / amax)[:, None]).clamp(-448, 448).to(torch.float8_e4m3fn)
    return q.view(torch.uint8), scale


@pytest.mark.parametrize("M,K", SIZES)
def test_quant(M, K):
    from opsagent_amd.ops import hip_lib

    x = _rows(M, 2 * K, M * K)
    x[0] = 0                                   # a row of zeros keeps a finite scale
    act = ops.silu_mul(x[:, :K].contiguous(), x[:, K:].contiguous())
    q, s = torch.empty(M, K, dtype=torch.uint8, device="cuda"), torch.empty(M, device="cuda")
    assert hip_lib.get_lib().oa_silu_quant_fp8(
        hip_lib.current_stream_ptr(), x.data_ptr(), q.data_ptr(), s.data_ptr(), M, K) == 0
    q2, s2 = ops.quant_fp8(act)
    want_q, want_s = _quantized(act)
    assert torch.equal(q, q2) and torch.equal(s, s2)
    # A float32 division on either side (one ulp each), a product more in a code: a code
    # may differ only where the exact value lies within 2^-21 of the middle between the two
    # (bf16 values often lie on it, so how many differ is not bounded).
    assert ((s - want_s).abs() <= 2.0 ** -22 * want_s).all()
    value = lambda c: c.view(torch.float8_e4m3fn).double()  # noqa: E731
    mid = (value(q) + value(want_q)) / 2
    exact = act.double() * (448.0 / act.double().abs().amax(1, keepdim=True).clamp_min(1e-8))
    near = (exact - mid).abs() <= 2.0 ** -21 * mid.abs()
    assert bool(((q == want_q) | ((q.int() - want_q.int()).abs() == 1) & near).all())


def test_mlp_fp8_is_its_parts():
    M, K, I = 33, 256, 384
    x = _rows(M, K, 6)
    wq, ws = ops.quant_fp8(_rows(2 * I, K, 7))
    dq, ds = ops.quant_fp8(_rows(K, I, 8))
    parts = ops.linear_fp8(ops.gateup_silu_fp8(x, wq, ws, I), dq, ds)
    assert torch.equal(ops.mlp_fp8(x, wq, ws, I, dq, ds), parts)


@pytest.mark.gpu
@pytest.mark.parametrize("T,K", [(1, 8), (7, 128), (5, 512), (5, 520), (4095, 1024), (4097, 1024),
                                 (4099, 2040), (4096, 2048), (2, 16392)])
def test_quantization_by_waves_and_blocks(T, K):
    """Short rows by a wave, long ones by a block: the same scales and bytes as in torch, and
    of the activation as of its rounded result."""
    gen = torch.Generator(device="cuda").manual_seed(T + K)
    gu = torch.randn(T, 2 * K, generator=gen, device="cuda").bfloat16()
    act = ops.silu_halves(gu, K)
    q8 = torch.empty(T, K, dtype=torch.uint8, device="cuda")
    s8 = torch.empty(T, dtype=torch.float32, device="cuda")
    lib, hip = ops._lib()
    hip.check(lib.oa_silu_quant_fp8(hip.current_stream_ptr(), gu.data_ptr(), q8.data_ptr(),
                                    s8.data_ptr(), T, K), "oa_silu_quant_fp8")
    q, s = ops.quant_fp8(act)
    assert torch.equal(q, q8) and torch.equal(s, s8)
    amax = act.float().abs().amax(-1).clamp_min(1e-8)
    top = torch.full_like(amax, 448.0)               # a scalar would be multiplied by its inverse
    assert torch.equal(s, amax / top)
    want = (act.float() * (top / amax)[:, None]).clamp(-448, 448).to(torch.float8_e4m3fn)
    assert torch.equal(q.view(torch.float8_e4m3fn).float(), want.float())


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [640, 896])
def test_mlp_refuses_other_gate_rows(rows):
    """gate-up weights of other than 2 I rows: an error, as of the split that was there."""
    x = _rows(33, 256, 9)
    wq, ws = ops.quant_fp8(_rows(rows, 256, 10))
    dq, ds = ops.quant_fp8(_rows(256, 384, 11))
    with pytest.raises(RuntimeError):
        ops.mlp_fp8(x, wq, ws, 384, dq, ds)
