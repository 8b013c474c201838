"""The fp8 gate-up product whose tiles make the activation, against the plain product and the activation of
its bf16 rows: the same bits, edges of rows and of strips of 128 outputs, the fewest steps and more."""

import pytest
import torch

from opsagent_amd import ops
from opsagent_amd.ops import hip_lib


def operand(g, rows, K):
    v = torch.randn(rows, K, generator=g, device="cuda").to(torch.float8_e4m3fn)
    return v.view(torch.uint8), 0.01 + torch.rand(rows, generator=g, device="cuda")


@pytest.mark.gpu
@pytest.mark.parametrize("form", [0, 1, 2])
@pytest.mark.parametrize("M,I,K", [(1, 8, 128), (129, 128, 256), (192, 136, 384), (193, 1000, 512), (257, 1408, 1152),
                                   (700, 2048, 640)])
def test_bits(M, I, K, form):
    g = torch.Generator(device="cuda").manual_seed(M + I)
    (x, xs), (w, ws) = operand(g, M, K), operand(g, 2 * I, K)
    xs, ws = xs * K ** -0.25, ws * K ** -0.25
    lib, stream = hip_lib.get_lib(), hip_lib.current_stream_ptr()
    gu = torch.empty(M, 2 * I, dtype=torch.bfloat16, device="cuda")
    assert lib.oa_tile_gemm_fp8(stream, x.data_ptr(), xs.data_ptr(), w.data_ptr(), ws.data_ptr(), gu.data_ptr(),
                                M, 2 * I, K, form) == 0
    got = torch.full((M + 1, I), 7.0, dtype=torch.bfloat16, device="cuda")
    assert lib.oa_tile_gemm_fp8_silu(stream, x.data_ptr(), xs.data_ptr(), w.data_ptr(), ws.data_ptr(),
                                     got.data_ptr(), M, I, K, form) == 0
    assert torch.equal(got[:M], ops.silu_halves(gu, I)) and (got[M] == 7.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,I,H", [(700, 14336, 512), (130, 256, 512), (300, 2048, 1024)])
def test_feed_forward(M, I, H, monkeypatch):
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, H, generator=g, device="cuda").bfloat16()
    (gw, gs), (dw, ds) = operand(g, 2 * I, H), operand(g, H, I)
    got = ops.mlp_fp8(x, gw, gs, I, dw, ds)
    rows = ops.mlp_fp8(ops.QuantRows(*ops.quant_fp8(x)), gw, gs, I, dw, ds)
    monkeypatch.setattr(ops, "_tile_form_fp8", lambda *a: -1)
    assert torch.equal(got, ops.mlp_fp8(x, gw, gs, I, dw, ds)) and torch.equal(rows, got)
