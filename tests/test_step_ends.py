"""The first and the last launch of a hybrid step: embedding with the norm behind it, logits as float32."""

import pytest
import torch

from opsagent_amd import ops
from opsagent_amd.ops import mixer_ops as mx

DEVICES = [pytest.param("cpu", id="cpu"), pytest.param("cuda", id="gpu", marks=pytest.mark.gpu)]


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,C,scale", [(1, 8, 1.0), (1, 2048, 2.5), (3, 30, 1.0), (2, 7, 0.5), (130, 4100, 45.25)])
def test_embedding_and_norm(device, dtype, T, C, scale):
    g = torch.Generator().manual_seed(C)
    table = torch.randn(50, C, generator=g).to(device, dtype)
    nxt = tuple(t.to(device) for t in (1 + 0.1 * torch.randn(C, generator=g), 0.1 * torch.randn(C, generator=g),
                                       torch.full((1,), 0.5)))
    ids = torch.randint(0, 50, (T,), generator=g).to(device)
    x, h = mx.embed_dyt_norm(table, ids, scale, nxt, dtype)
    want = mx.embed_rows(table, ids, scale)
    assert torch.equal(x, want) and x.dtype == torch.float32
    ref = mx.dyt_norm(want, nxt, dtype)
    assert h.dtype == dtype
    # a product and a sum may be one instruction here and two there
    assert torch.allclose(h.float(), ref.float(), rtol=2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -20, atol=2.0 ** -20)
    assert dtype == torch.float32 or (h != ref).float().mean() < 0.01


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("M,N,K", [(1, 1, 2048), (1, 4100, 2048), (1, 32000, 4096), (1, 65, 14336), (1, 40, 96), (3, 64, 2048)])
def test_logits(device, M, N, K):
    g = torch.Generator().manual_seed(N)
    x, w = (torch.randn(r, K, generator=g).bfloat16().to(device) for r in (M, N))
    got = ops.linear_float(x, w)
    assert got.dtype == torch.float32 and torch.equal(got, ops.linear(x, w).float())
