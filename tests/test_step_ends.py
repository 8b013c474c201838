"""The first and the last launch of a hybrid step: embedding with the norm behind it, logits as float32."""

import dataclasses

import pytest
import torch

import test_vazilorn as V
from opsagent_amd import ops
from opsagent_amd.engine.config import apply_tensor_shapes, vazilorn_spec_from_dict
from opsagent_amd.engine.hybrid import HybridForCausalLM
from opsagent_amd.engine.model import ForwardBatch
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


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("start", ["plain", "normed", "positions"])
def test_sandwich_models_of_every_embedding(device, start):
    """Embeddings that no launch shares with the first norm: the norm runs by itself. Against the layers one
    by one, each norm as the reference has it."""
    V._skip_if_wrong_device(device)
    cfg = V.make_cfg(pattern="dm")
    W = V.O.random_weights(cfg, seed=5)
    spec = apply_tensor_shapes(vazilorn_spec_from_dict(cfg), {k: tuple(v.shape) for k, v in W.items()})
    change = {"plain": {}, "normed": {"embed_norm": True, "embed_scale": 1.0}, "positions": {"sinusoid": True}}
    spec = dataclasses.replace(spec, **change[start])
    m = HybridForCausalLM(spec, dtype=torch.float32, device=device)
    toks = torch.tensor(V.tokens_for(cfg, 9, 4), device=device)
    sb = V.one_seq_batch(9, 0, device)

    def caches():
        return [tuple(torch.zeros(16, 8, g, d, device=device) for d in (dk, dv)) for g, dk, dv in m.kv_layer_shapes()]

    fb = ForwardBatch(kind="mixed", input_ids=toks, positions=torch.arange(9, dtype=torch.int32, device=device),
                      slot_mapping=sb.slot_mapping, seq_batch=sb)
    got = m(fb, caches(), [{} for _ in m.layers])
    if start == "normed":
        row = m.embed[toks].double()
        x = (row / (row.pow(2).mean(-1, keepdim=True) + spec.norm_eps).sqrt() * (1 + m.embed_norm_w.double())).float()
    else:
        x = mx.embed_rows(m.embed, toks, spec.embed_scale, m.pos_freq, sb)
    kv = caches()
    w, b, a = m.layers[0].first_norm()
    h = torch.tanh(a * x) * w + b
    for i, layer in enumerate(m.layers):
        nxt = m.layers[i + 1].first_norm() if i + 1 < len(m.layers) else None
        x, h = layer(x, h, sb, kv[i], {}, nxt)
    # float32 through two layers, sums and square roots in another order at the start
    assert torch.allclose(got, x, rtol=1e-4, atol=1e-4 * x.abs().max().item())
