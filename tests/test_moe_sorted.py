"""Sorted expert tiles (ops.moe_sorted_mlp) against the float64 sum over a
token's experts, at the edges of row tiles, weight strips and expert counts."""

import pytest
import torch

from opsagent_amd import ops
from opsagent_amd.ops import torch_ref


def _reference(x, w13, w2, idx, wts, act, more):
    x = x.double()
    out = torch.zeros(x.shape[0], w2.shape[1], dtype=torch.float64, device=x.device)
    for e in range(w13.shape[0]):
        rows, place = (idx == e).nonzero(as_tuple=True)
        if not rows.numel():
            continue
        h = x[rows] @ w13[e].double().T
        if act == "relu2":
            a = torch.relu(h) ** 2
        else:
            g, u = h.chunk(2, -1)
            if isinstance(act, tuple):
                _, limit, alpha = act
                g, u = g.clamp(max=limit), u.clamp(-limit, limit)
                a = g * torch.sigmoid(alpha * g) * (u + 1.0)
            else:
                a = g * torch.sigmoid(g) * u
        out.index_add_(0, rows, wts[rows, place, None].double() * (a @ w2[e].double().T))
    return out if more is None else out + more.double()


@pytest.mark.gpu
@pytest.mark.parametrize("T,E,top,K", [(1, 16, 4, 2048), (13, 64, 6, 2048), (3, 5, 5, 200),
                                       (65, 130, 8, 1000), (1025, 64, 6, 2048), (1027, 8, 1, 8192),
                                       (4, 3, 1, 8), (17, 257, 6, 1032), (128, 64, 6, 2048),
                                       (129, 66, 6, 2048), (2, 1024, 6, 16512)])
def test_route(T, E, top, K):
    """Against float64: weights to float32 rounding of K products (the chosen
    scores lie in 0..1, so 1e-5 holds at K = 8192 with logits of a few units),
    experts wherever the choice is clearer than that."""
    gen = torch.Generator(device="cuda").manual_seed(T + E)
    x = torch.randn(T, K, generator=gen, device="cuda").bfloat16()
    rw = torch.randn(E, K, generator=gen, device="cuda") * (2.0 * K ** -0.5)
    assert ops.moe_route_ok(x, rw, top)
    idx, wts, tok = ops.moe_route(x, rw, top)
    score = torch.softmax(x.double() @ rw.double().T, -1)
    want = score.topk(min(top + 1, E), -1)
    clear = torch.ones(T, dtype=torch.bool, device="cuda")
    if E > top:
        clear = want.values[:, top - 1] - want.values[:, top] > 1e-5
    assert clear.float().mean() > 0.9
    assert torch.equal(idx[clear].sort(-1).values, want.indices[clear, :top].int().sort(-1).values)
    picked = score.gather(1, idx.long())
    assert (wts - picked / picked.sum(-1, keepdim=True)).abs().max() < 1e-5
    assert torch.equal(tok, torch.arange(T, device="cuda", dtype=torch.int32)[:, None].expand(T, top))


@pytest.mark.gpu
@pytest.mark.parametrize("E,top", [(64, 6), (5, 5), (130, 1)])
def test_route_of_odd_rows(E, top):
    """A NaN, an infinite or no finite logit makes a row's weights NaN, as softmax does,
    with experts that exist; equal logits go to the lower experts."""
    K = 256
    gen = torch.Generator(device="cuda").manual_seed(E)
    x = torch.randn(6, K, generator=gen, device="cuda").bfloat16()
    rw = torch.randn(E, K, generator=gen, device="cuda") * K ** -0.5
    rw[:, 0], rw[2, 1], x[:, :2] = 0.0, 0.0, 0.0
    rw[2, 0], rw[3, 1] = float("nan"), float("inf")
    bad = ops.moe_route(x, rw, top)                  # 0 * NaN: one logit of every row
    assert torch.isnan(bad[1]).all() and (bad[0] >= 0).all() and (bad[0] < E).all()
    rw[2, 0] = 0.0
    x[1, 1] = 1.0                                    # one infinite logit; others 0 * inf
    idx, wts, _ = ops.moe_route(x, rw, top)
    assert torch.isnan(wts).all() and (idx >= 0).all() and (idx < E).all()
    rw[3, 1] = 0.0
    x[4], x[5, 5] = 0.0, float("nan")                # equal logits; a NaN activation
    idx, wts, _ = ops.moe_route(x, rw, top)
    assert torch.isfinite(wts[:5]).all() and torch.isnan(wts[5]).all()
    assert torch.equal(idx[4].cpu(), torch.arange(top, dtype=torch.int32))
    assert (wts[4] - 1.0 / top).abs().max() < 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("T,E,top,H,I,act,spread", [
    (65, 8, 2, 128, 128, None, "even"),             # one K step, one strip
    (64, 4, 1, 256, 128, None, "one"),              # every row in one expert: a full tile
    (65, 4, 1, 256, 384, None, "one"),              # ... and one row more
    (300, 64, 6, 512, 256, None, "even"),           # many small experts
    (5, 16, 2, 256, 256, None, "even"),             # 16-row tiles, experts without rows
    (17, 4, 1, 256, 128, None, "one"),              # ... one row past a 16-row tile
    (700, 5, 3, 384, 640, "relu2", "skew"),         # odd step counts, ungated
    (1100, 4, 3, 256, 256, ("clamp_swish", 7.0, 1.702), "skew"),   # 128-row tiles
    (129, 3, 1, 128, 128, None, "one"),             # an expert without rows on each side
])
def test_sorted_experts(fp8, T, E, top, H, I, act, spread):
    gen = torch.Generator(device="cuda").manual_seed(T * 7 + I)
    rn = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    x = rn(T, H).bfloat16()
    w13 = (rn(E, I if act == "relu2" else 2 * I, H) * H ** -0.5).bfloat16()
    w2 = (rn(E, H, I) * I ** -0.5).bfloat16()
    score = rn(T, E)
    if spread == "skew":
        score += torch.linspace(3, 0, E, device="cuda")
    elif spread == "one":
        score[:, E // 2] += 100.0
    idx = score.topk(top, -1).indices.to(torch.int32)
    wts = torch.softmax(score, -1).gather(1, idx.long()).contiguous()
    more = rn(T, H).bfloat16() if T % 2 else None
    s13 = s2 = None
    d13, d2 = w13, w2
    if fp8:
        w13, s13 = ops.quant_fp8(w13)
        w2, s2 = ops.quant_fp8(w2)
        s13, s2 = s13.view(E, -1), s2.view(E, -1)
        d13, d2 = torch_ref.dequant_fp8(w13, s13), torch_ref.dequant_fp8(w2, s2)
    assert ops.moe_sorted_ok(x, w13, w2, act)
    got = ops.moe_sorted_mlp(x, w13, s13, w2, s2, idx, wts, act, more)
    again = ops.moe_sorted_mlp(x, w13, s13, w2, s2, idx, wts, act, more)
    assert torch.equal(got, again)                  # no sum depends on placement
    want = _reference(x, d13, d2, idx, wts, act, more)
    # bf16 rounds the middle activation, a pair's row and the sum: three independent
    # errors, 0.0016 of a value each in the mean (at most 2^-8), 0.0028 together
    err = (got.double() - want).norm() / want.norm()
    assert err < 4e-3, float(err)



@pytest.mark.gpu
@pytest.mark.parametrize("E,top,T,form", [
    (1030, 6, 3, "plain"),        # more experts than the routing kernels hold
    (96, 65, 2, "plain"),         # more choices than a wave has lanes
    (16, 4, 5, "strided"), (16, 4, 70, "strided"),
    (16, 4, 5, "offset"),         # rows that start off 16 bytes
])
def test_layer_without_host_waits(E, top, T, form):
    """What a decode step may hold runs without waiting for the GPU, as a captured step
    has to, whatever the input's strides and the router's size."""
    from opsagent_amd.engine.config import ModelSpec
    from opsagent_amd.engine.moe import MoEMLP
    from opsagent_amd.parallel import state

    state.set_tp_state(0, 1, None)
    H, I = 256, 128
    spec = ModelSpec(name="moe", max_seq_len=64, hidden_size=H, num_heads=2, num_kv_heads=2,
                     head_dim=128, intermediate_size=256, num_layers=1, vocab_size=64,
                     moe_num_experts=E, moe_top_k=top, moe_intermediate_size=I,
                     moe_shared_experts=0, moe_dtype="bf16")
    moe = MoEMLP(spec, torch.bfloat16, torch.Generator(device="cuda").manual_seed(E)).to("cuda")
    gen = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn(T, 2 * H, generator=gen, device="cuda").bfloat16()
    if form == "strided":
        x = x[:, H:]
    elif form == "offset":
        x = x.flatten()[1 : 1 + T * H].view(T, H)
    else:
        x = x[:, :H].contiguous()
    moe(x)
    torch.cuda.synchronize()
    torch.cuda.set_sync_debug_mode("error")
    try:
        got = moe(x, decode=True)
    finally:
        torch.cuda.set_sync_debug_mode("default")
    score, idx = torch.softmax(x.double() @ moe.router_w.double().T, -1).topk(top, -1)
    wts = score / score.sum(-1, keepdim=True)
    want = _reference(x, moe.w13, moe.w2, idx, wts, None, None)
    # the roundings of test_sorted_experts
    assert float((got.double() - want).norm() / want.norm()) < 4e-3


@pytest.mark.gpu
@pytest.mark.parametrize("T", [17, 70])
def test_layer_asks_the_front_for_few_tokens(monkeypatch, T):
    """Routing beside the shared expert takes up to 16 tokens: more go to the routing launches at once."""
    from opsagent_amd.engine.config import ModelSpec
    from opsagent_amd.engine.moe import MoEMLP
    from opsagent_amd.parallel import state

    state.set_tp_state(0, 1, None)
    H, E, top = 256, 16, 4
    spec = ModelSpec(name="moe", max_seq_len=64, hidden_size=H, num_heads=2, num_kv_heads=2,
                     head_dim=128, intermediate_size=256, num_layers=1, vocab_size=64,
                     moe_num_experts=E, moe_top_k=top, moe_intermediate_size=128,
                     moe_shared_experts=1, moe_dtype="bf16")
    moe = MoEMLP(spec, torch.bfloat16, torch.Generator(device="cuda").manual_seed(E)).to("cuda")
    x = torch.randn(T, H, generator=torch.Generator(device="cuda").manual_seed(T), device="cuda").bfloat16()
    asked, front = [], ops.moe_front
    monkeypatch.setattr(ops, "moe_front", lambda x, *a: asked.append(x.shape[0]) or front(x, *a))
    monkeypatch.setattr(ops, "moe_sorted_wins", lambda *a: True)
    got = moe(x)
    assert not asked
    moe(x[:16])
    assert asked == [16]
    score, idx = torch.softmax(x.double() @ moe.router_w.double().T, -1).topk(top, -1)
    want = _reference(x, moe.w13, moe.w2, idx, score / score.sum(-1, keepdim=True), None, moe.shared(x))
    # the roundings of test_sorted_experts
    assert float((got.double() - want).norm() / want.norm()) < 4e-3


def test_sorted_experts_refuse():
    """CPU tensors and activations that the kernels do not have stay on the
    general path."""
    x = torch.zeros(4, 128, dtype=torch.bfloat16)
    w13 = torch.zeros(2, 256, 128, dtype=torch.bfloat16)
    w2 = torch.zeros(2, 128, 128, dtype=torch.bfloat16)
    assert not ops.moe_sorted_ok(x, w13, w2)
    assert ops._moe_act("gelu_tanh") is None and ops._moe_act(None) == (0, 0.0, 0.0)


@pytest.mark.gpu
def test_mismatches_are_refused():
    """A router or experts on another device or of another width are errors of the general
    path, not addresses that a kernel reads."""
    x = torch.zeros(3, 256, dtype=torch.bfloat16, device="cuda")
    router = torch.zeros(8, 256, device="cuda")
    assert ops.moe_route_ok(x, router, 2)
    for other in (router.cpu(), router[:, :128].contiguous(), torch.zeros(8, 264, device="cuda")):
        with pytest.raises(RuntimeError):
            ops.moe_route(x, other, 2)
    w13 = torch.zeros(8, 256, 256, dtype=torch.bfloat16, device="cuda")
    w2 = torch.zeros(8, 256, 128, dtype=torch.bfloat16, device="cuda")
    assert ops.moe_sorted_ok(x, w13, w2)
    assert not ops.moe_sorted_ok(x, w13.cpu(), w2) and not ops.moe_sorted_ok(x, w13, w2.cpu())


def test_ring_rows():
    """Tiles grow with the rows an expert has, later for small matrices; wide ones of 128
    rows are for bf16 alone."""
    rows = ops._moe_ring_rows
    big, small = 1408 * 2048, 512 * 1024
    assert [rows(p, 64, big, False) for p in (48, 512, 513, 1536, 1537, 4095, 4096)] == [
        16, 16, 32, 32, 64, 64, 128]
    assert [rows(p, 64, big, True) for p in (512, 513, 1536, 1537, 99999)] == [16, 32, 32, 64, 64]
    assert [rows(p, 16, small, False) for p in (256, 257, 1536, 1537, 9999)] == [16, 32, 32, 64, 64]


@pytest.mark.gpu
@pytest.mark.parametrize("fp8,tiles", [(False, (16, 32, 64, 128)), (True, (16, 32, 64))])
@pytest.mark.parametrize("T,E,top,H,I", [
    (5, 7, 2, 128, 128),          # fewer steps than the ring holds, experts without rows
    (33, 9, 3, 256, 192 + 64),    # one row past a tile of 32
    (131, 5, 2, 384, 128),        # odd steps; several tiles of most sizes an expert
])
def test_tiles_agree(monkeypatch, fp8, tiles, T, E, top, H, I):
    """A pair's sums run over the columns in one order whatever the tile: the same bits."""
    gen = torch.Generator(device="cuda").manual_seed(T + E)
    rn = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    x = rn(T, H).bfloat16()
    w13, w2 = (rn(E, 2 * I, H) * H ** -0.5).bfloat16(), (rn(E, H, I) * I ** -0.5).bfloat16()
    s13 = s2 = None
    d13, d2 = w13, w2
    if fp8:
        (w13, s13), (w2, s2) = ops.quant_fp8(w13), ops.quant_fp8(w2)
        s13, s2 = s13.view(E, -1), s2.view(E, -1)
        d13, d2 = torch_ref.dequant_fp8(w13, s13), torch_ref.dequant_fp8(w2, s2)
    wts, idx = torch.softmax(rn(T, E), -1).topk(top, -1)
    idx = idx.to(torch.int32)
    outs = []
    for rows in tiles:
        monkeypatch.setattr(ops, "_moe_ring_rows", lambda *a, rows=rows: rows)
        outs.append(ops.moe_sorted_mlp(x, w13, s13, w2, s2, idx, wts))
    for o in outs[1:]:
        assert torch.equal(o, outs[0])
    want = _reference(x, d13, d2, idx, wts, None, None)
    # the roundings of test_sorted_experts
    assert float((outs[0].double() - want).norm() / want.norm()) < 4e-3


@pytest.mark.gpu
@pytest.mark.parametrize("T,E,top,H,I,beside", [
    (3, 64, 6, 2048, 2816, True), (13, 64, 6, 2048, 2816, True),
    (16, 5, 5, 512, 768, True),      # fewer experts than a block of the logits
    (16, 100, 64, 1024, 1408, True),     # as many pairs as there are places
    (7, 256, 8, 2048, 512, True),    # as many experts as there are places
    (9, 8, 1, 512, 2048, True),      # long rows: four waves a strip
    (2, 64, 6, 2048, 2816, False), (1, 40, 40, 264, 0, False), (16, 64, 6, 512, 0, False),
])
def test_front(T, E, top, H, I, beside):
    """Routing, sort and the shared expert in shared launches: the bits of the separate ones, and
    lists that name every pair once, in its expert's place."""
    gen = torch.Generator(device="cuda").manual_seed(T + E)
    rn = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    x, rw = rn(T, H).bfloat16(), rn(E, H) * (2.0 * H ** -0.5)
    gate_up = (rn(2 * I, H) * H ** -0.5).bfloat16() if I else None
    down = (rn(H, I) * I ** -0.5).bfloat16() if I else None
    idx, wts, lists, shared = ops.moe_front(x, rw, top, 1408 * 2048, False, gate_up, down)
    ref_idx, ref_wts, _ = ops.moe_route(x, rw, top)
    assert torch.equal(idx, ref_idx) and torch.equal(wts, ref_wts)
    assert (shared is not None) == beside
    if beside:
        act = ops._skinny(x, gate_up, 1, gateup=True)
        assert torch.equal(shared, ops._skinny(act, down, 1))
    P = T * top
    bm, max_tiles, size = ops._moe_lists(P, E, 1408 * 2048, False)
    off, pre, tile_e, perm = (t.cpu() for t in lists.split([E + 1, E + 1, max_tiles, P]))
    count = torch.bincount(idx.flatten().cpu().long(), minlength=E)
    tiles = (count + bm - 1) // bm
    assert torch.equal(off[1:].long(), count.cumsum(0)) and off[0] == pre[0] == 0
    assert torch.equal(pre[1:].long(), tiles.cumsum(0))
    assert torch.equal(tile_e[: pre[-1]].long(), torch.arange(E).repeat_interleave(tiles))
    assert torch.equal(perm.sort().values.long(), torch.arange(P))
    assert torch.equal(idx.flatten().cpu()[perm.long()].long(), torch.arange(E).repeat_interleave(count))


@pytest.mark.gpu
def test_front_refuses():
    """What the shared launches do not hold goes through the separate ones."""
    x = torch.zeros(4, 512, dtype=torch.bfloat16, device="cuda")
    rw = torch.zeros(257, 512, device="cuda")
    assert ops.moe_front(x, rw, 2, 0, False) is None and ops.moe_front(x, rw[:256], 2, 0, False)
    assert ops.moe_front(x.repeat(5, 1)[:17], rw[:16], 2, 0, False) is None
    assert ops.moe_front(x[:, ::2], rw[:16, :256].contiguous(), 2, 0, False) is None
    w = torch.zeros(2048, 512, dtype=torch.bfloat16, device="cuda")
    down = torch.zeros(512, 1024, dtype=torch.bfloat16, device="cuda")
    assert ops.moe_front(x, rw[:16], 2, 0, False, w, down)[3] is not None
    for a, b in ((w.float(), down), (w, down.float()), (w, down.t().contiguous().t()),
                 (torch.nn.Parameter(w), down)):      # other types, strides, gradients asked for
        assert ops.moe_front(x, rw[:16], 2, 0, False, a, b)[3] is None
