"""The group norm that adds up a product's parts and takes the next layer's convolution along, and the
attention preparation that holds its row: against the launches apart and the reference."""

import pytest
import torch

from opsagent_amd import ops
from opsagent_amd.ops import mixer_ops as mx, torch_ref


def step_batch(past, rows, device):
    """One token per sequence, padded to `rows` as a captured step is."""
    B = len(past)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=device)  # noqa: E731
    pad = [0] * (rows - B)
    return mx.SeqBatch(cu=list(range(rows + 1)), past=past + pad, slots=list(range(B)) + pad,
                       cu_t=i32([min(i, B) for i in range(rows + 1)]), past_t=i32(past + pad),
                       slots_t=i32(list(range(B)) + pad), seq_of_t=i32(list(range(B)) + pad),
                       slot_mapping=i32([7 * b + 3 for b in range(B)] + [3] * len(pad)),
                       block_table=i32([[0]] * rows), max_chunk=1, max_total=64)


@pytest.mark.gpu
@pytest.mark.parametrize("taps", [0, 2, 3, 4])
@pytest.mark.parametrize("parts", [0, 1, 5])
@pytest.mark.parametrize("C,groups", [(120, 5), (512, 1), (2048, 1), (4096, 4), (6144, 3), (8192, 1)])
def test_norm_and_convolution(C, groups, parts, taps):
    past, T = [0, 1, 2, 3, 900], 8
    g = torch.Generator(device="cuda").manual_seed(C + taps)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    y, w, residual = rand(max(parts, 1), T, C), (1 + 0.2 * rand(C)).bfloat16(), rand(T, C)
    sb = step_batch(past, T, "cuda")
    total = y[0].clone()
    for plane in y[1:]:
        total += plane
    conv = (rand(C, taps).bfloat16(), rand(len(past), taps - 1, C)) if taps else None
    want_state = conv[1].clone() if taps else None
    want, want_copy = mx.group_rms_norm(total.bfloat16(), w, groups, 1e-5, residual.clone())
    x, copy, h = mx.group_norm_step(ops.PlaneSum(y) if parts else total.bfloat16(), w, groups, 1e-5,
                                    residual, True, conv, sb)
    assert x.data_ptr() == residual.data_ptr()
    # the sum of squares in another order (float32), and an add and a product in one instruction or two
    assert torch.allclose(x, want, rtol=2.0 ** -20, atol=2.0 ** -18)
    assert (copy != want_copy).float().mean() < 0.01
    if not taps:
        assert h is None
        return
    B = len(past)
    want_h = mx.causal_conv_seq(want, conv[0], want_state, sb, True, False)
    assert torch.allclose(h[:B].float(), want_h[:B].float(), rtol=2.0 ** -7, atol=2.0 ** -14)
    assert (h[:B] != want_h[:B]).float().mean() < 0.01
    assert torch.allclose(conv[1], want_state, rtol=2.0 ** -20, atol=2.0 ** -18)


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D,Dv,extra", [(1, 1, 8, 8, 8), (6, 2, 24, 64, 8), (32, 8, 128, 128, 32),
                                            (16, 4, 128, 128, 16), (32, 4, 128, 512, 1536)])
@pytest.mark.parametrize("parts", [0, 1, 5])
def test_attention_preparation(H, G, D, Dv, extra, parts, monkeypatch):
    past, T, eps = [0, 5, 900], 4, 1e-5
    n = (H + G) * D + G * Dv
    g = torch.Generator(device="cuda").manual_seed(n + parts)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    planes = rand(max(parts, 1), T, n + extra)
    bias, qw, kw = (0.1 * rand(n)).bfloat16(), rand(H * D).bfloat16(), rand(G * D).bfloat16()
    caches = [torch.zeros(4, 8, G, D, device="cuda").bfloat16(), torch.zeros(4, 8, G, Dv, device="cuda").bfloat16()]
    sb = step_batch(past, T, "cuda")
    total = planes[0].clone()
    for plane in planes[1:]:
        total += plane
    row = total.bfloat16()
    monkeypatch.setattr(ops, "linear_parts", lambda x, w: ops.PlaneSum(planes) if parts else row)
    x, w = torch.empty(T, 64, device="cuda").bfloat16(), torch.empty(n + extra, 64, device="cuda").bfloat16()
    q, gate = mx.attn_proj_prepare(x, w, bias, qw, kw, H, G, D, Dv, eps, *caches, sb)
    B = len(past)
    assert torch.equal(gate, row[:, n:])
    far = [torch.zeros(c.shape, dtype=torch.float64) for c in caches]
    want = torch_ref.attn_qkv_prepare(row[:B].double().cpu(), bias.double().cpu(), qw.double().cpu(),
                                      kw.double().cpu(), H, G, D, Dv, eps, *far, sb.slot_mapping[:B].cpu())
    # one rounding to bf16, and float32 before it
    for got, ref in ((q[:B], want), *zip(caches, far)):
        assert torch.allclose(got.double().cpu(), ref.double(), rtol=2.0 ** -8 + 2.0 ** -18, atol=2.0 ** -18)


class Plain(torch.nn.Module):
    """A layer of another class, as a user's program may put around one: it takes what layers take."""

    def __init__(self, layer):
        super().__init__()
        self.layer = layer
        self.canon_w = layer.canon_w

    def forward(self, x, sb, kv, state):
        return self.layer(x, sb, kv, state)


@pytest.mark.parametrize("device", [pytest.param("cpu", id="cpu"), pytest.param("cuda", id="gpu", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("way", ["class", "hook"])
def test_layers_that_are_looked_at(device, way):
    """Each then starts with its own convolution, and a hook's rows are what the next one reads."""
    import test_povazen as P

    P._skip_if_wrong_device(device)
    cfg = P.make_cfg(pattern="DaA")
    W = P.other_ranks(cfg, P.O.random_weights(cfg, seed=3))
    toks = P.tokens_for(cfg, 9, 4)
    schedule = [(toks[:6], [5])] + [([t], [0]) for t in toks[6:]]

    def logits(change):
        eng = P.build_engine(cfg, W)
        change(eng.model)
        rp = P.TraceReplayer(eng)
        return torch.cat([rp.step([{"id": "a", "tokens": t, "want": w}], []).cpu() for t, w in schedule])

    want = logits(lambda m: None)

    def wrap(m):
        m.layers[1] = Plain(m.layers[1])

    if way == "class":
        assert torch.allclose(logits(wrap), want, rtol=1e-5, atol=1e-5)
        return
    seen = []
    look = lambda mod, args, out: seen.append(out.shape)  # noqa: E731
    assert torch.allclose(logits(lambda m: m.layers[0].register_forward_hook(look)), want, rtol=1e-5, atol=1e-5)
    assert seen
    double = logits(lambda m: m.layers[0].register_forward_hook(lambda mod, args, out: 2 * out))
    assert not torch.allclose(double, want, rtol=1e-3)
