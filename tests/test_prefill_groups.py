"""Prefill attention in one, two and four key groups a block, at the edges of query tiles, key
tiles and groups, against float64: groups that see no key of a row, groups without a tile."""

import pytest
import torch

from opsagent_amd import ops

D = 128


@pytest.mark.gpu
@pytest.mark.parametrize("variant", [7, 8, 10, 11, 0])   # steady, 1, 2, 4 groups, by the rule
@pytest.mark.parametrize("B,Hq,Hk,Sq,Skv", [
    (1, 4, 4, 1, 1),              # one key: three of four groups have no tile
    (1, 4, 2, 33, 33),            # a second wave of one row, groups behind the diagonal
    (2, 6, 2, 65, 97),            # three heads a key head, a tile of one key more
    (1, 3, 1, 129, 191),
    (1, 16, 2, 64, 64),
    (3, 8, 8, 257, 257),          # a query tile of one row in every form
    (1, 8, 1, 127, 300),
    (1, 32, 8, 700, 740),         # more blocks than CUs
])
def test_forms(monkeypatch, variant, B, Hq, Hk, Sq, Skv):
    if variant:
        monkeypatch.setenv("OPSAGENT_PREFILL_VARIANT", str(variant))
    gen = torch.Generator(device="cuda").manual_seed(Sq + Skv)
    q = torch.randn(B, Sq, Hq + 1, D, generator=gen, device="cuda").bfloat16()[:, :, :Hq]
    kv = torch.randn(B, Skv, 2 * Hk, D, generator=gen, device="cuda").bfloat16()
    k, v = kv[:, :, :Hk], kv[:, :, Hk:]
    check(ops.attention_prefill(q, k, v), q, k, v)


def check(got, q, k, v):
    (B, Sq, Hq, _), (Skv, Hk) = q.shape, k.shape[1:3]
    i = torch.arange(Skv - Sq, Skv, device="cuda")[:, None]
    hidden = torch.arange(Skv, device="cuda")[None] > i
    for b in range(B):
        for h in range(Hq):
            g = h // (Hq // Hk)
            s = (q[b, :, h].double() @ k[b, :, g].double().T * D ** -0.5).masked_fill(hidden, -1e30)
            want = torch.softmax(s, -1) @ v[b, :, g].double()
            # weights enter the value product in bf16 (2^-8 at most, 0.0016 in the
            # mean, over many keys of either sign) and the result is rounded once
            err = (got[b, :, h].double() - want).norm() / want.norm()
            assert err < 6e-3, (b, h, float(err))


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hk,Sq,Skv", [(8, 2, 40, 700), (8, 2, 128, 383), (8, 2, 300, 1600),
                                          (32, 8, 130, 200), (32, 8, 1100, 1100)])
def test_steady(Hq, Hk, Sq, Skv):
    """What 8-bit models call: split and not, 128 rows and 256."""
    gen = torch.Generator(device="cuda").manual_seed(Sq)
    q, k, v = (torch.randn(1, n, h, D, generator=gen, device="cuda").bfloat16()
               for n, h in ((Sq, Hq), (Skv, Hk), (Skv, Hk)))
    check(ops.attention_prefill(q, k, v, steady=True), q, k, v)


@pytest.mark.gpu
@pytest.mark.parametrize("variant", [7, 8, 9, 10, 11, 0])
@pytest.mark.parametrize("steady", [False, True])
@pytest.mark.parametrize("Hq,Hk,Sq,Skv", [(8, 2, 1, 1), (8, 4, 33, 129), (16, 2, 200, 257),
                                          (8, 2, 70, 900), (8, 2, 300, 1700)])
def test_cache_rows(monkeypatch, variant, steady, Hq, Hk, Sq, Skv):
    """Keys and values read from the cache's rows, split and not: bit for bit the results of
    gathered ones."""
    if variant:
        monkeypatch.setenv("OPSAGENT_PREFILL_VARIANT", str(variant))
    gen = torch.Generator(device="cuda").manual_seed(Sq + Skv)
    q, k, v = (torch.randn(n, h, D, generator=gen, device="cuda").bfloat16()
               for n, h in ((Sq, Hq), (Skv + 40, Hk), (Skv + 40, Hk)))
    slots = torch.randperm(Skv + 40, generator=gen, device="cuda")[:Skv].contiguous()
    want = ops.attention_prefill(q[None], k[slots][None], v[slots][None], steady=steady)
    assert torch.equal(ops.attention_prefill(q[None], k, v, steady=steady, slots=slots), want)
    apart = torch.stack([slots, slots], 1)[:, 0]         # rows that are not side by side
    assert torch.equal(ops.attention_prefill(q[None], k, v, steady=steady, slots=apart), want)


def test_cache_rows_on_the_host():
    gen = torch.Generator().manual_seed(0)
    q, k, v = (torch.randn(n, 2, 16, generator=gen) for n in (5, 20, 20))
    slots = torch.randperm(20, generator=gen)[:9]
    assert torch.equal(ops.attention_prefill(q[None], k, v, slots=slots),
                       ops.attention_prefill(q[None], k[slots][None], v[slots][None]))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["host", "int32", "below 0", "wider rows", "off the grid", "mask"])
def test_any_index_of_rows(kind):
    """Every index that a gather takes: on the host, of 32 bits, from the end; caches that the kernel
    cannot read in place."""
    gen = torch.Generator(device="cuda").manual_seed(len(kind))
    Hq, Hk, Sq, Skv, rows = 8, 2, 70, 410, 450
    q = torch.randn(1, Sq, Hq, D, generator=gen, device="cuda").bfloat16()
    k, v = (torch.randn(rows, Hk, D + 8, generator=gen, device="cuda").bfloat16() for _ in range(2))
    if kind == "wider rows":
        k, v = k[:, :, :D], v[:, :, :D]
    elif kind == "off the grid":
        k, v = (t.flatten()[1:1 + rows * Hk * D].view(rows, Hk, D) for t in (k, v))
    else:
        k, v = k[:, :, :D].contiguous(), v[:, :, :D].contiguous()
    slots = torch.randperm(rows, generator=gen, device="cuda")[:Skv].contiguous()
    if kind == "host":
        slots = slots.cpu()
    elif kind == "int32":
        slots = slots.int()
    elif kind == "below 0":
        slots[::3] -= rows
    elif kind == "mask":
        slots = torch.zeros(rows, dtype=torch.bool, device="cuda").index_fill(0, slots, True)
    want = ops.attention_prefill(q, k[slots].view(1, Skv, Hk, D), v[slots].view(1, Skv, Hk, D))
    assert torch.equal(ops.attention_prefill(q, k, v, slots=slots), want)


@pytest.mark.gpu
@pytest.mark.parametrize("steady", [False, True])
def test_rows_outside(steady):
    """A slot outside the caches reads their last row, on either side; of more bits the low 32 count."""
    gen = torch.Generator(device="cuda").manual_seed(3)
    Sq, Skv, rows = 40, 700, 750
    q, k, v = (torch.randn(n, 2, D, generator=gen, device="cuda").bfloat16() for n in (Sq, rows, rows))
    slots = torch.randperm(rows, generator=gen, device="cuda")[:Skv].contiguous()
    far = slots.clone()
    for i, at in ((5, rows), (133, 2 ** 31 - 1), (300, -rows - 1), (450, -2 ** 31), (699, 2 ** 40 + rows)):
        slots[i], far[i] = rows - 1, at
    want = ops.attention_prefill(q[None], k[slots][None], v[slots][None], steady=steady)
    assert torch.equal(ops.attention_prefill(q[None], k, v, steady=steady, slots=far), want)


def _attend(device, dtype, gather, past=24, T=9, block=8, heads=2):
    """One attention sublayer over T rows behind a past, its caches' rows named by gather(list)."""
    from opsagent_amd.engine import model as m
    from opsagent_amd.engine.config import get_model_spec

    spec = get_model_spec("llama3-tiny") if dtype == torch.float32 else get_model_spec("llama3-micro")
    gen = torch.Generator().manual_seed(1)
    layer = m.Attention(spec, dtype, gen).to(device)
    hd, rows = spec.head_dim, 6 * block
    caches = [torch.randn(6, block, spec.num_kv_heads, hd, generator=gen).to(dtype).to(device) for _ in "kv"]
    cos, sin = (torch.randn(past + T, hd // 2, generator=gen).to(device) for _ in "cs")
    slots = torch.randperm(rows, generator=gen)[:past + T]
    x = torch.randn(T, spec.hidden_size, generator=gen).to(dtype).to(device)
    fb = m.ForwardBatch(kind="prefill", input_ids=torch.zeros(T, dtype=torch.int64, device=device),
                        positions=torch.arange(past, past + T, dtype=torch.int32, device=device),
                        slot_mapping=slots[past:].int().to(device), prefill_past_len=past,
                        prefill_slot_gather=gather(slots.to(device), rows))
    with torch.no_grad():
        return layer(x, cos, sin, *caches, fb)


GATHERS = {"host": lambda s, n: s.cpu(), "int32": lambda s, n: s.int(), "table": lambda s, n: s.view(3, -1),
           "below 0": lambda s, n: s - n}


@pytest.mark.parametrize("device,dtype", [("cpu", torch.float32), pytest.param(
    "cuda", torch.bfloat16, marks=pytest.mark.gpu)])
def test_rows_of_a_past(device, dtype):
    """What a sublayer's caller may hand in as the rows of a past, and lengths that are refused."""
    want = _attend(device, dtype, lambda s, n: s)
    for name, gather in GATHERS.items():
        assert torch.equal(_attend(device, dtype, gather), want), name
    for wrong in (lambda s, n: s[:-1], lambda s, n: torch.cat([s, s[:1]]), lambda s, n: s[:0], lambda s, n: None):
        with pytest.raises(RuntimeError):
            _attend(device, dtype, wrong)


@pytest.mark.gpu
@pytest.mark.parametrize("steady", [False, True])
@pytest.mark.parametrize("scale", [-1.0, -0.0, 0.0])
@pytest.mark.parametrize("Hq,Hk,Sq,Skv", [(8, 2, 40, 900), (32, 8, 300, 4000), (32, 8, 1100, 1100),
                                          (48, 16, 1500, 1500), (4, 4, 65, 65)])
def test_scales_that_turn_scores(Hq, Hk, Sq, Skv, scale, steady):
    """Negative and zero scales, where the largest score has not the largest weight: split over many
    and few queries, blocks of a key head, of 256 rows and of fewer."""
    gen = torch.Generator(device="cuda").manual_seed(Sq)
    q, k, v = (torch.randn(1, n, h, D, generator=gen, device="cuda").bfloat16()
               for n, h in ((Sq, Hq), (Skv, Hk), (Skv, Hk)))
    got = ops.attention_prefill(q, k, v, scale=scale, steady=steady)
    check(got, q.double() * (scale * D ** 0.5), k, v)
    slots = torch.randperm(Skv, generator=gen, device="cuda")
    back = torch.argsort(slots)                          # row slots[i] is key i
    assert torch.equal(ops.attention_prefill(q, k[0][back], v[0][back], scale=scale, steady=steady,
                                             slots=slots), got)


def test_scales_have_one_form():
    for Hq, Hk, Sq, Skv in ((32, 8, 300, 4000), (32, 8, 40, 900), (32, 8, 2048, 2048), (4, 4, 5, 5)):
        assert ops._prefill_plan(1, Hq, Hk, Sq, Skv, scaled=True)[1] == 2
        assert ops._prefill_plan(1, Hq, Hk, Sq, Skv, True, True)[1] == 2


@pytest.mark.gpu
@pytest.mark.parametrize("variant", [10, 11])
def test_scores_that_do_not_compare(monkeypatch, variant):
    """A row with a NaN or a positive infinite score is NaN in whichever group the score lies,
    and so is the softmax of no key; other rows of its block are not."""
    monkeypatch.setenv("OPSAGENT_PREFILL_VARIANT", str(variant))
    gen = torch.Generator(device="cuda").manual_seed(variant)
    Sq, Skv = 60, 340
    q, k, v = (torch.randn(1, n, 2, D, generator=gen, device="cuda").bfloat16()
               for n in (Sq, Skv, Skv))
    q[0, 3, 1, 5] = float("nan")
    k[0, 70, 0, 7] = float("inf")
    v[0, 100, 1, 9] = float("nan")
    bad = torch.zeros(1, Sq, 2, D, dtype=torch.bool, device="cuda")
    bad[0, 3, 1] = True
    bad[0, :, 0] |= (q[0, :, 0, 7] > 0)[:, None]
    bad[0, :, 1, 9] = True
    assert torch.equal(torch.isnan(ops.attention_prefill(q, k, v)), bad)
    # ten rows in front of the first key
    got = ops.attention_prefill(q[:, :, :1], k[:, :50, 1:], v[:, :50, :1])
    assert torch.isnan(got[0, :10]).all() and torch.isfinite(got[0, 10:]).all()


def test_few_splits():
    """Splits only where they beat key groups: more tiles where few splits fill the chip or
    where many rows leave sums; the steady form by its own rule."""
    plan = ops._prefill_plan
    for Hq, Sq, n, least in ((32, 1000, 2, 64), (32, 520, 3, 20), (32, 400, 4, 28),
                             (16, 700, 5, 18), (32, 300, 6, 16)):
        assert plan(1, Hq, Hq // 4, Sq, 128 * least) == (n, 1)
        assert plan(1, Hq, Hq // 4, Sq, 128 * (least - 1)) == (1, 1)
        assert plan(1, Hq, Hq // 4, Sq, 128 * (least - 1), True) == (n, 1)
    assert plan(1, 32, 8, 77, 1264) == (8, 0) and plan(1, 32, 8, 77, 1264, True) == (8, 2)
    assert plan(1, 80, 20, 128, 768) == (1, 0) and plan(1, 80, 20, 128, 768, True) == (3, 2)
    assert plan(1, 80, 20, 40, 2048) == (3, 0) and plan(1, 6, 2, 300, 4000) == (1, 0)
