"""A q | k | v product whose float32 parts its reader adds up, against the product by itself: the decode
attention and the rotation, whose results are the same bits."""

import pytest
import torch

from opsagent_amd import ops

HEAD = 128


def rand(seed, *shape):
    return torch.randn(*shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda")


def added(planes):
    total = planes[0].clone()
    for plane in planes[1:]:
        total += plane
    return total.bfloat16()


def heads(rows, Hq, Hk, D):
    q, k, v = rows.split([Hq * D, Hk * D, Hk * D], dim=-1)
    return q.view(-1, Hq, D), k.view(-1, Hk, D), v.view(-1, Hk, D)


@pytest.mark.gpu
@pytest.mark.parametrize("parts", [1, 5, 8, 9, 16])
@pytest.mark.parametrize("B,Hq,Hk,block", [(2, 4, 4, 16), (3, 8, 4, 32), (8, 32, 8, 32), (7, 8, 1, 8)])
def test_decode_attention(B, Hq, Hk, block, parts):
    lengths = [1, 2, 65, 700, 64, 333, 1, 1025][:B]
    mb = 40 * 32 // block
    table = torch.randperm(B * mb, generator=torch.Generator().manual_seed(B)).view(B, mb).int().cuda()
    seq = torch.tensor(lengths, dtype=torch.int32, device="cuda")
    at = [n - 1 for n in lengths]
    slots = torch.tensor([int(table[b, a // block]) * block + a % block for b, a in enumerate(at)],
                         dtype=torch.int32, device="cuda")
    planes = rand(parts + B, parts, B, (Hq + 2 * Hk) * HEAD)
    cos, sin = (t.cuda() for t in ops.rope_cos_sin(2048, HEAD, 500000.0))
    caches = [rand(s, B * mb, block, Hk, HEAD).bfloat16() for s in (1, 2)]
    other = [c.clone() for c in caches]
    assert ops.decode_takes_parts(B, Hq, Hk, HEAD)
    got = ops.attention_decode_parts(ops.PlaneSum(planes), Hq, Hk, HEAD, *caches, table, seq, cos, sin,
                                     slots, HEAD ** -0.5)
    want = ops.attention_decode_rope(*heads(added(planes), Hq, Hk, HEAD), *other, table, seq, cos, sin, slots)
    assert torch.equal(got, want)
    assert all(torch.equal(a, b) for a, b in zip(caches, other))


@pytest.mark.parametrize("B,Hk,takes", [(1, 8, True), (8, 8, True), (64, 1, True), (9, 8, False), (65, 1, False),
                                        (4096, 8, False), (4097, 8, False), (5000, 1, False)])
def test_steps_that_add_up_parts(B, Hk, takes):
    assert ops.decode_takes_parts(B, 4 * Hk, Hk, HEAD) == takes
    assert not ops.decode_takes_parts(B, 4 * Hk, Hk, 64) and not ops.decode_takes_parts(B, 3 * Hk, Hk, HEAD)


@pytest.mark.gpu
@pytest.mark.parametrize("T,Hq,Hk,D,parts", [(1, 1, 1, 16, 1), (3, 4, 2, 64, 2), (77, 32, 8, 128, 5), (128, 16, 4, 128, 16)])
def test_rotation(T, Hq, Hk, D, parts):
    planes = rand(T + parts, parts, T, (Hq + 2 * Hk) * D)
    positions = torch.arange(100, 100 + T, dtype=torch.int32, device="cuda")
    slots = torch.randperm(160, generator=torch.Generator().manual_seed(T))[:T].int().cuda()
    cos, sin = (t.cuda() for t in ops.rope_cos_sin(512, D, 500000.0))
    caches = [rand(s, 5, 32, Hk, D).bfloat16() for s in (1, 2)]
    other = [c.clone() for c in caches]
    got = ops.rope_kv_parts(ops.PlaneSum(planes), Hq, Hk, D, *caches, cos, sin, positions, slots)
    want = ops.rope_kv_fused(*heads(added(planes), Hq, Hk, D), *other, cos, sin, positions, slots)
    assert all(torch.equal(a, b) for a, b in zip((*got, *caches), (*want, *other)))

