"""Key-split prefill attention at the edges of query tiles, key tiles and splits,
against float64: splits that show a row none of its keys, uneven splits, batches."""

import pytest
import torch

from opsagent_amd import ops

D = 128


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hk,Sq,Skv", [
    (1, 8, 2, 1, 257),            # one query, three key tiles
    (1, 32, 8, 77, 1264),
    (1, 8, 2, 128, 383),          # most rows see nothing of the last split
    (1, 8, 1, 128, 2048),
    (1, 4, 4, 100, 3000),         # no shared key heads
    (2, 4, 2, 33, 900),
    (1, 8, 4, 129, 1600),         # merged form, two, four and eight heads a block
    (1, 8, 2, 300, 1537),
    (1, 8, 1, 400, 1500),
    (1, 4, 1, 1700, 1700),        # the causal diagonal through every split
    (3, 4, 2, 140, 1700),
])
def test_split_prefill(B, Hq, Hk, Sq, Skv):
    splits, _ = ops._prefill_splits(B, Hq, Hk, Sq, Skv)
    assert splits > 1
    gen = torch.Generator(device="cuda").manual_seed(Sq + Skv)
    # head slices of one fused buffer, as the model hands them over
    q = torch.randn(B, Sq, Hq + 3, D, generator=gen, device="cuda").bfloat16()[:, :, :Hq]
    kv = torch.randn(B, Skv, 2 * Hk, D, generator=gen, device="cuda").bfloat16()
    k, v = kv[:, :, :Hk], kv[:, :, Hk:]
    got = ops.attention_prefill(q, k, v)
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
@pytest.mark.parametrize("Hq,Hk,Sq,Skv", [(8, 2, 40, 900), (8, 2, 300, 1600), (8, 4, 300, 1600)])
def test_scores_that_do_not_compare(Hq, Hk, Sq, Skv):
    """A row with a NaN or a positive infinite score is NaN, as softmax makes it, in
    whichever split the score lies; a negative infinite score is a weight of zero."""
    assert ops._prefill_splits(1, Hq, Hk, Sq, Skv)[0] > 1
    gen = torch.Generator(device="cuda").manual_seed(Sq)
    q = torch.randn(1, Sq, Hq, D, generator=gen, device="cuda").bfloat16()
    k, v = (torch.randn(1, Skv, Hk, D, generator=gen, device="cuda").bfloat16() for _ in range(2))
    q[0, 3, 1, 5] = float("nan")
    k[0, 200, 0, 7] = float("inf")                   # every row sees key 200 of key head 0
    v[0, 500, 1, 9] = float("nan")                   # one channel, of key head 1's rows
    bad = torch.zeros(1, Sq, Hq, D, dtype=torch.bool, device="cuda")
    bad[0, 3, 1] = True
    bad[0, :, : Hq // Hk] |= (q[0, :, : Hq // Hk, 7] > 0)[..., None]
    bad[0, :, Hq // Hk : 2 * (Hq // Hk), 9] = True
    assert torch.equal(torch.isnan(ops.attention_prefill(q, k, v)), bad)


def test_rule():
    split = ops._prefill_splits
    assert split(1, 32, 8, 77, 1264) == (8, False) and split(1, 32, 8, 128, 256) == (1, False)
    assert split(1, 32, 8, 300, 4000) == (6, True) and split(1, 32, 8, 1024, 1024) == (1, False)
    assert split(1, 32, 8, 2048, 6144) == (1, True)
    assert split(1, 6, 2, 300, 4000) == (1, False)            # three heads a key head
    assert split(64, 32, 8, 77, 1264) == (1, False)


def test_lines_by_rows():
    """More key tiles where more rows leave sums: both sides of each line."""
    split = ops._prefill_splits
    for B, Hq, Sq, least in ((1, 16, 128, 3), (1, 32, 77, 3), (1, 32, 128, 4), (1, 64, 77, 4),
                             (8, 16, 16, 4), (1, 80, 77, 5), (1, 64, 128, 5), (4, 32, 77, 6),
                             (4, 32, 128, 6)):
        assert split(B, Hq, Hq, Sq, 128 * least - 20)[0] > 1
        assert split(B, Hq, Hq, Sq, 128 * (least - 1) - 20) == (1, False)
    assert split(1, 8, 2, 0, 300)[0] >= 1 and split(2, 0, 1, 16, 900)[0] >= 1
