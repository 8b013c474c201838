"""Paged decode attention at the edges of tiles (16 keys), waves (64), splits and
cache blocks, against float64."""

import pytest
import torch

from opsagent_amd import ops

D = 128


def _case(lens, Hk, G, bs, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rn = lambda *s: torch.randn(*s, generator=gen, device="cuda").bfloat16()  # noqa: E731
    need = [(n + bs - 1) // bs for n in lens]
    order = torch.randperm(sum(need), generator=torch.Generator().manual_seed(seed)).tolist()
    table = torch.zeros(len(lens), max(need) + 1, dtype=torch.int32)
    at = 0
    for b, k in enumerate(need):
        table[b, :k] = torch.tensor(order[at : at + k])
        at += k
    kc, vc = rn(at, bs, Hk, D), rn(at, bs, Hk, D)
    qkv = rn(len(lens), (Hk * G + 2 * Hk) * D)
    q, k, v = (t.view(len(lens), -1, D) for t in qkv.split([Hk * G * D, Hk * D, Hk * D], -1))
    slots = [int(table[b, (n - 1) // bs]) * bs + (n - 1) % bs for b, n in enumerate(lens)]
    return (q, k, v, kc, vc, table.cuda(), torch.tensor(lens, dtype=torch.int32, device="cuda"),
            torch.tensor(slots, dtype=torch.int32, device="cuda"))


def _attend(q, ks, vs, G):
    """q [Hq, D], ks/vs [n, Hk, D], float64."""
    s = torch.einsum("hgd,nhd->hgn", q.view(-1, G, D), ks) * D ** -0.5
    return torch.einsum("hgn,nhd->hgd", torch.softmax(s, -1), vs).reshape(-1, D)


def _rotate(x, pos, cos, sin):
    c, s = cos[pos].double(), sin[pos].double()
    a, b = x[..., : D // 2], x[..., D // 2 :]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


@pytest.mark.gpu
@pytest.mark.parametrize("G", [1, 2, 4, 8])
@pytest.mark.parametrize("lens,bs,nsplit", [
    ([1], 32, 32),                                   # the new key alone
    ([2, 16, 17, 18, 64, 65, 66], 32, 32),           # a tile and a wave more or less
    ([127, 128, 129, 130, 257, 513, 1025], 16, 32),  # a split more or less
    ([900, 3, 700], 8, 3),                           # blocks smaller than a tile, few splits
    ([200] * 20 + [1, 65], 32, 1),                   # one split, many sequences
    ([1500 - 61 * i for i in range(24)], 64, 4),     # large splits, ragged
])
def test_decode_attention(G, lens, bs, nsplit):
    Hk = 4
    q, k, v, kc, vc, table, lens_t, slots = _case(lens, Hk, G, bs, seed=sum(lens) + G)
    cos, sin = (t.cuda() for t in ops.rope_cos_sin(2048, D))
    flat_k, flat_v = kc.view(-1, Hk, D), vc.view(-1, Hk, D)
    rows = lambda b, n: (table[b, torch.arange(n, device="cuda") // bs].long() * bs  # noqa: E731
                         + torch.arange(n, device="cuda") % bs)
    plain, roped, new_k = [], [], []
    for b, n in enumerate(lens):
        r = rows(b, n)
        ks, vs = flat_k[r].double(), flat_v[r].double()
        plain.append(_attend(q[b].double(), ks, vs, G))
        new_k.append(_rotate(k[b].double(), n - 1, cos, sin))
        ks, vs = torch.cat([ks[:-1], new_k[-1][None]]), torch.cat([vs[:-1], v[b].double()[None]])
        roped.append(_attend(_rotate(q[b].double(), n - 1, cos, sin), ks, vs, G))

    # the result is one bf16 rounding of a float32 sum: 0.0016 in the mean over the 512
    # values and more of each call (a second one would make it 0.0023)
    def check(got, want):
        want = torch.stack(want)
        err = (got.double() - want).norm() / want.norm()
        assert err < 2e-3, float(err)

    check(ops.attention_decode_paged(q, kc, vc, table, lens_t, nsplit=nsplit), plain)
    check(ops.attention_decode_paged(q, kc, vc, table, lens_t, nsplit=nsplit, fused_combine=True),
          plain)
    check(ops.attention_decode_rope(q, k, v, kc, vc, table, lens_t, cos, sin, slots,
                                    nsplit=nsplit), roped)
    check(flat_k[slots.long()], new_k)               # the new key and value are cached
    assert torch.equal(flat_v[slots.long()], v)


@pytest.mark.gpu
def test_decode_scores_in_32_bits():
    """Scores far beyond what 16-bit queries would keep apart: two keys differ by
    2^-12 of a query of 64, and the softmax is steep."""
    Hk, G, n = 1, 4, 33
    q = torch.zeros(1, G, D, device="cuda", dtype=torch.bfloat16)
    k = torch.zeros(1, Hk, D, device="cuda", dtype=torch.bfloat16)
    v = torch.zeros_like(k)
    q[0, :, 3] = 1.0
    cos = torch.full((64, D // 2), 0.7071067811865476, device="cuda")
    sin = cos.clone()                                # rotated queries are no bf16 values
    kc = torch.zeros(2, 32, Hk, D, device="cuda", dtype=torch.bfloat16)
    kc[:, :, 0, 3] = 4096.0
    kc[0, 7, 0, 3 + D // 2] = 64.0                   # 64 * 0.7071 above the others
    vc = torch.randn(2, 32, Hk, D, device="cuda").bfloat16()
    table = torch.tensor([[0, 1]], dtype=torch.int32, device="cuda")
    lens = torch.tensor([n], dtype=torch.int32, device="cuda")
    slots = torch.tensor([32], dtype=torch.int32, device="cuda")
    got = ops.attention_decode_rope(q, k, v, kc, vc, table, lens, cos, sin, slots, scale=0.25)
    qr = _rotate(q[0].double(), 0, cos, sin)
    ks = torch.cat([kc[0, :, :].double(), _rotate(k.double(), 0, cos, sin)])
    vs = torch.cat([vc[0].double(), v.double()])
    s = torch.einsum("hd,nd->hn", qr, ks[:, 0]) * 0.25
    want = torch.softmax(s, -1) @ vs[:, 0]
    # scores are near 724, float32 keeps 6e-5 of them: weights to 1e-4, then one bf16
    # rounding
    assert ((got[0].double() - want).norm() / want.norm()) < 2.0 ** -8 + 2e-4


@pytest.mark.gpu
@pytest.mark.parametrize("G", [1, 2, 4, 8])
def test_infinite_keys(G):
    """A cached key with an infinite channel has weight zero for the heads whose score it
    makes minus infinity, and leaves the other keys theirs."""
    Hk, n, bs = 2, 300, 32
    q, _, _, kc, vc, table, lens, _ = _case([n], Hk, G, bs, seed=G)
    rows = lambda m: table[0, torch.arange(m, device="cuda") // bs].long() * bs + (  # noqa: E731
        torch.arange(m, device="cuda") % bs)
    q = q.clone()
    q[..., 5] = -q[..., 5].abs() - 0.25
    flat_k, flat_v = kc.view(-1, Hk, D), vc.view(-1, Hk, D)
    at = rows(n)
    flat_k[at[[7, 130, n - 1]], :, 5] = float("inf")
    keep = torch.ones(n, dtype=torch.bool, device="cuda")
    keep[[7, 130, n - 1]] = False
    want = _attend(q[0].double(), flat_k[at[keep]].double(), flat_v[at[keep]].double(), G)
    for nsplit in (1, 4):
        got = ops.attention_decode_paged(q, kc, vc, table, lens, nsplit=nsplit)[0].double()
        assert float((got - want).norm() / want.norm()) < 2.1e-3     # 256 values and more


@pytest.mark.gpu
@pytest.mark.parametrize("lens,nsplit,Hk", [
    ([9000, 4600, 1, 64], 128, 4),                   # 71 splits: more than lanes, asked for ahead
    ([10300, 257] + [5] * 18, 40, 4),                # 33 of 40 beside many short sequences
    ([2000, 33], 32, 32),                            # 64 pairs, asked for ahead
    ([2000, 33, 300], 32, 32),                       # 96 pairs, not
])
def test_combine_of_many_splits(lens, nsplit, Hk):
    G, bs = 2, 32
    q, _, _, kc, vc, table, lens_t, _ = _case(lens, Hk, G, bs, seed=sum(lens))
    want = []
    for b, n in enumerate(lens):
        at = torch.arange(n, device="cuda")
        r = table[b, at // bs].long() * bs + at % bs
        want.append(_attend(q[b].double(), kc.view(-1, Hk, D)[r].double(),
                            vc.view(-1, Hk, D)[r].double(), G))
    got = ops.attention_decode_paged(q, kc, vc, table, lens_t, nsplit=nsplit).double()
    want = torch.stack(want)
    assert (got - want).norm() / want.norm() < 2e-3      # as above: one bf16 rounding


@pytest.mark.gpu
@pytest.mark.parametrize("lens,nsplit,Hk", [([1], 32, 4), ([331], 32, 4), ([64, 700, 129], 8, 4), ([700, 20, 513] * 8, 4, 4),
                                            ([700, 1000, 30, 512] * 8, 32, 8), ([65, 600, 900] * 21, 32, 8)])
@pytest.mark.parametrize("G", [1, 4])
def test_plain_splits_leave_no_marks(lens, nsplit, Hk, G):
    """Under 512 (sequence, key head) pairs sequences are split one by one and the combine counts the
    splits: a launch writes the places that it has and no others, and what stood in those is not
    looked at."""
    bs, B = 32, len(lens)
    q, k, v, kc, vc, table, lens_t, slots = _case(lens, Hk, G, bs, seed=sum(lens))
    cos, sin = (t.cuda() for t in ops.rope_cos_sin(1024, D))
    pairs = B * Hk                                   # keys of a split at these sizes: by the pairs
    least = 64 if pairs <= 8 else 128 if pairs <= 32 else 256 if pairs <= 128 else 512

    def check(call):
        got = []
        for mark in (7.0, -2.0):
            ws = (torch.full((B * Hk * nsplit, G, D), mark, device="cuda"),
                  torch.full((B * Hk * nsplit, G, 2), mark, device="cuda"))
            got.append(call(kc.clone(), vc.clone(), ws))
            for b, n in enumerate(lens):
                used = -(-n // max(least, -(-n // nsplit // 64) * 64))
                rest = [w.view(B, Hk, nsplit, -1)[b, :, used:] for w in ws]
                assert all((r == mark).all() for r in rest), (b, used)
        assert torch.equal(*got)

    check(lambda kc, vc, ws: ops.attention_decode_rope(q, k, v, kc, vc, table, lens_t, cos, sin, slots,
                                                       workspace=ws, nsplit=nsplit))
    if ops.decode_takes_parts(B, Hk * G, Hk, D):
        planes = torch.stack([torch.cat([t.reshape(B, -1) for t in (q, k, v)], -1).float()] * 2)
        planes[1] = 0.0
        check(lambda kc, vc, ws: ops.attention_decode_parts(
            ops.PlaneSum(planes), Hk * G, Hk, D, kc, vc, table, lens_t, cos, sin, slots, D ** -0.5,
            workspace=ws, nsplit=nsplit))


@pytest.mark.gpu
@pytest.mark.parametrize("G,Hk,lens", [(4, 8, [700, 65, 130]), (8, 4, [513, 64]), (1, 33, [1, 90]), (4, 25, [700, 65, 130])])
def test_copies_of_the_first_row(G, Hk, lens):
    """Rows that repeat the first are answered by its results; rows that write its slot but differ
    in a query or an earlier page are answered by themselves."""
    bs, B = 32, 24
    cos, sin = (t.cuda() for t in ops.rope_cos_sin(1024, D))

    def batch(rows):
        q, k, v, kc, vc, table, n, slots = _case(lens, Hk, G, bs, seed=G)
        at = torch.tensor(rows, device="cuda")
        return [x[at].contiguous() for x in (q, k, v)] + [kc, vc, table[at], n[at], cos, sin, slots[at]]

    plain = ops.attention_decode_rope(*batch(range(len(lens))), nsplit=4)
    args = batch([*range(len(lens)), *[0] * (B - len(lens))])
    got = ops.attention_decode_rope(*args, nsplit=4)
    rel = (got[: len(lens)].float() - plain.float()).norm() / plain.float().norm()
    assert rel < 2e-3                                 # splits of other sizes: one bf16 rounding apart
    assert torch.equal(got[len(lens):], got[:1].expand_as(got[len(lens):]))

    args = batch([*range(len(lens)), *[0] * (B - len(lens))])
    args[0][B - 1, 0, 5] += 1.0                       # one query of one head
    if lens[0] > bs:
        args[5][B - 2, 0] = args[5][1, 0]             # another first page
    other = ops.attention_decode_rope(*args, nsplit=4)
    assert torch.equal(other[: B - 2], got[: B - 2])
    alone = [x[-2:].contiguous() for x in (*args[:3], *args[5:7], args[9])]
    want = ops.attention_decode_rope(*alone[:3], args[3], args[4], *alone[3:5], cos, sin, alone[5],
                                     nsplit=4)
    assert (other[-2:].float() - want.float()).norm() / want.float().norm() < 2e-3
    assert lens[0] == 1 or not torch.equal(other[-1], got[0])
    assert lens[0] <= bs or not torch.equal(other[-2], got[0])


@pytest.mark.gpu
@pytest.mark.parametrize("G,Hk", [(4, 8), (8, 4), (1, 33), (4, 25)])
def test_rows_that_are_nearly_copies(G, Hk):
    """Rows with the first row's slot that differ from it in one thing alone (a query, the new key
    or value of one key head, the length, the last page) are answered by themselves. The marks in
    the workspace say which (row, key head) was taken for a copy; a copy's partial results stay as
    they were before the launch."""
    bs, B, n, nsplit = 32, 24, 700, 4
    cos, sin = (t.cuda() for t in ops.rope_cos_sin(1024, D))
    q, k, v, kc, vc, table, lens, slots = _case([n, 65], Hk, G, bs, seed=Hk)
    at = torch.tensor([0, 1] + [0] * (B - 2), device="cuda")
    q, k, v, table, lens, slots = (x[at].contiguous() for x in (q, k, v, table, lens, slots))
    copied = torch.ones(B, Hk, dtype=torch.bool, device="cuda")
    copied[:2] = False
    q[3, Hk * G - 1, D - 1] += 1.0                    # last channel of the last head
    copied[3, Hk - 1] = False
    k[4, 1, 0] += 1.0
    copied[4, 1] = False
    v[5, 0, D - 1] += 1.0
    copied[5, 0] = False
    lens[6] -= 1                                      # its cached keys end before the shared slot
    table[7, (n - 1) // bs] = table[1, 0]
    copied[6:8] = False
    ws = (torch.full((B * Hk * nsplit, G, D), 7.0, device="cuda"),
          torch.full((B * Hk * nsplit, G, 2), 7.0, device="cuda"))
    got = ops.attention_decode_rope(q, k, v, kc.clone(), vc.clone(), table, lens, cos, sin, slots,
                                    workspace=ws, nsplit=nsplit)
    marks = ws[1].view(B, Hk, nsplit, G, 2)[:, :, 0, :, 1]
    assert torch.equal(marks == -1.0, copied[..., None].expand(B, Hk, G))
    assert (ws[0].view(B, Hk, -1)[copied] == 7.0).all()

    by_head = got.view(B, Hk, -1)
    assert torch.equal(by_head[copied], by_head[0].expand(B, -1, -1)[copied])
    for b in range(3, 8):
        alone = [x[b : b + 1] for x in (q, k, v, table, lens, slots)]
        want = ops.attention_decode_rope(*alone[:3], kc.clone(), vc.clone(), *alone[3:5], cos, sin,
                                         alone[5], nsplit=nsplit).view(Hk, -1)
        own = ~copied[b]                              # splits of other sizes: one bf16 rounding apart
        diff = (by_head[b] - want)[own].float().norm() / want[own].float().norm()
        assert diff < 2e-3 and not torch.equal(by_head[b][own], by_head[0][own])


@pytest.mark.gpu
@pytest.mark.parametrize("G", [1, 4, 8])
@pytest.mark.parametrize("lens,Hk,bs,nsplit", [
    ([3000, 1, 63, 64, 65, 2111, 128, 129, 1500, 16, 17, 900, 2500, 700, 31, 1023, 1024, 1025, 2048,
      5, 640], 4, 32, 32),                           # runs that end in, at and across rows
    ([2000 - 27 * i for i in range(70)], 2, 16, 32),  # more rows than lanes
    ([4000] + [900 + 7 * i for i in range(16)], 4, 8, 2),     # two places a row
    ([1 + 9 * i for i in range(66)], 2, 32, 32),     # short rows: units, more rows than lanes
    ([5000] + [5, 64, 65, 513, 1100] * 13, 4, 64, 3),         # units larger for one long row
    ([200] * 3 + [4000], 100, 32, 32),               # more key heads than runs for them
    ([3000, 1, 63, 64, 65, 2111, 128, 129, 1500, 16, 17, 900, 2500, 700, 31, 1023, 1024, 1025, 2048,
      5, 640], 25, 32, 32),                          # 512 pairs and more: the rows of before
    ([2000 - 27 * i for i in range(70)], 8, 16, 32),
    ([4000] + [900 + 7 * i for i in range(16)], 33, 8, 2),
    ([1 + 9 * i for i in range(66)], 8, 32, 32),
    ([3000] + [5, 64, 65, 513, 1100] * 13, 8, 64, 3),
    ([200] * 3 + [4000], 130, 32, 32),
])
def test_runs_over_sequences(G, lens, Hk, bs, nsplit):
    """512 (sequence, key head) pairs and more: blocks go over the tiles of all sequences."""
    q, k, v, kc, vc, table, lens_t, slots = _case(lens, Hk, G, bs, seed=len(lens) + G)
    cos, sin = (t.cuda() for t in ops.rope_cos_sin(8192, D))
    flat_k, flat_v = kc.view(-1, Hk, D), vc.view(-1, Hk, D)
    plain, roped = [], []
    for b, n in enumerate(lens):
        at = torch.arange(n, device="cuda")
        r = table[b, at // bs].long() * bs + at % bs
        ks, vs = flat_k[r].double(), flat_v[r].double()
        plain.append(_attend(q[b].double(), ks, vs, G))
        new = _rotate(k[b].double(), n - 1, cos, sin)
        ks, vs = torch.cat([ks[:-1], new[None]]), torch.cat([vs[:-1], v[b].double()[None]])
        roped.append(_attend(_rotate(q[b].double(), n - 1, cos, sin), ks, vs, G))
    # every row by itself: a bf16 rounding is 2^-9 at the most of each value, 0.0017 over a row
    for got, want in [(ops.attention_decode_paged(q, kc, vc, table, lens_t, nsplit=nsplit), plain),
                      (ops.attention_decode_rope(q, k, v, kc.clone(), vc.clone(), table, lens_t, cos,
                                                 sin, slots, nsplit=nsplit), roped)]:
        for b, w in enumerate(want):
            assert float((got[b].double() - w).norm() / w.norm()) < 2.0 ** -9 + 1e-4, (b, lens[b])

    empty = lens_t.clone()                           # a row without keys is answered by zeros
    empty[1::3] = 0
    got = ops.attention_decode_paged(q, kc, vc, table, empty, nsplit=nsplit)
    for b, w in enumerate(plain):
        if b % 3 == 1:
            assert not got[b].any()
        else:
            assert float((got[b].double() - w).norm() / w.norm()) < 2.0 ** -9 + 1e-4, (b, lens[b])


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hk,G,longest,common", [(64, 8, 4, 1500, 1024), (56, 16, 1, 1500, 1024), (100, 6, 2, 900, 640),
                                                   (64, 8, 4, 1500, 96), (16, 32, 1, 2500, 2016)])
def test_runs_over_shared_pages(B, Hk, G, longest, common):
    """Rows that share the page at their mean length are split in units that go in step, others in runs:
    the marks in the workspace say how many places a row has."""
    bs, nsplit = 32, 32
    lens = [max(1, round(longest * (1 - 0.75 * ((0.618034 * b) % 1.0)))) for b in range(B)]
    q, k, v, kc, vc, table, lens_t, slots = _case(lens, Hk, G, bs, seed=B + Hk)
    cos, sin = (t.cuda() for t in ops.rope_cos_sin(4096, D))
    for b, n in enumerate(lens):
        own = (n - 1) // bs                          # the page that the new key goes to
        table[b, : min(common // bs, own)] = table[0, : min(common // bs, own)]
    ws = (torch.full((B * Hk * nsplit, G, D), 7.0, device="cuda"),
          torch.full((B * Hk * nsplit, G, 2), 7.0, device="cuda"))
    got = ops.attention_decode_rope(q, k, v, kc.clone(), vc.clone(), table, lens_t, cos, sin, slots, workspace=ws,
                                    nsplit=nsplit)
    flat_k, flat_v = kc.view(-1, Hk, D), vc.view(-1, Hk, D)
    for b, n in enumerate(lens):
        at = torch.arange(n, device="cuda")
        r = table[b, at // bs].long() * bs + at % bs
        ks, vs = flat_k[r].double(), flat_v[r].double()
        new = _rotate(k[b].double(), n - 1, cos, sin)
        ks, vs = torch.cat([ks[:-1], new[None]]), torch.cat([vs[:-1], v[b].double()[None]])
        want = _attend(_rotate(q[b].double(), n - 1, cos, sin), ks, vs, G)
        # as above: one bf16 rounding of every row
        assert float((got[b].double() - want).norm() / want.norm()) < 2.0 ** -9 + 1e-4, (b, n)
    tiles = [(n + 63) // 64 for n in lens]
    size = max(8, -(-sum(tiles) // (3 * B)))         # 512 keys, or what the launch's blocks ask for
    units = [-(-n // size) for n in tiles]
    sums = ws[1].view(B, Hk, nsplit, G, 2)[..., 1]
    marked = [bool((sums[b, :, u] == -2.0).all()) and not bool((sums[b, :, :u] == -2.0).any()) for b, u in enumerate(units)]
    assert all(marked) == (common > sum(tiles) * 64 / B)
