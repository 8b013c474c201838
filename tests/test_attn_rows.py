"""Decode attention with the keys and values in registers (attn_rows_kernel) against 64 bits:
contexts around a piece, a page and a round of eight waves, pages smaller than a piece, every
option of the call, split and whole. The rule of the splits is checked by itself."""

import ctypes
import os

import pytest
import torch

from opsagent_amd.ops import mixer_ops as mx

LIB = os.path.join(os.path.dirname(mx.__file__), "libopsagent_mixers.so")


@pytest.mark.skipif(not os.path.exists(LIB), reason="mixers .so not built")
def test_splits():
    splits = ctypes.CDLL(LIB).oa_attn_rows_splits
    assert splits(16, 1, 128, 128, 0, 1, 1, 4000) == 0      # 16 heads a kv head: columns of a tile
    assert splits(8, 2, 128, 64, 0, 1, 1, 4000) == 0        # value heads of another size
    assert splits(8, 2, 96, 96, 0, 1, 1, 4000) == 0
    assert splits(8, 2, 128, 128, 1, 1, 1, 4000) == 0       # float32
    assert splits(8, 2, 128, 128, 0, 2, 1, 4000) == 0       # not a decode step
    for H, G in ((1, 1), (15, 1), (12, 2), (14, 2), (32, 8), (64, 64)):
        hb = 4 if H // G % 4 == 0 else (2 if H // G % 2 == 0 else 1)
        for D in (64, 128, 256):
            for rows in (1, 3, 16, 300):
                for reach in (1, 256, 512, 513, 2000, 100000):
                    n = splits(H, G, D, D, 0, 1, rows, reach)
                    assert 1 <= n <= 64
                    assert n == 1 or rows * H // hb * n <= 256
                    assert n == 1 or reach > 16 * (16 if D == 256 else 32)


def _exact(q, k, v, table, past, page, scale, slopes, gate, window, sinks, softcap, keep, channels):
    """(result, largest score magnitude) in 64 bits; k, v [pages, page, heads, D]"""
    T, H, D = q.shape
    G, Gv, out, big = k.shape[2], v.shape[2], [], 0.0
    for t in range(T):
        pos = torch.arange(past[t] + 1)
        at = torch.tensor(table[t])[pos // page], pos % page
        kt = k[at].double().repeat_interleave(H // G, 1)
        vt = v[at].double()[:, torch.arange(G) % Gv].repeat_interleave(H // G, 1)
        s = torch.einsum("hd,nhd->hn", q[t].double(), kt) * scale
        big = max(big, float(torch.einsum("hd,nhd->hn", q[t].double().abs(), kt.abs()).max()) * scale)
        if softcap:
            s = softcap * torch.tanh(s / softcap)
        if slopes is not None:
            s = s - slopes.double()[:, None] * (past[t] - pos)
        if window:
            s[:, (past[t] - pos >= window) & (pos >= keep)] = -float("inf")
        norm = torch.logsumexp(s, 1)
        if sinks is not None:
            norm = torch.logaddexp(norm, sinks.double())
        o = torch.einsum("hn,nhd->hd", torch.exp(s - norm[:, None]), vt)
        if gate is not None:
            o = o * torch.sigmoid(gate[t].double().view(H, -1))
        out.append(o.reshape(-1))
    return torch.stack(out), big


@pytest.mark.gpu
@pytest.mark.parametrize("splits", [None, 1, 3])
@pytest.mark.parametrize("ctx,H,G,D,page,opts", [
    ([1, 32, 33, 64, 513], 32, 8, 128, 32, dict(slopes=True, gate="heads")),
    ([257, 16, 700], 6, 2, 128, 8, dict(sinks=True)),                     # pages below a piece
    ([2005, 511], 16, 4, 128, 32, dict(window=512, sinks=True)),
    ([31, 300, 1], 12, 2, 64, 16, dict(window=40, keep=5, gate="channels", softcap=20.0)),
    ([129, 1030], 4, 4, 64, 64, dict(window=33, keep=70, value_heads=2)),
    ([17, 128, 500], 15, 1, 256, 32, dict(slopes=True, wide_values=True)),
    ([8300], 2, 2, 256, 16, dict()),                                      # above 64 pieces a wave
    ([40, 95], 14, 2, 128, 32, dict(gate="heads", sinks=True, keep=64, window=1)),
])
def test_rows(monkeypatch, splits, ctx, H, G, D, page, opts):
    g = torch.Generator().manual_seed(sum(ctx) + D)
    rn = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    need = [(c + page - 1) // page for c in ctx]
    perm = torch.randperm(sum(need), generator=g).tolist()
    table = [perm[sum(need[:i]):sum(need[:i + 1])] for i in range(len(ctx))]
    past = [c - 1 for c in ctx]
    T, Gv = len(ctx), opts.get("value_heads", G)
    q, k = rn(T, H, D).bfloat16(), rn(sum(need), page, G, D).bfloat16()
    v = rn(sum(need), page, Gv, D * (2 if opts.get("wide_values") else 1)).bfloat16()
    v = v[..., :D]                                   # the leading channels of wider rows
    slopes = 0.1 * torch.rand(H, generator=g) if opts.get("slopes") else None
    sinks = rn(H) if opts.get("sinks") else None
    gate = opts.get("gate") and rn(T, H * (D if opts["gate"] == "channels" else 1)).bfloat16()
    window, softcap, keep = (opts.get(n, 0) for n in ("window", "softcap", "keep"))
    want, big = _exact(q, k, v, table, past, page, D ** -0.5, slopes, gate, window, sinks, softcap,
                       keep, opts.get("gate") == "channels")

    lib = mx._lib()[0]
    assert lib.oa_attn_rows_splits(H, G, D, D, 0, 1, T, max(ctx)) > 0
    if splits:
        monkeypatch.setattr(lib, "oa_attn_rows_splits", lambda *args: splits)
    sb = mx.SeqBatch.build([(p, 1, i, t) for i, (p, t) in enumerate(zip(past, table))], page, "cuda")
    dev = lambda x: None if x is None else x.cuda()  # noqa: E731
    vd = torch.empty(sum(need), page, Gv, 2 * D, dtype=torch.bfloat16, device="cuda")
    vd = vd[..., :D] if opts.get("wide_values") else torch.empty(v.shape, dtype=v.dtype, device="cuda")
    vd.copy_(v)
    got = mx.attention_paged(dev(q), dev(k), vd, sb, D ** -0.5, dev(slopes), dev(gate), window or None,
                             dev(sinks), softcap or None, keep_first=keep,
                             gate_channels=opts.get("gate") == "channels").cpu().double()
    # a float32 sum of n terms is off by about 4 sqrt(n) 2^-24 of their size: the scores (D terms),
    # the cap (2 softcap log2(e) within 2^-21), the distance (exact to 2^-23), the weights and
    # their sums (a term a key). A weight's relative error moves the result twice: in the sum
    # over the values, at most their largest in size, and in the normaliser
    rel = (4 * D ** 0.5 * 2.0 ** -24 * big + 3 * softcap * 2.0 ** -21 + 0.1 * max(ctx) * 2.0 ** -23
           + 4 * max(ctx) ** 0.5 * 2.0 ** -24 + 2.0 ** -21)
    bound = want.abs() * 2.0 ** -8 + 2 * rel * float(v.float().abs().max())
    assert ((got - want).abs() <= bound).all(), ((got - want).abs() / bound).max()


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("H,G,chunks,page,opts", [
    (4, 1, [(0, 17), (63, 2), (100, 64)], 32, dict(slopes=True)),
    (6, 3, [(0, 130), (5, 1)], 8, dict(window=33, keep=5, sinks=True)),   # pages below a tile's 64 keys
    (3, 1, [(190, 3)], 64, dict(softcap=20.0, gate="heads")),
    (40, 2, [(300, 1), (16, 1), (0, 1)], 32, dict(slopes=True, sinks=True)),   # heads in the columns
])
def test_prompts(D, H, G, chunks, page, opts):
    """The tile kernel at the head sizes that it is built for, against 64 bits."""
    g = torch.Generator().manual_seed(D + H)
    rn = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    need = [(p + n + page - 1) // page for p, n in chunks]
    perm = torch.randperm(sum(need), generator=g).tolist()
    table = [perm[sum(need[:i]):sum(need[:i + 1])] for i in range(len(chunks))]
    T = sum(n for _, n in chunks)
    q, k, v = rn(T, H, D).bfloat16(), rn(sum(need), page, G, D).bfloat16(), rn(sum(need), page, G, D).bfloat16()
    slopes = 0.1 * torch.rand(H, generator=g) if opts.get("slopes") else None
    sinks = rn(H) if opts.get("sinks") else None
    gate = rn(T, H).bfloat16() if opts.get("gate") else None
    window, softcap, keep = (opts.get(n, 0) for n in ("window", "softcap", "keep"))
    rows = [(t, p + i) for t, (p, n) in zip(table, chunks) for i in range(n)]
    want, big = _exact(q, k, v, [t for t, _ in rows], [p for _, p in rows], page, D ** -0.5, slopes, gate,
                       window, sinks, softcap, keep, False)
    sb = mx.SeqBatch.build([(p, n, i, t) for i, ((p, n), t) in enumerate(zip(chunks, table))], page, "cuda")
    dev = lambda x: None if x is None else x.cuda()  # noqa: E731
    got = mx.attention_paged(q.cuda(), k.cuda(), v.cuda(), sb, D ** -0.5, dev(slopes), dev(gate), window or None,
                             dev(sinks), softcap or None, keep_first=keep).cpu().double()
    # as above; a weight enters its product as two bf16, within 2^-15 of itself
    ctx = max(p + n for p, n in chunks)
    rel = (4 * D ** 0.5 * 2.0 ** -24 * big + 3 * softcap * 2.0 ** -21 + 0.1 * ctx * 2.0 ** -23
           + 4 * ctx ** 0.5 * 2.0 ** -24 + 2.0 ** -21 + 2.0 ** -15)
    bound = want.abs() * 2.0 ** -8 + 2 * rel * float(v.float().abs().max())
    assert ((got - want).abs() <= bound).all(), ((got - want).abs() / bound).max()


def _counted(monkeypatch, lib):
    """The launches of a decode step's preparation and attention, as they are made."""
    calls = []
    for name in ("oa_attn_rows_rope", "oa_attn_rope_prepare", "oa_attn_bias_paged"):
        inner = getattr(lib, name)
        monkeypatch.setattr(lib, name, lambda *a, name=name, inner=inner: calls.append(name) or inner(*a))
    return calls


@pytest.mark.gpu
@pytest.mark.parametrize("splits", [None, 1, 3])
@pytest.mark.parametrize("ctx,H,G,D,page,window,nfreq,sinks", [
    ([1, 32, 33, 64, 513], 32, 8, 128, 32, None, 64, False),
    ([257, 16, 700, 1], 6, 2, 128, 8, 40, 20, True),             # pages below a piece
    ([2005, 511], 16, 4, 128, 32, 512, 64, True),
    ([31, 300, 1], 12, 2, 64, 16, 1, 32, False),
    ([129, 1030], 4, 4, 64, 64, 33, 0, True),
])
def test_from_the_projection(monkeypatch, splits, ctx, H, G, D, page, window, nfreq, sinks):
    """Head norms, rotation and cache writes inside the launch: the rows that are written, and the
    result, against the two launches; every other row of the cache stays, and what lies in the new
    token's slots before does not matter."""
    g = torch.Generator(device="cuda").manual_seed(sum(ctx) + D)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    need = [(c + page - 1) // page for c in ctx]
    perm = torch.randperm(sum(need), generator=torch.Generator().manual_seed(1)).tolist()
    table = [perm[sum(need[:i]):sum(need[:i + 1])] for i in range(len(ctx))]
    past, T = [c - 1 for c in ctx], len(ctx)
    qkv = rn(T, (H + 2 * G) * D + 8).bfloat16()[:, :(H + 2 * G) * D]        # rows apart
    qw, kw = 1 + 0.1 * rn(D), 1 + 0.1 * rn(D)
    freq = mx.rotary_inv_freq(2 * nfreq, 10000.0).cuda() if nfreq else torch.empty(0, device="cuda")
    k, v = rn(sum(need), page, G, D).bfloat16(), rn(sum(need), page, G, D).bfloat16()
    sk = rn(H) if sinks else None
    sb = mx.SeqBatch.build([(p, 1, i, t) for i, (p, t) in enumerate(zip(past, table))], page, "cuda")
    lib = mx._lib()[0]
    if splits:
        monkeypatch.setattr(lib, "oa_attn_rows_splits", lambda *args: splits)
    k1, v1, k2, v2 = k.clone(), v.clone(), k.clone(), v.clone()
    q = mx.attn_rope_prepare(qkv, qw, kw, freq, H, G, D, D, 1e-6, k1, v1, sb)
    want = mx.attention_paged(q, k1, v1, sb, D ** -0.5, window=window, sinks=sk)
    slots = sb.slot_mapping.long()
    k2.view(-1, G, D)[slots] = float("nan")
    v2.view(-1, G, D)[slots] = float("nan")
    calls = _counted(monkeypatch, lib)
    got = mx.attn_rope_rows(qkv, qw, kw, freq, H, G, D, D, 1e-6, k2, v2, sb, D ** -0.5,
                            window=window, sinks=sk)
    assert calls == ["oa_attn_rows_rope"]
    # the sums of squares in another order: a few queries and keys round to the other neighbour
    assert torch.equal(v2, v1)
    assert torch.allclose(k2.float(), k1.float(), rtol=2.0 ** -7, atol=0)
    assert (k2 != k1).float().mean() < 0.01
    assert (got.float() - want.float()).norm() <= 2.0 ** -8 * want.float().norm()
    assert (got.float() - want.float()).abs().max() <= 2.0 ** -6 * v.float().abs().max()


@pytest.mark.gpu
@pytest.mark.parametrize("other", ["float32", "prompt", "256", "value heads", "16 heads", "rows off the grid",
                                   "weights off the grid"])
def test_others_take_two_launches(monkeypatch, other):
    """What the fused launch does not take is prepared and attended as before, bit for bit."""
    g = torch.Generator(device="cuda").manual_seed(2)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    dtype = torch.float32 if other == "float32" else torch.bfloat16
    H, G, D, page, past, new = 8, 2, 128, 16, 37, 2 if other == "prompt" else 1
    D, Dv = {"256": (256, 256), "value heads": (128, 64)}.get(other, (D, D))
    H = 32 if other == "16 heads" else H
    n = (H + G) * D + G * Dv
    qkv = rn(new, n + 7).to(dtype)[:, :n] if other == "rows off the grid" else rn(new, n).to(dtype)
    off = int(other == "weights off the grid")
    qw, kw = ((1 + 0.1 * rn(D + off))[off:] for _ in "qk")
    freq = mx.rotary_inv_freq(D, 10000.0).cuda()
    sb = mx.SeqBatch.build([(past, new, 0, [2, 0, 1])], page, "cuda")
    k, v = rn(3, page, G, D).to(dtype), rn(3, page, G, Dv).to(dtype)
    k1, v1, k2, v2 = k.clone(), v.clone(), k.clone(), v.clone()
    q = mx.attn_rope_prepare(qkv, qw, kw, freq, H, G, D, Dv, 1e-6, k1, v1, sb)
    want = mx.attention_paged(q, k1, v1, sb, D ** -0.5, window=20)
    calls = _counted(monkeypatch, mx._lib()[0])
    got = mx.attn_rope_rows(qkv, qw, kw, freq, H, G, D, Dv, 1e-6, k2, v2, sb, D ** -0.5, window=20)
    assert calls == ["oa_attn_rope_prepare", "oa_attn_bias_paged"]
    assert torch.equal(got, want) and torch.equal(k1, k2) and torch.equal(v1, v2)
