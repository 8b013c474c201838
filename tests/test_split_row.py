"""The output product that merges an attention row's key splits, against the merge in a launch of its own."""

import pytest
import torch

from opsagent_amd.ops import mixer_ops as mx

PAGE = 32


@pytest.mark.gpu
@pytest.mark.parametrize("past", [0, 31, 256, 511, 513, 800, 1535])
@pytest.mark.parametrize("H,G,D,N,window,sink,last", [
    (16, 4, 128, 2048, 512, True, False), (16, 4, 128, 4100, 512, False, False), (32, 8, 64, 8, 700, True, True),
    (32, 8, 128, 4096, None, True, False), (32, 32, 128, 520, 512, False, True)])
def test_merge(H, G, D, N, window, sink, last, past):
    g = torch.Generator(device="cuda").manual_seed(past + N)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    pages = 1536 // PAGE
    sb = mx.SeqBatch.build([(past, 1, 0, torch.randperm(pages, generator=torch.Generator().manual_seed(N)).tolist())],
                           PAGE, "cuda")
    sb.max_total = 1536                              # as a captured step sizes its launches
    qkv = rand(1, (H + 2 * G) * D).bfloat16()
    qw, kw, sinks = 1 + 0.1 * rand(D), 1 + 0.1 * rand(D), rand(H) if sink else None
    inv = mx.rotary_inv_freq(D, 10000.0).to("cuda")
    w = (rand(N, H * D) * (H * D) ** -0.5).bfloat16()
    post, nxt = (tuple([1 + 0.1 * rand(N), 0.1 * rand(N), torch.full((1,), 0.5, device="cuda")]) for _ in "pn")
    kv = [rand(pages, PAGE, G, D).bfloat16() for _ in "kv"]
    res = rand(1, N)
    got = []
    for merges in (False, True):
        caches, x = [c.clone() for c in kv], res.clone()
        row = mx.attn_rope_rows(qkv, qw, kw, inv, H, G, D, D, 1e-6, *caches, sb, D ** -0.5, window=window,
                                sinks=sinks, merges=merges and mx.merges_split_row(w, x, torch.bfloat16))
        assert isinstance(row, mx.SplitRow) == merges
        h = mx.linear_dyt_norm(row, w, x, None if last else nxt, torch.bfloat16, post)
        got.append((x, h, *caches))
    (x0, h0, *c0), (x1, h1, *c1) = got
    assert all(torch.equal(a, b) for a, b in zip(c0, c1))
    # values of the row meet in another order and may round to bf16's neighbour: 2^-9 of each, random in
    # sign, over a product of unit size, and then the product's own rounding
    assert (x0 - x1).abs().max() <= 2.0 ** -6 and (x0 - x1).norm() <= 2.0 ** -8 * (x0 - res).norm()
    assert (h0 is None) == last and (last or (h0.float() - h1.float()).abs().max() <= 2.0 ** -5)
