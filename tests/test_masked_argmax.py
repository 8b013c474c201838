"""The greedy choice over bf16 rows (masked_argmax_kernel): rows shorter than a block, ragged last
groups and passes, ties, signed zeros, NaN, infinities, and masks that leave one token or none."""

import pytest
import torch

from opsagent_amd import ops


@pytest.mark.gpu
@pytest.mark.parametrize("V", [8, 40, 8192, 8200, 65536 + 8, 128256, 152064])
@pytest.mark.parametrize("masked", [False, True])
def test_masked_argmax(V, masked):
    g = torch.Generator().manual_seed(V)
    B = 9
    x = torch.randn(B, V, generator=g).bfloat16()      # many ties at this width
    allow = torch.rand(B, V, generator=g) < 0.5 if masked else torch.ones(B, V, dtype=torch.bool)
    x[1, V - 1], allow[1, V - 1] = 100.0, True         # the last token
    x[2] = float("-inf")
    x[3] = float("nan")
    x[3, V // 2] = -5.0
    allow[3, V // 2] = True
    x[4] = -1.0
    x[4, V // 3], x[4, V // 3 + 1] = -0.0, 0.0         # one value: the first of them
    allow[4, V // 3] = True
    x[5, V // 4] = float("inf")
    if masked:
        allow[6] = False
        allow[7] = False
        allow[7, V // 2 + 1] = True
        x[8, 0], allow[8, 0] = 100.0, False            # the largest is not allowed
    words = torch.zeros(B, (V + 31) // 32 * 32, dtype=torch.int64)
    words[:, :V] = allow
    words = (words.view(B, -1, 32) << torch.arange(32)).sum(-1)
    words = torch.where(words >= 2 ** 31, words - 2 ** 32, words).to(torch.int32)
    got = ops.greedy_sample_masked(x.cuda(), words.cuda() if masked else None).tolist()
    for b in range(B):
        ok = allow[b] & ~x[b].isnan() & (x[b] != -float("inf"))
        v = torch.where(ok, x[b].float(), torch.tensor(-float("inf")))
        assert got[b] == (int((v == v.max()).nonzero()[0]) if ok.any() else -1), b


@pytest.mark.gpu
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("V", [8, 8200])
def test_signaling_nan(V, masked):
    """It is never chosen and hides no other token, whatever its place in a group of 8."""
    x = torch.full((4, V), -1.0, dtype=torch.bfloat16)
    bits = x.view(torch.int16)
    bits[0] = 0x7f81
    x[0, 5] = -3.0
    bits[1, 0], bits[1, 6] = 0x7f81, 0x7fa0
    x[1, 7] = 2.0
    bits[2, 3], bits[2, 7] = -0x7f, 0x7fbf            # 0xff81: the sign set
    x[2, 4] = 5.0
    bits[3] = 0x7f81
    words = torch.full((4, (V + 31) // 32), -1, dtype=torch.int32, device="cuda") if masked else None
    assert ops.greedy_sample_masked(x.cuda(), words).tolist() == [5, 7, 4, -1]
