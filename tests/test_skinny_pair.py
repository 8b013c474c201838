"""Two products of one size in one launch, against each by itself: the same bits, and other sizes apart."""

import pytest
import torch

from opsagent_amd import ops
from opsagent_amd.ops import hip_lib

DEVICES = [pytest.param("cpu", id="cpu"), pytest.param("cuda", id="gpu", marks=pytest.mark.gpu)]


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("M,N,K,apart,one", [(2, 4096, 256, 904, True), (3, 2048, 128, 400, True), (4, 2056, 128, 0, True),
                                             (16, 4096, 256, 904, True), (17, 4096, 256, 904, False),
                                             (1, 4096, 256, 904, False), (5, 40, 96, 200, False)])
def test_pair(device, M, N, K, apart, one, monkeypatch):
    g = torch.Generator().manual_seed(M + N)
    wide = torch.randn(M, 2 * K + apart, generator=g).bfloat16().to(device)
    x0, x1 = (wide[:, :K], wide[:, K : 2 * K]) if apart else (wide[:, :K].contiguous(), wide[:, K:].contiguous())
    w0, w1 = (torch.randn(N, K, generator=g).bfloat16().to(device) for _ in "01")
    want = ops.linear(x0, w0), ops.linear(x1, w1)
    calls = []
    if device == "cuda":
        lib = hip_lib.get_lib()
        inner = lib.oa_skinny_pair
        monkeypatch.setattr(lib, "oa_skinny_pair", lambda *a: calls.append(1) or inner(*a))
    got = ops.linear_pair(x0, w0, x1, w1)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert bool(calls) == (one and device == "cuda")
