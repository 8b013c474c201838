"""The fp8 tile product against its operands in float64: row and column remainders, one
tile and many, as few K-steps as the ring has buffers and fewer, and all four tilings (one
or two blocks of 128 x 128 a CU, 128 x 256, 256 x 256)."""

import pytest
import torch

from opsagent_amd import ops


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [
    (9, 16, 128), (77, 130, 256), (128, 128, 384), (129, 256, 512), (33, 1000, 640),
    (200, 384, 2048),             # one step to fifteen more than the ring holds
    (2048, 2048, 256),            # 256 tiles: the last that take four steps
    (2049, 2048, 128), (2049, 2048, 256), (2049, 2100, 384), (300, 12500, 1024),
    (1030, 4100, 384), (1500, 12288, 128),                        # two blocks a CU; in rounds
    (500, 16300, 128), (1000, 8190, 640), (520, 12270, 256),      # 128 x 256
    (1025, 7700, 128), (2100, 6100, 384), (513, 16384, 256),      # 256 x 256
])
def test_tile_product(M, N, K):
    torch.manual_seed(M + N + K)
    from opsagent_amd.ops import hip_lib

    # Whole numbers up to 2 and scales that are powers of two: every product and every
    # sum (at most 4 K, far below 2^24) is exact, also where the matrix unit aligns its
    # 64 products to the largest and drops low bits, so the result is the exact one
    # rounded once.
    def operand(rows):
        v = torch.randint(-2, 3, (rows, K), device="cuda").float().to(torch.float8_e4m3fn)
        return v.view(torch.uint8), torch.exp2(torch.randint(-3, 4, (rows,), device="cuda").float())

    (xq, xs), (wq, ws) = operand(M), operand(N)
    got = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device="cuda")
    rc = hip_lib.get_lib().oa_gemm_fp8(
        hip_lib.current_stream_ptr(), xq.data_ptr(), wq.data_ptr(), xs.data_ptr(),
        ws.data_ptr(), got.data_ptr(), M, N, K)
    assert rc == 0
    xd = xq.view(torch.float8_e4m3fn).double() * xs.double()[:, None]
    wd = wq.view(torch.float8_e4m3fn).double() * ws.double()[:, None]
    assert torch.equal(got[:M], (xd @ wd.T).to(torch.bfloat16))
    assert (got[M] == 7.0).all()      # the row after the last stays untouched


def test_ring_or_tiles():
    choice = ops._ring_choice_fp8
    assert choice(80, 28672, 4096) == (96, 1) and choice(81, 28672, 4096) is None
    assert choice(32, 4096, 1024) == (32, 1) and choice(33, 4096, 1024) is None
    assert choice(128, 4096, 3072) == (128, 6) and choice(129, 4096, 3072) is None
    assert choice(129, 2048, 2816) == (128, 5) and choice(200, 2048, 2816) is None
    assert choice(512, 4096, 14336) == (128, 2) and choice(700, 4096, 14336) is None
