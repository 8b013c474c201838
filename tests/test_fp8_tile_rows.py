"""The fp8 tile product in tiles of 96 rows (one round of the CUs at most): edges of rows and columns, fewer
steps than the ring holds and more, the last size that it takes and the first that it leaves."""

import pytest
import torch

from opsagent_amd.ops import hip_lib


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [
    (1, 1, 128), (95, 127, 256), (96, 128, 384), (97, 129, 512), (192, 250, 640), (193, 1000, 1536),
    (767, 4096, 256), (768, 4096, 640), (769, 4096, 384), (1536, 2048, 512), (1537, 2048, 128),
])
def test_rows_of_96(M, N, K):
    torch.manual_seed(M + N + K)

    # whole numbers up to 2, scales that are powers of two: every sum (at most 4 K) is exact
    def operand(rows):
        v = torch.randint(-2, 3, (rows, K), device="cuda").float().to(torch.float8_e4m3fn)
        return v.view(torch.uint8), torch.exp2(torch.randint(-3, 4, (rows,), device="cuda").float())

    (xq, xs), (wq, ws) = operand(M), operand(N)
    got = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device="cuda")
    assert hip_lib.get_lib().oa_gemm_fp8(
        hip_lib.current_stream_ptr(), xq.data_ptr(), wq.data_ptr(), xs.data_ptr(), ws.data_ptr(),
        got.data_ptr(), M, N, K) == 0
    xd = xq.view(torch.float8_e4m3fn).double() * xs.double()[:, None]
    wd = wq.view(torch.float8_e4m3fn).double() * ws.double()[:, None]
    assert torch.equal(got[:M], (xd @ wd.T).to(torch.bfloat16))
    assert (got[M] == 7.0).all()      # the row after the last stays untouched
