"""Products on the transfer ring against float64: row tiles, strip and row remainders,
fewer steps than the ring holds, column splits, both activations, rows apart; and which
products take it."""

import pytest
import torch

from opsagent_amd import ops

# M, N, K, rows of a tile, splits
FORMS = [
    (2, 8, 64, 32, 1), (32, 128, 192, 32, 2), (17, 264, 320, 32, 5),
    (33, 136, 384, 64, 1), (64, 256, 448, 64, 7), (65, 72, 640, 64, 3), (127, 384, 1024, 64, 16),
    (66, 200, 256, 96, 2), (96, 128, 1088, 96, 1), (97, 392, 512, 128, 1), (128, 1000, 4096, 128, 5),
    (200, 128, 256, 64, 2), (47, 4096, 1024, 64, 4),
]


def _whole(rows, cols, scale=1.0):
    """Whole numbers up to 2 times a power of two: every product and sum is exact."""
    return (torch.randint(-2, 3, (rows, cols), device="cuda") * scale).to(torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,tile,splits", FORMS)
def test_plain(M, N, K, tile, splits):
    torch.manual_seed(M + N + K)
    wide = _whole(M, K + 8)
    w = _whole(N, K)
    for x in (wide[:, :K].contiguous(), wide[:, :K]):      # rows apart as well
        got = ops._ring(x, w, (tile, splits))
        assert torch.equal(got, (x.double() @ w.double().T).to(torch.bfloat16))


@pytest.mark.gpu
@pytest.mark.parametrize("act", [1, 2])
@pytest.mark.parametrize("M,N,K,tile,splits", FORMS)
def test_gateup(M, N, K, tile, splits, act):
    torch.manual_seed(M + N + K)
    x, w = _whole(M, K), _whole(2 * N, K, 2.0 ** -5)
    got = ops._ring(x, w, (tile, splits), act).double()
    g, u = (x.double() @ w.double().T).split(N, 1)
    f = torch.nn.functional.silu(g) if act == 1 else torch.nn.functional.gelu(g, approximate="tanh")
    # one rounding to bf16, and some float32 roundings (exp of up to |g| / ln 2 scaled
    # bits, 1 + tanh near -1) of the exact halves
    bound = 2.0 ** -8 * (f * u).abs() + 2.0 ** -20 * (1 + g.abs()) * (g * u).abs()
    assert ((got - f * u).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [
    (9, 8, 128), (17, 132, 256), (33, 264, 1024), (64, 128, 1536), (65, 2048, 2816),
    (128, 1000, 640), (129, 256, 2048), (200, 4096, 4096), (300, 520, 1152),
])
def test_fp8(M, N, K):
    """Whole numbers and scales that are powers of two: exact sums, one rounding."""
    torch.manual_seed(M + N + K)

    def operand(rows):
        v = torch.randint(-2, 3, (rows, K), device="cuda").float().to(torch.float8_e4m3fn)
        return v.view(torch.uint8), torch.exp2(torch.randint(-3, 4, (rows,), device="cuda").float())

    (xq, xs), (wq, ws) = operand(M), operand(N)
    assert ops._ring_plan_fp8(M, N, K) is not None
    got = ops._gemm_fp8(xq, xs, wq, ws)
    xd = xq.view(torch.float8_e4m3fn).double() * xs.double()[:, None]
    wd = wq.view(torch.float8_e4m3fn).double() * ws.double()[:, None]
    assert torch.equal(got, (xd @ wd.T).to(torch.bfloat16))


def test_fp8_plans():
    for M in list(range(1, 140)) + [256, 257, 384, 700, 2048]:
        for N in (4, 1024, 4096, 6144, 14336, 28672):
            for K in (128, 2048, 4096, 14336):
                plan = ops._ring_plan_fp8(M, N, K)
                if plan:
                    tile, splits = plan
                    assert tile in (32, 64, 96, 128) and (M <= tile or tile == 128)
                    assert 1 <= splits <= K // 128 and splits * M * N * 4 <= 64 << 20
    assert ops._ring_plan_fp8(128, 4096, 14336) == (128, 8)
    assert ops._ring_plan_fp8(512, 4096, 14336) == (128, 2)
    assert ops._ring_plan_fp8(513, 4096, 14336) is None
    assert ops._ring_plan_fp8(129, 28672, 4096) is None
    assert ops._ring_plan_fp8(77, 6, 4096) is None


def test_plans_stay_in_range():
    """Tiles cover the rows, splits have steps of their own, parts stay small."""
    for gateup in (False, True):
        for K in (256, 512, 2048, 4096, 7168, 14336, 28672):
            for N in (8, 1024, 2048, 4096, 6144, 8192, 12288, 14336, 32000, 128256):
                for M in range(1, 130):
                    plan = ops._ring_plan(M, N, K, gateup)
                    if plan is None:
                        continue
                    tile, splits = plan
                    assert 1 < M <= 128 and tile in (32, 64, 96, 128)
                    assert 1 <= splits <= K // 64
                    assert -(-M // tile) == 1 or tile == 64
                    if splits > 1:
                        assert splits * M * N * (2 if gateup else 1) * 4 <= 64 << 20


def test_plans_at_the_lines():
    assert ops._ring_plan(1, 4096, 14336) is None
    assert ops._ring_plan(8, 4096, 14336) == (32, 8)
    assert ops._ring_plan(2, 4096, 14336) is None
    assert ops._ring_plan(2, 6144, 4096) is None and ops._skinny_form(2, 6144, 4096) == 0
    assert ops._ring_plan(3, 6144, 4096) == (32, 5) and ops._skinny_form(2, 4096, 14336) == 1
    assert ops._ring_plan(47, 14336, 4096, True) == (64, 1)
    assert ops._ring_plan(128, 14336, 4096, True) is None
    assert ops._ring_plan(8, 14336, 4096, True) is None
    assert ops._ring_plan(96, 4096, 4096) == (64, 4)
    assert ops._ring_plan(8, 4096, 4096) is None
    assert ops._ring_plan(32, 12288, 4096) is None
    assert ops._ring_plan(129, 4096, 14336) is None


def test_lines_between_the_forms():
    """Shapes on both sides of the lines at _ring_plan and _skinny_form, among them those
    where a form would be slower than the one it replaced."""
    def forms(M, N, K, gateup=False):
        return ops._ring_plan(M, N, K, gateup), ops._skinny_form(M, N, K, gateup)

    # runs of a multiple of 4 KiB: twice the splits, or the library
    assert ops._ring_plan(8, 16384, 4096) == (32, 4) and ops._ring_plan(8, 8192, 8192) == (32, 8)
    assert ops._ring_plan(64, 8192, 8192) is None and ops._ring_plan(128, 8192, 8192) == (128, 4)
    assert ops._ring_plan(64, 4096, 16384) == (64, 8)
    assert ops._ring_plan(24, 4096, 8192, True) is None and forms(8, 4096, 8192, True) == (None, 1)
    # short wide weights and many rows
    assert ops._ring_plan(48, 8192, 2048) is None and ops._ring_plan(48, 8192, 3072) == (64, 4)
    assert ops._ring_plan(80, 8192, 3072) is None and ops._ring_plan(80, 16384, 1024) == (64, 1)
    assert ops._ring_plan(96, 32000, 1024) == (96, 1) and ops._ring_plan(112, 32000, 1024) is None
    assert ops._ring_plan(96, 128256, 2048) is None and ops._ring_plan(96, 128256, 4096) == (96, 1)
    assert ops._ring_plan(80, 5120, 5120) == (96, 6) and ops._ring_plan(112, 5120, 5120) == (64, 3)
    assert ops._ring_plan(80, 2816, 2048, True) == (96, 5)
    assert ops._ring_plan(112, 2816, 2048, True) is None
    # few strips or long ones: the library; short rows in many rounds: the staged GEMV
    assert forms(3, 5120, 13824) == (None, 0) and forms(2, 5120, 13824) == (None, 0)
    assert forms(32, 1024, 4096) == (None, 0) and forms(16, 2048, 5632) == (None, 0)
    assert forms(28, 1024, 2816) == (None, 1) and forms(32, 1024, 2816) == (None, 0)
    assert forms(32, 1024, 4096, True) == (None, 0) and forms(4, 1024, 4096, True) == (None, 1)
    assert forms(8, 32000, 1024) == (None, 0) and ops._bf16_mfma_ok(8, 1024)
    assert forms(9, 16384, 1024) == (None, 0) and forms(9, 8192, 1024) == (None, 1)
    # three to eight rows that found no form
    assert forms(8, 12288, 6144) == forms(8, 18432, 5120) == (None, 1)
    assert forms(7, 128256, 2048) == (None, 1)
    assert forms(8, 18432, 7168, True) == (None, 0)
    for N, K, gateup in ((512, 1024, True), (18432, 5120, False), (256, 2048, False)):
        assert forms(2, N, K, gateup) == (None, 0)
    # two rows of few columns, and two that lie apart
    assert forms(2, 2048, 128) == forms(2, 4112, 256) == forms(2, 1024, 256, True) == (None, 1)
    assert forms(2, 2048, 512) == (None, 1) and forms(2, 2064, 512) == (None, 0)
    assert forms(2, 512, 512, True) == forms(2, 1024, 1024) == (None, 0)
    assert [ops._skinny_form(2, N, K, strided=True) for N, K in
            ((2048, 128), (2064, 512), (4096, 4096), (8192, 4096), (512, 480))] == [1, 1, 1, 1, 0]
    # strips of short rows in several rounds
    assert forms(8, 14336, 128) == forms(31, 16384, 128) == forms(17, 32000, 512) == (None, 1)
    assert forms(32, 16384, 128) == forms(8, 32000, 64) == forms(8, 65536, 256) == (None, 0)
    assert forms(5, 8192, 1408) == forms(24, 14336, 768) == (None, 1)
    assert forms(16, 14336, 768) == forms(24, 16384, 768) == forms(5, 8208, 1408) == (None, 0)
    assert [ops._skinny_form(8, 8192, 1024, strided=far) for far in (False, True)] == [0, 1]
    # two tiles of 64 rows on light gate-up weights
    assert ops._ring_plan(128, 8192, 640, True) == (64, 1)
    assert ops._ring_plan(128, 4096, 1408, True) == (64, 2)
    assert ops._skinny_form(8, 8192, 4096, strided=True) == 2


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(3, 16384, 1024), (8, 16400, 1024), (8, 8192, 8192),
                                   (32, 4096, 16384), (8, 18432, 5120), (64, 4096, 16384)])
def test_lines_agree(M, N, K):
    gen = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K, generator=gen, device="cuda").bfloat16()
    w = (torch.randn(N, K, generator=gen, device="cuda") * K ** -0.5).bfloat16()
    want = x.double() @ w.double().T
    # one bf16 rounding of a float32 sum: 0.0016 in the mean
    assert float((ops.linear(x, w).double() - want).norm() / want.norm()) < 2e-3


NARROW = [(3, 8, 64, 32, 1), (32, 200, 320, 32, 2), (33, 72, 448, 64, 3), (64, 264, 1024, 64, 1),
          (17, 64, 4096, 32, 8), (48, 1000, 256, 64, 4)]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,tile,splits", NARROW)
def test_narrow_strips(M, N, K, tile, splits):
    """Strips of 64 weight rows, two blocks a CU: fewer steps than the ring holds, runs that
    differ by a step, strips and tiles part filled, rows of x that lie apart."""
    torch.manual_seed(M + N + K)
    wide, w = _whole(M, K + 8), _whole(N, K)
    for x in (wide[:, :K].contiguous(), wide[:, :K]):
        got = ops._ring(x, w, (tile, splits, True))
        assert torch.equal(got, (x.double() @ w.double().T).to(torch.bfloat16))
    x, w = _whole(M, K), _whole(2 * N, K, 2.0 ** -5)
    g, u = (x.double() @ w.double().T).split(N, 1)
    for act in (1, 2):
        got = ops._ring(x, w, (tile, splits, True), act).double()
        f = torch.nn.functional.silu(g) if act == 1 else torch.nn.functional.gelu(g, approximate="tanh")
        # as in test_gateup
        bound = 2.0 ** -8 * (f * u).abs() + 2.0 ** -20 * (1 + g.abs()) * (g * u).abs()
        assert ((got - f * u).abs() <= bound).all()


def test_narrow_plans():
    choice = ops._ring_choice
    assert choice(8, 14336, 4096, True) == (32, 1, True) and choice(48, 14336, 4096, True) == (64, 1, True)
    assert choice(49, 14336, 4096, True) == (64, 1, False) and choice(2, 14336, 4096, True) is None
    assert choice(8, 11008, 4096, True) is None                # 344 blocks: a round two thirds full
    assert choice(24, 2048, 2048) is None                      # under 10 MB
    assert choice(24, 8192, 4096) == (32, 4, False)            # two splits of 2048 columns each
    assert choice(24, 4096, 4096) == (32, 4, True) and choice(8, 4096, 4096) is None
    assert choice(48, 2048, 8192) == (64, 8, True) and choice(49, 2048, 8192)[2] is False
    assert choice(64, 16384, 4096) == (64, 1, True)           # the library's otherwise
    assert choice(32, 8192, 28672)[2] is False and choice(8, 16384, 4096)[2] is False
    assert choice(8, 32000, 4096) == (32, 1, True) and choice(48, 32000, 4096) == (64, 1, True)
    assert choice(24, 8192, 2048, True)[2] is False and choice(24, 8192, 3072, True) == (32, 1, True)
    assert choice(24, 2560, 1024, True) is None and choice(40, 2560, 1024, True) == (64, 3, True)
    assert choice(24, 2816, 3520, True)[2] is False            # 176 blocks beside 220
    # as many rounds and nothing to add up; eight waves a block beside four
    assert choice(24, 28160, 5632)[2] is choice(48, 31056, 4224)[2] is choice(33, 7768, 6208)[2] is False
    assert choice(17, 3072, 2048) is None and choice(40, 3072, 2048) == (64, 5, True)
    assert choice(40, 2560, 2560) is None and choice(40, 2048, 3584) == (64, 8, True)
    for gateup in (False, True):
        for K in (64, 640, 1408, 2048, 4096, 14336):
            for N in (8, 1024, 3072, 6144, 32000, 128256):
                for M in range(1, 130):
                    plan = choice(M, N, K, gateup)
                    if plan and plan[2]:
                        assert 2 < M <= plan[0] <= 64 and 1 <= plan[1] <= K // 64


def test_choices_are_those_of_the_rules(monkeypatch):
    """Asked again, a size is answered as the rules answer it; two rows follow the GEMV switch."""
    for gateup in (False, True):
        for N, K in ((3072, 2048), (4096, 14336), (14336, 4096), (1408, 2048), (7, 64)):
            for M in (1, 2, 3, 16, 47, 64, 65, 128, 129):
                fresh = ops._ring_sizes.__wrapped__(M, N, K, gateup)
                assert ops._ring_choice(M, N, K, gateup) == ops._ring_choice(M, N, K, gateup) == fresh
    before = ops._ring_choice(2, 6144, 4096)
    monkeypatch.setenv("OPSAGENT_GEMV_MAX_M", "1")
    assert before is None and ops._ring_choice(2, 6144, 4096)[:2] == ops._ring_plan(2, 6144, 4096)
