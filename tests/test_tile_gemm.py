"""Tile products of more than 128 rows against float64: every form, row and strip remainders, fewer
steps than a ring holds, odd and even numbers of them, column splits, both activations, rows
apart; and which products take them."""

import pytest
import torch

from opsagent_amd import ops

FORMS = range(10)
FORMS8 = range(5)
# M, N, K, splits
SIZES = [(129, 8, 64, 1), (256, 520, 128, 1), (300, 136, 192, 1), (161, 264, 448, 3),
         (513, 392, 512, 2), (700, 1000, 1088, 1), (200, 1104, 1984, 1)]


def _whole(rows, cols, scale=1.0):
    """Whole numbers up to 2 times a power of two: every product and sum is exact."""
    return (torch.randint(-2, 3, (rows, cols), device="cuda") * scale).to(torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,splits", SIZES)
@pytest.mark.parametrize("form", FORMS)
def test_plain(form, M, N, K, splits):
    torch.manual_seed(M + N + K)
    wide, w = _whole(M, K + 8), _whole(N, K)
    for x in (wide[:, :K].contiguous(), wide[:, :K]):      # rows apart as well
        want = x.double() @ w.double().T
        assert torch.equal(ops._tile(x, w, form * 256 + splits), want.to(torch.bfloat16))
        if splits > 1:
            parts = ops._tile(x, w, form * 256 + splits, parts=True)
            assert parts.shape == (splits, M, N) and torch.equal(parts.double().sum(0), want)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,splits", SIZES)
@pytest.mark.parametrize("form", FORMS)
def test_gateup(form, M, N, K, splits):
    torch.manual_seed(M + N + K)
    x, w = _whole(M, K), _whole(2 * N, K, 2.0 ** -5)
    g, u = (x.double() @ w.double().T).split(N, 1)
    for act in (1, 2):
        got = ops._tile(x, w, form * 256 + 1, act).double()
        f = torch.nn.functional.silu(g) if act == 1 else torch.nn.functional.gelu(g, approximate="tanh")
        # one rounding to bf16, and some float32 roundings (exp of up to |g| / ln 2 scaled
        # bits, 1 + tanh near -1) of the exact halves
        bound = 2.0 ** -8 * (f * u).abs() + 2.0 ** -20 * (1 + g.abs()) * (g * u).abs()
        assert ((got - f * u).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,splits", SIZES)
@pytest.mark.parametrize("form", FORMS8)
def test_fp8(form, M, N, K, splits):
    """Bit for bit what the one-barrier tiles answer, on rows whose sums round."""
    torch.manual_seed(M + N + K)
    K *= 2
    x, w = (torch.randn(rows, K, device="cuda") * torch.randn(rows, K, device="cuda").exp()
            for rows in (M, N))
    (a, sa), (b, sb) = ops.quant_fp8(x.bfloat16()), ops.quant_fp8(w.bfloat16())
    lib, hip = ops._lib()
    got, want = (torch.empty(M, N, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    hip.check(lib.oa_tile_gemm_fp8(hip.current_stream_ptr(), a.data_ptr(), sa.data_ptr(), b.data_ptr(),
                                   sb.data_ptr(), got.data_ptr(), M, N, K, form), "oa_tile_gemm_fp8")
    hip.check(lib.oa_gemm_fp8(hip.current_stream_ptr(), a.data_ptr(), b.data_ptr(), sa.data_ptr(),
                              sb.data_ptr(), want.data_ptr(), M, N, K), "oa_gemm_fp8")
    assert torch.equal(got, want)

    def values(q, scale):
        return q.view(torch.float8_e4m3fn).double() * scale.double()[:, None]

    exact = values(a, sa) @ values(b, sb).T
    assert (got.double() - exact).norm() <= 2.0 ** -8 * exact.norm()     # one rounding to bf16
    if M > 128:
        assert torch.equal(ops._gemm_fp8(a, sa, b, sb), want) or ops._ring_choice_fp8(M, N, K)


@pytest.mark.gpu
def test_dispatch():
    """The public products take the tiles, parts reach the norm behind them, and the results are
    those of the library's product to the rounding of bf16."""
    torch.manual_seed(0)
    x = torch.randn(333, 8192, device="cuda").bfloat16()
    w = (torch.randn(2048, 8192, device="cuda") / 90).bfloat16()
    want = x.double() @ w.double().T
    assert ops._tile_choice(333, 2048, 8192) & 255 > 1
    parts = ops.linear_parts(x, w)
    assert isinstance(parts, ops.PlaneSum)
    for got in (ops.linear(x, w), ops._added_up(parts)):
        assert (got.double() - want).norm() <= 2.0 ** -8 * want.norm()
    grad = w.clone().requires_grad_()
    ops.linear(x, grad).sum().backward()                 # gradients go through the library
    assert grad.grad is not None


def test_whole_tiles_of_the_library():
    """Plain products in unsplit tiles of 256 x 256 are the library's, but for short rows."""
    plan = ops._lib()[0].oa_tile_gemm_plan
    for M, N, K, taken in ((2048, 8192, 4096, False), (1966, 16384, 2048, False), (1024, 14336, 4096, False),
                           (1430, 10296, 640, True)):
        assert plan(M, N, K, 0, 0) == 1 and (ops._tile_choice(M, N, K) is not None) == taken
    assert plan(2048, 4096, 14336, 0, 0) == 2 == ops._tile_choice(2048, 4096, 14336)      # split in two
    assert plan(3900, 8192, 2048, 1, 0) == 1 == ops._tile_choice(3900, 8192, 2048, gateup=True)


def test_light_weights():
    for N, K in ((2048, 2048), (2560, 2560), (3072, 2048), (2048, 2816)):
        assert ops._tile_choice(499, N, K) is None and ops._tile_choice(500, N, K) is not None
    assert ops._tile_choice(512, 2816, 2048, gateup=True) is not None
    assert ops._tile_choice(512, 2048, 8192) is not None


def test_idle_units():
    """Products in few unsplit tiles are the library's, out of 2048 to 8192 columns: plain ones of 160 x
    256 and 256 x 128; on whole steps of its columns those of 96 x 128, but for whole 32s of up to 256
    plain rows, and of heavy weights and more rows those of 128 x 64."""
    plan = ops._lib()[0].oa_tile_gemm_plan
    for M, N, K, form, tiles, taken in ((640, 12288, 4096, 3, 192, False), (514, 12288, 4096, 3, 192, False),
                                        (486, 12288, 4096, 4, 192, False), (517, 11072, 5760, 3, 176, False),
                                        (640, 13056, 4096, 3, 204, True), (514, 12288, 1984, 3, 192, True),
                                        (279, 17856, 12736, 3, 140, True), (283, 6144, 4096, 8, 144, False),
                                        (268, 6144, 3136, 8, 144, True), (283, 6656, 4096, 8, 156, True),
                                        (191, 9088, 4096, 8, 142, False), (192, 9088, 4096, 8, 142, True),
                                        (512, 2880, 4352, 9, 180, False), (382, 4032, 3328, 9, 189, False),
                                        (700, 2048, 2816, 9, 192, True), (250, 6144, 4096, 9, 192, True)):
        rows, cols = {3: (160, 256), 4: (256, 128), 8: (96, 128), 9: (128, 64)}[form]
        assert plan(M, N, K, 0, 0) == form * 256 + 1 and -(-M // rows) * -(-N // cols) == tiles
        assert (ops._tile_choice(M, N, K) is not None) == taken
    for M, N, K, form, tiles, taken in ((190, 5120, 5888, 8, 160, False), (192, 5120, 5888, 8, 160, False),
                                        (150, 4928, 3840, 8, 154, True), (209, 1024, 2048, 9, 64, True)):
        rows, cols = {8: (96, 128), 9: (128, 64)}[form]
        assert plan(M, N, K, 1, 0) == form * 256 + 1 and -(-M // rows) * -(-2 * N // cols) == tiles
        assert (ops._tile_choice(M, N, K, gateup=True) is not None) == taken
    assert ops._tile_choice(514, 6144, 4096, gateup=True) is not None


def test_rounds_of_the_library():
    """Large gate-up products: the library's where its tiles of 256 x 256 fill every round."""
    for M, N, K, blocks, taken in ((8192, 14336, 4096, 14 * 256, False), (8193, 14336, 4096, 3696, True),
                                   (7937, 14336, 4096, 14 * 256, False), (10319, 14336, 4096, 18 * 256 - 16, True),
                                   (12288, 14336, 4096, 21 * 256, False), (13195, 13824, 5120, 22 * 256 - 16, True),
                                   (14976, 13824, 5120, 25 * 256 - 28, True)):
        assert -(-M // 256) * (2 * N // 256) == blocks
        assert (ops._tile_choice(M, N, K, gateup=True) is not None) == taken


@pytest.mark.gpu
def test_rows_far_apart():
    """One token of each of many long sequences, 8 MB apart and a step less."""
    g = torch.Generator(device="cuda").manual_seed(1)
    w = (torch.randn(4096, 4096, generator=g, device="cuda") / 64).bfloat16()
    rows = torch.randn(160, 4096, generator=g, device="cuda").bfloat16()
    want = rows.double() @ w.double().T
    for step in (2 ** 22 - 8, 2 ** 22, 2 ** 22 + 8):
        x = torch.empty(160 * step, dtype=torch.bfloat16, device="cuda").view(160, step)[:, :4096]
        x.copy_(rows)
        parts = ops.linear_parts(x, w)
        for got in (ops.linear(x, w), ops._added_up(parts) if isinstance(parts, ops.PlaneSum) else parts):
            assert (got.double() - want).norm() <= 2.0 ** -8 * want.norm()     # one rounding


def test_plan_within_reach():
    """A plan is a product that the launch takes: what its 32-bit places do not span has none."""
    plan = ops._lib()[0].oa_tile_gemm_plan
    for M in (129, 4000):
        for N, K in ((2 ** 21, 1024), (2 ** 21 - 256, 1024), (2 ** 21 - 264, 1024), (2 ** 18, 8192),
                     (512, 2 ** 22), (512, 2 ** 22 - 64), (8, 2 ** 23), (2 ** 20, 2048)):
            for gateup in (0, 1):
                within = K < 2 ** 22 and (gateup * N + 256) * K * 2 < 2 ** 32
                assert within or plan(M, N, K, gateup, 0) == -1, (M, N, K, gateup)
                assert not within or gateup or plan(M, N, K, 0, 0) >= 0
    assert ops._tile_choice(1000, 2 ** 21, 1024, gateup=True) is None
    for step in (64, 2 ** 22 - 8, 2 ** 22):
        x = torch.empty_strided((200, 64), (step, 1), dtype=torch.bfloat16, device="meta")
        assert ops._near_rows(x) == (step < 2 ** 22)


def test_plan():
    """Sizes that no form takes, and what the rule answers for those it takes: a form of the table,
    splits that leave every block eight steps and no more blocks than CUs."""
    plan = ops._lib()[0].oa_tile_gemm_plan
    for args in ((0, 64, 512), (200, 12, 512), (200, 64, 448), (200, 64, 520)):
        assert plan(*args, 0, 0) == -1
    tiles = [(256, 256), (224, 256), (192, 256), (160, 256), (256, 128), (224, 128), (160, 128),
             (128, 128), (96, 128), (128, 64)]
    for M in (129, 200, 333, 800, 2048, 8192):
        for N, K in ((2048, 2048), (4096, 14336), (12288, 4096), (128256, 4096), (264, 576)):
            for gateup in (0, 1):
                for summed in (0, 1):
                    answer = plan(M, N, K, gateup, summed)
                    if answer < 0:
                        assert gateup                    # left to splits and the activation kernel
                        continue
                    form, splits = divmod(answer, 256)
                    bm, bn = tiles[form]
                    blocks = -(-M // bm) * -(-N * (1 + gateup) // bn) * splits
                    assert splits == 1 or (not gateup and blocks <= 256 and K // 64 // splits >= 8)
                if K % 128 == 0:
                    assert ops._tile_form_fp8(M, N, K) in (-1, *FORMS8)
    for args in ((0, 64, 512), (200, 12, 512), (200, 64, 384), (200, 64, 576)):
        assert ops._tile_form_fp8(*args) == -1
    assert ops._tile_choice(128, 4096, 14336) is None    # the ring's
    assert ops._tile_choice(200, 2048, 2048) is None     # light weights, few rows: the library
    for args, taken in (((8192, 14336, 4096), False), ((7500, 14336, 4096), True),
                        ((9200, 14336, 4096), True), ((4000, 14336, 4096), True), ((8192, 2816, 2048), True),
                        ((8192, 4096, 14336), False), ((5500, 4096, 14336), True), ((8000, 3584, 8192), True)):
        assert (ops._tile_choice(*args, gateup=True) is not None) == taken
