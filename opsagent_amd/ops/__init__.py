"""Op dispatch layer.

GPU (ROCm) path → hand-written HIP/CDNA4 kernels from the in-tree library
(fails LOUDLY if the library is missing — no silent eager fallback on a GPU
box, per the build contract). CPU path → opsagent_amd.ops.torch_ref (also the
numerics oracle for the GPU parity tests).

GEMM-shaped work (QKV/O/MLP projections, lm_head) takes the kernels of its number of rows
(linear, gateup_silu); what they do not take, and every call under gradients, goes through
torch.nn.functional.linear → hipBLASLt/rocBLAS. The fused hot ops (norms, RoPE,
attention, activation, sampling) are the HIP kernels here.
"""

from __future__ import annotations

import functools
import os
from typing import NamedTuple, Optional, Tuple, Union

import torch
from torch.autograd import forward_ad

from opsagent_amd.ops import torch_ref

__all__ = [
    "rms_norm",
    "fused_add_rms_norm",
    "rope_apply_",
    "silu_mul",
    "kv_cache_write",
    "attention_prefill",
    "attention_decode_paged",
    "greedy_sample_masked",
    "rope_cos_sin",
]

rope_cos_sin = torch_ref.rope_cos_sin

# VALU-gemv M instantiations (the dot-per-lane form; measured crossover
# notes below). More rows go to the matrix-core forms (linear).
_GEMV_MS = frozenset(range(1, 9))

# Measured crossover vs hipBLASLt (concurrent bench, within-box A/B):
#   M=1: custom ~2.5x faster        M=2: custom +19% (c=2 3.42 vs 2.88 t/s)
#   M=4: tie (5.20 vs 5.28)         M=8: custom ~2x SLOWER (c=8 4.6 vs 9.2)
# The per-lane-dot form goes VALU-bound as M grows; hipBLASLt's MFMA kernels
# take over. Default cap 2; OPSAGENT_GEMV_MAX_M overrides for experiments.


# The mapping under os.environ, which changes with it: a lookup in it takes 0.05 us, one
# through os.environ, where a variable is not set, 0.6 (it raises inside), and a product
# of a short prompt makes several.
_ENV = os.environ._data


def _bf16_mfma_ok(M: int, K: int, gateup: bool = False) -> bool:
    """Mirror of gemv.hip's gemv_bf16_use_mfma: the staged MFMA kernel (M 3..8 unless
    OPSAGENT_BF16_GEMV_MFMA asks for others)."""
    e = _ENV.get(b"OPSAGENT_BF16_GEMV_MFMA", b"")
    if e == b"0":
        return False
    min_m = int(e[1:]) if e.startswith(b"m") else 3
    if M < min_m or M > 16:
        return False
    if K % (512 if gateup else 1024) != 0:
        return False
    if not e.startswith(b"m"):
        # measured win region only (see gemv.hip's gemv_bf16_use_mfma)
        if K > 6144 or M > 8:
            return False
    return M * (K * 2 + 16) <= 147456


def _gemv_m_ok(M: int) -> bool:
    cap = int(_ENV.get(b"OPSAGENT_GEMV_MAX_M", 2))
    return M in _GEMV_MS and M <= cap


def _gemv_switched() -> bool:
    """OPSAGENT_BF16_GEMV_MFMA or OPSAGENT_GEMV_MAX_M is set: the two choose between the
    staged GEMVs and the library, and the newer forms step aside for both."""
    return b"OPSAGENT_BF16_GEMV_MFMA" in _ENV or b"OPSAGENT_GEMV_MAX_M" in _ENV


def _two_rows_valu(M: int, N: int, K: int, gateup: bool = False) -> bool:
    """Two rows that the VALU GEMV takes better than the matrix-core forms (us, VALU /
    best of those, 2 GB of weights in turn: gate-up 2 x 14336 x 4096 41.1 / 45.3, 6144 x
    4096 10.7 / 12.7, 5120 x 5120 10.7 / 13.5, 32000 x 2048 25.1 / 26.0, 4096 x 4096 8.5 /
    8.2, 14336 x 384 5.0 / 5.6), long rows (4096 x 14336 26.6 / 23.0), short ones (2048 x 128
    2.7 / 2.1, 14336 x 256 4.6 / 4.5; gate-up 2 x 2048 x 128 3.1 / 2.4, 2 x 512 x 512 2.9 /
    3.2) and few of them (1024 x 640 3.2 / 2.8, 1024 x 1024 3.2 / 3.8) apart."""
    if M != 2 or K > 8192 or K <= 256 or (not gateup and K < 1024 and N * K <= 2 ** 20):
        return False
    return _gemv_m_ok(M)


def _skinny_form(M: int, N: int, K: int, gateup: bool = False, strided: bool = False) -> int:
    """Which form of the skinny product (skinny.hip; figures there) takes M rows
    of K columns against N (gate-up: 2N) weight rows: 0 none, 1 strips, 2
    persistent.

    Strips: a block of 16 weight rows (gate-up: 32) takes a time of its own per column
    and row of x, blocks of one CU add up, and past 4.75 TB/s memory bounds all of them;
    measured over 64 weights this holds to a tenth. The library's best times over the same
    weights are 5 us + its bytes at 5.9 TB/s (gate-up with its activation 7.3 and 5.4), and
    no less than `least` (another of its kernels takes over at 32 rows). Strips take what
    they finish sooner: 4096 x 4096, M = 16 10.6 against 15.5 and 32 15.2 against 13.3;
    1024 x 2816, 28 10.3 / 10.9 and 32 10.9 / 9.3; 5120 x 13824, 3 39.1 / 28.4. Up to eight rows the staged
    GEMV is the other form where it runs, and strips are the faster one (12288 x 6144, 8
    35.0 / 41.2), except for rows too short to pipeline, four steps a wave, in more than
    one round (32000 x 1024, 8 19.9 / 16.0; the library 17.2). Against the library strips
    of rows under 2048 columns pay in two rounds (8192 x 1408, 5 8.3 / 10.1), in more of
    them with up to 512 columns (14336 x 128, 8 3.5 / 5.0, 31 4.3 / 4.4; 32000 x 512, 17
    14.5 / 17.9; but 32000 x 64, 8 4.8 / 4.6, 65536 x 256, 8 14.1 / 10.4), and with up to 768
    from 17 rows on (14336 x 768, 16 10.1 / 8.4, 24 11.9 / 17.4; 16384 x 768, 24 12.3 / 10.7).
    The persistent form is for blocks that go over several strips: gate-up from N = 8192
    on (2 x 11008, 8 36.2 / 38.4; 2 x 3584 16.5 / 13.8) and N >= 6144 up to 16 rows, N >= 16384 up to 32. Under 2^18
    weights the library stays for its order of sums, not for its speed: a pair of equal
    choices in a small routed model falls the other way with strips, which take 2.5 us
    against 4.3 (480 x 512, 3 rows; 512 x 512 2.5 / 4.3, 64 x 2048, 32 rows 7.1 / 7.9).
    strided: rows of x that lie apart, which the VALU GEMV does not take. Two of them go to
    strips (us, strips / library: 2048 x 128 2.1 / 3.4, 2048 x 2048 4.8 / 10.9, 8192 x 4096
    14.1 / 16.9; the persistent form 18.4, the ring 14.0)."""
    R = 2 if gateup else 1
    two = M == 2 and strided
    if M < 1 or M > 32 or K % 32 != 0 or R * N * K < 2 ** 18 or (
            not two and _two_rows_valu(M, N, K, gateup)):
        return 0
    if K == 4096 and not two and (M <= 16 and N >= 8192 if gateup else N >= (6144 if M <= 16 else 16384)):
        return 2
    blocks = -(-N // 16)
    staged = M > 2 and _bf16_mfma_ok(M, K, gateup)
    if K < 2048 and not gateup and blocks > 256:
        if K <= 512:
            rounds = (4 if K < 256 else 8) if M < 32 else 3.5 if K <= 128 else 2
        else:
            rounds = 2 if M <= 16 or K > 768 else 3.5
        if (staged and not strided) or blocks > 256 * rounds:
            return 0
        if K <= 512:
            return 1
    if staged:
        return 1
    if M <= 16:
        col = (2.5 + 0.06 * M) if gateup else (1.3 + 0.05 * M)
    else:
        col = (2.9 + 0.06 * M) if gateup else (1.6 + 0.045 * M)
    mb = R * N * K * 2e-6
    strips = max(1.8 + -(-blocks // 256) * K / 1024 * col, mb / (5.0 if M > 2 else 4.75))
    if gateup:
        library = max(17.6 if K >= 4096 and M <= 24 else 13.5, 7.3 + mb / 5.4)
    else:
        least = 10.4 if M <= 16 else 8.4 if M == 32 else 12.6 if K >= 4096 else 10.2
        library = max(least, 5 + mb / 5.9)
    return int(strips < library)


_PLAIN = (torch.Tensor, torch.nn.Parameter)
_compiling = torch.compiler.is_compiling
_traced = torch._C._get_tracing_state
_transform = torch._C._functorch.maybe_current_level
_modes = torch._C._len_torch_dispatch_stack


def _plain_call(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Nobody asks for gradients or tangents, traces or transforms the call: a kernel sees
    addresses alone, the library's product is an operation that all of these know."""
    return not (
        _compiling() or _traced() is not None or _transform() is not None
        or _modes() or forward_ad._current_level >= 0
        or ((x.requires_grad or w.requires_grad) and torch.is_grad_enabled())
    ) and type(x) in _PLAIN and type(w) in _PLAIN


def _skinny_ok(x: torch.Tensor, w: torch.Tensor) -> bool:
    """16-byte loads of the rows of both operands, on one device, a call that nothing
    records, and no switch that asks for other forms."""
    return (
        _plain_call(x, w) and x.is_cuda and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16
        and w.device == x.device and w.dim() == 2 and w.is_contiguous() and x.dim() >= 1 and x.shape[-1] == w.shape[1]
        and (x.is_contiguous() or (x.dim() == 2 and x.stride(1) == 1
                                   and x.stride(0) >= x.shape[1] and x.stride(0) % 8 == 0))
        and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0 and not _gemv_switched()
    )


def _skinny(x: torch.Tensor, w: torch.Tensor, form: int, gateup: bool = False,
            act: int = 0) -> torch.Tensor:
    lib, hip = _lib()
    K = x.shape[-1]
    M, N = x.numel() // K, w.shape[0] // (2 if gateup else 1)
    out = torch.empty(*x.shape[:-1], N, dtype=x.dtype, device=x.device)
    hip.check(lib.oa_skinny(hip.current_stream_ptr(), x.data_ptr(),
                            K if x.is_contiguous() else x.stride(0), w.data_ptr(), out.data_ptr(),
                            M, N, K, int(gateup), act, form), "oa_skinny")
    return out


def _ring_plan(M: int, N: int, K: int, gateup: bool = False) -> Optional[Tuple[int, int]]:
    """(rows of a tile, column splits) of the product on the transfer ring
    (ring_gemm.hip; figures there) in strips of 128 weight rows, of M rows of K columns against
    N (gate-up: 2N) weight rows, None where these lines leave it to the other forms.

    The lines were drawn at 2 to 128 rows over 64 weights, 2 GB of them in turn, when all strips
    started together; _ring_form looks past them where strips apart are faster by its estimate.
    What they go by, with today's us, best other form / this one: light weights end before the ring
    pays for its start (4096 x 4096, M = 8 9.2 / 11.0, 24 13.3 / 12.1; gate-up 2 x 2816 x 2048, 24
    10.7 / 11.3, 47 15.5 / 13.7, 112 17.0 / 16.2; but where two tiles of 64 rows fill the CUs 2 x
    8192 x 640, 128 14.7 / 10.0, 2 x 4096 x 1408 19.1 / 14.0), short rows at few rows too (2 x
    8192 x 2048, 8 15.4 / 15.9; 2 x 8192 x 3072 24.3 / 21.3), long ones less (2048 x 8192, 8 12.9 /
    11.9). Column splits fill the CUs; unsplit, a round filled to less than 0.8 loses (12288 x 4096,
    24 23.4 / 29.4, in two 21.9), and at two or three rows adding up many splits does (4096 x
    14336, 2 23.2 / 23.8). Runs of a multiple of 2048 columns, 4 KiB, kept all blocks on the same
    channels: twice as many splits mended it up to 32 rows, and above and for gate-up the library
    was faster on weights of no fewer rows than columns. Apart that matters less (16384 x 4096, M = 8
    30.3 / 26.9 in two splits, 28.2 in four; 8192 x 8192 30.7 / 30.2 in four, 27.3 in eight, 64 32.9 /
    31.5, 128 48.3 / 37.2; 2 x 4096 x 8192, 8 30.0 / 29.2; 4096 x 16384, 64 42.2 / 35.0), and so do many
    rows on short wide weights that need splits (8192 x 2048, 48 14.9 / 13.5; 8192 x 3072, 48 18.3 /
    16.1, 80 19.3 / 18.6).
    Up to 16 rows of 4096 the persistent skinny form was the better one where no split is needed
    (2 x 14336, 8 47.5 / 39.9 now), under eight shorter rows the strips (32000 x 2048, 4 27.2 / 23.6
    now). Two tiles of 64 rows beat a tile of 128 under 64 MB of weights and one of 96 under 32 MB
    (us, one / two: 2048 x 8192, 80 16.9 / 16.5, 128 19.2 / 16.7; 2 x 3584 x 4096, 80 21.9 / 22.7), as
    long as both read a strip in the same round (32000 x 1024, 112 18.1 / 24.5). Without splits
    tiles of 96 pay in one round or from rows of 4096 on (128256 x 2048, 96 129 / 128, 32000 x 2048
    35.0 / 27.9, 128256 x 4096 233 / 224); tiles of 128 did not (2 x 14336 x 4096, 62.7 / 53.6 now)."""
    if not 1 < M <= 128 or K % 64 or K < 256 or N % 8 or _two_rows_valu(M, N, K, gateup):
        return None
    weights = (2 if gateup else 1) * N * K
    if M <= 16:
        ok = weights >= (2 ** 24 if K >= 8192 else 24e6 if K >= 4096 else 40e6 if K >= 3072 else 60e6)
    else:
        ok = weights >= (10e6 if gateup and M > 32 else 2 ** 24)
    if not ok:
        return None
    strips = -(-N // (64 if gateup else 128))
    one = 32 * -(-M // 32)
    two = M > 64 and weights < (2 ** 25 if M > 96 else 2 ** 24 + 1)
    if gateup and M > 80 and weights < 2 ** 24:
        one = 64
    for tile in (64, one) if two else (one,):
        tiles = strips * -(-M // tile)
        splits = max(1, min(256 // tiles, K // 256))
        blocks = tiles * splits
        if blocks < 0.8 * 256 * -(-blocks // 256):
            continue
        if splits == 1:
            if tile == 128 or M <= 16 and K == 4096 or M < 8 and K < 4096:
                continue
            if blocks > 256 and M > 64 and (K < 4096 or tile == 64):
                continue
        else:
            if not gateup and (M > 64 and 2 * K < N or M > 40 and 3 * K < N):
                continue
            if K % (splits * 2048) == 0:
                if M <= 32 and not gateup:
                    splits *= 2
                elif weights >= K * K and M < (113 if gateup else 96):
                    continue
            if M < 4 and splits > 5:
                continue
        return tile, splits
    return None


def _ring_narrow(M: int, N: int, K: int, gateup: bool, wide) -> Optional[int]:
    """Column splits of the ring product in strips of 64 weight rows, two blocks a CU
    (ring_gemm.hip), None where strips of 128 (wide: their plan) or the other forms stay.

    What decides is, in this order, how full the CUs are, how many columns a split has, and what
    the other form is. Drawn from 190 weights, 150 of them random, at 3 to 64 rows, 0.7 GB of them in
    turn, when all strips started together; today's us, other / narrow:

    One round of half the blocks (12288 x 4096, M = 8 22.1 / 21.5 with 192), or rounds of 512
    (gate-up 2 x 14336 x 4096, 8 39.9 / 40.7 with 448; 2 x 11008, 8 32.4 / 38.3 with 344), and
    against strips of 128 that fill them better no fewer (2 x 2816 x 3520, 24 13.6 / 13.6 with
    176). Weights under 10 MB end before it starts (2048 x 2048, 24 7.5 / 7.3); wide weights of
    many splits run as fast in one deep ring (8192 x 28672, 32 79.4 / 78.6).

    Against strips of 128 in as many rounds it halves the splits or has none to add up: short
    ones gain most (4096 x 4096, 24 12.1 / 10.6; 2 x 7704 x 1216, 24 .73 of the time). Above 32
    rows eight waves a block carry those strips, and only splits of up to 1700 columns are better
    here (4096 x 4096, 48 13.8 / 12.3; 4096 x 14336, 33 1.04 of the time; 7768 x 6208 1.08). Where
    neither form splits it has nothing to save (28160 x 5632, 24 1.11, 48 1.17); strips of 128 that
    started together on rows of 4 KiB were the slower ones, which _ring_form knows they are no
    longer (32000 x 4096, 24 41.7 / 41.8, 48 41.8 / 45.3; 2 x 14336 x 4096, 32 38.3 / 40.2). Splits of
    such a size started together too (8192 x 4096, 24 15.4 / 14.3 in two, 15.0 in four; 4096 x 8192
    17.3 / 16.8).

    Strips of skinny.hip are the faster form of short rows: up to 16 rows (4096 x 4096, 8 9.2 /
    10.1; but 32000 x 2048, 6 27.0 / 22.7 now), up to 32 where columns of gate-up would be split (2 x
    2560 x 1024, 24 1.14 of the time; 2 x 3072 x 1536 1.01) or rows of 4 KiB are cut to a few hundred
    columns (3072 x 2048, 17 1.10, 24 1.06, 32 .93)."""
    if not 2 < M <= (64 if wide is None else 48) or K % 64 or N % 8:
        return None
    weights = (2 if gateup else 1) * N * K
    strips = -(-N // (32 if gateup else 64))
    splits = max(1, min(256 // strips, K // 256))
    blocks, many = strips * splits, M > 32
    if blocks > 256:
        full = 0.84 * 512 * -(-blocks // 512)
    else:
        full = 256 * (0.85 if splits > 1 and not gateup else 0.8 if wide and not many else 0.68)
    if blocks < full or weights < 5e6 or K >= 8192 and N >= 8192:
        return None
    if wide and (K % 2048 if wide[1] == 1 else many and K // splits > 1700):
        return None
    if gateup:
        if splits == 1 and K >= 3072 and weights >= 45e6:
            ok = M <= (48 if K < 8192 else 32)       # 2 x 6144 x 12288, 40 1.16 of the time
        elif M <= 16:
            ok = wide is None and K >= 4096 and weights < 24e6
        else:
            ok = (wide is None or weights < 24e6) and (many or splits == 1 or K >= 2048)
    elif splits == 1:
        if M <= 16:
            ok = wide is None and weights >= 45e6 and (K >= 3072 or M >= 8)
        else:
            ok = K >= 2048 and not many or K >= 4096 and strips <= 512 and blocks >= 0.9 * 256
    elif M <= 16:
        ok = K % (splits * 2048) != 0 and (K >= 5120 or K >= 3072 and weights >= 24e6)
    else:
        # the library is the best form of a square weight in one of its rounds (2560 x 2560, 48
        # 1.08 of the time)
        ok = K >= (2048 if M > 24 or weights >= 1e7 else 2049) and not (
            wide and K % (splits * 2048) == 0) and not (wide is None and K == N and 32 < M <= 48)
    return splits if ok else None


@functools.lru_cache(maxsize=4096)
def _ring_sizes(M: int, N: int, K: int, gateup: bool):
    wide = _ring_plan(M, N, K, gateup)
    splits = _ring_narrow(M, N, K, gateup, wide)
    if splits:
        return 32 * -(-M // 32), splits, True
    return wide and (*wide, False)


def _ring_choice(M: int, N: int, K: int, gateup: bool = False):
    """(rows of a tile, column splits, whether in strips of 64 weight rows) of the product on
    the transfer ring, None where the other forms are faster. The sizes alone decide, so that
    the rules are gone through once for each (2 to 3 us, 17 times in a prompt of four layers,
    which up to some tens of rows takes as long as its host), but for two rows, where a switch
    has a say."""
    if M == 2:
        return _ring_sizes.__wrapped__(M, N, K, gateup)
    return _ring_sizes(M, N, K, gateup)


# us of a step of 64 columns where a block is alone on its CU's part of the chip, of starting and
# ending a round, and the share of the first that is left where few blocks run; by rows of a
# tile and whether strips are of 64 weight rows
_RING_STEPS = {(32, False): (0.443, 1.5, 0.85), (32, True): (0.306, 1.3, 0.69),
               (64, False): (0.472, 1.9, 0.86), (64, True): (0.527, 2.5, 0.20),
               (96, False): (0.688, 2.0, 0.72), (128, False): (0.754, 1.5, 0.77)}


def _ring_us(M: int, N: int, K: int, gateup: bool, tile: int, splits: int, narrow: bool) -> float:
    """The ring product's time by rounds of its blocks: a step takes what a CU needs for it or
    what memory needs for all of them (6.46 TB/s; where some CUs have two blocks and others one,
    partly for two each), splits 2.3 us and their sums on top. Least squares over 7600 times of
    130 weights at 3 to 128 rows, 6% rms."""
    step, ends, few = _RING_STEPS[tile, narrow]
    slots, rows, mtiles = 512 if narrow else 256, N * (1 + gateup), -(-M // tile)
    height = 64 if narrow else 128
    rounds, rest = divmod(-(-rows // height) * mtiles * splits, slots)
    steps, us = K / 64 / splits, 2.0
    for blocks, times in ((slots, rounds), (rest, int(rest > 0))):
        busy = blocks / slots if not narrow else 1.0 if blocks > 256 else 0.5
        full = blocks + 0.3 * (512 - blocks) if narrow and blocks > 256 else blocks
        read = height * 128 / mtiles * full / 6.46e6
        us += times * (steps * max(step * (few + (1 - few) * busy), read) + ends)
    if splits == 1:
        return us * 1.08 if tile == 64 and narrow else us
    return us + 2.3 + splits * M * rows * 1.7e-6


@functools.lru_cache(maxsize=4096)
def _ring_fastest(M: int, N: int, K: int, gateup: bool):
    if K % 64 or K < 256 or N % 8:
        return None
    forms = []
    for tile, narrow in {(32 * -(-M // 32), False), (64, False), (32 * -(-M // 32), True)}:
        if tile > 32 * -(-M // 32) or narrow and tile > 64:
            continue
        tiles = -(-N // ((64 if gateup else 128) // (1 + narrow))) * -(-M // tile)
        for splits in {1, 256 // tiles, 256 // tiles * 2, 512 // tiles if narrow else 1}:
            if 1 <= splits <= min(16, K // 256) and (splits == 1 or tiles * splits <= 520):
                forms.append((_ring_us(M, N, K, gateup, tile, splits, narrow), tile, splits, narrow))
    us, *form = min(forms)
    plan = _ring_choice(M, N, K, gateup)
    if plan:
        full = plan[0] == 128 and form == [64, 1, False] and N > 64 * 112
        short = plan[2] and form[0] == 64 and not form[2] and min(plan[1], form[1]) > 1 and K <= 2048
        ahead = 0.9 if gateup and (full or short) else 0.97
        return tuple(form) if us < ahead * _ring_us(M, N, K, gateup, *plan) else plan
    stream = N * (1 + gateup) * K * 2 / 6.2e6 + 3.0
    near = 1.3 if M > 32 and not form[2] else 1.2
    return tuple(form) if K >= (1536 if M <= 16 else 1024) and us < near * stream else None


def _ring_form(M: int, N: int, K: int, gateup: bool = False):
    """The ring's form that the products take, laid out as _ring_choice's answer.

    Those lines were drawn where all blocks read the same columns at a time; since strips start at
    steps of their own (ring_gemm.hip) the wide forms run up to a quarter faster, and an
    estimate finds the form: over 130 weights at 3 to 128 rows, 105 of them drawn, 0.957 of the
    time of _ring_choice's, 1.035 of the best form's, 1.11 of _ring_choice's at the most. Its form
    is taken where it is 3 per cent ahead of that one's by the same estimate, and where that is
    none, if it comes within 1.2 (above 32 rows, where those are slower, 1.3) of reading the
    weights at 6.2 TB/s; skinny.hip is the better one for up to 16 short rows (2 x 25088 x 1024, 3
    19.8 / 22.5). us, _ring_choice's form or the others / here: gate-up 2 x 14336 x 4096, M = 47 44.2
    / 38.1, 128 58.3 / 48.2; 32000 x 4096, 47 48.5 / 41.5, 112 76.6 / 51.8; 20288 x 1664, 16 41.5 /
    15.2; 12584 x 3520, 40 32.7 / 21.6; but 2 x 5632 x 2048, 48 14.2 / 15.7.

    Two tiles of 64 gate-up rows on more than 224 of the CUs take up to 15 per cent longer than it
    says; against splits of 128-row tiles, as full, they have to be 10 per cent ahead (us, splits
    / two tiles: 2 x 7552 x 3648, M = 103 34.4 / 37.7, 2 x 8128 x 4160, 128 39.3 / 44.7, 2 x 8192 x
    4032, 112 37.0 / 41.7; on fewer CUs 2 x 6720 x 3264, 128 35.2 / 32.7, 2 x 7040 x 3264 35.7 /
    33.3; far ahead 2 x 8192 x 2048, 128 23.0 / 20.9). So do splits of 128-row strips against those of 64,
    where rows have 2048 columns and fewer (strips of 64 / 128: 2 x 2816 x 2048, 47 12.8 / 13.8, 34 12.4 /
    12.8; 2 x 2816 x 1664, 46 11.8 / 13.7; 2 x 3008 x 1344, 34 11.3 / 11.7; but 2 x 2880 x 2240, 40 14.4 /
    13.4, 2 x 3008 x 3136, 38 17.2 / 14.8)."""
    return _ring_choice(M, N, K, gateup) if M == 2 else _ring_fastest(M, N, K, gateup)


def _ring(x: torch.Tensor, w: torch.Tensor, plan: Tuple[int, ...], act: int = 0,
          parts: bool = False) -> torch.Tensor:
    """x @ w^T, or act 1 (silu), 2 (tanh gelu) of the gate rows times the up rows. plan: (rows
    of a tile, column splits), and whether in strips of 64 weight rows. parts: the float32
    parts of a split product [splits, M, N], not added up."""
    lib, hip = _lib()
    K, (tile, splits), narrow = x.shape[-1], plan[:2], len(plan) > 2 and plan[2]
    M, N = x.numel() // K, w.shape[0] // (2 if act else 1)
    out = None if parts else torch.empty(*x.shape[:-1], N, dtype=x.dtype, device=x.device)
    # at most 256 tiles of 128 x 128 float32 (gate and up): 17 MB
    part = None if splits == 1 else torch.empty(splits, M, w.shape[0], dtype=torch.float32,
                                                device=x.device)
    hip.check(lib.oa_ring_gemm(hip.current_stream_ptr(), x.data_ptr(),
                               K if x.is_contiguous() else x.stride(0), w.data_ptr(),
                               None if parts else out.data_ptr(),
                               None if part is None else part.data_ptr(),
                               M, N, K, tile, int(narrow), splits, act), "oa_ring_gemm")
    return part if parts else out


# unsplit forms that leave CUs idle, to the library's gain, by (form, gateup): rows and weight rows of
# a tile, up to how many tiles, from how many columns on
_TILES_IDLE = {(3, False): (160, 256, 192, 2048), (4, False): (256, 128, 192, 2048),
               (8, False): (96, 128, 153, 2048), (9, False): (128, 64, 192, 2048),
               (8, True): (96, 128, 160, 4224)}


@functools.lru_cache(maxsize=4096)
def _tile_sizes(M: int, N: int, K: int, gateup: bool, summed: bool) -> Optional[int]:
    weights = N * K * (2 if gateup else 1)
    if summed and K < 2 * N:             # deep products split, others hardly
        return None
    if weights < (2 ** 22 if gateup or summed or M >= 500 else 9e6) or (
            M >= 3500 and not gateup):
        return None
    if gateup and M > 4000 and M * weights >= 7.2e11:
        tiles = -(-M // 256) * -(-2 * N // 256)
        if K >= 8192 or K >= 4096 and tiles % 256 == 0:
            return None
    plan = _lib()[0].oa_tile_gemm_plan(M, N, K, int(gateup), int(summed))
    if plan < 0 or plan == 1 and K >= 2048 and not gateup:       # tiles of 256 x 256, unsplit
        return None
    form, splits = plan >> 8, plan & 255
    rows, cols, most, least = _TILES_IDLE.get((form, gateup), (1, 1, 0, 0))
    if splits == 1 and least <= K <= 8192 and -(-M // rows) * -(-N * (1 + gateup) // cols) <= most:
        # small tiles: where nothing of what costs the library a quarter and more is in the sizes
        ahead = M > 256 and weights >= 9e6 if form == 9 else gateup or M > 256 or M % 32
        if form < 8 or K % 128 == 0 and ahead:
            return None
    return plan


def _tile_choice(M: int, N: int, K: int, gateup: bool = False, summed: bool = False) -> Optional[int]:
    """Form and column splits of the tile product (tile_gemm.hip; figures and the rule by sizes
    there) of more than 128 rows, None where the library is faster: light weights at few rows (us,
    library / tiles: 2048 x 2048, 256 rows 10.1 / 13.0, 800 15.3 / 14.5; between 500 and 800 level to 2.5 us
    ahead, 512 11.4 / 13.9, 599 13.6 / 14.0, 2816 x 1664, 550 16.7 / 12.8, which its first call of a number
    of rows, 76 us of the host where the tiles take 9, outweighs in a model of a few dozen layers; deep
    ones with a norm behind them split, 1024 x 4096, 338 16.9 / 15.0), and from some thousand rows on,
    where power bounds both (4096 x 4096, 4067 92 / 103, 2900 79 / 78), but for gate-up, whose activation
    rides along.
    So do products that would run in whole tiles of 256 x 256, the library's own form and faster
    there (8192 x 4096, 2048 rows 93 / 101; 16384 x 2048, 922 53 / 53, 1966 99 / 105, 2987 156 / 170; 14336 x
    4096, 1024 89 / 94, 2092 180 / 194; 10240 x 8192, 3072 337 / 358), but for short rows, where it is
    not (10296 x 640, 1430 35 / 23). And tiles of 160 x 256 and 256 x 128 that leave a quarter of the
    CUs idle: of 340 such products of 2048 to 8192 columns, on two cards, three in four were 3 per cent
    and more slower, 1.05 times on average, and one in 25 faster (12288 x 4096, 514 61 / 68, 640 63 /
    70, 486 57 / 58; 11072 x 5760, 517 87 / 92; 16640 x 3648, 315 61 / 66). With 193 tiles and more
    they are ahead again, by 5 per cent, and on rows of 12000 columns the library is up to 1.5 times
    slower (17856 x 12736, 279 293 / 191). Tiles of 96 x 128 with two in five idle go there too, where
    rows are whole steps of 128 columns (6144 x 4096, 262 30.1 / 33.9, 283 30.4 / 35.2; 9088 x 4096, 191
    32.7 / 36.9; of 141 on two cards 128 were 3 per cent and more slower, 1.1 times on average): half a
    step over costs the library a quarter (6144 x 3136, 268 31.4 / 27.9), and so do whole 32s of up to
    256 rows (9088 x 4096, 192 40.5 / 36.6). So do, above 256 rows and but for light weights, those of 128 x
    64 with a quarter idle (2880 x 4352, 512 26.7 / 31.3; 4032 x 3328, 382 21.9 / 24.9; 3072 x 5120, 497 32 /
    36), and gate-up of 4224 columns on in 160 of 96 x 128 (library and activation / tiles: 2 x 5120 x 5888,
    190 50.3 / 55.1; 2 x 3072 x 5888, 278 44.9 / 50.6; 101 of them 1.09 on average).
    Of gate-up the largest of more than 4000 rows go there where columns are many (library and
    activation / tiles: 8000 rows of 4096 x 14336 1281 / 1371, 8192 of 7168 x 8192 1315 / 1385, 16000 of
    28672 x 8192 10213 / 10959, 9395 of 16848 x 13952 6023 / 6735; smaller ones not, 5500 of 4096 x 14336
    1049 / 964) or where its tiles, 256 x 256 by its kernel's name, which splits those left over by
    columns, leave none over (14336 x 4096, 8000 rows 1403 / 1449, 8192 1412 / 1459, 12288 2084 / 2114;
    7500 1404 / 1377, 8193 1576 / 1507, 9200 1601 / 1601, 10319, 16 tiles of 4608 short, 1935 / 1796;
    13195 of 13824 x 5120, 16 of 5632 short, 3038 / 2680). Over 113 products of 3000 to 16384 rows, 52 of
    them drawn, the choice is 0.5 per cent from the better of the two on average; many columns in
    part of a round lose up to 6 (5084 rows of 8424 x 9984, 1346 / 1266).
    Of 33110 plain products at 129 to 3500 rows, 3000 weights but 19 of them drawn, 23000 are taken, 1.2
    times as fast as the library on average (1.16 on whole steps of 128 columns), 4 in 100 of them 3 per
    cent and more slower, 7 in 1000 more than 10 (16704 x 5120, 283 rows 81 / 98: three row tiles of
    96 in a round and a half); gate-up 1.2 times, hardly one slower. summed: for linear_parts, where a
    norm adds up the splits."""
    return _tile_sizes(M, N, K, gateup, summed) if M > 128 else None


def _near_rows(x: torch.Tensor) -> bool:
    """Rows of x that the tile product's 32-bit places span (tile_gemm.hip): less than 8 MB apart.
    Others, one token of each of many long sequences, go to the library."""
    return x.is_contiguous() or x.stride(0) < 2 ** 22


def _tile(x: torch.Tensor, w: torch.Tensor, plan: int, act: int = 0,
          parts: bool = False) -> torch.Tensor:
    """x @ w^T, or act 1 (silu), 2 (tanh gelu) of the gate rows times the up rows, in the form
    and splits of plan. parts: the float32 parts of a split product, as of _ring."""
    lib, hip = _lib()
    K, splits = x.shape[-1], plan & 255
    M, N = x.numel() // K, w.shape[0] // (2 if act else 1)
    out = None if parts else torch.empty(*x.shape[:-1], N, dtype=x.dtype, device=x.device)
    # at most 256 tiles of 256 x 256 float32: 67 MB
    part = None if splits == 1 else torch.empty(splits, M, N, dtype=torch.float32, device=x.device)
    hip.check(lib.oa_tile_gemm(hip.current_stream_ptr(), x.data_ptr(),
                               K if x.is_contiguous() else x.stride(0), w.data_ptr(),
                               None if parts else out.data_ptr(),
                               None if part is None else part.data_ptr(), M, N, K, plan, act),
              "oa_tile_gemm")
    return part if parts else out


@functools.lru_cache(maxsize=4096)
def _shallow_parts(M: int, N: int, K: int) -> Optional[int]:
    """The tile product's plan of more than 128 rows whose parts a norm adds up, for products of K < 2 N
    that would be tiles anyway: where splits of more than one are the faster way by the same estimate.
    They save the launch that would add them up, or fill CUs that one split leaves idle. us a prompt of
    four layers, without / with: 4096 x 4096 in all, 130 rows 659 / 647, 256 797 / 779, 300 826 / 810,
    512 1044 / 1038; 2048 x 2048, 512 516 / 498, and with 2048 x 2816 behind 64 experts 1330 / 1312. Larger
    results cost as much to write in parts as splits gain (4096 x 4096, 600 1273 / 1276, 800 1555 / 1555)."""
    if K >= 2 * N or M * N > 2200000 or _tile_sizes(M, N, K, False, False) is None:
        return None
    plan = _lib()[0].oa_tile_gemm_plan(M, N, K, 0, 1)
    return plan if plan & 255 > 1 else None


def shallow_parts(x: torch.Tensor, w: torch.Tensor) -> Optional[PlaneSum]:
    """linear_parts' parts for more than 128 rows of less than 2 N columns, None where the product is
    not split for the norm. (A caller who wants the product then, too, asks linear_parts with `shallow`:
    it looks the operands over once.)"""
    M = x.numel() // x.shape[-1]
    if M > 128 and x.dim() == 2 and w.shape[0] <= 8192 and _skinny_ok(x, w) and _near_rows(x):
        tile = _shallow_parts(M, *w.shape)
        if tile:
            return PlaneSum(_tile(x, w, tile, parts=True))
    return None


def _rows_product(x: torch.Tensor, w: torch.Tensor, M: int, parts: bool = False,
                  shallow: bool = False) -> Union[torch.Tensor, PlaneSum, None]:
    """x @ w^T of M > 1 rows on the ring, in strips or in tiles, None where none of them takes it;
    parts, shallow: see linear_parts."""
    if not _skinny_ok(x, w):
        return None
    N, K = w.shape
    if M <= 128:
        plan = _ring_form(M, N, K)
        if plan:
            y = _ring(x, w, plan, parts=parts and plan[1] > 1)
            return PlaneSum(y) if parts and plan[1] > 1 else y
        form = _skinny_form(M, N, K, strided=not x.is_contiguous())
        return _skinny(x, w, form) if form else None
    if not _near_rows(x):
        return None
    if parts:
        plan = shallow and _shallow_parts(M, N, K) or _tile_choice(M, N, K, summed=True)
        if plan and plan & 255 > 1:
            return PlaneSum(_tile(x, w, plan, parts=True))
    plan = _tile_choice(M, N, K)
    return None if plan is None else _tile(x, w, plan)


def linear_parts(x: torch.Tensor, w: torch.Tensor,
                 shallow: bool = False) -> Union[torch.Tensor, PlaneSum]:
    """x @ w^T for rows x [T, K] that go through fused_add_rms_norm next: bf16 [T, N], or the
    product's float32 column parts, which the norm adds up, where the transfer ring or, of deep
    products (shallow: of those of fewer columns too, _shallow_parts), the tiles split it."""
    M = x.numel() // x.shape[-1]
    y = _rows_product(x, w, M, x.dim() == 2 and w.shape[0] <= 8192, shallow) if M > 1 else None
    return _other_product(x, w, M) if y is None else y


def linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """F.linear with custom HIP paths for decode shapes: the VALU GEMV at M = 1
    (hipBLASLt's M=1 kernels run ~2.5x off the HBM roofline on gfx950), the transfer
    ring up to 128 rows and the skinny matrix-core products up to 32 where they win
    (_ring_form, _skinny_form), the VALU GEMV for what two rows are left and the
    matrix-core GEMV for what 3 to 8 are, the tile product for more than 128 (_tile_choice);
    everything else goes to hipBLASLt."""
    M = x.numel() // x.shape[-1]
    y = _rows_product(x, w, M) if M > 1 else None
    return _other_product(x, w, M) if y is None else y


def _other_product(x: torch.Tensor, w: torch.Tensor, M: int) -> torch.Tensor:
    """What _rows_product leaves: the VALU and staged GEMVs or the library."""
    if (
        x.is_cuda
        and x.dtype == torch.bfloat16
        and (_gemv_m_ok(M) or _bf16_mfma_ok(M, x.shape[-1]))
        and x.shape[-1] % 8 == 0
        # the kernels read whole rows one after the other, 16 bytes at a time: a
        # column slice of a wider buffer has gaps and may start anywhere
        and w.is_contiguous()
        and x.is_contiguous()
        and x.data_ptr() % 16 == 0
        and w.data_ptr() % 16 == 0
    ):
        from opsagent_amd.ops import hip_lib

        lib = hip_lib.get_lib()
        N, K = w.shape
        out = torch.empty(*x.shape[:-1], N, dtype=x.dtype, device=x.device)
        rc = lib.oa_gemv(
            hip_lib.current_stream_ptr(), x.data_ptr(), w.data_ptr(), out.data_ptr(),
            M, N, K,
        )
        hip_lib.check(rc, "oa_gemv")
        return out
    return torch.nn.functional.linear(x, w)


def linear_pair(x0: torch.Tensor, w0: torch.Tensor, x1: torch.Tensor,
                w1: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """linear(x0, w0) and linear(x1, w1): in one launch where both are skinny strips of one size."""
    M, (N, K) = x0.numel() // x0.shape[-1], w0.shape
    if not (1 < M <= 16 and x0.shape == x1.shape and w0.shape == w1.shape and x0.dim() == 2
            and x0.stride() == x1.stride() and x0.device == x1.device
            and _skinny_ok(x0, w0) and _skinny_ok(x1, w1) and not _ring_form(M, N, K)
            and _skinny_form(M, N, K, strided=not x0.is_contiguous()) == 1):
        return linear(x0, w0), linear(x1, w1)
    lib, hip = _lib()
    out = torch.empty(2, M, N, dtype=x0.dtype, device=x0.device)
    hip.check(lib.oa_skinny_pair(
        hip.current_stream_ptr(), x0.data_ptr(), x1.data_ptr(), K if x0.is_contiguous() else x0.stride(0),
        w0.data_ptr(), w1.data_ptr(), out[0].data_ptr(), out[1].data_ptr(), M, N, K), "oa_skinny_pair")
    return out[0], out[1]


def linear_float(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """linear(x, w).float(), of one bf16 row in the product's own launch where gemv.hip takes it."""
    N, K = w.shape
    if not (x.is_cuda and x.dim() == 2 and x.shape == (1, K) and K % 2048 == 0 and K <= 16384
            and x.dtype == w.dtype == torch.bfloat16 and x.device == w.device
            and _gemv_m_ok(1) and _plain_call(x, w) and x.is_contiguous() and w.is_contiguous()
            and (x.data_ptr() | w.data_ptr()) % 16 == 0):
        return linear(x, w).float()
    lib, hip = _lib()
    out = torch.empty(1, N, dtype=torch.float32, device=x.device)
    hip.check(lib.oa_gemv_float(hip.current_stream_ptr(), x.data_ptr(), w.data_ptr(), out.data_ptr(),
                                N, K), "oa_gemv_float")
    return out


def _is_gpu(t: torch.Tensor) -> bool:
    return t.is_cuda


_hip = None


def _lib():
    global _hip
    if _hip is None:                 # the import statement takes 0.7 us, 33 times a prompt
        from opsagent_amd.ops import hip_lib

        _hip = hip_lib
    return _hip.get_lib(), _hip


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float = 1e-5) -> torch.Tensor:
    if not _is_gpu(x):
        return torch_ref.rms_norm(x, weight, eps)
    assert x.dtype == torch.bfloat16 and x.is_contiguous()
    lib, hip = _lib()
    rows = x.numel() // x.shape[-1]
    out = torch.empty_like(x)
    rc = lib.oa_rmsnorm(
        hip.current_stream_ptr(), x.data_ptr(), weight.data_ptr(), out.data_ptr(),
        rows, x.shape[-1], eps,
    )
    hip.check(rc, "oa_rmsnorm")
    return out


def embed_rms_norm(ids: torch.Tensor, table: torch.Tensor, weight: torch.Tensor,
                   eps: float = 1e-5) -> Tuple[torch.Tensor, torch.Tensor]:
    """(table[ids], its rms_norm) for token ids [T]; rows of NaN for ids outside the table
    (the GPU path, which cannot raise)."""
    D = table.shape[1]
    if not (table.is_cuda and table.dtype == torch.bfloat16 and weight.dtype == table.dtype
            and table.is_contiguous() and weight.is_contiguous()
            and ids.dim() == 1 and ids.is_contiguous()
            and ids.dtype in (torch.int64, torch.int32) and ids.device == table.device
            and D % 8 == 0 and D <= 8192 and (table.data_ptr() | weight.data_ptr()) % 16 == 0
            and table.shape[0] > 0):
        x = torch.nn.functional.embedding(ids, table)
        return x, rms_norm(x, weight, eps)
    lib, hip = _lib()
    x, out = torch.empty(2, ids.numel(), D, dtype=table.dtype, device=table.device)
    hip.check(lib.oa_embed_rmsnorm(
        hip.current_stream_ptr(), table.data_ptr(), ids.data_ptr(), int(ids.dtype == torch.int64),
        table.shape[0], weight.data_ptr(), x.data_ptr(), out.data_ptr(), ids.numel(), D, eps),
        "oa_embed_rmsnorm")
    return x, out


class PlaneSum(NamedTuple):
    """A product whose float32 column parts [parts, T, N] the norm behind it adds up."""

    planes: torch.Tensor


class PairSum(NamedTuple):
    """A sum that the norm behind it takes: for each token its `top` rows of y
    [T * top, H], bf16, plus its row of `more`, which may be a product's parts."""

    y: torch.Tensor
    top: int
    more: Union[torch.Tensor, PlaneSum, None]


def _added_up(x: Union[PlaneSum, PairSum]) -> torch.Tensor:
    """The hidden rows that x stands for, bf16, in the order of the norms' kernels."""
    if isinstance(x, PairSum):
        return moe_combine(x.y, x.top, x.more)
    total = x.planes[0].clone()
    for plane in x.planes[1:]:
        total += plane
    return total.to(torch.bfloat16)


def _add_norm_parts(x: Union[PlaneSum, PairSum], residual: torch.Tensor, weight: torch.Tensor,
                    eps: float) -> Optional[torch.Tensor]:
    """fused_add_rms_norm's first result from what is not added up yet, None where the
    kernels do not take the residual or the weight."""
    rows, dim = residual.shape
    planes = isinstance(x, PlaneSum)
    data, n = (x.planes, x.planes.shape[0]) if planes else (x.y, x.top)
    assert data.shape == ((n, rows, dim) if planes else (rows * n, dim)) and weight.numel() == dim
    assert residual.dtype == weight.dtype == torch.bfloat16 and data.dtype == (
        torch.float32 if planes else torch.bfloat16)
    assert data.get_device() == residual.get_device() == weight.get_device()
    assert data.is_contiguous() and residual.is_contiguous() and weight.is_contiguous()
    at, w = residual.data_ptr(), weight.data_ptr()
    if dim % 8 or dim > 8192 or (at | w) % 16:
        return None
    lib, hip = _lib()
    out = torch.empty_like(residual)
    if planes:
        hip.check(lib.oa_add_rmsnorm_parts(
            hip.current_stream_ptr(), data.data_ptr(), n, at, w, out.data_ptr(), rows, dim, eps),
            "oa_add_rmsnorm_parts")
    elif isinstance(x.more, PlaneSum):
        more = x.more.planes
        assert more.shape[1:] == (rows, dim) and more.dtype == torch.float32
        assert more.is_contiguous() and more.get_device() == residual.get_device()
        hip.check(lib.oa_add_rmsnorm_pairs_parts(
            hip.current_stream_ptr(), data.data_ptr(), n, more.data_ptr(), more.shape[0], at, w,
            out.data_ptr(), rows, dim, eps), "oa_add_rmsnorm_pairs_parts")
    else:
        hip.check(lib.oa_add_rmsnorm_pairs(
            hip.current_stream_ptr(), data.data_ptr(), n,
            x.more.data_ptr() if x.more is not None else None, at, w, out.data_ptr(), rows, dim, eps),
            "oa_add_rmsnorm_pairs")
    return out


def fused_add_rms_norm(
    x: Union[torch.Tensor, PlaneSum, PairSum], residual: torch.Tensor, weight: torch.Tensor,
    eps: float = 1e-5
) -> Tuple[torch.Tensor, torch.Tensor]:
    """Returns (rmsnorm(x+residual), x+residual). GPU path updates `residual`
    in place as the new residual stream and returns it. x may be a product's parts
    (linear_parts) or a sum over pairs (moe_combine) that is not added up yet."""
    if not isinstance(x, torch.Tensor):
        out = _add_norm_parts(x, residual, weight, eps) if _is_gpu(residual) else None
        if out is not None:
            return out, residual
        x = _added_up(x)
    if not _is_gpu(x):
        return torch_ref.fused_add_rms_norm(x, residual, weight, eps)
    assert x.dtype == torch.bfloat16 and x.is_contiguous() and residual.is_contiguous()
    lib, hip = _lib()
    rows = x.numel() // x.shape[-1]
    out = torch.empty_like(x)
    rc = lib.oa_fused_add_rmsnorm(
        hip.current_stream_ptr(), x.data_ptr(), residual.data_ptr(), weight.data_ptr(),
        out.data_ptr(), rows, x.shape[-1], eps,
    )
    hip.check(rc, "oa_fused_add_rmsnorm")
    return out, residual


class QuantRows(NamedTuple):
    """Hidden rows for fp8 products: 8-bit numbers [T, K] and a float32 scale a row."""

    rows: torch.Tensor
    scales: torch.Tensor

    @property
    def shape(self):
        return self.rows.shape

    @property
    def is_cuda(self) -> bool:
        return self.rows.is_cuda


def fp8_rows_ok(rows: int, K: int) -> bool:
    """Whether linear_fp8 of as many rows of K columns quantizes them first."""
    return rows > 8 and K % 128 == 0 and not _fp8_mfma_ok(rows, K)


def fused_add_rms_norm_fp8(
    x: Union[torch.Tensor, PlaneSum, PairSum], residual: torch.Tensor, weight: torch.Tensor,
    eps: float = 1e-5
) -> Tuple[Union[torch.Tensor, QuantRows], torch.Tensor]:
    """fused_add_rms_norm for fp8 products that quantize their rows (fp8_rows_ok): its first result
    quantized, the bits of quant_fp8, in the same launch; as it is where the kernel does not take it."""
    rows, dim = residual.shape
    if not (isinstance(x, torch.Tensor) and x.is_cuda and x.shape == residual.shape and rows
            and weight.numel() == dim and dim % 8 == 0 and dim <= 8192
            and all(t.dtype == torch.bfloat16 and t.device == x.device and t.is_contiguous()
                    and t.data_ptr() % 16 == 0 for t in (x, residual, weight))):
        return fused_add_rms_norm(x, residual, weight, eps)
    lib, hip = _lib()
    q = torch.empty(rows, dim, dtype=torch.uint8, device=x.device)
    scales = torch.empty(rows, dtype=torch.float32, device=x.device)
    hip.check(lib.oa_fused_add_rmsnorm_fp8(
        hip.current_stream_ptr(), x.data_ptr(), residual.data_ptr(), weight.data_ptr(), q.data_ptr(),
        scales.data_ptr(), rows, dim, eps), "oa_fused_add_rmsnorm_fp8")
    return QuantRows(q, scales), residual


def rope_apply_(
    q: torch.Tensor,
    k: torch.Tensor,
    cos: torch.Tensor,
    sin: torch.Tensor,
    positions: torch.Tensor,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """In-place on GPU; q [T, Hq, D], k [T, Hk, D], positions int32 [T]."""
    if not _is_gpu(q):
        return torch_ref.rope_apply(q, k, cos, sin, positions)
    assert q.dtype == torch.bfloat16 and q.is_contiguous() and k.is_contiguous()
    assert cos.dtype == torch.float32 and positions.dtype == torch.int32
    lib, hip = _lib()
    T, Hq, D = q.shape
    Hk = k.shape[1]
    rc = lib.oa_rope(
        hip.current_stream_ptr(), q.data_ptr(), k.data_ptr(), cos.data_ptr(),
        sin.data_ptr(), positions.data_ptr(), T, Hq, Hk, D,
    )
    hip.check(rc, "oa_rope")
    return q, k


def silu_mul(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    if not _is_gpu(gate):
        return torch_ref.silu_mul(gate, up)
    assert gate.dtype == torch.bfloat16 and gate.is_contiguous() and up.is_contiguous()
    lib, hip = _lib()
    out = torch.empty_like(gate)
    rc = lib.oa_silu_mul(
        hip.current_stream_ptr(), gate.data_ptr(), up.data_ptr(), out.data_ptr(),
        gate.numel(),
    )
    hip.check(rc, "oa_silu_mul")
    return out


def silu_halves(gu: torch.Tensor, i_local: int) -> torch.Tensor:
    """silu(gu[..., :I]) * gu[..., I:]; on the GPU the halves are read in place where
    their rows keep 16-byte alignment."""
    if (
        _is_gpu(gu) and gu.dtype == torch.bfloat16 and gu.is_contiguous() and gu.numel()
        and i_local % 8 == 0 and gu.shape[-1] == 2 * i_local and gu.data_ptr() % 16 == 0
    ):
        lib, hip = _lib()
        out = torch.empty(*gu.shape[:-1], i_local, dtype=gu.dtype, device=gu.device)
        hip.check(lib.oa_silu_halves(hip.current_stream_ptr(), gu.data_ptr(), out.data_ptr(),
                                     out.numel() // i_local, i_local), "oa_silu_halves")
        return out
    gate, up = gu.split([i_local, i_local], dim=-1)
    return silu_mul(gate.contiguous(), up.contiguous())


def quant_fp8(x: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """Per-row OCP e4m3 quantization: bf16 [T, K] -> (uint8 [T, K], f32 [T])."""
    T = x.numel() // x.shape[-1]
    K = x.shape[-1]
    if not _is_gpu(x):
        return torch_ref.quant_fp8(x)
    assert x.dtype == torch.bfloat16 and x.is_contiguous() and K % 8 == 0
    lib, hip = _lib()
    q = torch.empty(*x.shape, dtype=torch.uint8, device=x.device)
    scales = torch.empty(T, dtype=torch.float32, device=x.device)
    rc = lib.oa_quant_fp8(
        hip.current_stream_ptr(), x.data_ptr(), q.data_ptr(), scales.data_ptr(), T, K
    )
    hip.check(rc, "oa_quant_fp8")
    return q, scales


def linear_fp8(
    x: Union[torch.Tensor, QuantRows], w8: torch.Tensor, w_scale: torch.Tensor
) -> torch.Tensor:
    """out = (x @ dequant(w8)^T) with per-row weight scales.

    GPU: M <= 8 -> fp8 weight-streaming GEMV (half the bytes of bf16);
    M <= 16 -> the same GEMV padded to the next instantiation (catch-up /
    speculative verify passes); larger M -> quantize x per token and run the
    fp8 product on the transfer ring or in MFMA tiles (_gemm_fp8). (A dequant-to-bf16 + hipBLASLt
    variant was measured and REVERTED: 70B fp8 turn 723 ms vs 573 with the
    tile GEMM — the per-call dequant round-trip costs more than the GEMM's
    tile-pipeline inefficiency.)
    CPU: dequantized torch reference. x may be quantized already (fused_add_rms_norm_fp8)."""
    if isinstance(x, QuantRows):
        assert x.shape[1] == w8.shape[1]
        return _gemm_fp8(x.rows, x.scales, w8, w_scale)
    M = x.numel() // x.shape[-1]
    K = x.shape[-1]
    N = w8.shape[0]
    if not _is_gpu(x):
        return torch_ref.linear_fp8(x, w8, w_scale)
    assert x.dtype == torch.bfloat16 and x.is_contiguous() and K % 64 == 0
    lib, hip = _lib()
    # NOTE: the bf16 _gemv_m_ok cap (M<=2) encodes the crossover vs
    # hipBLASLt, which does not apply here — for fp8 weights the alternative
    # pays a dequant round-trip. Keep bf16-activation GEMV for skinny M.
    # M>8 goes to the MX tile GEMM: the padded M=12/16 gemv instantiations
    # are VALU-bound (16 dots/lane) and measured 276 us/call on the 70B
    # jump-ahead catch-up passes vs ~80-150 us through the tile GEMM.
    if (M <= 8 or _fp8_mfma_ok(M, K)) and K % 16 == 0:
        out = torch.empty(*x.shape[:-1], N, dtype=x.dtype, device=x.device)
        rc = lib.oa_gemv_fp8(
            hip.current_stream_ptr(), x.data_ptr(), w8.data_ptr(),
            w_scale.data_ptr(), out.data_ptr(), M, N, K,
        )
        hip.check(rc, "oa_gemv_fp8")
        return out
    if K % 128 != 0:
        # the pipelined tile GEMM unrolls K in 128-byte steps; shapes below
        # that (tiny test experts) chunk through the skinny-M gemv instead
        xm = x.reshape(M, K).contiguous()
        parts = [
            linear_fp8(xm[m0 : m0 + 8].contiguous(), w8, w_scale)
            for m0 in range(0, M, 8)
        ]
        return torch.cat(parts, dim=0).reshape(*x.shape[:-1], N)
    a8, a_scale = quant_fp8(x.reshape(M, K))
    return _gemm_fp8(a8, a_scale, w8, w_scale).view(*x.shape[:-1], N)


def _ring_plan_fp8(M: int, N: int, K: int) -> Optional[Tuple[int, int]]:
    """(rows of a tile, column splits) of the fp8 product on the transfer ring, None
    for the tile product. Up to 128 rows the ring is faster everywhere (figures at
    its kernel); more rows take it while the tiles leave half of the CUs idle. Two
    splits of short rows are not worth adding up (16384 x 2048, M = 47 12.6 us
    unsplit, 14.8)."""
    if N % 4 or K % 128:
        return None
    tile = min(128, 32 * -(-M // 32))
    tiles = -(-N // 128) * -(-M // tile)
    if M > 128 and tiles > 128:
        return None
    splits = max(1, min(256 // tiles, K // 512))
    return tile, 1 if splits == 2 and K < 4096 else splits


def _ring_choice_fp8(M: int, N: int, K: int) -> Optional[Tuple[int, int]]:
    """The ring's plan where it is faster than the tile product (fp8_moe.hip). Us, ring / tiles:
    without splits its one block a CU, of eight waves above 32 rows, falls behind with the rows,
    sooner with short ones (4096 x 1024, 32 7.8 / 8.0, 48 8.4 / 8.2, 128 11.6 / 8.7; 16384 x 2048,
    64 13.0 / 13.5, 80 15.2 / 14.0, 128 17.7 / 15.5; 28672 x 4096, 64 29.1 / 31.7, 80 30.9 / 31.8,
    96 31.2 / 31.8, 128 33.0 / 33.0): 80 rows lie between. Splits of short rows cost more than they
    fill (3072 x 2048, 80 11.0 / 11.5, 128 13.1 / 11.9, 200 14.5 / 11.8; 2048 x 2816, 128 13.2 /
    14.3, 200 14.4 / 14.3; 4096 x 3072, 200 18.7 / 17.9), long rows do not (4096 x 14336, 512 47.8
    / 67; 2048 x 8192, 512 22.7 / 38.5)."""
    plan = _ring_plan_fp8(M, N, K)
    if plan and (M > (32 if K < 2048 else 80) if plan[1] == 1
                 else K < 4096 and M > 128 and M * N >= 390000):
        return None
    return plan


@functools.lru_cache(maxsize=4096)
def _tile_form_fp8(M: int, N: int, K: int) -> int:
    return _lib()[0].oa_tile_gemm_fp8_form(M, N, K)


def _gemm_fp8(a8: torch.Tensor, a_scale: torch.Tensor, w8: torch.Tensor,
              w_scale: torch.Tensor) -> torch.Tensor:
    """The product of fp8 rows a8 [M, K] (K % 128 == 0) and w8 [N, K] with their row
    scales, bf16 [M, N]: on the transfer ring where its column splits fill the chip, above 128
    rows in tiles of one kind or the other (tile_gemm.hip; the rule there), bit for bit the
    same."""
    (M, K), N = a8.shape, w8.shape[0]
    lib, hip = _lib()
    out = torch.empty(M, N, dtype=torch.bfloat16, device=a8.device)
    plan = _ring_choice_fp8(M, N, K)
    if plan and w8.data_ptr() % 16 == 0 and a8.data_ptr() % 16 == 0:
        tile, splits = plan
        # at most 256 tiles of 128 x 128 float32: 17 MB
        part = None if splits == 1 else torch.empty(splits * M * N, dtype=torch.float32,
                                                    device=a8.device)
        hip.check(lib.oa_ring_gemm_fp8(
            hip.current_stream_ptr(), a8.data_ptr(), a_scale.data_ptr(), w8.data_ptr(),
            w_scale.data_ptr(), out.data_ptr(), None if part is None else part.data_ptr(),
            M, N, K, tile, splits), "oa_ring_gemm_fp8")
        return out
    form = _tile_form_fp8(M, N, K) if M > 128 else -1
    if form >= 0 and w8.data_ptr() % 16 == 0 and a8.data_ptr() % 16 == 0:
        hip.check(lib.oa_tile_gemm_fp8(
            hip.current_stream_ptr(), a8.data_ptr(), a_scale.data_ptr(), w8.data_ptr(),
            w_scale.data_ptr(), out.data_ptr(), M, N, K, form), "oa_tile_gemm_fp8")
        return out
    rc = lib.oa_gemm_fp8(
        hip.current_stream_ptr(), a8.data_ptr(), w8.data_ptr(),
        a_scale.data_ptr(), w_scale.data_ptr(), out.data_ptr(), M, N, K,
    )
    hip.check(rc, "oa_gemm_fp8")
    return out


def mlp_fp8_rows_ok(rows: int, K: int, i_local: int, gate_up_q: torch.Tensor) -> bool:
    """Whether mlp_fp8 runs both products on quantized rows."""
    return (fp8_rows_ok(rows, K) and i_local % 128 == 0 and gate_up_q.shape[0] == 2 * i_local
            and not _fp8_mfma_ok(rows, i_local))


def mlp_fp8(
    x: Union[torch.Tensor, QuantRows], gate_up_q: torch.Tensor, gate_up_s: torch.Tensor, i_local: int,
    down_q: torch.Tensor, down_s: torch.Tensor,
) -> torch.Tensor:
    """(silu(x @ gate8^T) * (x @ up8^T)) @ down8^T. Where both products are tile
    products (prefill rows), the activation is made by the wide tiles of the first one or
    quantized as it is made: the same bf16 values, rows and scales as quantizing it afterwards.
    x may be quantized already, where mlp_fp8_rows_ok says so."""
    if isinstance(x, QuantRows):
        M, tiles = x.shape[0], True
    else:
        M = x.numel() // x.shape[-1]
        tiles = M > 8 and _is_gpu(x) and mlp_fp8_rows_ok(M, x.shape[-1], i_local, gate_up_q)
    if not tiles:
        return linear_fp8(gateup_silu_fp8(x, gate_up_q, gate_up_s, i_local), down_q, down_s)
    lib, hip = _lib()
    lead, K = x.shape[:-1], x.shape[-1]
    if not isinstance(x, QuantRows):
        assert x.dtype == torch.bfloat16 and x.is_contiguous()
        x = QuantRows(*quant_fp8(x.reshape(M, K)))
    form = -1
    if M > 128 and not _ring_choice_fp8(M, 2 * i_local, K) and (i_local + 256) * K < 2 ** 32:
        form = _tile_form_fp8(M, 2 * i_local, K)
    if 0 <= form <= 2 and (x.rows.data_ptr() | gate_up_q.data_ptr()) % 16 == 0:
        act = torch.empty(M, i_local, dtype=torch.bfloat16, device=x.rows.device)
        hip.check(lib.oa_tile_gemm_fp8_silu(
            hip.current_stream_ptr(), x.rows.data_ptr(), x.scales.data_ptr(), gate_up_q.data_ptr(),
            gate_up_s.data_ptr(), act.data_ptr(), M, i_local, K, form), "oa_tile_gemm_fp8_silu")
        a8, a_scale = quant_fp8(act)
    else:
        gu = linear_fp8(x, gate_up_q, gate_up_s)
        a8 = torch.empty(M, i_local, dtype=torch.uint8, device=gu.device)
        a_scale = torch.empty(M, dtype=torch.float32, device=gu.device)
        hip.check(lib.oa_silu_quant_fp8(hip.current_stream_ptr(), gu.data_ptr(), a8.data_ptr(),
                                        a_scale.data_ptr(), M, i_local), "oa_silu_quant_fp8")
    return _gemm_fp8(a8, a_scale, down_q, down_s).view(*lead, down_q.shape[0])


def linear_norm(
    x: torch.Tensor, norm_w: torch.Tensor, eps: float, w: torch.Tensor
) -> torch.Tensor:
    """rmsnorm(x) @ W^T with the norm fused into the GEMV prologue (decode
    fast path: the standalone norm kernel + its output round-trip disappear).
    Fused form normalizes in fp32 without the intermediate bf16 rounding of
    the two-kernel form (slightly MORE precise)."""
    M = x.numel() // x.shape[-1]
    if M == 1 and _bf16_prenorm():
        return linear(rms_norm(x, norm_w, eps), w)
    if (
        x.is_cuda and x.dtype == torch.bfloat16
        and (_gemv_m_ok(M) or _bf16_mfma_ok(M, x.shape[-1]))
        and x.shape[-1] % 8 == 0 and x.is_contiguous() and w.is_contiguous()
    ):
        from opsagent_amd.ops import hip_lib

        lib = hip_lib.get_lib()
        N, K = w.shape
        out = torch.empty(*x.shape[:-1], N, dtype=x.dtype, device=x.device)
        rc = lib.oa_gemv_ex(
            hip_lib.current_stream_ptr(), x.data_ptr(), w.data_ptr(), out.data_ptr(),
            norm_w.data_ptr(), None, M, N, K, eps, 1,
        )
        hip_lib.check(rc, "oa_gemv_ex(norm)")
        return out
    return linear(rms_norm(x, norm_w, eps), w)


def linear_addres(x: torch.Tensor, w: torch.Tensor, res: torch.Tensor) -> torch.Tensor:
    """x @ W^T + res — the projection emits the new residual stream directly."""
    M = x.numel() // x.shape[-1]
    if (
        x.is_cuda and x.dtype == torch.bfloat16
        and (_gemv_m_ok(M) or _bf16_mfma_ok(M, x.shape[-1]))
        and x.shape[-1] % 8 == 0 and x.is_contiguous() and w.is_contiguous()
        and res.is_contiguous()
    ):
        from opsagent_amd.ops import hip_lib

        lib = hip_lib.get_lib()
        N, K = w.shape
        out = torch.empty(*x.shape[:-1], N, dtype=x.dtype, device=x.device)
        rc = lib.oa_gemv_ex(
            hip_lib.current_stream_ptr(), x.data_ptr(), w.data_ptr(), out.data_ptr(),
            None, res.data_ptr(), M, N, K, 0.0, 2,
        )
        hip_lib.check(rc, "oa_gemv_ex(addres)")
        return out
    return linear(x, w) + res


def gateup_silu_norm(
    x: torch.Tensor, norm_w: torch.Tensor, eps: float, gate_up_w: torch.Tensor,
    i_local: int
) -> torch.Tensor:
    """silu(norm(x) @ gate^T) * (norm(x) @ up^T), norm fused in the prologue."""
    M = x.numel() // x.shape[-1]
    if M == 1 and _bf16_prenorm():
        return gateup_silu(rms_norm(x, norm_w, eps), gate_up_w, i_local)
    if (
        x.is_cuda and x.dtype == torch.bfloat16
        and (_gemv_m_ok(M) or _bf16_mfma_ok(M, x.shape[-1]))
        and x.shape[-1] % 8 == 0 and x.is_contiguous() and gate_up_w.is_contiguous()
    ):
        from opsagent_amd.ops import hip_lib

        lib = hip_lib.get_lib()
        out = torch.empty(*x.shape[:-1], i_local, dtype=x.dtype, device=x.device)
        rc = lib.oa_gemv_gateup_ex(
            hip_lib.current_stream_ptr(), x.data_ptr(), gate_up_w.data_ptr(),
            out.data_ptr(), norm_w.data_ptr(), M, i_local, x.shape[-1], eps, 1,
        )
        hip_lib.check(rc, "oa_gemv_gateup_ex(norm)")
        return out
    return gateup_silu(rms_norm(x, norm_w, eps), gate_up_w, i_local)


def _moe_act(act):
    """(kernel's activation number, limit, alpha) of an expert activation, None
    if the kernels have no such activation."""
    if isinstance(act, tuple) and act[0] == "clamp_swish":
        return 2, float(act[1]), float(act[2])
    if act == "relu2":
        return 3, 0.0, 0.0
    return (0, 0.0, 0.0) if act in (None, "silu") else None


def moe_route_ok(x: torch.Tensor, router_w: torch.Tensor, top: int) -> bool:
    """Whether the routing kernels take this router."""
    E, K = router_w.shape
    return (
        x.is_cuda and x.dtype == torch.bfloat16 and x.dim() == 2 and x.is_contiguous()
        and router_w.dtype == torch.float32 and router_w.is_contiguous()
        and router_w.device == x.device and x.shape[1] == K
        and K % 8 == 0 and E <= 1024 and top <= min(E, 64)
        and x.data_ptr() % 16 == 0 and router_w.data_ptr() % 16 == 0
    )


def moe_route(x: torch.Tensor, router_w: torch.Tensor, top: int):
    """Softmax routing of bf16 rows x [T, K] by float32 router_w [E, K]: experts
    int32, weights float32 (normalised over the chosen) and tokens int32, each
    [T, top]. Static shapes and no host sync in either form: routers that the kernels do
    not take go through the library."""
    T, K = x.shape
    E = router_w.shape[0]
    if not moe_route_ok(x, router_w, top):
        probs = torch.softmax(torch.nn.functional.linear(x.float(), router_w), dim=-1)
        wts, idx = probs.topk(top, dim=-1)
        tok = torch.arange(T, device=x.device, dtype=torch.int32)[:, None].expand(T, top)
        return idx.int(), wts / wts.sum(dim=-1, keepdim=True), tok.contiguous()
    lib, hip = _lib()
    idx, tok = torch.empty(2, T, top, dtype=torch.int32, device=x.device)
    wts = torch.empty(T, top, dtype=torch.float32, device=x.device)
    scratch = torch.empty(lib.oa_moe_route_scratch(T, E, K), dtype=torch.float32, device=x.device)
    hip.check(lib.oa_moe_route(hip.current_stream_ptr(), x.data_ptr(), router_w.data_ptr(),
                               scratch.data_ptr(), idx.data_ptr(), wts.data_ptr(), tok.data_ptr(),
                               T, E, K, top), "oa_moe_route")
    return idx, wts, tok


def moe_combine(y: torch.Tensor, top: int, more: Union[torch.Tensor, PlaneSum, None] = None,
                parts: bool = False) -> Union[torch.Tensor, PairSum]:
    """out[t] = sum of rows t * top .. + top of y [T * top, H] (+ more[t]), bf16
    with float32 sums in one order. With `parts` it may be left to the norm that follows."""
    T, H = y.shape[0] // top, y.shape[1]
    assert y.is_cuda and y.dtype == torch.bfloat16 and y.is_contiguous()
    if isinstance(more, PlaneSum):
        if parts and H % 8 == 0 and H <= 8192 and more.planes.shape[1:] == (T, H):
            return PairSum(y, top, more)
        more = _added_up(more)
    assert more is None or (more.shape == (T, H) and more.dtype == y.dtype
                            and more.is_contiguous())
    if parts and H % 8 == 0 and H <= 8192 and (more is None or more.data_ptr() % 16 == 0):
        return PairSum(y, top, more)
    lib, hip = _lib()
    out = torch.empty(T, H, dtype=y.dtype, device=y.device)
    hip.check(lib.oa_moe_combine(hip.current_stream_ptr(), y.data_ptr(),
                                 more.data_ptr() if more is not None else None, out.data_ptr(),
                                 T, top, H), "oa_moe_combine")
    return out


def moe_sorted_wins(pairs: int, experts: int, fp8: bool, weights: int = 0) -> bool:
    """Sorted tiles against a weight stream per pair; weights is the size of one expert
    matrix, 0 if unknown. Us in graphs, both products, the sort and the sum, pairs / sorted.
    64 experts of 1408 x 2048, fp8: 6 pairs 22 / 28, 12 33 / 30, 24 53 / 44; bf16: 24 pairs
    77 / 77, 36 107 / 96. 128 of 768 x 2048, fp8: 24 36 / 38, 32 44 / 39; bf16: 40 73 / 71, 48
    87 / 84. 16 of 1024 x 2048, fp8: 12 24 / 25, 16 29 / 25; bf16: 12 34 / 37, 16 40 / 38. 8 of
    14336 x 4096, fp8: 2 pairs 83 / 98, 4 148 / 123; bf16: 4 193 / 217, 6 322 / 255. Small
    matrices are launches either way: 16 of 512 x 1024, fp8: 24 17 / 18, 32 20 / 18; bf16: 24
    19 / 21, 32 22 / 21."""
    heavy = 3 * weights * pairs >= 10 ** 8
    if fp8:
        return pairs >= max(32, experts // 4) or heavy and pairs >= max(4, experts // 6)
    return pairs >= max(32, 3 * experts // 8) or heavy and pairs >= max(6, experts // 2)


def _moe_ring_rows(pairs: int, experts: int, weights: int, fp8: bool) -> int:
    """Rows of a tile of moe_sorted_mlp, by the rows that an expert has on average; weights
    is the size of one expert matrix. The same bits with any of them.

    A narrow tile costs a strip read again for every further tile of its expert, a wide one
    LDS reads for rows that are not there. Both products in graphs, us with 16 / 32 / 64 rows.
    fp8, 64 experts of 1408 x 2048: 2 rows 83 / 84 / 97, 8 90 / 92 / 100, 16 112 / 95 / 105, 24
    134 / 102 / 107, 32 153 / 128 / 116; 8 of 14336 x 4096: 8 rows 216 / 219 / 295, 24 311 / 227 /
    298, 32 391 / 326 / 304. bf16: 2 rows 160 / 158 / 167, 8 181 / 183 / 188, 16 207 / 187 / 191,
    24 234 / 192 / 195, 32 270 / 218 / 202. Small matrices have too few strips to go round the
    CUs, so that narrow tiles pay for longer: 16 fp8 experts of 512 x 1024, 16 rows 13.4 / 15.0 /
    19.8, 32 15.7 / 15.5 / 20.6, 96 24.4 / 18.2 / 20.7, 192 39 / 30 / 25; bf16 96 rows 31 / 22 / 22.
    64 / 128 rows, bf16 (fp8 has no room for a second block of 128): 64 experts of 1408 x 2048,
    48 rows 213 / 239, 64 263 / 252, 192 429 / 404; 128 of 768 x 2048, 48 rows 242 / 255, 64 287 /
    286; 16 of 512 x 1024, 192 rows 27 / 34."""
    small = weights < 2 ** 20
    if pairs <= (16 if small else 8) * experts:
        return 16
    if pairs <= (96 if small else 24) * experts:
        return 32
    return 64 if small or fp8 or pairs < 64 * experts else 128


def _moe_lists(pairs: int, experts: int, weights: int, fp8: bool) -> Tuple[int, int, int]:
    """Rows of a tile, the most tiles, and the int32s of the sorted pairs' lists."""
    bm = _moe_ring_rows(pairs, experts, weights, fp8)
    max_tiles = pairs // bm + min(experts, pairs)
    return bm, max_tiles, 2 * experts + 2 + max_tiles + pairs


def _moe_list_ptrs(ints: torch.Tensor, experts: int, max_tiles: int) -> Tuple[int, int, int, int]:
    """Addresses of offsets and tile counts [E + 1], tiles' experts and the order in _moe_lists' ints."""
    at = ints.data_ptr()
    return (at, at + 4 * (experts + 1), at + 8 * (experts + 1), at + 4 * (2 * experts + 2 + max_tiles))


def moe_front(x: torch.Tensor, router_w: torch.Tensor, top: int, weights: int, fp8: bool,
              gate_up_w: Optional[torch.Tensor] = None, down_w: Optional[torch.Tensor] = None):
    """Routing of up to 16 tokens x [T, K] with its pairs sorted for moe_sorted_mlp, and a shared
    expert down(silu(gate x) * up x) beside it where its products are strips: (experts and weights as of
    moe_route, lists, the shared expert's rows or None), None where the kernels do not take it.
    weights: size of one expert matrix. Choice and sort are one block's launch, and with the shared
    expert two launches do for five (moe_grouped.hip; figures there)."""
    T, K = x.shape
    E = router_w.shape[0]
    if not (T <= 16 and E <= 256 and moe_route_ok(x, router_w, top)):
        return None
    lib, hip = _lib()
    stream, dev = hip.current_stream_ptr(), x.device
    beside = False
    if gate_up_w is not None and K == gate_up_w.shape[1]:
        H, I = down_w.shape
        if gate_up_w.shape[0] == 2 * I and _gateup_form(x, gate_up_w, I) == ("skinny", 1):
            mid = torch.empty(T, I, dtype=x.dtype, device=dev)
            beside = (_skinny_ok(mid, down_w) and not _ring_form(T, H, I)
                      and _skinny_form(T, H, I) == 1)
    idx = torch.empty(T, top, dtype=torch.int32, device=dev)
    wts = torch.empty(T, top, dtype=torch.float32, device=dev)
    scratch = torch.empty(lib.oa_moe_route_scratch(T, E, K), dtype=torch.float32, device=dev)
    bm, max_tiles, size = _moe_lists(T * top, E, weights, fp8)
    lists = torch.empty(size, dtype=torch.int32, device=dev)
    shared = torch.empty(T, H, dtype=x.dtype, device=dev) if beside else None
    up = (gate_up_w.data_ptr(), mid.data_ptr(), I) if beside else (None, None, 0)
    down = (mid.data_ptr(), down_w.data_ptr(), shared.data_ptr(), H, I) if beside else (None,) * 3 + (0, 0)
    hip.check(lib.oa_moe_front_up(stream, x.data_ptr(), router_w.data_ptr(), scratch.data_ptr(), T, E, K,
                                  *up), "oa_moe_front_up")
    hip.check(lib.oa_moe_front_down(stream, scratch.data_ptr(), idx.data_ptr(), wts.data_ptr(), T, E, K,
                                    top, bm, *_moe_list_ptrs(lists, E, max_tiles), *down),
              "oa_moe_front_down")
    return idx, wts, lists, shared


def moe_sorted_ok(x: torch.Tensor, w13: torch.Tensor, w2: torch.Tensor, act=None) -> bool:
    """Whether moe_sorted_mlp takes these experts: both products run over
    128-column steps, a gate strip holds 64 rows."""
    return (
        x.is_cuda and x.dtype == torch.bfloat16 and x.dim() == 2 and x.is_contiguous()
        and w13.device == w2.device == x.device
        and w13.is_contiguous() and w2.is_contiguous() and w13.dtype == w2.dtype
        and w13.dtype in (torch.bfloat16, torch.uint8) and _moe_act(act) is not None
        and x.shape[1] % 128 == 0 and w2.shape[2] % 128 == 0 and w13.shape[0] <= 1024
        and all(t.data_ptr() % 16 == 0 for t in (x, w13, w2))
    )


def moe_sorted_mlp(
    x: torch.Tensor,
    w13: torch.Tensor,
    w13_scale: Optional[torch.Tensor],
    w2: torch.Tensor,
    w2_scale: Optional[torch.Tensor],
    expert_ids: torch.Tensor,
    pair_weights: torch.Tensor,
    act=None,
    more: Union[torch.Tensor, PlaneSum, None] = None,
    parts: bool = False,
    lists: Optional[torch.Tensor] = None,
) -> Union[torch.Tensor, PairSum]:
    """Routed experts of a prompt-sized batch (GPU): out[t] = sum over token t's
    choices j of weight_tj * W2[e_tj] act(W13[e_tj] x_t), plus more[t] if given.
    x [T, H] bf16; expert_ids int32 and pair_weights float32 [T, top]; experts as
    in moe_grouped_mlp, bf16 or fp8 with row scales. Pairs are sorted by expert
    on the GPU and every expert's rows run as matrix-core tiles: no host sync,
    static shapes. With `parts` the sum may be left to the norm that follows. lists: the pairs
    sorted already (moe_front)."""
    T, H = x.shape
    top = expert_ids.shape[1]
    E, I = w13.shape[0], w2.shape[2]
    actk, limit, alpha = _moe_act(act)
    assert w13.shape[1] == (I if actk == 3 else 2 * I) and w13.shape[2] == H and w2.shape[1] == H
    assert expert_ids.dtype == torch.int32 and expert_ids.is_contiguous()
    assert pair_weights.dtype == torch.float32 and pair_weights.is_contiguous()
    assert expert_ids.shape == pair_weights.shape == (T, top)
    assert (w13.dtype == torch.uint8) == (w13_scale is not None) == (w2_scale is not None)
    P = T * top
    bm, max_tiles, size = _moe_lists(P, E, I * H, w13_scale is not None)
    lib, hip = _lib()
    stream, dev = hip.current_stream_ptr(), x.device
    if lists is None:
        ints = torch.empty(size, dtype=torch.int32, device=dev)
        ptrs = _moe_list_ptrs(ints, E, max_tiles)
        hip.check(lib.oa_moe_sort(stream, expert_ids.data_ptr(), P, E, bm, *ptrs), "oa_moe_sort")
    else:
        assert lists.shape == (size,) and lists.dtype == torch.int32 and lists.device == dev
        ptrs = _moe_list_ptrs(lists, E, max_tiles)
    mid = torch.empty(P, I, dtype=x.dtype, device=dev)
    y = torch.empty(P, H, dtype=x.dtype, device=dev)
    ptr = lambda t: t.data_ptr() if t is not None else None  # noqa: E731
    hip.check(lib.oa_moe_grouped(stream, x.data_ptr(), w13.data_ptr(), ptr(w13_scale), *ptrs, None,
                                 mid.data_ptr(), E, I, H, top, bm, max_tiles,
                                 2 if actk == 3 else 1, actk, limit, alpha), "oa_moe_grouped(up)")
    hip.check(lib.oa_moe_grouped(stream, mid.data_ptr(), w2.data_ptr(), ptr(w2_scale), *ptrs,
                                 pair_weights.data_ptr(), y.data_ptr(), E, H, I, top, bm, max_tiles,
                                 0, 0, 0.0, 0.0), "oa_moe_grouped(down)")
    return moe_combine(y, top, more, parts)


def moe_grouped_mlp(
    x: torch.Tensor,
    w13: torch.Tensor,
    w13_scale: Optional[torch.Tensor],
    w2: torch.Tensor,
    w2_scale: Optional[torch.Tensor],
    expert_ids: torch.Tensor,
    token_ids: torch.Tensor,
    pair_weights: torch.Tensor,
    i_local: int,
    fp8: bool,
    num_experts: int = 0,
    act=None,
) -> torch.Tensor:
    """Grouped MoE expert MLP (GPU decode path): one gateup launch + one down
    launch for ALL (token, expert) pairs of a layer — no per-expert loop, no
    host sync, shape-static (graph-capturable). Returns y [P, H] to be
    index_add-ed into the output by token.

    Two kernel families, both static-shaped:
      * pair-major (default): one block column per PAIR; the expert's weight
        rows stream once per pair — lowest latency at tiny P
      * expert-major (P > OPSAGENT_MOE_EMAJ_MIN_P, needs num_experts): one
        block column per EXPERT; weights stream once per GROUP of 8 matched
        pairs, cutting the weight traffic up to 8x at big decode batches
    act: None / "silu", or ("clamp_swish", limit, alpha) for the clamped gate
    g' = min(g, limit), u' = clamp(u, -limit, limit), g' sigmoid(alpha g') (u' + 1),
    or "relu2" for UNGATED experts: w13 is [E, I, K] (up rows alone) and the
    middle activation is relu(up x)^2.
    """
    actk, limit, alpha = _moe_act(act)
    assert actk != 3 or w13.shape[1] == i_local
    assert x.is_cuda and x.dtype == torch.bfloat16 and x.is_contiguous()
    # stride-0 expand views have a data_ptr that covers ONE element — the
    # kernels index these linearly, so contiguity is load-bearing
    assert expert_ids.is_contiguous() and expert_ids.dtype == torch.int32
    assert token_ids.is_contiguous() and token_ids.dtype == torch.int32
    assert pair_weights.is_contiguous() and pair_weights.dtype == torch.float32
    lib, hip = _lib()
    P = expert_ids.shape[0]
    K = x.shape[-1]
    H = w2.shape[1]
    emaj_min = int(os.environ.get("OPSAGENT_MOE_EMAJ_MIN_P", "64"))
    use_emaj = num_experts > 0 and P >= emaj_min and P <= 2048
    mid = torch.empty(P, i_local, dtype=x.dtype, device=x.device)
    if use_emaj:
        rc = lib.oa_moe_gateup_emaj_act(
            hip.current_stream_ptr(), x.data_ptr(), w13.data_ptr(),
            w13_scale.data_ptr() if fp8 else None,
            expert_ids.data_ptr(), token_ids.data_ptr(), mid.data_ptr(),
            P, num_experts, i_local, K, 1 if fp8 else 0, actk, limit, alpha,
        )
        hip.check(rc, "oa_moe_gateup_emaj")
    else:
        rc = lib.oa_moe_gateup_act(
            hip.current_stream_ptr(), x.data_ptr(), w13.data_ptr(),
            w13_scale.data_ptr() if fp8 else None,
            expert_ids.data_ptr(), token_ids.data_ptr(), mid.data_ptr(),
            P, i_local, K, 1 if fp8 else 0, actk, limit, alpha,
        )
        hip.check(rc, "oa_moe_gateup")
    y = torch.empty(P, H, dtype=x.dtype, device=x.device)
    if use_emaj:
        rc = lib.oa_moe_down_emaj(
            hip.current_stream_ptr(), mid.data_ptr(), w2.data_ptr(),
            w2_scale.data_ptr() if fp8 else None,
            expert_ids.data_ptr(), pair_weights.data_ptr(), y.data_ptr(),
            P, num_experts, H, i_local, 1 if fp8 else 0,
        )
        hip.check(rc, "oa_moe_down_emaj")
    else:
        rc = lib.oa_moe_down(
            hip.current_stream_ptr(), mid.data_ptr(), w2.data_ptr(),
            w2_scale.data_ptr() if fp8 else None,
            expert_ids.data_ptr(), pair_weights.data_ptr(), y.data_ptr(),
            P, H, i_local, 1 if fp8 else 0,
        )
        hip.check(rc, "oa_moe_down")
    return y


def rope_kv_fused(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    cos: torch.Tensor,
    sin: torch.Tensor,
    positions: torch.Tensor,
    slot_mapping: torch.Tensor,
) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """Fused RoPE(q,k in place) + paged KV write of k,v. Returns (q, k, v).

    q/k/v may be head-slices of ONE fused [T, (Hq+2Hk)*D] qkv buffer sharing
    a token stride — no .contiguous() copies (those cost ~5.8 ms per 736-token
    prefill). Requires contiguous (head, dim) inner layout and equal token
    strides across q/k/v."""
    if not _is_gpu(q):
        q2, k2 = torch_ref.rope_apply(q, k, cos, sin, positions)
        torch_ref.kv_cache_write(k_cache, v_cache, k2, v, slot_mapping.long())
        return q2, k2, v
    T, Hq, D = q.shape
    Hk = k.shape[1]
    assert q.dtype == torch.bfloat16
    assert q.stride(2) == 1 and q.stride(1) == D, "q heads must be inner-contiguous"
    assert k.stride(2) == 1 and k.stride(1) == D and v.stride(2) == 1 and v.stride(1) == D
    assert cos.dtype == torch.float32
    assert positions.dtype == torch.int32 and slot_mapping.dtype == torch.int32
    lib, hip = _lib()
    rc = lib.oa_rope_kv(
        hip.current_stream_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
        k_cache.data_ptr(), v_cache.data_ptr(), cos.data_ptr(), sin.data_ptr(),
        positions.data_ptr(), slot_mapping.data_ptr(), T, Hq, Hk, D,
        q.stride(0), k.stride(0), v.stride(0),
    )
    hip.check(rc, "oa_rope_kv")
    return q, k, v


def rope_kv_parts(parts: PlaneSum, Hq: int, Hk: int, D: int, k_cache: torch.Tensor,
                  v_cache: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
                  positions: torch.Tensor, slot_mapping: torch.Tensor
                  ) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """rope_kv_fused of a q | k | v product that is not added up yet (linear_parts)."""
    planes = parts.planes
    n, T, width = planes.shape
    assert width == (Hq + 2 * Hk) * D and planes.is_contiguous() and planes.dtype == torch.float32
    assert cos.dtype == torch.float32 and k_cache.dtype == v_cache.dtype == torch.bfloat16
    assert positions.dtype == torch.int32 and slot_mapping.dtype == torch.int32
    lib, hip = _lib()
    qkv = torch.empty(T, width, dtype=k_cache.dtype, device=planes.device)
    hip.check(lib.oa_rope_kv_parts(
        hip.current_stream_ptr(), planes.data_ptr(), n, qkv.data_ptr(), k_cache.data_ptr(),
        v_cache.data_ptr(), cos.data_ptr(), sin.data_ptr(), positions.data_ptr(),
        slot_mapping.data_ptr(), T, Hq, Hk, D), "oa_rope_kv_parts")
    q, k, v = qkv.split([Hq * D, Hk * D, Hk * D], dim=-1)
    return q.view(T, Hq, D), k.view(T, Hk, D), v.view(T, Hk, D)


def gateup_silu(x: torch.Tensor, gate_up_w: torch.Tensor, i_local: int) -> torch.Tensor:
    """silu(x @ gate^T) * (x @ up^T) with gate_up_w = [gate; up] rows.

    GPU decode: one fused HIP kernel, no [*, 2I] intermediate, where gateup_fused
    says so. Otherwise: library GEMM + the silu_mul kernel."""
    form = _gateup_form(x, gate_up_w, i_local)
    if form:
        return gateup_act(x, gate_up_w, i_local, form=form)
    return silu_halves(linear(x, gate_up_w), i_local)


def _gateup_form(x: torch.Tensor, gate_up_w: torch.Tensor, i_local: int):
    """What takes this product in one launch, None if nothing does: ("ring", plan) and
    ("skinny", form), the transfer ring and the skinny matrix-core product where they win,
    ("tile", plan), the tile product of more than 128 rows;
    ("staged", None), the VALU GEMV up to two rows and the staged matrix-core GEMV for what
    3 to 8 rows are left."""
    K = x.shape[-1]
    M = x.numel() // K
    if not (x.is_cuda and x.dtype == torch.bfloat16 and K % 8 == 0 and x.is_contiguous()
            and gate_up_w.is_contiguous()):
        return None
    if M > 128 and _skinny_ok(x, gate_up_w) and gate_up_w.shape[0] == 2 * i_local:
        plan = _tile_choice(M, i_local, K, gateup=True)
        return None if plan is None else ("tile", plan)
    if 1 < M <= 128 and _skinny_ok(x, gate_up_w) and gate_up_w.shape[0] == 2 * i_local:
        plan = _ring_form(M, i_local, K, gateup=True)
        if plan:
            return "ring", plan
        form = _skinny_form(M, i_local, K, gateup=True)
        if form:
            return "skinny", form
    return ("staged", None) if _gemv_m_ok(M) or _bf16_mfma_ok(M, K, gateup=True) else None


def gateup_fused(x: torch.Tensor, gate_up_w: torch.Tensor, i_local: int) -> bool:
    """Whether gateup_act takes this product in one launch."""
    return _gateup_form(x, gate_up_w, i_local) is not None


def gateup_act(x: torch.Tensor, gate_up_w: torch.Tensor, i_local: int,
               act: str = "silu", form=None) -> torch.Tensor:
    """act(x @ gate^T) * (x @ up^T), act "silu" | "gelu_tanh", for decode-sized
    bf16 batches that gateup_fused names: one launch. form: _gateup_form's answer, where the
    caller has asked it."""
    from opsagent_amd.ops import hip_lib

    M = x.numel() // x.shape[-1]
    assert x.is_cuda and x.dtype == torch.bfloat16 and x.is_contiguous()
    assert act in ("silu", "gelu_tanh")
    kind, plan = form or _gateup_form(x, gate_up_w, i_local) or ("staged", None)
    if kind == "ring":
        return _ring(x, gate_up_w, plan, act=1 + int(act == "gelu_tanh"))
    if kind == "skinny":
        return _skinny(x, gate_up_w, plan, gateup=True, act=int(act == "gelu_tanh"))
    if kind == "tile":
        return _tile(x, gate_up_w, plan, act=1 + int(act == "gelu_tanh"))
    lib = hip_lib.get_lib()
    out = torch.empty(*x.shape[:-1], i_local, dtype=x.dtype, device=x.device)
    rc = lib.oa_gemv_gateup_act(
        hip_lib.current_stream_ptr(), x.data_ptr(), gate_up_w.data_ptr(),
        out.data_ptr(), M, i_local, x.shape[-1], int(act == "gelu_tanh"),
    )
    hip_lib.check(rc, "oa_gemv_gateup_act")
    return out


def kv_cache_write(
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    slot_mapping: torch.Tensor,
) -> None:
    """k/v: [T, Hk, D]; caches [num_blocks, block_size, Hk, D]; slots int32 [T]."""
    if not _is_gpu(k):
        torch_ref.kv_cache_write(k_cache, v_cache, k, v, slot_mapping.long())
        return
    assert k.dtype == torch.bfloat16 and k.is_contiguous() and v.is_contiguous()
    assert slot_mapping.dtype == torch.int32
    lib, hip = _lib()
    T, Hk, D = k.shape
    rc = lib.oa_kv_write(
        hip.current_stream_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
        k.data_ptr(), v.data_ptr(), slot_mapping.data_ptr(), T, Hk, D,
    )
    hip.check(rc, "oa_kv_write")


def _prefill_splits(B: int, Hq: int, Hk: int, Sq: int, Skv: int) -> Tuple[int, bool]:
    """(key splits, merged form) of prefill attention; (1, False): not split.

    Few queries over many keys leave most CUs idle. Up to 128 queries: blocks of a
    head, from three tiles of 128 keys on (32 heads on 8, us before / split: 3 over
    300 14.4 / 11.1, 16 over 2000 64 / 21, 77 over 1264 40.4 / 20.9), more tiles where
    the rows that leave sums of their own, heads times queries, are many (64 x 77, 3 tiles
    16.4 / 17.3, 4 20.0 / 19.6; 80 x 77, 4 20.3 / 21.0, 5 23.9 / 23.3; 128 x 128, 5 28.7 /
    31.8, 6 33.1 / 32.0) or two splits share three (128 x 16 16.0 / 16.9). More: blocks
    of a key head, from twelve tiles on (300 over 4000 142 / 54, 1024 over 5000 171 /
    116; 1024 over 1024 would take 44 instead of 38.5)."""
    if Hk < 1 or Hq % Hk:
        return 1, False
    tiles = (Skv + 127) // 128
    if Sq <= 128:
        rows, splits = B * Hq * Sq, max(1, min(tiles, 256 // max(1, B * Hq)))
        least = 6 if rows > 8192 else 5 if rows > 5200 else 4 if rows > 3200 or splits < 3 else 3
        return (splits if tiles >= least else 1), False
    group = Hq // Hk
    if group not in (2, 4, 8) or tiles < 12:
        return 1, False
    blocks = -(-Sq // (256 // group)) * B * Hk
    return max(1, min(tiles, 256 // max(1, blocks))), True


@functools.lru_cache(maxsize=4096)
def _prefill_plan(
    B: int, Hq: int, Hk: int, Sq: int, Skv: int, steady: bool = False, scaled: bool = False
) -> Tuple[int, int]:
    """(key splits, form) of prefill attention: form 0 in key groups, 1 merged, 2 steady, which alone
    takes the maxima of scaled scores (scaled).

    What :func:`_prefill_splits` splits, the steady form as it says; the others where that is
    faster than key groups within a block, which halve and quarter a chain of tiles without
    sums in memory. Up to 128 queries by the estimates below, us: over 260 sizes (4 to 128
    heads, 2 to 128 queries, 3 to 24 tiles) 0.2 per cent from the better of the two on average
    and 12 at the most (4 heads, 128 queries, 3 tiles, not split / split: 11.8 / 13.2; both
    sides: 80 heads, 128 queries, 6 tiles 18.2 / 25.8, 4 heads, 16 queries, 11 tiles 22.3 /
    12.2). More queries: where few splits fill the chip, from as many tiles as make up for the
    sums that they leave, lines drawn with keys that the caches hold. Not split / split, and with
    0.3 GB of keys in turn, 32 heads on 8 or 16 on 4: in two, 1000 queries of 32 heads and 50 and 64
    tiles 134 / 139, 177 / 168 (163 / 147, 207 / 180); in three, 520 of 32, 16 and 20 tiles 43 / 45, 52 / 49
    (47 / 46, 57 / 49); in four, 400 of 32, 24 and 28 46 / 45, 51 / 50 (57 / 47, 65 / 51), 1000 of 16, 28
    and 34 52 / 54, 62 / 61 (65 / 53, 78 / 60); in five, 700 of 16, 16, 18 and 20 32 / 37, 35 / 38, 38 / 37
    (41 / 38, 44 / 38, 48 / 38); in six, 300 of 32, 12, 16 and 20 26 / 29, 32 / 33, 38 / 37 (31 / 29, 40 / 33,
    50 / 39). Keys from memory would draw them up to ten tiles, 15 per cent of a launch, lower."""
    splits, merged = _prefill_splits(B, Hq, Hk, Sq, Skv)
    if scaled:
        return splits, 2
    if steady or splits == 1:
        return splits, 1 if merged else 2 * steady
    tiles = (Skv + 127) // 128
    if merged:
        least = (0, 0, 64, 20, 28, 18, 16)
        worth = splits >= len(least) or tiles >= least[splits]
    else:
        sums = B * Hq * Sq * splits * 520e-6          # MB
        chain = (2.0 if Sq <= 64 else 2.6) * -(-tiles // splits)
        worth = chain + 6.0 + 0.6 * sums < 1.85 * tiles + 4.0
    return (splits if worth else 1), int(merged)


def _rows_in_place(k: torch.Tensor, v: torch.Tensor, slots: torch.Tensor, D: int) -> bool:
    """Whether the prefill kernel may read rows ``slots`` of k and v [rows, Hk, D] where they lie: a
    list of int64 beside them, heads side by side, rows from 16 bytes to 16 bytes. Everything else
    that an index of a tensor may be is gathered."""
    steps = k.stride()
    return (len(steps) == 3 and steps[1:] == (D, 1) and 0 < steps[0] < 2 ** 31 and steps[0] % 8 == 0
            and v.stride() == steps and v.shape == k.shape and 0 < k.shape[0] < 2 ** 31
            and (k.data_ptr() | v.data_ptr()) % 16 == 0
            and slots.dtype == torch.int64 and slots.dim() == 1 and slots.is_contiguous()
            and slots.get_device() == k.get_device() == v.get_device())


def attention_prefill(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    scale: Optional[float] = None,
    causal: bool = True,
    steady: bool = False,
    slots: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """q [B, Sq, Hq, D]; k, v [B, Skv, Hk, D] (token-major layouts; the CPU
    reference uses [B, H, S, D], so the dispatch transposes for it). ``steady``: a row's keys
    added up in the one order that callers with 8-bit activations are held to: any other
    rounding of a weight moves some of those to the next 8-bit value. ``slots``: [Skv],
    key i of the one sequence is row slots[i] of the caches k, v [rows, Hk, D], counted from the
    end below 0; the kernel reads them where they lie (us, two gathers and attention / here, 32 heads
    on 8: 77 queries of 1264 keys 20.6 / 15.3, 800 of 1056 33.9 / 29.1, 2048 of 6144 215 / 204; whole
    prompts of 5 to 2048 tokens behind 100 to 6000 0.90 to 1.0 of the time with gathers, but 16 heads on
    4 and 1500 tokens or more behind 1800 1.007, 1500 behind 6000 1.02), and takes the last
    row for a slot outside the caches (by its low 32 bits), where a gather has no answer."""
    if slots is not None and not (_is_gpu(q) and _rows_in_place(k, v, slots, q.shape[-1])):
        k, v, slots = k[slots], v[slots], None
        k, v = k.unsqueeze(0), v.unsqueeze(0)
    if not _is_gpu(q):
        out = torch_ref.attention_prefill(
            q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2), scale, causal
        )
        return out.transpose(1, 2).contiguous()
    assert causal, "GPU prefill kernel is causal-only"
    assert q.dtype == torch.bfloat16
    B, Sq, Hq, D = q.shape
    if slots is not None:
        assert B == 1
        Skv, Hk, at, rows = slots.shape[0], k.shape[1], slots.data_ptr(), k.shape[0]
    else:
        Skv, Hk, at, rows = k.shape[1], k.shape[2], None, 0
    k_step, v_step = k.stride(-3), v.stride(-3)
    for t, name in ((q, "q"), (k, "k"), (v, "v")) if slots is None else ((q, "q"),):
        assert t.stride(3) == 1 and t.stride(2) == D, f"{name} heads must be inner-contiguous"
        assert t.shape[0] == 1 or t.stride(0) == t.shape[1] * t.stride(1), f"{name} batch stride"
    scale = scale if scale is not None else D ** -0.5
    lib, hip = _lib()
    out = torch.empty(B, Sq, Hq, D, dtype=q.dtype, device=q.device)
    # where a larger score is no larger weight, maxima before the scale would not bound the weights
    splits, form = _prefill_plan(B, Hq, Hk, Sq, Skv, steady, not scale > 0.0)
    if splits > 1 and D == 128 and "OPSAGENT_PREFILL_VARIANT" not in os.environ:
        part = torch.empty(splits, B, Sq, Hq, D + 2, dtype=torch.float32, device=q.device)
        sums = splits * B * Sq * Hq * D * 4
        rc = lib.oa_attention_prefill_split(
            hip.current_stream_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
            out.data_ptr(), part.data_ptr(), part.data_ptr() + sums, B, Hq, Hk, Sq, Skv, D,
            scale, q.stride(1), k_step, v_step, splits, form, at, rows,
        )
        hip.check(rc, "oa_attention_prefill_split")
        return out
    rc = lib.oa_attention_prefill(
        hip.current_stream_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
        out.data_ptr(), B, Hq, Hk, Sq, Skv, D, scale,
        q.stride(1), k_step, v_step, int(steady), at, rows,
    )
    hip.check(rc, "oa_attention_prefill")
    return out


def decode_nsplit(batch: int, n_kv_heads: int, max_len: int) -> int:
    """The most splits of a sequence's keys: blocks for the 256 CUs, a couple each. Target
    512, not more: every split leaves a partial result that the combine reads again.
    The kernel gives a split at least 64 keys (16 per wave), more for larger launches
    (decode_chunk in attention_decode.hip), so short sequences use fewer."""
    tgt_blocks = int(os.environ.get("OPSAGENT_DECODE_NSPLIT_TARGET", "512"))
    target = max(1, tgt_blocks // max(1, batch * n_kv_heads))
    return int(max(1, min(target, (max_len + 63) // 64)))


def attention_decode_paged(
    q: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    block_table: torch.Tensor,
    seq_lens: torch.Tensor,
    scale: Optional[float] = None,
    workspace: Optional[Tuple[torch.Tensor, ...]] = None,
    nsplit: Optional[int] = None,
    fused_combine: bool = False,
) -> torch.Tensor:
    """q [B, Hq, D]; caches [num_blocks, block_size, Hk, D]; out [B, Hq, D].

    fused_combine folds the split reduction into the attention launch via the
    in-launch G16 release/acquire hand-off (one kernel + a memset node
    instead of two kernels per layer). Measured on MI355X it is ~0.4 ms/step
    SLOWER than the two-kernel form at 8B decode (the single last-arriving
    block serializes a reduction the combine kernel spreads over B*Hq blocks)
    — kept as a correct, tested option; default off."""
    if not _is_gpu(q):
        return torch_ref.attention_decode_paged(q, k_cache, v_cache, block_table, seq_lens, scale)
    assert q.dtype == torch.bfloat16
    assert q.stride(2) == 1 and q.stride(1) == q.shape[2], "q heads must be inner-contiguous"
    assert block_table.dtype == torch.int32 and seq_lens.dtype == torch.int32
    B, Hq, D = q.shape
    nb, block_size, Hk, _ = k_cache.shape
    G = Hq // Hk
    scale = scale if scale is not None else D ** -0.5
    if nsplit is None:
        nsplit = decode_nsplit(B, Hk, int(block_table.shape[1] * block_size))
    if workspace is None:
        o_part = torch.empty(B * Hk * nsplit, G, D, dtype=torch.float32, device=q.device)
        ml_part = torch.empty(B * Hk * nsplit, G, 2, dtype=torch.float32, device=q.device)
        cnt_ws = torch.empty(B * Hk, dtype=torch.int32, device=q.device)
    else:
        o_part, ml_part, cnt_ws = workspace
    lib, hip = _lib()
    out = torch.empty(B, Hq, D, dtype=q.dtype, device=q.device)
    rc = lib.oa_attention_decode(
        hip.current_stream_ptr(), q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
        block_table.data_ptr(), seq_lens.data_ptr(), o_part.data_ptr(),
        ml_part.data_ptr(), cnt_ws.data_ptr(), out.data_ptr(), B, Hq, Hk, D,
        block_table.shape[1], block_size, nsplit, scale, q.stride(0),
        1 if fused_combine else 0,
    )
    hip.check(rc, "oa_attention_decode")
    return out


def _bf16_prenorm() -> bool:
    """OPSAGENT_BF16_PRENORM=1: at M=1 run rmsnorm as its own pass and the
    PLAIN bf16 gemv (A/B knob mirroring the fp8 M=1 prenorm win)."""
    return os.environ.get("OPSAGENT_BF16_PRENORM", "0") == "1"


def _fp8_mfma_ok(M: int, K: int, gateup: bool = False) -> bool:
    """Mirror of fp8_moe.hip's gemv_fp8_use_mfma for the M 9..16 range
    (the VALU kernels have no 9-11/13-15 instantiations — those batch
    sizes are only reachable through the MFMA stream)."""
    # unlike bf16 (whose M>8 alternative is a decent hipBLASLt skinny
    # kernel), fp8's M 9..16 alternative is the 128-row tile GEMM on an
    # underfilled grid — in-engine c16 fp8: MFMA gemv 8.93 t/s vs 7.40
    # through the GEMM. Keep the full M 2..16 range here.
    # (The sizes first: a look at the environment is a microsecond of the host.)
    if not 2 <= M <= 16 or M * K > 131072 or K % 512 != 0 or (K // 512) % (4 if gateup else 8) != 0:
        return False
    return os.environ.get("OPSAGENT_FP8_GEMV_MFMA", "") != "0"


def _fp8_gemv_ok(x: torch.Tensor) -> bool:
    M = x.numel() // x.shape[-1]
    K = x.shape[-1]
    return (
        x.is_cuda and x.dtype == torch.bfloat16
        and (M <= 8 or _fp8_mfma_ok(M, K))
        and K % 16 == 0 and x.is_contiguous()
    )


def _fp8_gemv1_ok(x: torch.Tensor, N: int) -> bool:
    """Mirror of fp8_moe.hip's gemv1_fp8_ok for one row x and N weight rows."""
    return x.shape[-1] % 2048 == 0 and x.shape[-1] <= 16384 and N % 2 == 0 and x.data_ptr() % 16 == 0


def linear_norm_fp8(
    x: torch.Tensor, norm_w: torch.Tensor, eps: float,
    w8: torch.Tensor, w_scale: torch.Tensor,
) -> torch.Tensor:
    """rmsnorm(x) @ dequant(W8)^T with the norm fused into the fp8 GEMV
    prologue (fp8 decode fast path): at M=1 where the one-row kernel takes the
    shape (once per block; _fp8_gemv1_ok). Elsewhere at M=1 the VALU stream
    kernel would run the norm per ELEMENT inside the weight loop (measured 2.7 vs
    5.1 TB/s on the 70B qkv shape), so a rmsnorm pass + the plain kernel wins;
    the M>=2 MFMA path fuses the norm into its one-shot x-quant instead."""
    if not _fp8_gemv_ok(x):
        return linear_fp8(rms_norm(x, norm_w, eps), w8, w_scale)
    lib, hip = _lib()
    M = x.numel() // x.shape[-1]
    if M == 1 and not _fp8_gemv1_ok(x, w8.shape[0]):
        return linear_fp8(rms_norm(x, norm_w, eps), w8, w_scale)
    N, K4 = w8.shape[0], x.shape[-1]
    out = torch.empty(*x.shape[:-1], N, dtype=x.dtype, device=x.device)
    rc = lib.oa_gemv_fp8_ex(
        hip.current_stream_ptr(), x.data_ptr(), w8.data_ptr(),
        w_scale.data_ptr(), out.data_ptr(), norm_w.data_ptr(), None,
        M, N, K4, eps, 1,
    )
    hip.check(rc, "oa_gemv_fp8_ex(norm)")
    return out


def linear_addres_fp8(
    x: torch.Tensor, w8: torch.Tensor, w_scale: torch.Tensor,
    res: torch.Tensor,
) -> torch.Tensor:
    """x @ dequant(W8)^T + res (fp8 residual-producing projection)."""
    if not (_fp8_gemv_ok(x) and res.is_contiguous()):
        return linear_fp8(x, w8, w_scale) + res
    lib, hip = _lib()
    M = x.numel() // x.shape[-1]
    N = w8.shape[0]
    out = torch.empty(*x.shape[:-1], N, dtype=x.dtype, device=x.device)
    rc = lib.oa_gemv_fp8_ex(
        hip.current_stream_ptr(), x.data_ptr(), w8.data_ptr(),
        w_scale.data_ptr(), out.data_ptr(), None, res.data_ptr(),
        M, N, x.shape[-1], 0.0, 2,
    )
    hip.check(rc, "oa_gemv_fp8_ex(addres)")
    return out


def gateup_silu_fp8(
    x: torch.Tensor, w8: torch.Tensor, w_scale: torch.Tensor, i_local: int,
    norm_w: Optional[torch.Tensor] = None, eps: float = 0.0,
) -> torch.Tensor:
    """silu(x @ gate8^T) * (x @ up8^T) with fp8 [gate; up] weights; optional
    fused rmsnorm prologue. Falls back to linear_fp8 + silu_mul."""
    use_norm = norm_w is not None
    _Mgu = x.numel() // x.shape[-1]
    if not _fp8_gemv_ok(x) or (
        _Mgu in (5, 7) and not _fp8_mfma_ok(_Mgu, x.shape[-1], gateup=True)
    ):
        xin = rms_norm(x, norm_w, eps) if use_norm else x
        return silu_halves(linear_fp8(xin, w8, w_scale), i_local)
    lib, hip = _lib()
    M = x.numel() // x.shape[-1]
    if use_norm and M == 1 and not _fp8_gemv1_ok(x, 2):  # see linear_norm_fp8
        x = rms_norm(x, norm_w, eps)
        norm_w = None
        use_norm = False
    out = torch.empty(*x.shape[:-1], i_local, dtype=x.dtype, device=x.device)
    rc = lib.oa_gemv_gateup_fp8(
        hip.current_stream_ptr(), x.data_ptr(), w8.data_ptr(),
        w_scale.data_ptr(), out.data_ptr(),
        norm_w.data_ptr() if use_norm else None,
        M, i_local, x.shape[-1], eps, 1 if use_norm else 0,
    )
    hip.check(rc, "oa_gemv_gateup_fp8")
    return out


def attention_decode_rope(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    block_table: torch.Tensor,
    seq_lens: torch.Tensor,
    cos: torch.Tensor,
    sin: torch.Tensor,
    slots: torch.Tensor,
    scale: Optional[float] = None,
    workspace: Optional[Tuple[torch.Tensor, ...]] = None,
    nsplit: Optional[int] = None,
) -> torch.Tensor:
    """Fully-fused decode attention: RoPE(q, k) + paged-KV scatter + split-K
    attention + combine in two launches, replacing the separate rope_kv
    launch per layer. q [B, Hq, D], k/v [B, Hk, D] are the RAW (un-roped)
    GEMV outputs (head-slice views of the fused qkv buffer are fine —
    per-tensor token strides); slots [B] int32 gives the new token's cache
    slot. CPU path: rope_kv then the torch reference attention."""
    if not _is_gpu(q):
        positions = (seq_lens.to(torch.int64) - 1).to(torch.int32)
        q2, k2 = torch_ref.rope_apply(q, k, cos, sin, positions)
        torch_ref.kv_cache_write(k_cache, v_cache, k2, v, slots.long())
        return torch_ref.attention_decode_paged(
            q2, k_cache, v_cache, block_table, seq_lens, scale
        )
    assert q.dtype == torch.bfloat16
    assert q.stride(2) == 1 and q.stride(1) == q.shape[2]
    assert k.stride(2) == 1 and k.stride(1) == k.shape[2]
    assert v.stride(2) == 1 and v.stride(1) == v.shape[2]
    assert block_table.dtype == torch.int32 and seq_lens.dtype == torch.int32
    assert slots.dtype == torch.int32
    B, Hq, D = q.shape
    nb, block_size, Hk, _ = k_cache.shape
    G = Hq // Hk
    scale = scale if scale is not None else D ** -0.5
    if nsplit is None:
        nsplit = decode_nsplit(B, Hk, int(block_table.shape[1] * block_size))
    if workspace is None:
        o_part = torch.empty(B * Hk * nsplit, G, D, dtype=torch.float32, device=q.device)
        ml_part = torch.empty(B * Hk * nsplit, G, 2, dtype=torch.float32, device=q.device)
    else:
        o_part, ml_part = workspace[0], workspace[1]
    lib, hip = _lib()
    out = torch.empty(B, Hq, D, dtype=q.dtype, device=q.device)
    rc = lib.oa_attention_decode_rope(
        hip.current_stream_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
        k_cache.data_ptr(), v_cache.data_ptr(), block_table.data_ptr(),
        seq_lens.data_ptr(), cos.data_ptr(), sin.data_ptr(), slots.data_ptr(),
        o_part.data_ptr(), ml_part.data_ptr(), out.data_ptr(), B, Hq, Hk, D,
        block_table.shape[1], block_size, nsplit, scale, q.stride(0),
        k.stride(0), v.stride(0),
    )
    hip.check(rc, "oa_attention_decode_rope")
    return out


def decode_takes_parts(batch: int, Hq: int, Hk: int, D: int) -> bool:
    """Whether attention_decode_parts takes the step: up to 64 (sequence, key head) pairs."""
    return bool(_lib()[0].oa_attention_decode_takes_parts(batch, Hq, Hk, D))


def attention_decode_parts(
    parts: PlaneSum, Hq: int, Hk: int, D: int, k_cache: torch.Tensor, v_cache: torch.Tensor,
    block_table: torch.Tensor, seq_lens: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
    slots: torch.Tensor, scale: float,
    workspace: Optional[Tuple[torch.Tensor, ...]] = None, nsplit: Optional[int] = None,
) -> torch.Tensor:
    """attention_decode_rope of a q | k | v product that is not added up yet (linear_parts), where
    decode_takes_parts says so."""
    planes = parts.planes
    n, B, width = planes.shape
    block_size, G = k_cache.shape[1], Hq // Hk
    assert width == (Hq + 2 * Hk) * D and planes.is_contiguous() and planes.dtype == torch.float32
    assert k_cache.shape[2:] == v_cache.shape[2:] == (Hk, D) and cos.dtype == torch.float32
    assert block_table.dtype == seq_lens.dtype == slots.dtype == torch.int32
    if nsplit is None:
        nsplit = decode_nsplit(B, Hk, int(block_table.shape[1] * block_size))
    if workspace is None:
        o_part = torch.empty(B * Hk * nsplit, G, D, dtype=torch.float32, device=planes.device)
        ml_part = torch.empty(B * Hk * nsplit, G, 2, dtype=torch.float32, device=planes.device)
    else:
        o_part, ml_part = workspace[0], workspace[1]
    lib, hip = _lib()
    out = torch.empty(B, Hq, D, dtype=k_cache.dtype, device=planes.device)
    hip.check(lib.oa_attention_decode_parts(
        hip.current_stream_ptr(), planes.data_ptr(), n, k_cache.data_ptr(), v_cache.data_ptr(),
        block_table.data_ptr(), seq_lens.data_ptr(), cos.data_ptr(), sin.data_ptr(), slots.data_ptr(),
        o_part.data_ptr(), ml_part.data_ptr(), out.data_ptr(), B, Hq, Hk, D, block_table.shape[1],
        block_size, nsplit, scale), "oa_attention_decode_parts")
    return out


def greedy_sample_masked(
    logits: torch.Tensor, mask_bits: Optional[torch.Tensor]
) -> torch.Tensor:
    """logits [B, V] bf16 (GPU) / any float (CPU); mask_bits uint32-packed
    [B, ceil(V/32)] on GPU, bool [B, V] on CPU. Returns int32/int64 [B]."""
    if not _is_gpu(logits):
        return torch_ref.greedy_sample_masked(logits, mask_bits)
    lib, hip = _lib()
    B, V = logits.shape
    out = torch.empty(B, dtype=torch.int32, device=logits.device)
    if logits.dtype == torch.float32:
        # float32 rows of any width (hybrid models' soft-capped logits)
        assert logits.is_contiguous()
        if mask_bits is not None:
            assert mask_bits.dtype == torch.int32 and mask_bits.is_contiguous()
        ws32 = torch.empty(B * 16 * 2, dtype=torch.int32, device=logits.device)
        rc = lib.oa_masked_argmax_f32(
            hip.current_stream_ptr(), logits.data_ptr(),
            mask_bits.data_ptr() if mask_bits is not None else None,
            ws32.data_ptr(), out.data_ptr(), B, V,
        )
        hip.check(rc, "oa_masked_argmax_f32")
        return out
    assert logits.dtype == torch.bfloat16 and logits.is_contiguous()
    mask_ptr = mask_bits.data_ptr() if mask_bits is not None else None
    if mask_bits is not None:
        assert mask_bits.dtype == torch.int32 and mask_bits.is_contiguous()
    rc = lib.oa_masked_argmax(
        hip.current_stream_ptr(), logits.data_ptr(), mask_ptr, out.data_ptr(), B, V,
    )
    hip.check(rc, "oa_masked_argmax")
    return out


def token_logprobs(logits: torch.Tensor, tokens: torch.Tensor, top: int):
    """Log-softmax of logits [B, V] at tokens [B], and of the `top` most likely tokens of
    each row: (logprobs [B], indices [B, top] int32, their logprobs [B, top]) on the host,
    float32. Equal values go by index; NaN where a token is none (negative)."""
    B, V = logits.shape
    top = max(0, min(top, V))
    if not (_is_gpu(logits) and logits.dtype in (torch.bfloat16, torch.float32)
            and logits.stride(1) == 1 and 0 < B <= 65535 and top <= 32):
        lp = torch.log_softmax(logits.float(), dim=-1)
        t = tokens.long().to(lp.device)
        at = torch.where((t >= 0) & (t < V), lp.gather(1, t.clamp(0, V - 1)[:, None])[:, 0], torch.nan)
        val, idx = torch.topk(lp, top)
        return at.cpu(), idx.to(torch.int32).cpu(), val.cpu()
    lib, hip = _lib()
    assert tokens.dtype == torch.int32 and tokens.is_contiguous() and tokens.shape == (B,)
    ws = torch.empty(B * -(-V // 1024) * (top + 1), dtype=torch.int64, device=logits.device)
    out = torch.empty(B, 1 + 2 * top, dtype=torch.int32, device=logits.device)
    hip.check(lib.oa_token_logprobs(
        hip.current_stream_ptr(), logits.data_ptr(), logits.stride(0), tokens.data_ptr(),
        ws.data_ptr(), out.data_ptr(), B, V, top, int(logits.dtype == torch.float32)),
        "oa_token_logprobs")
    host = out.cpu()
    values = host.view(torch.float32)
    return values[:, 0], host[:, 1::2], values[:, 2::2]
