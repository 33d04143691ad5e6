"""The kernel and tiles that kd_mm_run launches (kandinsky.cpp_amd/csrc/
kd_mm_host.cpp), on the host alone."""
import math
import random

import pytest

from mm_plan import plan
from test_gpu_mm_tiles import CASES, DEEP, ENDS


@pytest.mark.parametrize("M,N,K", [(2 ** 31 - 1, 4, 32), (2 ** 31 - 255, 4, 32), (1, 2 ** 31 - 4, 32),
                                   (200, 2 ** 31 - 128, 64), (5, 2 ** 28 + 4, 32)])
def test_sizes_within_a_tile_of_2_31(M, N, K):
    p = plan(M, N, K)
    tn, tm = 32 * (p.tile // 10), 32 * (p.tile % 10)
    assert p.tiles_m == -(-M // tm) and p.tiles_n == -(-N // tn)
    assert p.n_blocks == p.tiles_m * p.tiles_n <= 2 ** 23   # 256 threads each: a grid of less than 2^32
    assert p.cols == (p.tiles_n if p.kernel == "mm_bf16" and p.tiles_n <= 8 else 4)
    # the last tile's row and output indexes are 32-bit
    assert p.tiles_m * tm <= 2 ** 31 and p.tiles_n * tn <= 2 ** 31


@pytest.mark.parametrize("M,N,K", [(60000, 4, 32), (59971, 24, 64), (60000, 64, 32), (60000, 64, 256),
                                   (60000, 64, 512)])
def test_few_outputs_of_many_tokens_take_one_round(M, N, K):
    """The large tile's time is mostly stores: with few outputs its one round
    beats several of small tiles (60,000 x 4 x 32: 8.3 us against 11.4), also
    where x's way from HBM bounds both (60,000 x 64 x 512: 27.0 against 28.9)."""
    assert plan(M, N, K)[:2] == ("mm_bf16", 88)


def test_both_types_of_x_take_the_same_tile():
    """F32 x has the bits of its BF16 rounding (a kernel sums both in one
    order, but the kernels not in the same)."""
    rng = random.Random(11)
    for _ in range(3000):
        M, N, K = (int(math.exp(rng.uniform(math.log(a), math.log(b)))) for a, b in ((1, 70000), (4, 20000), (32, 17000)))
        N, K = N // 4 * 4, K // 32 * 32
        assert plan(M, N, K, True) == plan(M, N, K, False), (M, N, K)
    for M in range(40000, 64000, 500):
        for K in (256, 512, 1024, 2048, 4096):
            assert plan(M, 64, K, True) == plan(M, 64, K, False), (M, 64, K)


# the tile (outputs, tokens in units of 32) of test_gpu_mm_tiles.py's cases of more than 16 tokens
TILE = {(17, 32): 11, (33, 100): 11, (31, 8200): 21, (130, 4100): 22, (300, 4096): 23, (850, 2100): 42, (700, 4100): 44,
        (1030, 8000): 43, (1540, 4100): 84, (1700, 4096): 84, (2047, 4004): 84, (3900, 4080): 88, (3841, 4064): 88,
        (4090, 4064): 88,
        (33001, 132): 88, (33, 112): 11, (34, 4144): 21, (99, 4184): 22, (3347, 260): 23, (291, 4148): 42, (3274, 524): 43, (4048, 648): 44,
        (3601, 1044): 84, (4057, 2180): 88}
LDS = 160 * 1024


def _stages(tile, x_f32):
    """LDS stages of an mm_ksplit instance, as the kernel sizes its ring."""
    return min(5, LDS // (tile // 10 * 4096 + tile % 10 * 32 * (256 if x_f32 else 128)))


@pytest.mark.parametrize("x_f32", [True, False], ids=["f32", "bf16"])
def test_gpu_cases_take_their_tiles(x_f32):
    for M, N, K in CASES + DEEP + ENDS:
        p = plan(M, N, K, x_f32)
        assert (p.kernel == "mm_skinny") == (M <= 16)
        assert M <= 16 or p.tile == TILE[M, N], (M, N, K, p)
    # every instance runs its steady loop and refills every buffer of its ring
    deep = {}
    for M, N, K in DEEP:
        nk = -(-K // 64)
        if M <= 16:
            wide = -(-N // 64) >= 256
            stages = {(True, 8): 4, (False, 8): 3, (True, 16): 3, (False, 16): 5}[wide, 8 if M <= 8 else 16]
            assert nk // 4 >= 2 * stages + 1
            deep.setdefault((wide, M <= 8), set()).add(K % 64)
        else:
            tile = TILE[M, N]
            if tile < 84:
                assert nk >= 2 * _stages(tile, x_f32) + 3
            else:
                assert K // 32 >= 2 * 6 + 3
            deep.setdefault(tile, set()).add(K % 64)
    assert len(deep) == 4 + 9 and all(k == {0, 32} for k in deep.values())
