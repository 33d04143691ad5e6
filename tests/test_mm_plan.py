"""The kernel and tiles that kd_mm_run launches (kandinsky.cpp_amd/csrc/
kd_mm_host.cpp), on the host alone."""
import pytest

from mm_plan import plan


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
                                   (61442, 64, 4096), (60000, 64, 512)])
def test_few_outputs_of_many_tokens_take_one_round(M, N, K):
    """The large tile's time is mostly stores: with few outputs its one round
    beats several of small tiles (60,000 x 4 x 32: 8.3 us against 11.4), also
    where x's way from HBM bounds both (60,000 x 64 x 4096: 178 against 184)."""
    assert plan(M, N, K)[:2] == ("mm_bf16", 88)
