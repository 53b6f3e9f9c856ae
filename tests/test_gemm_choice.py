"""Which kernel a row-ragged launch takes, where the choice has a line."""
import ctypes
from itertools import accumulate

import pytest

FOUR, TWO, ONE, SMALL_TILES, LARGE_TILES, SHARED, HIGHER = 2, 7, 8, 0, 1, 5, 6


def choice(M, N, steps, E=1, grouped=0, b_rows=0, workspace=0, splits=None, c_dtype=0):
    from atorch_amd import _probes

    offsets = (ctypes.c_int64 * (E + 1))(0, *accumulate(splits)) if splits else None
    return _probes.lib().aamd_tuning_grouped_gemm_choice(M, N, 128 * steps, E, grouped, b_rows, workspace, c_dtype, offsets)


@pytest.mark.parametrize("grouped", [0, 1])
@pytest.mark.parametrize("steps", [3, 4, 8, 12, 16, 19])
def test_blocks_that_are_known_and_fill_a_round(grouped, steps):
    """Without groups, or with one, the 64 x 64 blocks are counted, not expected: 512 are a round of two blocks of four waves to a CU, 1024
    of four blocks of two."""
    for M, N in ((2048, 1024), (1024, 2048), (512, 4096), (256, 8192), (64, 32768)):
        assert choice(M, N, steps, grouped=grouped) == FOUR
        assert choice(M, N + 128, steps, grouped=grouped) in (TWO, SMALL_TILES)
    assert choice(64, 32896, steps, grouped=grouped) == TWO and choice(128, 16512, steps, grouped=grouped) == TWO
    if steps >= 4:
        assert choice(64, 65536, steps, grouped=grouped) in (TWO, SMALL_TILES)
        assert choice(64, 65664, steps, grouped=grouped) in (ONE, SMALL_TILES)


# (us, 128 x 128 tiles and one wave to a block)
@pytest.mark.parametrize("M,N,steps,E,c_dtype,one_wave", [
    (8195, 21760, 2, 2, 0, False), (8192, 14336, 2, 16, 0, False), (94295, 2048, 2, 55, 0, False), (8907, 13312, 2, 44, 0, False),  # 137, 163; 94, 117; 163, 194; 116, 131
    (9600, 8192, 2, 32, 1, False), (24000, 5120, 1, 4, 1, False),  # 78, 118; 101, 104: outputs of 315 and 492 MB
    (9600, 8192, 2, 32, 0, True), (8192, 4096, 2, 8, 1, True), (3072, 27776, 2, 1, 0, True), (410, 25728, 4, 56, 0, True),  # 76, 59; 34, 31; 73, 62; 193, 142
    (30000, 4096, 2, 1, 0, False), (11718, 1024, 2, 1, 0, False), (40000, 1024, 2, 4, 0, False), (20000, 4096, 2, 4, 0, True),  # 85, 112, rows of 7.7 MB in a group; of 3 and 2.6 MB; of 1.3
])  # fmt: skip
def test_one_wave_where_the_caches_hold_what_it_needs(M, N, steps, E, c_dtype, one_wave):
    got = choice(M, N, steps, E, 1, c_dtype=c_dtype)
    assert got == (ONE if one_wave else SMALL_TILES)


# (us, tiles of 256 rows and of up to 288)
@pytest.mark.parametrize("splits,N,K,workspace,higher", [
    ([485, 505, 513, 520, 500, 516, 515, 542], 28672, 4096, 0, True),  # 524, 474
    ([496, 493, 518, 511, 526, 505, 521, 526], 28672, 4096, 0, True), ([519, 512, 516, 485, 521, 506, 489, 548], 28672, 4096, 0, True),  # 510, 500; 523, 507
    ([496, 493, 518, 511, 526, 505, 521, 526], 4096, 14336, 1, True),  # 266, 253
    ([802], 21120, 2560, 0, True),  # 66, 52: 249 tiles, of which no XCD has more than 32
    ([264] * 8, 28672, 4096, 0, True), ([520] * 8, 28672, 4096, 0, True), ([280, 277, 265], 15488, 3584, 0, True),  # 373, 302; 558, 489; 82, 62
    ([285, 300, 276, 310, 292, 281, 302, 293], 16128, 11392, 1, False),  # 555, 625
    ([1250, 1296], 9344, 7680, 1, False),  # 185, 225
    ([1160, 1130, 1135], 9984, 4224, 0, False),  # 153, 179: 507 tiles, of which an XCD has 65
    ([820] * 8, 4096, 7424, 1, False), ([512] * 8, 28672, 4096, 0, False), ([640] * 8, 28672, 4096, 0, False),  # 200, 237; 449, 473; 595, 632
])  # fmt: skip
def test_higher_tiles_where_they_are_faster(splits, N, K, workspace, higher):
    got = choice(sum(splits), N, K // 128, len(splits), 1, 0, workspace, splits)
    assert got == HIGHER if higher else got in (LARGE_TILES, SHARED)


def test_higher_tiles_of_one_group_and_of_none():
    for M, N, steps, workspace, higher in ((1288, 12032, 8, 0, True), (1032, 13312, 48, 1, True), (1280, 12032, 8, 0, False), (1300, 16384, 32, 0, False)):
        assert (choice(M, N, steps, workspace=workspace) == HIGHER) == higher
        assert (choice(M, N, steps, 1, 1, 0, workspace, [M]) == HIGHER) == higher
