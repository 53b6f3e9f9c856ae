"""Which kernel a row-ragged launch takes, where the choice has a line."""
import pytest

FOUR, TWO, ONE, SMALL_TILES = 2, 7, 8, 0


def choice(M, N, steps, E=1, grouped=0, b_rows=0, workspace=0):
    from atorch_amd import _probes

    return _probes.lib().aamd_tuning_grouped_gemm_choice(M, N, 128 * steps, E, grouped, b_rows, workspace)


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
