"""The workspace that a row-ragged GEMM asks for: none where no tile's contraction can be shared out."""
import pytest


def _bytes(M, N, K, E, grouped, b_rows=0):
    from atorch_amd import _lib

    return _lib.lib().aamd_grouped_gemm_fp8_ws_bytes(M, N, K, E, grouped, b_rows)


@pytest.mark.parametrize("b_rows", [0, 1])
def test_launches_of_one_round_with_a_workgroup_per_tile_ask_for_none(b_rows):
    assert _bytes(1667, 6656, 8832, 1, 1, b_rows) == 0  # 182 tiles for 256 workgroups, in a group
    assert _bytes(2229, 3456, 6784, 8, 1, b_rows) == 0  # about 170 in eight
    assert _bytes(4224, 4096, 6144, 1, 1, b_rows) > 0  # a second round of 16
    assert _bytes(4224, 4096, 6016, 1, 1, b_rows) == 0  # too short a contraction
