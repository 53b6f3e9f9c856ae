"""The last round of 256-row tiles, whose rows are shared by two or four workgroups where few tiles are left: bit-equal to the 128 x 128
tiles (the same sums in the same order) with full tiles and with tiles of 1 to 200 rows, of which some workgroups have no share, in it,
and for tiles of up to 288 rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# 16 tiles of outputs: 17 tiles of rows leave 2 of 34 tiles per XCD to four workgroups each, 24 leave 16 of 48 to two
@pytest.mark.parametrize("tile,splits", [
    (1, [4352]), (1, [6144]), (1, [256] * 12 + [1, 40, 65, 130, 200]), (1, [1, 40, 65, 130, 200] + [256] * 12), (1, [200, 1, 0, 60] * 8),
    (6, [280] * 16 + [40]), (6, [40] + [544] * 8), (6, [288] * 23 + [130]),
])  # fmt: skip
@pytest.mark.parametrize("K,out_dtype", [(1024, torch.bfloat16), (1152, torch.float32)])
@pytest.mark.parametrize("turned", [False, True])
def test_shares_of_rows_give_the_bits_of_small_tiles(dev, tile, splits, K, out_dtype, turned):
    from atorch_amd import kernels

    N, E, M = 4096, len(splits), sum(splits)
    g = torch.Generator(device=dev).manual_seed(M + K)
    qx, sx = kernels.tile_quant(torch.randn((M, K), generator=g, device=dev).bfloat16())
    w = torch.randn((E, K, N) if turned else (E, N, K), generator=g, device=dev).bfloat16() * 0.05
    q, s, q_t, s_t = kernels.block_quant_batched(w, return_transpose=True, written=kernels.STORED)
    ops, goff = (qx, sx, q_t, s_t) if turned else (qx, sx, q, s), kernels.group_offsets_from_splits(splits, dev)
    got = {}
    for t in (0, tile):
        out = torch.full((M + 3, N), 7.0, dtype=out_dtype, device=dev)  # rows behind the last one stay as they are
        with kernels.gemm_options(tile=t):
            kernels.grouped_gemm_nt(*ops, goff, out=out[:M])
        got[t] = out
    assert torch.equal(got[0], got[tile]) and torch.all(got[tile][M:] == 7.0)
