"""The row-ragged GEMM on 256 x 256 tiles, whose workgroups take one tile after the other (at most 256 of them): several tiles
per workgroup and less than one, even and odd numbers of 128-deep steps around the batches of eight blocks of scales, rows of
scales that are 16-byte aligned and not, half tiles of outputs, tiles of one row next to full ones, more than 64 groups and
empty ones.  The 128 x 128 tiles add the same products in the same order, so that the results are the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("splits,N,K", [
    ([1], 128, 1024), ([8192], 4096, 1152), ([8191], 4224, 1024), ([300, 0, 5000, 257, 1, 3000], 2176, 1280),
    ([800] * 60, 1024, 1408), ([257] * 70 + [0, 1, 255], 640, 2048), ([256, 1] * 32, 1152, 1664), ([4097, 4095], 2048, 2176),
    ([129] * 130, 384, 1920),
])  # fmt: skip
@pytest.mark.parametrize("out_dtype,bias", [(torch.bfloat16, None), (torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("turned", [False, True])
def test_large_tiles_give_the_bits_of_small_ones(dev, splits, N, K, out_dtype, bias, turned):
    from atorch_amd import kernels

    E, M = len(splits), sum(splits)
    g = torch.Generator(device=dev).manual_seed(7)
    qx, sx = kernels.tile_quant(torch.randn((M, K), generator=g, device=dev).bfloat16())
    w = torch.randn((E, K, N) if turned else (E, N, K), generator=g, device=dev).bfloat16() * 0.05
    q, s, q_t, s_t = kernels.block_quant_batched(w, return_transpose=True, written=kernels.STORED)
    if turned:
        q, s = q_t, s_t
    b = torch.randn((E, N), generator=g, device=dev).to(bias) if bias is not None else None
    goff = kernels.group_offsets_from_splits(splits, dev)
    got = {}
    for tile in (0, 1):
        out = torch.full((M + 3, N), 7.0, dtype=out_dtype, device=dev)  # rows behind the last one stay as they are
        with kernels.gemm_options(tile=tile):
            kernels.grouped_gemm_nt(qx, sx, q, s, goff, out=out[:M], bias=b)
        got[tile] = out
    assert torch.equal(got[0], got[1]) and torch.all(got[1][M:] == 7.0)


def test_output_rows_apart(dev):
    """Columns between the rows of a wider output are not touched."""
    from atorch_amd import kernels

    g = torch.Generator(device=dev).manual_seed(8)
    splits, N, K = [700, 3, 900], 640, 1024
    qx, sx = kernels.tile_quant(torch.randn((sum(splits), K), generator=g, device=dev).bfloat16())
    qw, sw, _, _ = kernels.block_quant_batched(torch.randn((3, N, K), generator=g, device=dev).bfloat16())
    goff = kernels.group_offsets_from_splits(splits, dev)
    wide = torch.full((sum(splits), N + 64), 7.0, dtype=torch.bfloat16, device=dev)
    with kernels.gemm_options(tile=1):
        kernels.grouped_gemm_nt(qx, sx, qw, sw, goff, out=wide[:, :N])
    with kernels.gemm_options(tile=0):
        want = kernels.grouped_gemm_nt(qx, sx, qw, sw, goff)
    assert torch.equal(wide[:, :N], want) and torch.all(wide[:, N:] == 7.0)
