"""Row tiles of up to 288 rows, which take the rows of a group beyond its full tiles: bit-equal to the 128 x 128 tiles (the same sums
in the same order) for remainders of one row to 32 a tile, one more than the tiles take, groups of less than a tile, empty ones, more
than 64, an odd number of steps, half tiles of outputs, weights along either side and a bias; with the last round's tiles in
parts; and where the groups' rows decide between them and tiles of 256."""
import pytest
import torch

from helpers import rel_err

pytestmark = pytest.mark.gpu


def operands(dev, splits, N, K, turned):
    from atorch_amd import kernels

    E, M = len(splits), sum(splits)
    g = torch.Generator(device=dev).manual_seed(M + N)
    qx, sx = kernels.tile_quant(torch.randn((M, K), generator=g, device=dev).bfloat16())
    w = torch.randn((E, K, N) if turned else (E, N, K), generator=g, device=dev).bfloat16() * 0.05
    q, s, q_t, s_t = kernels.block_quant_batched(w, return_transpose=True, written=kernels.STORED)
    return (qx, sx, q_t, s_t) if turned else (qx, sx, q, s)


@pytest.mark.parametrize("splits,N,K", [
    ([264], 256, 1024), ([288], 384, 1152), ([289], 256, 1024), ([520, 300, 0, 255, 256, 257, 1], 384, 1024), ([576, 577], 1152, 1408),
    ([2303, 256 * 9 + 33], 640, 1152), ([4100, 777, 0, 545], 1024, 2048), ([(37 * e) % 330 for e in range(70)], 384, 1024),
])  # fmt: skip
@pytest.mark.parametrize("out_dtype,bias", [(torch.bfloat16, None), (torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("turned", [False, True])
def test_higher_tiles_give_the_bits_of_small_ones(dev, splits, N, K, out_dtype, bias, turned):
    from atorch_amd import kernels

    E, M = len(splits), sum(splits)
    ops, goff = operands(dev, splits, N, K, turned), kernels.group_offsets_from_splits(splits, dev)
    b = torch.randn((E, N), generator=torch.Generator(device=dev).manual_seed(1), device=dev).to(bias) if bias is not None else None
    got = {}
    for tile in (0, 6):
        out = torch.full((M + 3, N), 7.0, dtype=out_dtype, device=dev)  # rows behind the last one stay as they are
        with kernels.gemm_options(tile=tile):
            kernels.grouped_gemm_nt(*ops, goff, out=out[:M], bias=b)
        got[tile] = out
    assert torch.equal(got[0], got[6]) and torch.all(got[6][M:] == 7.0)


# (the first two are worth it: 28 64ths of a tile a group against 5 for each tile; the others just not, or not with these rows)
@pytest.mark.parametrize("splits", [[264] * 8, [512, 513, 520, 0, 530], [768 + 30, 300], [545] * 4, [20000, 264, 264]])
@pytest.mark.parametrize("turned", [False, True])
def test_either_by_the_rows_of_the_groups(dev, splits, turned):
    from atorch_amd import kernels

    N, K = 20480, 1024
    ops, goff = operands(dev, splits, N, K, turned), kernels.group_offsets_from_splits(splits, dev)
    got = kernels.grouped_gemm_nt(*ops, goff)
    with kernels.gemm_options(tile=0):
        assert torch.equal(kernels.grouped_gemm_nt(*ops, goff), got)


@pytest.mark.parametrize("splits,N,K", [([264] * 17, 4096, 6144), ([520] * 9, 3968, 6272)])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("turned", [False, True])
def test_parts_of_higher_tiles(dev, splits, N, K, out_dtype, turned):
    """Tiles of more than 256 rows in the last round, in parts.  At most eight sums a row instead of one, of the same products: an fp32
    result may differ by the rounding of nkb additions, and a bf16 one by what its own rounding makes of that."""
    from atorch_amd import _lib, kernels

    E, M, nkb = len(splits), sum(splits), K // 128
    ops, goff = operands(dev, splits, N, K, turned), kernels.group_offsets_from_splits(splits, dev)
    ws = torch.full((1 << 24,), float("nan"), device=dev)
    out = torch.full((M + 3, N), 7.0, dtype=out_dtype, device=dev)
    _lib.check(_lib.lib().aamd_grouped_gemm_fp8_ws(
        ops[0].data_ptr(), K, ops[1].data_ptr(), ops[2].data_ptr(), ops[3].data_ptr(), int(turned), goff.data_ptr(), E, M, N, K,
        out.data_ptr(), kernels.dtype_code(out_dtype), N, None, _lib.NONE, ws.data_ptr(), ws.numel() * 4, _lib.stream()))  # fmt: skip
    assert torch.all(out[M:] == 7.0) and not torch.isnan(ws).all()
    with kernels.gemm_options(tile=0):
        want = kernels.grouped_gemm_nt(*ops, goff, out_dtype=out_dtype)
    # (sums of nkb products of like size: an addition rounds by at most 2^-24 of a partial sum, which stays below sqrt(nkb) of the
    # result's root mean square times 4; two sums on either side of a rounding give neighbours in bf16, up to 2^-7 apart)
    assert rel_err(out[:M], want) <= nkb * 2.0**-24 * 4 + (2.0**-7 if out_dtype == torch.bfloat16 else 0.0)


@pytest.mark.parametrize("splits", [[288], [287, 0, 1]])
def test_rows_as_far_apart_as_is_taken(dev, splits):
    """288 rows of nearly 8 MB: their last byte lies beyond what a signed 32-bit offset reaches."""
    from atorch_amd import kernels

    N, K, M, lda = 384, 1024, sum(splits), (1 << 23) - 16
    qx, *rest = operands(dev, splits, N, K, False)
    goff = kernels.group_offsets_from_splits(splits, dev)
    far = torch.empty((M - 1) * lda + K, dtype=torch.uint8, device=dev).view(qx.dtype).as_strided((M, K), (lda, 1))
    far.view(torch.uint8).copy_(qx.view(torch.uint8))
    with kernels.gemm_options(tile=0):
        want = kernels.grouped_gemm_nt(qx, *rest, goff)
    with kernels.gemm_options(tile=6):
        assert torch.equal(kernels.grouped_gemm_nt(far, *rest, goff), want)
