"""One written orientation of a weight's codes: the grouped GEMM on the transposed view of dense codes gives the bits it gives
on the transposed codes themselves, with each kernel both have (the split form of the one for few rows exists for the codes
only and adds the blocks in another order), at the edges of their tiles (half a tile of outputs, rows
around 32, 64, 128 and 256, contractions around the batches of eight blocks of scales, more than 64 groups); and the
quantiser writes the same codes whichever orientations it writes."""
import pytest
import torch

from helpers import randn_bf16, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("splits,N,K", [
    ([1], 128, 128), ([7, 0, 65], 128, 384), ([31, 33], 256, 1024), ([127, 129, 0], 384, 1152), ([255, 257], 640, 1920),
    ([300, 5], 256, 2176), ([3] * 63 + [0, 5, 40], 128, 1024), ([0] * 70 + [17], 384, 640), ([520], 896, 4096),
])  # fmt: skip
@pytest.mark.parametrize("out_dtype,bias", [(torch.float32, None), (torch.bfloat16, torch.bfloat16)])
def test_gemm_reads_the_view_as_the_codes(dev, splits, N, K, out_dtype, bias):
    from atorch_amd import kernels

    E, M = len(splits), sum(splits)
    qx, sx = kernels.tile_quant(randn_bf16((M, K), 1).to(dev))
    q, s, q_t, s_t = kernels.block_quant_batched(randn_bf16((E, K, N), 2, std=0.05).to(dev), return_transpose=True)
    b = randn_bf16((E, N), 3).to(dev) if bias is not None else None
    goff = kernels.group_offsets_from_splits(splits, dev)
    args = (goff, None, out_dtype, b)
    for tile in (0, 1, 2):
        with kernels.gemm_options(tile=tile):
            want = kernels.grouped_gemm_nt(qx, sx, q_t, s_t, *args)
            got = kernels.grouped_gemm_nt(qx, sx, q.transpose(1, 2), s.transpose(1, 2), *args)
        assert torch.equal(got, want), f"tile {tile}"
    # the library's own choice (the bars of the few-rows test: the order of the sum over blocks may differ), and scales or codes
    # that somebody has made dense meanwhile
    gemm = kernels.host().gemm_nt
    want, got = gemm(qx, sx, q_t, s_t, *args), gemm(qx, sx, q.transpose(1, 2), s.transpose(1, 2), *args)
    assert rel_err(got.float().cpu(), want.float().cpu()) <= (5e-4 if out_dtype == torch.float32 else 1e-2)
    assert torch.equal(gemm(qx, sx, q.transpose(1, 2), s_t, *args), got)
    assert torch.equal(gemm(qx, sx, q_t, s.transpose(1, 2), *args), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("E,N,K", [(1, 128, 128), (3, 256, 640), (9, 4096, 4096)])
def test_quantiser_writes_one_orientation_of_the_same_codes(dev, dtype, E, N, K):
    from atorch_amd import kernels

    w = torch.randn((E, N, K), generator=torch.Generator(device=dev).manual_seed(5), device=dev, dtype=torch.float32).to(dtype)
    want = kernels.block_quant_batched(w, return_transpose=True)
    for written in (kernels.STORED, kernels.TURNED):
        got = kernels.block_quant_batched(w, return_transpose=True, written=written)
        assert all(g.shape == t.shape and torch.equal(g.contiguous().view(torch.uint8), t.view(torch.uint8)) for g, t in zip(got, want))
        assert got[0].data_ptr() == got[2].data_ptr() and got[1].data_ptr() == got[3].data_ptr()
