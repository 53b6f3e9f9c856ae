"""The row permutes at the edges of their rules for lanes per row: 256 chunks of 16 bytes and one more, 512 and 1024 and one more, and
2048 tokens and one more; with copies that are dropped or lie beyond the output, whose places stay as they are."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 2048, 2049])
@pytest.mark.parametrize("chunks", [1, 255, 256, 257, 512, 513, 1024, 1025, 1792])
@pytest.mark.parametrize("dtype,topk", [(torch.bfloat16, 3), (torch.float32, 1)])
def test_permute_rows_copies_every_chunk(dev, T, chunks, dtype, topk):
    from atorch_amd import _lib, kernels

    n, cols = T * topk, chunks * 16 // dtype.itemsize
    g = torch.Generator().manual_seed(T + chunks)
    place = torch.randperm(n, generator=g).to(torch.int32)
    place[torch.rand(n, generator=g) < 0.1] = -1
    rows = n - n // 8  # of the output: places behind them are dropped
    x = torch.randn((T, cols), generator=g).to(dtype)
    want = torch.full((rows, cols), 7.0, dtype=dtype)
    kept = (place >= 0) & (place < rows)
    want[place[kept].long()] = x.repeat_interleave(topk, 0)[kept]
    held, got, place = x.to(dev), torch.full((rows + 1, cols), 7.0, dtype=dtype, device=dev), place.to(dev)
    _lib.check(_lib.lib().aamd_permute_rows(held.data_ptr(), kernels.dtype_code(dtype), T, cols, place.data_ptr(), topk, rows, got.data_ptr(), _lib.stream()))
    assert torch.equal(got[:rows].cpu(), want) and torch.all(got[rows] == 7.0)


@pytest.mark.parametrize("T", [1, 2048, 2049])
@pytest.mark.parametrize("eights", [1, 256, 257, 1024, 1025])
@pytest.mark.parametrize("dtype,out_dtype,topk", [(torch.bfloat16, torch.bfloat16, 3), (torch.float32, torch.bfloat16, 1), (torch.float32, torch.float32, 2), (torch.float32, torch.float32, 3)])
def test_permute_rows_scaled_rounds_one_product(dev, T, eights, dtype, out_dtype, topk):
    from atorch_amd import kernels

    n, cols = T * topk, eights * 8
    g = torch.Generator().manual_seed(T + eights)
    place = torch.randperm(n, generator=g)
    x, probs = torch.randn((T, cols), generator=g).to(dtype), torch.rand((T, topk), generator=g).to(dtype)
    want = torch.empty((n, cols), dtype=out_dtype)
    want[place] = (x.float().repeat_interleave(topk, 0) * probs.float().reshape(-1, 1)).to(out_dtype)
    got = kernels.permute_rows_scaled(x.to(dev), place.to(torch.int32).to(dev), topk, n, probs.to(dev), out_dtype)
    assert torch.equal(got.cpu(), want)
