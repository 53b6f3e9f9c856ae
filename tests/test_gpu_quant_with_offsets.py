"""The row quantiser that stores the groups' offsets on the side, against the two launches it stands for."""
import pytest
import torch

from helpers import randn_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("splits", [[1], [0], [5, 0, 7], [3] * 64, [2] * 65, [1000, 0, 24, 0]], ids=lambda s: f"{len(s)}groups_{sum(s)}rows")
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_offsets_and_codes(dev, splits, dtype):
    from atorch_amd import _lib, kernels

    M, K, E = sum(splits), 384, len(splits)
    x = randn_bf16((M, K), 1).to(dev).to(dtype)
    q, s = torch.empty((M, K), dtype=kernels.FP8, device=dev), torch.empty((M, K // 128), device=dev)
    goff = torch.full((E + 2,), -7, dtype=torch.int64, device=dev)
    counts = torch.tensor(splits, dtype=torch.int64)
    _lib.check(_lib.lib().aamd_quant_1x128_with_offsets(
        x.data_ptr(), kernels.dtype_code(dtype) if dtype != torch.float16 else _lib.F16, M, K, K, counts.data_ptr(), E, goff.data_ptr(),
        q.data_ptr(), s.data_ptr(), 0.0, _lib.stream()))  # fmt: skip
    assert goff.tolist() == [0, *torch.cumsum(counts, 0).tolist(), -7]
    if M:
        qw, sw = kernels.tile_quant(x)
        assert torch.equal(q.float(), qw.float()) and torch.equal(s, sw)
