"""The dense product with 1x128 scales on both sides, where large outputs take the weight-gradient kernel with the
scales turned round: bit-equal to the row-major kernel (the same sums in the same order), at the size where the one
takes over from the other, and the transpose of the scales at the edges of its 32 x 32 tiles."""
import pytest
import torch

from helpers import randn_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(128 * 64, 128 * 32, 128), (128 * 33, 128 * 63, 384), (128 * 64, 128 * 31, 256), (128 * 64 + 1, 128 * 33, 128)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_dense_product_with_row_scales_on_both_sides(dev, M, N, K, dtype):
    from atorch_amd import _lib, kernels

    a, sa = kernels.tile_quant(randn_bf16((M, K), 1).to(dev))
    b, sb = kernels.tile_quant(randn_bf16((N, K), 2).to(dev))
    got = kernels.fp8_gemm(a, sa, b, sb, dtype=dtype)
    want = torch.empty((M, N), dtype=dtype, device=dev)
    _lib.check(_lib.lib().aamd_grouped_gemm_fp8_nt(
        a.data_ptr(), K, sa.data_ptr(), b.data_ptr(), sb.data_ptr(), 1, None, 1, None, M, N, K, want.data_ptr(),
        _lib.dtype_code(dtype), N, None, _lib.NONE, _lib.stream()))  # fmt: skip
    assert torch.equal(got, want)


@pytest.mark.parametrize("rows,blocks", [(1, 1), (31, 33), (32, 32), (129, 7), (7, 129)])
def test_transpose_of_the_scales(dev, rows, blocks):
    from atorch_amd import kernels

    s = torch.randn(rows, blocks, device=dev)
    assert torch.equal(kernels.host().transpose_scales(s), s.t().contiguous())
