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


@pytest.mark.parametrize("M,K", [(1, 128), (127, 256), (128, 1152), (300, 2048)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_transposed_scales_written_row_major(dev, M, K, dtype):
    """The operator's transposed codes and scales, contiguous, against the quantiser that writes the scales block by block."""
    from atorch_amd import kernels, ops

    x = randn_bf16((M, K), 3).to(dev).to(dtype)
    q, s, q_t, s_t = kernels.tile_quant(x, return_transpose=True)
    got = ops.quantize_vector_blockwise(x, return_transpose=True)
    for a, b in zip(got, (q, s, q_t, s_t)):
        assert a.shape == b.shape and a.is_contiguous() and torch.equal(a.float(), b.float())


@pytest.mark.parametrize("rows,other,blocks", [(1, 33, 1), (64, 32, 40), (129, 31, 7)])
def test_two_transposes_in_one_launch(dev, rows, other, blocks):
    from atorch_amd import _lib

    a, b = torch.randn(rows, blocks, device=dev), torch.randn(other, blocks, device=dev)
    at, bt = torch.empty(blocks, rows, device=dev), torch.empty(blocks, other, device=dev)
    _lib.check(_lib.lib().aamd_transpose_scales_pair(a.data_ptr(), rows, at.data_ptr(), b.data_ptr(), other, bt.data_ptr(), blocks, _lib.stream()))
    assert torch.equal(at, a.t()) and torch.equal(bt, b.t())
