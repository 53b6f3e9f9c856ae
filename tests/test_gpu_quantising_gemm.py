"""The GEMM that quantises its few rows itself gives the bits of the quantiser followed by the GEMM: permuted rows, SwiGLU and GELU
rows; one row to the most it takes, all in one group or spread, groups of more rows than are requested ahead, both forms of the
kernel, rows of zeros, infinities and NaN, biases; and refuses other sizes."""
import pytest
import torch

from helpers import randn_bf16
from test_gemm_choice import FOUR, ONE, TWO, choice

pytestmark = pytest.mark.gpu

# (T, k, E, N, K) of 64 x 64 blocks with four waves, two and one: an odd number of steps, fewer steps than waves, groups of more rows than are
# requested ahead, and more than 64 groups
FEWER_WAVES = [((32, 2, 2, 8192, 1024), FOUR), ((8, 8, 32, 1408, 384), FOUR), ((8, 8, 64, 2048, 1408), TWO), ((8, 8, 256, 1024, 512), TWO), ((32, 2, 2, 16384, 1152), TWO),
               ((1, 8, 64, 8192, 128), TWO), ((8, 8, 128, 2048, 768), ONE), ((8, 8, 64, 4096, 1024), ONE), ((32, 2, 8, 8192, 384), ONE),
               ((40, 1, 3, 16384, 256), ONE)]  # fmt: skip


@pytest.mark.parametrize("shape,kernel", FEWER_WAVES)
def test_the_forms_of_these_sizes(shape, kernel):
    T, k, E, N, K = shape
    assert choice(T * k, N, K // 128, E, 1) == kernel


def fused(what, rows, sorted_idx, topk, q, s, goff, bias, M):
    from atorch_amd import _lib, kernels

    E, N, K = q.shape
    out = torch.full((M + 2, N), 7.0, dtype=torch.bfloat16, device=rows.device)
    rc = _lib.lib().aamd_quant_grouped_gemm_fp8_nt(
        what, rows.data_ptr(), rows.shape[1], sorted_idx.data_ptr() if sorted_idx is not None else None, topk, rows.shape[0], q.data_ptr(),
        s.data_ptr(), goff.data_ptr(), E, M, N, K, out.data_ptr(), N, bias.data_ptr() if bias is not None else None,
        kernels.dtype_code(bias.dtype) if bias is not None else _lib.NONE, _lib.stream())  # fmt: skip
    return rc, out


@pytest.mark.parametrize("T,k,E,N,K", [
    (1, 4, 60, 2816, 2048), (1, 1, 1, 128, 128), (16, 2, 2, 256, 1152), (32, 1, 1, 512, 640), (5, 3, 8, 4096, 1024), (8, 4, 64, 1024, 7168),
    (13, 2, 4, 1408, 384), (2, 8, 70, 2048, 1408),
    *[shape for shape, _ in FEWER_WAVES],
])  # fmt: skip
@pytest.mark.parametrize("what", [0, 1, 2], ids=["permuted", "swiglu", "gelu"])
@pytest.mark.parametrize("bias", [None, torch.bfloat16, torch.float32])
def test_bits_of_the_two_launches(dev, T, k, E, N, K, what, bias):
    from atorch_amd import kernels

    M = T * k
    g = torch.Generator().manual_seed(T + 100 * what)
    ids = torch.stack([torch.randperm(E, generator=g)[:k] if E >= k else torch.randint(E, (k,), generator=g) for _ in range(T)]).to(dev)
    sorted_idx, row_map, goff = kernels.moe_preprocess(ids, E)
    if (T, k, E, N, K) in dict(FEWER_WAVES):  # (many weights: made on the device)
        w = torch.randn((E, N, K), generator=torch.Generator(device=dev).manual_seed(3), device=dev).bfloat16() * 0.05
    else:
        w = randn_bf16((E, N, K), 3, std=0.05).to(dev)
    q, s, _, _ = kernels.block_quant_batched(w)
    b = torch.randn((E, N), generator=g).to(dev).to(bias) if bias is not None else None
    x = randn_bf16((T if what == 0 else M, K * (2 if what == 1 else 1)), 5).to(dev)
    x[0, :128] = 0.0  # a scale of one
    x[-1, -5] = float("inf")
    x[x.shape[0] // 2, -1] = float("nan")
    x[0, -3] = 3.0e38
    if what == 0:
        qx, sx = kernels.permute_tile_quant(x, row_map, k, M)
    elif what == 1:
        qx, sx = kernels.swiglu_tile_quant(x)[:2]
    else:
        qx, sx = kernels.gelu_tile_quant(x)[:2]
    want = kernels.grouped_gemm_nt(qx, sx, q, s, goff, out_dtype=torch.bfloat16, bias=b)
    rc, got = fused(what, x, sorted_idx if what == 0 else None, k, q, s, goff, b, M)
    assert rc == 0 and torch.all(got[M:] == 7.0)
    assert torch.equal(got[:M].view(torch.int16), want.view(torch.int16))


def test_other_sizes_are_refused(dev):
    from atorch_amd import _lib, kernels

    fits = _lib.lib().aamd_quant_grouped_gemm_fits
    assert fits(4, 2816, 2048, 60, 1) and not fits(65, 256, 256, 2, 8) and not fits(0, 256, 256, 2, 0) and not fits(32, 1024, 4096, 1, 32)
    x, w = randn_bf16((65, 256), 1).to(dev), randn_bf16((1, 256, 256), 2).to(dev)
    q, s, _, _ = kernels.block_quant_batched(w)
    rc, _ = fused(2, x, None, 0, q, s, kernels.group_offsets_from_splits([65], dev), None, 65)
    assert rc != 0
