"""The kernel for few rows with two waves and with one to a block of 64 x 64, for launches of many blocks of a short contraction: groups of
one row to three blocks, empty ones, a contraction of fewer steps than waves, of an odd number and of the most the choice takes, and what
the library chooses on both sides of its lines."""
import pytest
import torch

from helpers import rel_err
from test_gemm_choice import ONE, choice

pytestmark = pytest.mark.gpu


def operands(dev, splits, N, K):
    from atorch_amd import kernels

    g = torch.Generator(device=dev).manual_seed(sum(splits) + N + K)
    qx, sx = kernels.tile_quant(torch.randn((sum(splits), K), generator=g, device=dev).bfloat16())
    w = torch.randn((len(splits), N, K), generator=g, device=dev).bfloat16() * 0.05
    return (qx, sx, *kernels.block_quant_batched(w)[:2], kernels.group_offsets_from_splits(splits, dev))


def tolerance(K, out_dtype):
    # sums of K/128 products of like size in another order: an addition rounds by at most 2^-24 of a partial sum, which stays below
    # sqrt(K/128) of the result's root mean square times 4; two sums on either side of a rounding give neighbours in bf16
    return K / 128 * 2.0**-24 * 4 + (2.0**-7 if out_dtype == torch.bfloat16 else 0.0)


@pytest.mark.parametrize("splits,N", [([1], 128), ([63, 64, 65, 0, 130], 384), ([0, 192, 7], 640), ([(5 * e) % 70 for e in range(70)], 256)])
@pytest.mark.parametrize("K", [128, 256, 384, 2432])
@pytest.mark.parametrize("out_dtype,bias", [(torch.bfloat16, torch.float32), (torch.float32, None)])
def test_fewer_waves(dev, splits, N, K, out_dtype, bias):
    from atorch_amd import kernels

    ops, M = operands(dev, splits, N, K), sum(splits)
    b = torch.randn((len(splits), N), generator=torch.Generator(device=dev).manual_seed(1), device=dev).to(bias) if bias is not None else None
    got = {}
    for tile in (0, 7, 8):
        out = torch.full((M + 3, N), 7.0, dtype=out_dtype, device=dev)  # rows behind the last one stay as they are
        with kernels.gemm_options(tile=tile):
            kernels.grouped_gemm_nt(*ops, out=out[:M], bias=b)
        assert torch.all(out[M:] == 7.0)
        got[tile] = out
    assert torch.equal(got[0], got[8])  # one wave adds in the order of the contraction, like the tiles
    assert rel_err(got[7][:M], got[0][:M]) <= tolerance(K, out_dtype)


# 64 groups of six rows on average, 62 of which the library expects to have any: 498, 623, 747, 997, 1121, 1744 and 2243 blocks around its lines
# at 500, 724 and 1024, with 2 to 20 steps around those at 4, 14 (weights of 256 MB and more) and 20; and one group of 512, 516, 1024 and 1032
@pytest.mark.parametrize("splits,N", [([3, 0, 15, 2, 5, 8, 6, 9] * 8, n) for n in (512, 640, 768, 1024, 1152, 1792, 2304)]
                         + [([64], n) for n in (32768, 33024, 65536, 66048)])  # fmt: skip
@pytest.mark.parametrize("K", [256, 384, 512, 1664, 1792, 2432, 2560])
@pytest.mark.parametrize("out_dtype", [torch.float32])
def test_what_is_chosen_at_the_lines(dev, splits, N, K, out_dtype):
    from atorch_amd import kernels

    kernel = choice(sum(splits), N, K // 128, len(splits), 1)
    ops = operands(dev, splits, N, K)
    got = kernels.grouped_gemm_nt(*ops, out_dtype=out_dtype)
    with kernels.gemm_options(tile=kernel):  # the library takes what it says
        assert torch.equal(got, kernels.grouped_gemm_nt(*ops, out_dtype=out_dtype))
    with kernels.gemm_options(tile=0):
        want = kernels.grouped_gemm_nt(*ops, out_dtype=out_dtype)
    assert torch.equal(got, want) if kernel == ONE else rel_err(got, want) <= tolerance(K, out_dtype)
