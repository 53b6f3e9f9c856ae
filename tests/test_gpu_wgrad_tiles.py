"""Weight gradients on 256 x 256 tiles, whose workgroups take one tile after the other: bit-equal to the 128 x 128 tiles (the same
sums in the same order) for groups of no block, one (taken twice, the second time with scales of zero), two, odd and even
numbers, half tiles of either side, more tiles than workgroups, both operand layouts and an expert stride beyond the matrix."""
import pytest
import torch

from helpers import randn_bf16

pytestmark = pytest.mark.gpu

SPLITS = [
    [300, 0, 1111, 128, 77], [1], [700], [0], [0, 0, 129, 0], [256, 257, 384, 1, 0, 2000], [(37 * e) % 260 for e in range(64)],
]  # fmt: skip


def operands(dev, splits, N, K, blocked):
    from atorch_amd import kernels

    E, M = len(splits), sum(splits)
    goff = kernels.group_offsets_from_splits(splits, dev)
    ld = kernels.padded_bound(M, E)
    x, dy = randn_bf16((M, K), 1).to(dev), randn_bf16((M, N), 2, std=1e-2).to(dev)
    h = kernels.host()
    _, _, qx, sx = h.dual(x, goff, E, 0.0, ld, False, blocked)
    _, _, qd, sd = h.dual(dy, goff, E, 0.0, ld, False, blocked)
    return qd, sd, qx, sx, goff


@pytest.mark.parametrize("splits", SPLITS, ids=lambda s: f"{len(s)}groups_{sum(s)}rows")
@pytest.mark.parametrize("N,K", [(128, 128), (640, 384), (256, 2176), (1152, 4096)])
@pytest.mark.parametrize("blocked", [True, False], ids=["blocked", "rows"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_large_tiles_give_the_bits_of_small_ones(dev, splits, N, K, blocked, dtype):
    from atorch_amd import kernels

    ops = operands(dev, splits, N, K, blocked)
    got = {}
    for tile in (0, 1):
        wide = torch.full((len(splits), N * K + 64), 7.0, dtype=dtype, device=dev)
        out = wide[:, : N * K].view(len(splits), N, K) if len(splits) > 1 else torch.full((1, N, K), 7.0, dtype=dtype, device=dev)
        with kernels.gemm_options(tile=tile):
            kernels.grouped_gemm_wgrad(*ops, out=out, out_dtype=dtype)
        got[tile] = out
        assert len(splits) == 1 or torch.all(wide[:, N * K :] == 7.0)
    assert torch.equal(got[0], got[1])


@pytest.mark.parametrize("splits,N,K", [([1100, 1], 4096, 4096), ([5000, 0, 3000, 300], 2048, 2048), ([900] * 8, 1024, 4096)])
def test_launches_of_whole_rounds(dev, splits, N, K):
    """Sizes that the library itself gives to them, a workgroup for every tile."""
    from atorch_amd import kernels

    ops = operands(dev, splits, N, K, True)
    got = kernels.grouped_gemm_wgrad(*ops, out_dtype=torch.bfloat16)
    with kernels.gemm_options(tile=0):
        want = kernels.grouped_gemm_wgrad(*ops, out_dtype=torch.bfloat16)
    assert torch.equal(got, want)


def test_groups_beyond_the_operand_buffers_are_nan(dev):
    """Room for two token blocks: groups that do not fit are written as NaN, and read nowhere."""
    from atorch_amd import kernels

    splits, N, K = [128, 0, 100, 5000], 384, 256
    goff = kernels.group_offsets_from_splits(splits, dev)
    qd = torch.zeros((2, N, 128), dtype=torch.uint8, device=dev).view(kernels.FP8)
    qx = torch.zeros((2, K, 128), dtype=torch.uint8, device=dev).view(kernels.FP8)
    with kernels.gemm_options(tile=1):
        for dtype in (torch.float32, torch.bfloat16):
            dw = kernels.grouped_gemm_wgrad(qd, torch.ones((2, N), device=dev), qx, torch.ones((2, K), device=dev), goff, out_dtype=dtype)
            assert torch.all(dw[:3] == 0) and torch.all(torch.isnan(dw[3]))
