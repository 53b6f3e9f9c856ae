"""Weight gradients of groups without rows, written as zeros beside the tiles of the others: nothing of them is left, and nothing
beyond the matrix is touched, for gradients smaller and larger than one pass of the workgroups that write them."""
import pytest
import torch

from helpers import randn_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("splits", [[0] * 5, [0, 130, 0, 0, 1], [0] * 63 + [257], [300, 0]], ids=lambda s: f"{len(s)}groups_{sum(s)}rows")
@pytest.mark.parametrize("N,K", [(128, 128), (640, 384), (1152, 1024)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_zeros_of_groups_without_rows(dev, splits, N, K, dtype):
    from atorch_amd import kernels

    E, M = len(splits), sum(splits)
    goff = kernels.group_offsets_from_splits(splits, dev)
    ld = kernels.padded_bound(M, E)
    h = kernels.host()
    _, _, qx, sx = h.dual(randn_bf16((M, K), 1).to(dev), goff, E, 0.0, ld, False, True)
    _, _, qd, sd = h.dual(randn_bf16((M, N), 2).to(dev), goff, E, 0.0, ld, False, True)
    wide = torch.full((E, N * K + 64), 7.0, dtype=dtype, device=dev)
    out = wide[:, : N * K].view(E, N, K)
    kernels.grouped_gemm_wgrad(qd, sd, qx, sx, goff, out=out, out_dtype=dtype)
    with kernels.gemm_options(tile=0):  # (a workgroup for every tile)
        want = kernels.grouped_gemm_wgrad(qd, sd, qx, sx, goff, out_dtype=dtype)
    assert torch.equal(out, want) and torch.all(wide[:, N * K :] == 7.0)
    for e, m in enumerate(splits):
        assert torch.all(out[e] == 0) == (m == 0)


# (zeros beside the tiles, by 64 and by 96 workgroups, and as tiles: too few groups without rows, too long a contraction)
@pytest.mark.parametrize("splits", [[40] + [0] * 29, [2500, 0, 0] * 16, [300, 0, 7] * 10, [3000] + [0] * 29], ids=lambda s: f"{len(s)}groups_{sum(s)}rows")
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_zeros_by_either_way(dev, splits, dtype):
    from atorch_amd import kernels

    E, M = len(splits), sum(splits)
    N, K = (2048, 1536) if M == 40000 else (256, 384)
    goff = kernels.group_offsets_from_splits(splits, dev)
    ld = kernels.padded_bound(M, E)
    h = kernels.host()
    _, _, qx, sx = h.dual(torch.randn((M, K), device=dev, dtype=torch.bfloat16), goff, E, 0.0, ld, False, True)
    _, _, qd, sd = h.dual(torch.randn((M, N), device=dev, dtype=torch.bfloat16), goff, E, 0.0, ld, False, True)
    out = torch.full((E, N, K), 7.0, dtype=dtype, device=dev)
    kernels.grouped_gemm_wgrad(qd, sd, qx, sx, goff, out=out, out_dtype=dtype)
    with kernels.gemm_options(tile=0):  # (a workgroup for every tile)
        want = kernels.grouped_gemm_wgrad(qd, sd, qx, sx, goff, out_dtype=dtype)
    assert torch.equal(out, want)
    before = out.clone()
    kernels.grouped_gemm_wgrad(qd, sd, qx, sx, goff, out=out, out_dtype=dtype, accumulate=True)
    empty = torch.tensor(splits, device=dev) == 0
    assert torch.all(out[empty] == 0) and not torch.equal(out[~empty], before[~empty])
