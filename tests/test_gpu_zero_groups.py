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
