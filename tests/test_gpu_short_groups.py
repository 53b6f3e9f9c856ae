"""Weight gradients of groups of few rows, whose tiles a workgroup takes several at a time: bit-equal to the kernel of one
tile per workgroup (the same sums in the same order), for lists of short, long and empty groups in every order, runs that
cross a row of tiles and a group, one tile per group, one group, the most groups of the rule and one more."""
import pytest
import torch

from helpers import randn_bf16

pytestmark = pytest.mark.gpu

SPLITS = [
    [300, 0, 1111, 128, 77],  # long groups (more than 512 rows) between short ones, remainders of every kind
    [0, 0, 1, 0],
    [512, 513, 511, 640, 0, 129],
    [1],
    [700],
    [0],
    [0, 2000, 0, 1500, 1025],  # no short group but empty ones
    [(37 * e) % 260 for e in range(64)],
    [(53 * e) % 700 for e in range(65)],
]


@pytest.mark.parametrize("splits", SPLITS, ids=lambda s: f"{len(s)}groups_{sum(s)}rows")
@pytest.mark.parametrize("N,K", [(128, 128), (640, 384), (256, 2176)])
@pytest.mark.parametrize("blocked", [True, False], ids=["blocked", "rows"])
def test_weight_gradient_of_short_groups(dev, splits, N, K, blocked):
    from atorch_amd import kernels

    E, M = len(splits), sum(splits)
    goff = kernels.group_offsets_from_splits(splits, dev)
    ld = kernels.padded_bound(M, E)
    x, dy = randn_bf16((M, K), 1).to(dev), randn_bf16((M, N), 2, std=1e-2).to(dev)
    h = kernels.host()
    _, _, qx, sx = h.dual(x, goff, E, 0.0, ld, False, blocked)
    _, _, qd, sd = h.dual(dy, goff, E, 0.0, ld, False, blocked)
    base = torch.randn(E, N, K, generator=torch.Generator().manual_seed(3)).to(dev)

    def run():
        acc, acc16 = base.clone(), base.bfloat16()
        res = [kernels.grouped_gemm_wgrad(qd, sd, qx, sx, goff, out_dtype=t) for t in (torch.float32, torch.bfloat16)]
        for a in (acc, acc16):
            kernels.grouped_gemm_wgrad(qd, sd, qx, sx, goff, out=a, accumulate=True)
        return res + [acc, acc16]

    got = run()
    with kernels.gemm_options(tile=0):  # (the measurement library, one tile per workgroup)
        want = run()
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    for e, m in enumerate(splits):
        if m == 0:
            assert torch.all(got[0][e] == 0) and torch.equal(got[2][e], base[e])


@pytest.mark.parametrize("splits,fits", [([128, 256], [1, 0]), ([0, 128, 5000], [1, 1, 0])])
def test_groups_beyond_the_operand_buffers_are_nan(dev, splits, fits):
    """Room for one token block only: a short and a long group that do not fit are written as NaN, and read nowhere."""
    from atorch_amd import kernels

    E, N, K = len(splits), 256, 384
    goff = kernels.group_offsets_from_splits(splits, dev)
    qd = torch.zeros((1, N, 128), dtype=torch.uint8, device=dev).view(kernels.FP8)
    qx = torch.zeros((1, K, 128), dtype=torch.uint8, device=dev).view(kernels.FP8)
    dw = kernels.grouped_gemm_wgrad(qd, torch.ones((1, N), device=dev), qx, torch.ones((1, K), device=dev), goff, out_dtype=torch.float32)
    for e, ok in enumerate(fits):
        assert torch.all(dw[e] == 0) if ok else torch.all(torch.isnan(dw[e]))
