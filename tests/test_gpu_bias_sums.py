"""Bias gradients from the quantisers: the codes are those of the quantiser without sums, the sums those of the bf16
gradient per group, at partial tiles, empty groups and more than 64 groups.  An fp32 sum of n terms, added up tile by
tile, is off by at most n 2^-24 sum |g| (Higham's bound for any order); the bar is that, per column."""
import pytest
import torch

from helpers import randn_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("splits", [[1], [127, 128, 129], [0, 300, 0, 5], [3] * 70 + [0, 400]])
@pytest.mark.parametrize("activation", [None, "gelu", "swiglu"])
def test_column_sums_of_the_quantised_gradient(dev, splits, activation):
    from atorch_amd import kernels

    E, M, N = len(splits), sum(splits), 256
    goff = kernels.group_offsets_from_splits(splits, dev)
    x = randn_bf16((M, N), 1).to(dev)
    dh = randn_bf16((M, N // 2 if activation == "swiglu" else N), 2).to(dev) if activation else None
    q, s, q_t, s_t, sums = kernels.gradient_quant_with_sums(x, goff, E, dh=dh, activation=activation)
    if activation is None:
        g, want = x, kernels.tile_quant_dual_grouped(x, goff, E, blocked=True)
    elif activation == "gelu":
        *want, g = kernels.gelu_tile_quant_dual_grouped(x, goff, E, dh=dh, blocked=True, return_activation=True)
    else:
        *want, g = kernels.swiglu_bwd_tile_quant_dual_grouped(dh, x, goff, E, blocked=True, return_grad=True)
    tiles = sum((m + 127) // 128 for m in splits)
    assert torch.equal(q.view(torch.uint8), want[0].view(torch.uint8)) and torch.equal(s, want[1])
    assert torch.equal(q_t[:tiles].view(torch.uint8), want[2][:tiles].view(torch.uint8)) and torch.equal(s_t[:tiles], want[3][:tiles])
    half = kernels.gradient_quant_with_sums(x, goff, E, dh=dh, activation=activation, sums_dtype=torch.bfloat16)[4]
    assert torch.equal(half, sums.bfloat16())
    off = 0
    for e, m in enumerate(splits):
        part = g[off : off + m].double()
        bound = m * 2.0**-24 * part.abs().sum(0)
        assert torch.all((sums[e].double() - part.sum(0)).abs() <= bound)
        off += m
