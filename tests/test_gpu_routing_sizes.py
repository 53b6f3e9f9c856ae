"""The routing kernels at the sizes where another of them takes over, the group offsets, the search for a tile's group
past 64 groups, and the combine's backward in one pass, each against a host restatement or the kernels it fuses."""
import pytest
import torch

from helpers import randn_bf16

pytestmark = pytest.mark.gpu


# one workgroup up to 8192 ids (while the counts fit), histogram + placement up to 512 chunks of 1024, four launches beyond
@pytest.mark.parametrize("n,E", [(0, 3), (1, 1), (63, 60), (64, 64), (65, 65), (960, 1024), (1024, 1024), (1025, 60), (8192, 60),
                                 (8193, 60), (70001, 8), (524288, 64), (524289, 64), (30000, 1024)])  # fmt: skip
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32])
def test_preprocess_is_a_stable_counting_sort(dev, n, E, dtype):
    from atorch_amd import kernels

    g = torch.Generator().manual_seed(n + E)
    ids = torch.randint(-1, E + 1, (n,), generator=g)  # some out of range: dropped
    if n > 100:
        ids[: n // 3] = E - 1  # a long run of one expert, across chunks
    sorted_idx, row_map, goff = kernels.moe_preprocess(ids.to(dtype).to(dev), E)
    ok = (ids >= 0) & (ids < E)
    counts = torch.bincount(ids[ok], minlength=E)
    want_off = torch.cat([torch.zeros(1, dtype=torch.int64), counts.cumsum(0)])
    kept = torch.nonzero(ok).flatten()
    order = kept[torch.sort(ids[kept], stable=True).indices]
    want_map = torch.full((n,), -1, dtype=torch.int32)
    want_map[order] = torch.arange(order.numel(), dtype=torch.int32)
    assert torch.equal(goff.cpu(), want_off)
    assert torch.equal(row_map.cpu(), want_map)
    assert torch.equal(sorted_idx.cpu()[: order.numel()], order)


@pytest.mark.parametrize("E", [1, 63, 64, 65, 239, 240, 241, 700])
def test_group_offsets_from_host_and_device_counts(dev, E):
    from atorch_amd import kernels
    from atorch_amd.gmm import _offsets

    g = torch.Generator().manual_seed(E)
    counts = torch.randint(0, 3, (E,), generator=g) * torch.randint(0, 1 << 33, (E,), generator=g)
    want = torch.cat([torch.zeros(1, dtype=torch.int64), counts.cumsum(0)])
    assert torch.equal(kernels.group_offsets_from_splits(counts.tolist(), dev).cpu(), want)
    assert torch.equal(_offsets(counts, dev).cpu(), want)
    assert torch.equal(_offsets(counts.to(dev), dev).cpu(), want)


# 64 groups are one scan of a wave, more take several; the order of the weight gradient's groups changes there too
@pytest.mark.parametrize("E", [63, 64, 65, 130])
def test_grouped_kernels_find_their_group_around_64_groups(dev, E):
    from atorch_amd import kernels

    K, N = 128, 256
    g = torch.Generator().manual_seed(E)
    splits = (torch.randint(0, 3, (E,), generator=g) * torch.randint(1, 90, (E,), generator=g)).tolist()
    splits[E // 2] = 700  # one busy group, so that the groups fall into the classes of the order
    splits[0] = 0
    M = sum(splits)
    x, dy, w = randn_bf16((M, K), 1).to(dev), randn_bf16((M, N), 2).to(dev), randn_bf16((E, N, K), 3).to(dev)
    goff = kernels.group_offsets_from_splits(splits, dev)
    qx, sx, qx_t, sx_t = kernels.tile_quant_dual_grouped(x, goff, E, blocked=True)
    _, _, qd_t, sd_t = kernels.tile_quant_dual_grouped(dy, goff, E, blocked=True, rowwise=False)
    qw, sw, _, _ = kernels.block_quant_batched(w)
    y = kernels.grouped_gemm_nt(qx, sx, qw, sw, goff, out_dtype=torch.float32)
    dw = kernels.grouped_gemm_wgrad(qd_t, sd_t, qx_t, sx_t, goff)
    off = 0
    for e, m in enumerate(splits):
        if m:  # the group alone, without offsets or with its own
            q1, s1, q1_t, s1_t = kernels.host().dual(x[off : off + m], None, 1, 0.0, kernels.padded_total([m]), True, True)
            assert torch.equal(q1.view(torch.uint8), qx[off : off + m].view(torch.uint8))
            assert torch.equal(y[off : off + m], kernels.fp8_gemm(q1, s1, qw[e], sw[e], dtype=torch.float32))
            _, _, d1_t, t1_t = kernels.host().dual(dy[off : off + m], None, 1, 0.0, kernels.padded_total([m]), True, True)
            one = kernels.grouped_gemm_wgrad(d1_t, t1_t, q1_t, s1_t, kernels.group_offsets_from_splits([m], dev))
            assert torch.equal(dw[e], one[0])
        else:
            assert torch.all(dw[e] == 0)
        off += m


@pytest.mark.parametrize("T,H,k,rows,weights", [(1, 8, 1, "bf16", "bf16"), (33, 128, 2, "bf16", "f32"), (7, 7168, 5, "bf16", "bf16"),
                                                (5, 8200, 8, "f32", "bf16"), (3, 256, 13, "f32", "f32")])  # fmt: skip
@pytest.mark.parametrize("drop", [False, True])
def test_unpermute_backward_equals_the_two_kernels(dev, T, H, k, rows, weights, drop):
    from atorch_amd import kernels

    dt = {"bf16": torch.bfloat16, "f32": torch.float32}
    g = torch.Generator().manual_seed(T * k)
    M = T * k - (1 if drop and T * k > 1 else 0)
    row_map = torch.randperm(T * k, generator=g).to(torch.int32)
    row_map[row_map >= M] = -1
    y = randn_bf16((M, H), 1).to(dt[rows]).to(dev)
    probs = torch.rand((T, k), generator=g).to(dt[weights]).to(dev)
    dout = randn_bf16((T, H), 2).to(torch.promote_types(dt[rows], dt[weights])).to(dev)
    row_map = row_map.to(dev)
    d_rows, d_probs = kernels.unpermute_backward(dout, y, row_map, probs, k)
    assert torch.equal(d_rows, kernels.permute_rows_scaled(dout, row_map, k, M, probs, y.dtype))
    want = kernels.unpermute_probs_grad(dout, y, row_map, k).to(probs.dtype)
    # sums of the same fp32 products in the same order, lane by lane
    assert d_probs.dtype == probs.dtype and torch.equal(d_probs, want)
