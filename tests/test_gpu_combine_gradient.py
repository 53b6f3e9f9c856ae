"""The combine's gradient quantised without being written: the bits of the kernels that write it and quantise what was written, with the
column sums and the weights' gradient beside it, for dropped copies, partial tiles, empty groups and both types on either side."""
import pytest
import torch

from helpers import randn_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,k,E,H", [(1, 1, 1, 128), (130, 2, 4, 384), (77, 3, 66, 1024), (300, 8, 9, 128), (257, 1, 2, 1152)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("pd", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("drop", [False, True])
def test_bits_of_the_separate_kernels(dev, T, k, E, H, dt, pd, drop):
    from atorch_amd import _lib, kernels

    g = torch.Generator().manual_seed(T + k)
    ids = torch.randint(E + (1 if drop else 0), (T, k), generator=g).to(dev)  # id E: dropped
    sorted_idx, row_map, goff = kernels.moe_preprocess(ids, E)
    n, M = int(goff[-1]), T * k
    dout = torch.randn((T, H), generator=g).to(dt).to(dev)
    probs = torch.rand((T, k), generator=g).to(pd).to(dev)
    dout[0, :128] = 0.0
    dout[-1, -3] = float("inf")
    probs[T // 2, 0] = 0.0
    ld = kernels.padded_bound(M, E)
    rows = kernels.permute_rows_scaled(dout, row_map, k, M, probs, torch.bfloat16)
    q, s, q_t, s_t, _ = (kernels.host().dual_with_sums(0, rows, None, goff, E, ld, 0.0, torch.float32))
    tiles = sum((m + 127) // 128 for m in (goff[1:] - goff[:-1]).tolist())
    for sums in (False, True):
        got = [torch.full_like(t.view(torch.uint8) if t.dtype == kernels.FP8 else t, 7) for t in (q, s, q_t, s_t)]
        part = torch.zeros((ld // 128, H), device=dev)
        _lib.check(_lib.lib().aamd_combine_grad_quant_1x128_dual_grouped(
            dout.data_ptr(), kernels.dtype_code(dt), T, H, sorted_idx.data_ptr(), k, M, probs.data_ptr(), kernels.dtype_code(pd),
            goff.data_ptr(), E, *[t.data_ptr() for t in got], ld, 1, part.data_ptr() if sums else None, _lib.stream()))  # fmt: skip
        for a, b in zip(got, (q.view(torch.uint8), s, q_t.view(torch.uint8), s_t)):
            m = tiles if a.shape[0] == ld // 128 else n
            assert torch.equal(a[:m], b[:m])
        if sums:  # every tile of every group, in fp32 over its at most 128 rows
            at = 0
            for e in range(E):
                for first in range(int(goff[e]), int(goff[e + 1]), 128):
                    tile = rows[first : min(first + 128, int(goff[e + 1]))].double()
                    bound = 1e-5 * tile.abs().sum(0).nan_to_num(0, 0, 0)  # (128 roundings of 2^-24 of it at most)
                    finite = torch.isfinite(tile).all(0)
                    assert torch.all((part[at].double() - tile.sum(0)).abs()[finite] <= bound[finite])
                    assert torch.equal(torch.isfinite(part[at]), finite)
                    at += 1
            assert at == tiles
    y = randn_bf16((M, H), 2).to(dev)
    d_probs = torch.full_like(probs, 9.0)
    _lib.check(_lib.lib().aamd_unpermute_probs_grad_as(
        dout.data_ptr(), kernels.dtype_code(dt), y.data_ptr(), _lib.BF16, M, H, row_map.data_ptr(), T, k, d_probs.data_ptr(),
        kernels.dtype_code(pd), _lib.stream()))  # fmt: skip
    if dt == pd:  # the kernel that makes both gradients
        want = kernels.unpermute_backward(dout, y, row_map, probs, k)[1]
        torch.testing.assert_close(d_probs, want, rtol=0, atol=0, equal_nan=True)
    gone = (row_map < 0).view(T, k)
    products = y.double()[row_map.long().clamp(min=0)].view(T, k, H) * dout.double()[:, None]
    want = torch.where(gone, 0.0, products.sum(-1))
    finite = torch.isfinite(want)
    # (H roundings of 2^-24 of the products' sum at most, and that of the result)
    bound = H * 2.0**-24 * products.abs().sum(-1) + (2.0**-8 if pd == torch.bfloat16 else 2.0**-24) * want.abs()
    assert torch.all((d_probs.double() - want).abs()[finite] <= bound[finite]) and torch.equal(torch.isfinite(d_probs), finite)


@pytest.mark.parametrize("dt,yt", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.bfloat16), (torch.float32, torch.float32),
                                   (torch.bfloat16, torch.float32)])  # fmt: skip
@pytest.mark.parametrize("k", [1, 3, 8, 11])
def test_a_dropped_copy_has_no_gradient(dev, dt, yt, k):
    """Whatever its token's gradient holds: nothing is multiplied for a slot without a row."""
    from atorch_amd import kernels

    T, H, M = 9, 136, 9 * k
    g = torch.Generator().manual_seed(k)
    row_map = torch.randperm(M, generator=g).int()
    row_map[torch.rand(M, generator=g) < 0.5] = -1
    dout, y = torch.randn((T, H), generator=g).to(dt).to(dev), torch.randn((M, H), generator=g).to(yt).to(dev)
    dout[2], dout[4, 7], dout[5, 130] = float("inf"), float("-inf"), float("nan")
    row_map = row_map.to(dev)
    got = kernels.unpermute_probs_grad(dout, y, row_map, k)
    dropped = (row_map < 0).view(T, k)
    assert dropped[[2, 4, 5]].any() and torch.all(got[dropped] == 0)
    rows = y.float()[row_map.long().clamp(min=0)].view(T, k, H)
    want = torch.where(dropped, 0.0, (rows * dout.float()[:, None]).sum(-1))
    # (sums of 136 products of about 1 in two orders)
    torch.testing.assert_close(got, want, rtol=1e-4, atol=1e-4, equal_nan=True)


@pytest.mark.parametrize("pd", [torch.bfloat16, torch.float32])
def test_layer_with_dropped_copies_and_a_gradient_that_is_not_finite(dev, pd):
    """Expert ids out of range: the router weights' gradient is 0 there, and the layer's own unfused path (a shared expert that adds
    nothing) gives the same one."""
    from atorch_amd.moe_layer import Grouped_GEMM_MoE

    T, H, F, E, k = 96, 256, 128, 4, 2
    torch.manual_seed(3)
    layer = Grouped_GEMM_MoE(H, F, 0.0, E, k, use_swiglu=True, implementation_type="Megatron", device=dev, dtype=torch.bfloat16)
    ids = torch.stack([torch.randperm(E)[:k] for _ in range(T)])
    ids[::3, 1], ids[1::5, 0] = E, -1
    x, dout = randn_bf16((T, H), 4).to(dev), torch.randn(T, H).to(pd).to(dev)
    dout[0], dout[1, 3], dout[6, 9] = float("inf"), float("-inf"), float("nan")
    grads = []
    for kw in ({}, dict(se_fn1=lambda h: h, se_fn2=lambda h: torch.zeros_like(h))):
        probs = torch.full((T, k), 0.5, dtype=pd, device=dev, requires_grad=True)
        layer(x, probs, ids.to(dev), **kw).backward(dout)
        grads.append(probs.grad)
    assert torch.all(grads[0][(ids < 0) | (ids >= E)] == 0)
    torch.testing.assert_close(grads[0], grads[1], rtol=0, atol=0, equal_nan=True)


# (written first -> gathered: 20.4 -> 24.5 us, 396 -> 421, 9.9 -> 10.3, 29.4 -> 31.5; 107 -> 86, 92 -> 88, 16.0 -> 12.1)
@pytest.mark.parametrize("T,k,H,bf16,want_probs,gathers", [(500, 4, 4096, False, True, False), (16384, 8, 2048, False, True, False), (64, 2, 512, True, True, False),
                                                           (1000, 8, 2048, False, False, False), (8191, 4, 2048, True, True, True),
                                                           (8191, 4, 2048, False, False, True), (300, 8, 2048, False, False, True)])  # fmt: skip
def test_gathered_where_it_is_faster(T, k, H, bf16, want_probs, gathers):
    from atorch_amd import kernels

    assert kernels.host().gathers_gradient(T * k, H, k, bf16, want_probs) == gathers


# (below and above the lines of the rule)
@pytest.mark.parametrize("T,k,H,E", [(40, 2, 256, 4), (333, 8, 512, 9), (2100, 8, 512, 9)])
@pytest.mark.parametrize("pd", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("want_probs", [True, False])
@pytest.mark.parametrize("bias", [True, False])
def test_layer_gradients_are_those_of_its_parts(dev, T, k, H, E, pd, want_probs, bias):
    from atorch_amd.moe_layer import Grouped_GEMM_MoE

    torch.manual_seed(T)
    layer = Grouped_GEMM_MoE(H, 128, 0.0, E, k, use_swiglu=not bias, use_bias=bias, implementation_type="Megatron", device=dev, dtype=torch.bfloat16)
    ids = torch.stack([torch.randperm(E)[:k] for _ in range(T)])
    ids[::7, 0] = E
    x, dout, probs = randn_bf16((T, H), 4).to(dev), (torch.randn(T, H) * 0.1).to(pd).to(dev), torch.rand(T, k).to(pd).to(dev)
    grads = []
    for kw in ({}, dict(se_fn1=lambda h: h, se_fn2=lambda h: torch.zeros_like(h))):
        layer.zero_grad(set_to_none=True)
        xg, pg = x.clone().requires_grad_(True), probs.clone().requires_grad_(want_probs)
        layer(xg, pg, ids.to(dev), **kw).backward(dout)
        grads.append([xg.grad, pg.grad] + [p.grad for p in layer.parameters()])
    for a, b in zip(*grads):
        assert (a is None and b is None) or torch.equal(a, b)
