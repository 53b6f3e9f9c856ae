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
        if sums:
            for t, first in enumerate(range(0, M, 128)) if E == 1 and not drop else []:
                want = rows[first : first + 128].float().sum(0)
                assert torch.allclose(part[t], want, rtol=1e-5, atol=1e-4, equal_nan=True)
    y = randn_bf16((M, H), 2).to(dev)
    want = kernels.unpermute_probs_grad(dout, y, row_map, k).to(pd)
    d_probs = torch.full_like(probs, 9.0)
    _lib.check(_lib.lib().aamd_unpermute_probs_grad_as(
        dout.data_ptr(), kernels.dtype_code(dt), y.data_ptr(), _lib.BF16, M, H, row_map.data_ptr(), T, k, d_probs.data_ptr(),
        kernels.dtype_code(pd), _lib.stream()))  # fmt: skip
    assert torch.equal(d_probs, want) or (torch.isnan(d_probs) == torch.isnan(want)).all()
