"""The grouped GEMM for groups of few rows (one and both of its forms), at the edges of its tiles of 32 and 64 token
rows, its slabs of 8, its split of the contraction over 4 and 8 waves, and around 64 groups; against the float64
definition sum_kb dot_kb * a_s * b_s evaluated on the device.  fp32 outputs: 5e-4 of the larger of value and rms, the bar of
the other fp32 GEMM tests (the fp8 matrix instruction's 128-term dot product is not exactly rounded); bf16: 1e-2."""
import pytest
import torch

from helpers import TILE, randn_bf16, rel_err

pytestmark = pytest.mark.gpu


def _definition(qx, sx, qw, sw, splits, bias):
    xd = qx.float().double() * sx.double().repeat_interleave(TILE, 1)
    out = torch.empty(qx.shape[0], qw.shape[1], dtype=torch.float64, device=qx.device)
    off = 0
    for e, m in enumerate(splits):
        if m:
            wd = qw[e].float().double() * sw[e].double().repeat_interleave(TILE, 0).repeat_interleave(TILE, 1)
            out[off : off + m] = xd[off : off + m] @ wd.t() + (bias[e].double() if bias is not None else 0.0)
        off += m
    return out


@pytest.mark.parametrize("splits,N,K", [
    ([1], 128, 128), ([7, 8, 9], 128, 384), ([0, 31, 32, 33, 0], 256, 1024), ([63, 64, 65], 128, 1152), ([129, 0, 1], 384, 2176),
    ([3] * 63 + [0, 5, 40], 128, 256), ([0] * 70 + [17], 256, 640),
])  # fmt: skip
@pytest.mark.parametrize("form", [2, 3], ids=["tiles", "split"])
@pytest.mark.parametrize("out_dtype,bias", [(torch.float32, torch.bfloat16), (torch.bfloat16, None), (torch.bfloat16, torch.float32)])
def test_few_rows_gemm_matches_the_definition(dev, splits, N, K, form, out_dtype, bias):
    from atorch_amd import kernels

    E, M = len(splits), sum(splits)
    qx, sx = kernels.tile_quant(randn_bf16((M, K), 1).to(dev))
    qw, sw, _, _ = kernels.block_quant_batched(randn_bf16((E, N, K), 2, std=0.05).to(dev))
    b = randn_bf16((E, N), 3).to(bias).to(dev) if bias is not None else None
    goff = kernels.group_offsets_from_splits(splits, dev)
    ref = _definition(qx, sx, qw, sw, splits, b)
    bar = 5e-4 if out_dtype == torch.float32 else 1e-2
    with kernels.gemm_options(tile=form):
        got = kernels.grouped_gemm_nt(qx, sx, qw, sw, goff, out_dtype=out_dtype, bias=b)
        again = kernels.grouped_gemm_nt(qx, sx, qw, sw, goff, out_dtype=out_dtype, bias=b)
        assert rel_err(got.float().cpu(), ref.float().cpu()) <= bar and torch.equal(got, again)
        if E == 1 and b is None:  # one group without offsets
            assert torch.equal(got, kernels.fp8_gemm(qx, sx, qw[0], sw[0], dtype=out_dtype))
    # the library's own choice, whichever kernel it is
    got = kernels.grouped_gemm_nt(qx, sx, qw, sw, goff, out_dtype=out_dtype, bias=b)
    assert rel_err(got.float().cpu(), ref.float().cpu()) <= bar


def test_few_rows_gemm_leaves_other_rows_alone(dev):
    """Rows past the end of a group's tile are computed by no workgroup but their own: the output of rows that no group
    owns stays as it was."""
    from atorch_amd import kernels

    qx, sx = kernels.tile_quant(randn_bf16((50, 256), 1).to(dev))
    qw, sw, _, _ = kernels.block_quant_batched(randn_bf16((2, 128, 256), 2).to(dev))
    goff = torch.tensor([0, 5, 41], dtype=torch.int64, device=dev)
    for form in (2, 3):
        out = torch.full((50, 128), 1e4, dtype=torch.bfloat16, device=dev)
        with kernels.gemm_options(tile=form):
            kernels.grouped_gemm_nt(qx, sx, qw, sw, goff, out=out)
        assert torch.all(out[41:] == 1e4) and out[:41].float().abs().max() < 1e3
