"""The row-ragged GEMM on 256 x 256 tiles, whose workgroups take one tile after the other (at most 256 of them): several tiles
per workgroup and less than one, even and odd numbers of 128-deep steps around the batches of eight blocks of scales, rows of
scales that are 16-byte aligned and not, half tiles of outputs, tiles of one row next to full ones, more than 64 groups and
empty ones.  The 128 x 128 tiles add the same products in the same order, so that the results are the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("splits,N,K", [
    ([1], 128, 1024), ([8192], 4096, 1152), ([8191], 4224, 1024), ([300, 0, 5000, 257, 1, 3000], 2176, 1280),
    ([800] * 60, 1024, 1408), ([257] * 70 + [0, 1, 255], 640, 2048), ([256, 1] * 32, 1152, 1664), ([4097, 4095], 2048, 2176),
    ([129] * 130, 384, 1920),
])  # fmt: skip
@pytest.mark.parametrize("out_dtype,bias", [(torch.bfloat16, None), (torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("turned", [False, True])
def test_large_tiles_give_the_bits_of_small_ones(dev, splits, N, K, out_dtype, bias, turned):
    from atorch_amd import kernels

    E, M = len(splits), sum(splits)
    g = torch.Generator(device=dev).manual_seed(7)
    qx, sx = kernels.tile_quant(torch.randn((M, K), generator=g, device=dev).bfloat16())
    w = torch.randn((E, K, N) if turned else (E, N, K), generator=g, device=dev).bfloat16() * 0.05
    q, s, q_t, s_t = kernels.block_quant_batched(w, return_transpose=True, written=kernels.STORED)
    if turned:
        q, s = q_t, s_t
    b = torch.randn((E, N), generator=g, device=dev).to(bias) if bias is not None else None
    goff = kernels.group_offsets_from_splits(splits, dev)
    got = {}
    for tile in (0, 1):
        out = torch.full((M + 3, N), 7.0, dtype=out_dtype, device=dev)  # rows behind the last one stay as they are
        with kernels.gemm_options(tile=tile):
            kernels.grouped_gemm_nt(qx, sx, q, s, goff, out=out[:M], bias=b)
        got[tile] = out
    assert torch.equal(got[0], got[1]) and torch.all(got[1][M:] == 7.0)


@pytest.mark.parametrize("splits,N,K", [
    ([1], 128, 1024), ([2047], 1152, 1152), ([300, 0, 257, 1, 700], 896, 1280), ([33] * 70 + [0, 1, 255], 384, 2176),
])  # fmt: skip
@pytest.mark.parametrize("out_dtype,bias", [(torch.bfloat16, None), (torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("turned", [False, True])
def test_a_workgroup_per_tile_gives_the_same_bits(dev, splits, N, K, out_dtype, bias, turned):
    """The form that launches of one round of tiles take."""
    from atorch_amd import kernels

    E, M = len(splits), sum(splits)
    g = torch.Generator(device=dev).manual_seed(10)
    qx, sx = kernels.tile_quant(torch.randn((M, K), generator=g, device=dev).bfloat16())
    w = torch.randn((E, K, N) if turned else (E, N, K), generator=g, device=dev).bfloat16() * 0.05
    q, s, q_t, s_t = kernels.block_quant_batched(w, return_transpose=True, written=kernels.STORED)
    if turned:
        q, s = q_t, s_t
    b = torch.randn((E, N), generator=g, device=dev).to(bias) if bias is not None else None
    goff = kernels.group_offsets_from_splits(splits, dev)
    got = {}
    for tile in (0, 4):
        out = torch.full((M + 3, N), 7.0, dtype=out_dtype, device=dev)
        with kernels.gemm_options(tile=tile):
            kernels.grouped_gemm_nt(qx, sx, q, s, goff, out=out[:M], bias=b)
        got[tile] = out
    assert torch.equal(got[0], got[4]) and torch.all(got[4][M:] == 7.0)


def test_output_rows_apart(dev):
    """Columns between the rows of a wider output are not touched."""
    from atorch_amd import kernels

    g = torch.Generator(device=dev).manual_seed(8)
    splits, N, K = [700, 3, 900], 640, 1024
    qx, sx = kernels.tile_quant(torch.randn((sum(splits), K), generator=g, device=dev).bfloat16())
    qw, sw, _, _ = kernels.block_quant_batched(torch.randn((3, N, K), generator=g, device=dev).bfloat16())
    goff = kernels.group_offsets_from_splits(splits, dev)
    wide = torch.full((sum(splits), N + 64), 7.0, dtype=torch.bfloat16, device=dev)
    with kernels.gemm_options(tile=1):
        kernels.grouped_gemm_nt(qx, sx, qw, sw, goff, out=wide[:, :N])
    with kernels.gemm_options(tile=0):
        want = kernels.grouped_gemm_nt(qx, sx, qw, sw, goff)
    assert torch.equal(wide[:, :N], want) and torch.all(wide[:, N:] == 7.0)


# Tiles left in the last round of an XCD: 2, 4 and 5, 12, 8, 11 and 12 (more than 64 groups); the last two launches
# do not share.
@pytest.mark.parametrize("splits,N,K,shared", [
    ([4224], 4096, 6144, True), ([4097], 4224, 6528, True), ([300, 0, 2500, 257, 1, 1700], 4096, 6144, True),
    ([257, 257, 4096], 3968, 6272, True), ([256] * 69 + [1], 1280, 6144, True),
    ([4096, 2200], 4096, 6144, False), ([1, 600], 512, 14336, False),
])  # fmt: skip
@pytest.mark.parametrize("out_dtype,bias", [(torch.float32, None), (torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("turned", [False, True])
def test_parts_of_the_contraction(dev, splits, N, K, shared, out_dtype, bias, turned):
    """A split row has the same products in up to eight sums.  Against 64 bits both forms stay below the worst rounding of nkb
    sequential additions, and the split form's error, of shorter sums, is no larger on the whole.  Rows behind the last one and
    launches that do not split are as without a workspace."""
    from atorch_amd import _lib, kernels

    E, M, nkb = len(splits), sum(splits), K // 128
    g = torch.Generator(device=dev).manual_seed(9)
    qx, sx = kernels.tile_quant(torch.randn((M, K), generator=g, device=dev).bfloat16())
    w = torch.randn((E, K, N) if turned else (E, N, K), generator=g, device=dev).bfloat16() * 0.05
    q, s, q_t, s_t = kernels.block_quant_batched(w, return_transpose=True, written=kernels.STORED)
    b = torch.randn((E, N), generator=g, device=dev).to(bias) if bias is not None else None
    goff = kernels.group_offsets_from_splits(splits, dev)
    ws = torch.full((1 << 24,), float("nan"), device=dev)
    code, bias_code = kernels.dtype_code(out_dtype), kernels.dtype_code(b.dtype) if b is not None else _lib.NONE

    def run(ws):
        out = torch.full((M + 3, N), 7.0, dtype=out_dtype, device=dev)
        _lib.check(_lib.lib().aamd_grouped_gemm_fp8_ws(
            qx.data_ptr(), K, sx.data_ptr(), q.data_ptr(), s.data_ptr(), int(turned), goff.data_ptr(), E, M, N, K, out.data_ptr(), code, N,
            b.data_ptr() if b is not None else None, bias_code, ws.data_ptr() if ws is not None else None,
            ws.numel() * 4 if ws is not None else 0, _lib.stream()))  # fmt: skip
        return out

    with_ws, without = run(ws), run(None)
    assert torch.all(with_ws[M:] == 7.0)
    assert shared == (not torch.isnan(ws).all())
    if not shared:
        assert torch.equal(with_ws, without)
        return
    ws2 = torch.zeros_like(ws)
    assert torch.equal(run(ws2), with_ws)
    # 64-bit sums of the dequantised operands; |a||b| beside them for the bound
    at = 0
    err = {0: 0.0, 1: 0.0}
    for e, m in enumerate(splits):
        rows = slice(at, at + m)
        at += m
        if m == 0:
            continue
        x = (qx[rows].float().view(m, nkb, 128) * sx[rows].unsqueeze(-1)).view(m, K).double()
        sw = s[e].repeat_interleave(128, 0).repeat_interleave(128, 1)
        wt = (q[e].float() * sw).double()
        wt = wt if turned else wt.t().contiguous()
        want, size = x @ wt, x.abs() @ wt.abs()
        if b is not None:
            want, size = want + b[e].double(), size + b[e].double().abs()
        for i, got in enumerate((without, with_ws)):
            d = (got[rows].double() - want).abs()
            # (bf16 keeps 8 bits: rounding to nearest is off by at most 2^-8 of the value; 1.01 for the error of the value itself)
            half = want.abs() * 2.0**-8 * 1.01 if out_dtype == torch.bfloat16 else 0.0
            assert torch.all(d <= half + (nkb + 8) * 2.0**-23 * size)
            err[i] += float((d * d).sum())
    assert err[1] <= 1.02 * err[0]
