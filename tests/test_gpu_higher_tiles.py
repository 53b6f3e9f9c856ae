"""Row tiles of up to 288 rows, which take the rows of a group beyond its full tiles: bit-equal to the 128 x 128 tiles (the same sums
in the same order) for remainders of one row to 32 a tile, one more than the tiles take, groups of less than a tile, empty ones, more
than 64, an odd number of steps, half tiles of outputs, weights along either side and a bias; with the last round's tiles in
parts, with an eighth of every group for each XCD, and without groups; streamed past the caches; and where the groups' rows decide between
them and tiles of 256."""
import pytest
import torch

from helpers import rel_err
from test_gemm_choice import HIGHER, LARGE_TILES, SHARED, choice

pytestmark = pytest.mark.gpu


def operands(dev, splits, N, K, turned):
    from atorch_amd import kernels

    E, M = len(splits), sum(splits)
    g = torch.Generator(device=dev).manual_seed(M + N)
    qx, sx = kernels.tile_quant(torch.randn((M, K), generator=g, device=dev).bfloat16())
    w = torch.randn((E, K, N) if turned else (E, N, K), generator=g, device=dev).bfloat16() * 0.05
    q, s, q_t, s_t = kernels.block_quant_batched(w, return_transpose=True, written=kernels.STORED)
    return (qx, sx, q_t, s_t) if turned else (qx, sx, q, s)


@pytest.mark.parametrize("splits,N,K", [
    ([264], 256, 1024), ([288], 384, 1152), ([289], 256, 1024), ([520, 300, 0, 255, 256, 257, 1], 384, 1024), ([576, 577], 1152, 1408),
    ([2303, 256 * 9 + 33], 640, 1152), ([4100, 777, 0, 545], 1024, 2048), ([(37 * e) % 330 for e in range(70)], 384, 1024),
])  # fmt: skip
@pytest.mark.parametrize("out_dtype,bias", [(torch.bfloat16, None), (torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("turned", [False, True])
def test_higher_tiles_give_the_bits_of_small_ones(dev, splits, N, K, out_dtype, bias, turned):
    from atorch_amd import kernels

    E, M = len(splits), sum(splits)
    ops, goff = operands(dev, splits, N, K, turned), kernels.group_offsets_from_splits(splits, dev)
    b = torch.randn((E, N), generator=torch.Generator(device=dev).manual_seed(1), device=dev).to(bias) if bias is not None else None
    got = {}
    for tile in (0, 6):
        out = torch.full((M + 3, N), 7.0, dtype=out_dtype, device=dev)  # rows behind the last one stay as they are
        with kernels.gemm_options(tile=tile):
            kernels.grouped_gemm_nt(*ops, goff, out=out[:M], bias=b)
        got[tile] = out
    assert torch.equal(got[0], got[6]) and torch.all(got[6][M:] == 7.0)


# (slices of the groups for every XCD: the rule says yes, yes, yes, and no three times, of which the last is not asked: seven tiles a group)
@pytest.mark.parametrize("splits,yes", [([264] * 8, True), ([270, 513, 520, 0, 530, 264], True), ([260, 0, 513, 515, 288], True), ([768 + 30, 300], False),
                                        ([600, 640, 630, 10], False), ([20000, 264, 264], False)])  # fmt: skip
@pytest.mark.parametrize("turned", [False, True])
def test_either_by_the_rows_of_the_groups(dev, splits, yes, turned):
    from atorch_amd import kernels

    N, K = 20480, 1024
    assert (choice(sum(splits), N, K // 128, len(splits), 1, int(turned), 0, splits) == HIGHER) == yes
    ops, goff = operands(dev, splits, N, K, turned), kernels.group_offsets_from_splits(splits, dev)
    got = kernels.grouped_gemm_nt(*ops, goff)
    with kernels.gemm_options(tile=0):
        assert torch.equal(kernels.grouped_gemm_nt(*ops, goff), got)


def with_workspace(dev, ops, goff, E, M, N, K, out_dtype, turned, bias=None):
    from atorch_amd import _lib, kernels

    out, ws = torch.full((M + 3, N), 7.0, dtype=out_dtype, device=dev), torch.full((1 << 24,), float("nan"), device=dev)
    _lib.check(_lib.lib().aamd_grouped_gemm_fp8_ws(
        ops[0].data_ptr(), K, ops[1].data_ptr(), ops[2].data_ptr(), ops[3].data_ptr(), int(turned), goff.data_ptr() if goff is not None else None, E, M,
        N, K, out.data_ptr(), kernels.dtype_code(out_dtype), N, bias.data_ptr() if bias is not None else None,
        kernels.dtype_code(bias.dtype) if bias is not None else _lib.NONE, ws.data_ptr(), ws.numel() * 4, _lib.stream()))  # fmt: skip
    assert torch.all(out[M:] == 7.0)
    return out[:M], ws


def tolerance(K, out_dtype):
    # (sums of nkb products of like size: an addition rounds by at most 2^-24 of a partial sum, which stays below sqrt(nkb) of the
    # result's root mean square times 4; two sums on either side of a rounding give neighbours in bf16, up to 2^-7 apart)
    return K / 128 * 2.0**-24 * 4 + (2.0**-7 if out_dtype == torch.bfloat16 else 0.0)


# 16 R tiles (no slices), and 32 to 33, whose tiles an XCD takes by slices of every group: 4 to 11 of them in its last round
PARTS = [([264] * 17, 4096, 6144), ([520] * 9, 3968, 6272), ([257, 780, 780, 780, 520, 577, 530], 4224, 6272), ([264] * 9, 8192, 6144),
         ([300, 0, 780, 288, 288, 530, 520, 520, 0, 577, 300], 8320, 6144), ([288, 545, 530, 520, 281, 545, 545, 288, 0, 577, 270], 8320, 6272),
         ([257, 264, 780, 281, 520, 530, 520, 257, 281, 288, 264], 8448, 6144)]  # fmt: skip


@pytest.mark.parametrize("splits,N,K", PARTS)
@pytest.mark.parametrize("out_dtype,bias", [(torch.float32, None), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("turned", [False, True])
def test_parts_of_higher_tiles(dev, splits, N, K, out_dtype, bias, turned):
    """Tiles of more than 256 rows in the last round, in parts.  At most eight sums a row instead of one, of the same products: an fp32
    result may differ by the rounding of nkb additions, and a bf16 one by what its own rounding makes of that."""
    from atorch_amd import kernels

    E, M = len(splits), sum(splits)
    assert choice(M, N, K // 128, E, 1, int(turned), 1, splits) == HIGHER
    ops, goff = operands(dev, splits, N, K, turned), kernels.group_offsets_from_splits(splits, dev)
    b = torch.randn((E, N), generator=torch.Generator(device=dev).manual_seed(1), device=dev).to(bias) if bias is not None else None
    got, ws = with_workspace(dev, ops, goff, E, M, N, K, out_dtype, turned, b)
    assert not torch.isnan(ws).all()
    with kernels.gemm_options(tile=0):
        want = kernels.grouped_gemm_nt(*ops, goff, out_dtype=out_dtype, bias=b)
    assert rel_err(got, want) <= tolerance(K, out_dtype)


# The parts of the second XCD begin behind 28 places of 288 rows, or behind 32 of 256, of which these launches fill at most 30.
@pytest.mark.parametrize("splits,N,K,yes", [(*PARTS[0], True), (*PARTS[4], True), (*PARTS[6], True), ([270, 530, 513, 1, 300], 8448, 6272, False),
                                            ([288, 513, 257, 0, 577, 780, 545], 8320, 6272, False), ([512] * 9, 4096, 6144, False),
                                            ([1, 577, 513, 780, 530, 270, 257], 8448, 6272, False)])  # fmt: skip
def test_the_device_decides_as_the_rule_says(dev, splits, N, K, yes):
    from atorch_amd import kernels

    E, M = len(splits), sum(splits)
    assert choice(M, N, K // 128, E, 1, 0, 1, splits) == (HIGHER if yes else SHARED) and choice(M, N, K // 128, E, 1, 0, 1) in (LARGE_TILES, SHARED)
    ops, goff = operands(dev, splits, N, K, False), kernels.group_offsets_from_splits(splits, dev)
    _, ws = with_workspace(dev, ops, goff, E, M, N, K, torch.bfloat16, False)
    assert not torch.isnan(ws).all() and bool(torch.isnan(ws[28 * 288 * 256])) != yes


@pytest.mark.parametrize("M,N,K", [(264, 256, 1024), (288, 384, 1152), (289, 256, 1024), (545, 1152, 1152), (1288, 2176, 1408)])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("turned", [False, True])
def test_higher_tiles_without_groups(dev, M, N, K, out_dtype, turned):
    from atorch_amd import _lib, _probes, kernels

    ops = operands(dev, [M], N, K, turned)
    got = {}
    for tile in (0, 6):
        got[tile] = torch.full((M + 3, N), 7.0, dtype=out_dtype, device=dev)
        args = [ops[0].data_ptr(), K, ops[1].data_ptr(), ops[2].data_ptr(), ops[3].data_ptr()] + ([] if turned else [0]) + [None, 1] + ([] if turned else [None])
        entry = _probes.lib().aamd_tuning_grouped_gemm_fp8_nn if turned else _probes.lib().aamd_tuning_grouped_gemm_fp8_nt
        _probes.check(entry(*args, M, N, K, got[tile].data_ptr(), kernels.dtype_code(out_dtype), N, None, _lib.NONE, _probes.options_array({"tile": tile}), _lib.stream()))
    assert torch.equal(got[0], got[6]) and torch.all(got[6][M:] == 7.0)


# (with a workspace: 8, 2 and 4 tiles of an XCD in the last round, in parts)
@pytest.mark.parametrize("M,N,K,workspace", [(1288, 12032, 1024, False), (1045, 15360, 1152, False), (1032, 20480, 6144, True), (545, 34816, 6272, True),
                                             (520, 36864, 6144, True)])  # fmt: skip
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("turned", [False, True])
def test_higher_tiles_chosen_without_groups(dev, M, N, K, workspace, out_dtype, turned):
    from atorch_amd import _lib, kernels

    assert choice(M, N, K // 128, 1, 0, int(turned), int(workspace)) == HIGHER
    ops = operands(dev, [M], N, K, turned)
    with kernels.gemm_options(tile=0):
        want = kernels.grouped_gemm_nt(*ops, kernels.group_offsets_from_splits([M], dev), out_dtype=out_dtype)
    if workspace:
        got, ws = with_workspace(dev, ops, None, 1, M, N, K, out_dtype, turned)
        assert not torch.isnan(ws).all() and rel_err(got, want) <= tolerance(K, out_dtype)
        return
    got = torch.empty_like(want)
    _lib.check(_lib.lib().aamd_grouped_gemm_fp8_ws(
        ops[0].data_ptr(), K, ops[1].data_ptr(), ops[2].data_ptr(), ops[3].data_ptr(), int(turned), None, 1, M, N, K, got.data_ptr(),
        kernels.dtype_code(out_dtype), N, None, _lib.NONE, None, 0, _lib.stream()))  # fmt: skip
    assert torch.equal(got, want)


@pytest.mark.parametrize("K", [4096, 4224])
@pytest.mark.parametrize("out_dtype,N", [(torch.float32, 32768), (torch.bfloat16, 65536)])
def test_higher_tiles_streamed_past_the_caches(dev, K, out_dtype, N):
    """An output of 256 MB or more and 32 steps or more."""
    from atorch_amd import kernels

    splits = [1050, 0, 1022]
    assert sum(splits) * N * out_dtype.itemsize >= 1 << 28
    qx, sx, q, s = operands(dev, [sum(splits)], N, K, False)
    ops, goff = (qx, sx, q.expand(3, N, K).contiguous(), s.expand(3, *s.shape[1:]).contiguous()), kernels.group_offsets_from_splits(splits, dev)
    got = {}
    for tile in (0, 6):
        with kernels.gemm_options(tile=tile):
            got[tile] = kernels.grouped_gemm_nt(*ops, goff, out_dtype=out_dtype)
    assert torch.equal(got[0], got[6])


@pytest.mark.parametrize("splits", [[288], [287, 0, 1]])
def test_rows_as_far_apart_as_is_taken(dev, splits):
    """288 rows of nearly 8 MB: their last byte lies beyond what a signed 32-bit offset reaches."""
    from atorch_amd import kernels

    N, K, M, lda = 384, 1024, sum(splits), (1 << 23) - 16
    qx, *rest = operands(dev, splits, N, K, False)
    goff = kernels.group_offsets_from_splits(splits, dev)
    far = torch.empty((M - 1) * lda + K, dtype=torch.uint8, device=dev).view(qx.dtype).as_strided((M, K), (lda, 1))
    far.view(torch.uint8).copy_(qx.view(torch.uint8))
    with kernels.gemm_options(tile=0):
        want = kernels.grouped_gemm_nt(qx, *rest, goff)
    with kernels.gemm_options(tile=6):
        assert torch.equal(kernels.grouped_gemm_nt(far, *rest, goff), want)
