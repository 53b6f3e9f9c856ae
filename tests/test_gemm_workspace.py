"""The workspace that a row-ragged GEMM asks for: none where no tile's contraction can be shared out."""
import pytest


def _bytes(M, N, K, E, grouped, b_rows=0):
    from atorch_amd import _lib

    return _lib.lib().aamd_grouped_gemm_fp8_ws_bytes(M, N, K, E, grouped, b_rows)


@pytest.mark.parametrize("b_rows", [0, 1])
def test_launches_of_one_round_with_a_workgroup_per_tile_ask_for_none(b_rows):
    assert _bytes(1667, 6656, 8832, 1, 1, b_rows) == 0  # 182 tiles for 256 workgroups, in a group
    assert _bytes(2229, 3456, 6784, 8, 1, b_rows) == 0  # about 170 in eight
    assert _bytes(4224, 4096, 6144, 1, 1, b_rows) > 0  # a second round of 16
    assert _bytes(4224, 4096, 6016, 1, 1, b_rows) == 0  # too short a contraction


@pytest.mark.gpu
@pytest.mark.parametrize("turned", [False, True])
def test_without_memory_for_it_the_allocator_keeps_its_reserve(dev, turned):
    """A launch that would share its last round runs without, and what the allocator holds in reserve stays there."""
    import torch

    from atorch_amd import kernels

    M, N, K = 4224, 4096, 6144
    assert _bytes(M, N, K, 1, 1, int(turned)) > 16 << 20
    g = torch.Generator(device=dev).manual_seed(3)
    qx, sx = kernels.tile_quant(torch.randn((M, K), generator=g, device=dev).bfloat16())
    w = torch.randn((1, K, N) if turned else (1, N, K), generator=g, device=dev).bfloat16() * 0.05
    q, s, q_t, s_t = kernels.block_quant_batched(w, return_transpose=True, written=kernels.STORED)
    if turned:
        q, s = q_t, s_t
    goff = kernels.group_offsets_from_splits([M], dev)
    with kernels.gemm_options(tile=1):  # (the large tiles without a workspace)
        want = kernels.grouped_gemm_nt(qx, sx, q, s, goff)
    out = torch.empty_like(want)
    del w
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    spare = torch.empty(12 << 20, dtype=torch.uint8, device=dev)
    del spare  # (a reserve, too small for the workspace)
    held, total = torch.cuda.memory_reserved(), torch.cuda.mem_get_info()[1]
    before = torch.cuda.memory_stats()["num_alloc_retries"]
    torch.cuda.set_per_process_memory_fraction((held + (16 << 20)) / total)
    try:
        kernels.grouped_gemm_nt(qx, sx, q, s, goff, out=out)
        torch.cuda.synchronize()
        assert torch.cuda.memory_reserved() == held and torch.cuda.memory_stats()["num_alloc_retries"] == before
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(out, want)
    kernels.grouped_gemm_nt(qx, sx, q, s, goff, out=out)
    assert torch.cuda.memory_reserved() > held and not torch.equal(out, want)  # in parts: another order of the sums
