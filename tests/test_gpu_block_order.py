"""The order in which workgroups take the blocks of a weight of 2^27 elements and more: every block is quantised once, where
the blocks of a matrix are fewer than a turn of the XCDs (64), a whole number of turns, one more, and with rows of blocks
that a turn crosses; equal to the same blocks as matrices of their own, for which there is no order."""
import pytest
import torch

from helpers import randn_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,nb,kb", [(131, 7, 9), (128, 8, 8), (127, 5, 13), (127, 1, 65), (127, 65, 1), (1, 91, 91), (1, 8, 8)])
@pytest.mark.parametrize("transpose", [False, True])
def test_blocks_of_a_weight(dev, E, nb, kb, transpose):
    from atorch_amd import kernels

    w = randn_bf16((E, nb * 128, kb * 128), 1).to(dev)
    q, s, q_t, s_t = kernels.block_quant_batched(w, return_transpose=transpose)
    blocks = w.view(E, nb, 128, kb, 128).transpose(2, 3).reshape(-1, 128, 128).contiguous()
    bq, bs, bq_t, _ = kernels.block_quant_batched(blocks, return_transpose=transpose)
    u8 = lambda t: t.view(torch.uint8)  # noqa: E731
    assert torch.equal(u8(q).view(E, nb, 128, kb, 128).transpose(2, 3).reshape(-1, 128, 128), u8(bq))
    assert torch.equal(s, bs.view(E, nb, kb))
    if transpose:
        assert torch.equal(u8(q_t).view(E, kb, 128, nb, 128).permute(0, 3, 1, 2, 4).reshape(-1, 128, 128), u8(bq_t))
        assert torch.equal(s_t, s.transpose(1, 2))
