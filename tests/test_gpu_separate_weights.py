"""Weights of a grouped linear that do not share one buffer (moved, loaded or replaced one by one): the codes of a stack of
them, whichever way they are reached."""
import pytest
import torch

from helpers import randn_bf16

pytestmark = pytest.mark.gpu


def _own(w):
    return [t.clone() for t in w]


def _with_gaps(w):  # equally far apart
    n = w[0].numel()
    buf = torch.zeros((len(w), n + 64), dtype=w.dtype, device=w.device)
    return [row[:n].view(t.shape).copy_(t) for row, t in zip(buf, w)]


def _unequal(w):
    n = w[0].numel()
    buf = torch.zeros((len(w), n + 1024), dtype=w.dtype, device=w.device)
    return [row[64 * i * i : 64 * i * i + n].view(t.shape).copy_(t) for i, (row, t) in enumerate(zip(buf, w))]


def _misaligned(w):
    n = w[0].numel()
    buf = torch.zeros((len(w), n + 64), dtype=w.dtype, device=w.device)
    return [row[1 : 1 + n].view(t.shape).copy_(t) for row, t in zip(buf, w)]


def _transposed(w):
    return [t.t().contiguous().t() for t in w]


# (on both sides of the size from which a weight gets a launch of its own, 2^21 elements)
@pytest.mark.parametrize("E,N,K", [(1, 128, 128), (3, 256, 384), (3, 1024, 1920), (3, 1024, 2048), (2, 2048, 1152)])
@pytest.mark.parametrize("layout", [_own, _with_gaps, _unequal, _misaligned, _transposed])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
def test_codes_of_separate_weights(dev, E, N, K, layout, dtype):
    from atorch_amd import kernels
    from atorch_amd._lib import host

    w = randn_bf16((E, N, K), 1, std=0.02, dtype=dtype).to(dev)
    ws = layout(w)
    for transpose in (True, False):
        want = kernels.block_quant_batched(w, return_transpose=transpose)
        got = host().block_quant_list(ws, 0.0, transpose)
        for a, b in zip(got, want):
            assert (a is None) == (b is None) and (a is None or torch.equal(a.view(torch.uint8), b.view(torch.uint8)))


def test_weights_of_different_shapes_are_refused(dev):
    from atorch_amd._lib import host

    ws = [torch.zeros((256, 128), device=dev), torch.zeros((128, 256), device=dev)]
    with pytest.raises(AssertionError):
        host().block_quant_list(ws, 0.0, True)
    with pytest.raises(AssertionError):
        host().block_quant_list([ws[0], ws[0].bfloat16()], 0.0, True)


def test_module_moved_to_the_device_copies_no_large_weights(dev):
    """A module built on the CPU and moved: no copy of the weights ahead of their quantisation."""
    from atorch_amd.grouped_linear import ATorchGroupedLinear

    E, K, N = 3, 2048, 1024
    mod = ATorchGroupedLinear(E, K, N, bias=False, params_dtype=torch.bfloat16, device="cpu").to(dev)
    x = randn_bf16((100, K), 2).to(dev)
    with torch.no_grad():
        want = mod(x, [40, 0, 60], is_first_microbatch=True)
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        got = mod(x, [40, 0, 60], is_first_microbatch=None)
        peak = torch.cuda.max_memory_allocated() - before
    assert torch.equal(got, want)
    assert peak < E * N * K * 3 // 2  # (codes and scales are a byte and a bit per weight, a copy would be two more)
