"""Fused weight-gradient accumulation into main_grad buffers wherever they lie: what is equally far apart takes the gradient
in place, whatever is not gets it from a buffer of its own.  Either way the buffers hold the bits of dense ones."""
import pytest
import torch

from helpers import randn_bf16

E, K, N, SPLITS = 4, 256, 384, [70, 0, 129, 57]


def _dense(dev, dtype):
    return list(torch.full((E, N, K), 0.25, dtype=dtype, device=dev).unbind(0)), None


def _with_biases(dev, dtype):
    """One flat buffer as a distributed optimizer makes it: every weight's gradient with its bias' behind it."""
    flat = torch.full((E, N * K + N), 0.25, dtype=dtype, device=dev)
    return [row[: N * K].view(N, K) for row in flat], flat[:, N * K :]


def _flat(dev, dtype):
    flat = torch.full((E, N * K + N), 0.25, dtype=dtype, device=dev)
    return [row[: N * K] for row in flat], flat[:, N * K :]


def _one_by_one(dev, dtype):
    return [torch.full((N, K), 0.25, dtype=dtype, device=dev) for _ in range(E)], None


def _unequal(dev, dtype):
    flat = torch.full((E * (N * K + 64 * E),), 0.25, dtype=dtype, device=dev)
    at = [g * N * K + 64 * g * g for g in range(E)]
    return [flat[a : a + N * K].view(N, K) for a in at], flat[3 * N * K + 64 * 4 : 3 * N * K + 64 * 9]


def _misaligned(dev, dtype):
    flat = torch.full((E * N * K + 1,), 0.25, dtype=dtype, device=dev)
    return [flat[1 + g * N * K : 1 + (g + 1) * N * K].view(N, K) for g in range(E)], flat[:1]


def _backwards(dev, dtype):
    return list(torch.full((E, N, K), 0.25, dtype=dtype, device=dev).unbind(0))[::-1], None


LAYOUTS = [_dense, _with_biases, _flat, _one_by_one, _unequal, _misaligned, _backwards]


def test_what_counts_as_equally_far_apart():
    from atorch_amd._lib import host

    spaced = lambda layout, **kw: host().spaced(layout("cpu", torch.float32)[0], N * K, **kw)  # noqa: E731
    for layout, stride in ((_dense, N * K), (_with_biases, N * K + N), (_flat, N * K + N)):
        ts = layout("cpu", torch.float32)[0]
        assert host().spaced(ts, N * K) == (ts[0].data_ptr(), stride)
    for layout in (_unequal, _misaligned, _backwards):
        assert spaced(layout) is None
    ts = _dense("cpu", torch.float32)[0]
    assert host().spaced(ts[:1], N * K) == (ts[0].data_ptr(), N * K)
    assert host().spaced(ts, N * K - 1) is None and host().spaced([], N * K) is None
    assert host().spaced([ts[0], ts[0]], N * K) is None  # one buffer for two weights
    assert host().spaced([ts[0], ts[2], ts[3]], N * K) is None
    assert host().spaced([ts[0], ts[1].t(), ts[2]], N * K) is None
    assert host().spaced([ts[0], ts[1].view(torch.int32), ts[2]], N * K) is None


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("layout", LAYOUTS)
def test_main_grad_buffers(dev, layout, dtype):
    from atorch_amd.grouped_linear import ATorchGroupedLinear

    x, dy = randn_bf16((sum(SPLITS), K), 1).to(dev), randn_bf16((sum(SPLITS), N), 2, std=0.01).to(dev)
    layer = ATorchGroupedLinear(E, K, N, bias=False, params_dtype=torch.bfloat16, device=dev, fuse_wgrad_accumulation=True)
    results, peaks, gaps = [], [], None
    for make in (_dense, layout):
        mains, gaps = make(dev, dtype)
        for i, m in enumerate(mains):
            layer.get_parameter(f"weight{i}").main_grad = m
        for first in (None, True, False):  # added to what is there, written over it, added again
            out = layer(x.clone().requires_grad_(True), SPLITS, is_first_microbatch=first)
            torch.cuda.reset_peak_memory_stats()
            before = torch.cuda.memory_allocated()
            out.backward(dy)
            peaks.append(torch.cuda.max_memory_allocated() - before)
            results.append([m.clone() for m in mains])
    for got, want in zip(results[3:], results[:3]):
        for i in range(E):
            # (also from a buffer of its own: the sum is fp32 and rounded once)
            assert torch.equal(got[i].view(N, K), want[i])
    assert gaps is None or torch.all(gaps == 0.25)
    if layout in (_with_biases, _flat):  # in place: no more memory than dense buffers ask for
        assert max(peaks[3:]) - max(peaks[:3]) < E * N * K


@pytest.mark.gpu
def test_main_grad_of_another_size_is_refused(dev):
    from atorch_amd.grouped_linear import ATorchGroupedLinear

    layer = ATorchGroupedLinear(E, K, N, bias=False, params_dtype=torch.bfloat16, device=dev, fuse_wgrad_accumulation=True)
    for i in range(E):
        layer.get_parameter(f"weight{i}").main_grad = torch.zeros((N, K // 2), device=dev)
    out = layer(randn_bf16((sum(SPLITS), K), 1).to(dev).requires_grad_(True), SPLITS)
    with pytest.raises(AssertionError):
        out.backward(torch.zeros_like(out))
