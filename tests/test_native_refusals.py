"""The native call sequences refuse, before they launch anything, tensors on which the kernels would read or write out of
range.  On the CPU: a refusal is an AssertionError, and a sound call gets as far as the first use of the device."""
import pytest
import torch

from helpers import TILE

FP8, BF16, F32 = torch.float8_e4m3fn, torch.bfloat16, torch.float32
T, E, H, F, K = 6, 4, 256, 128, 2  # tokens, experts, hidden and feed-forward size, choices per token


def _host():
    from atorch_amd._lib import host

    return host()


def _codes(*shape):
    e, n, k = shape
    return torch.zeros(shape, dtype=torch.uint8).view(FP8), torch.ones(e, n // TILE, k // TILE)


def _layer(x=(T, H), probs=(T, K), ids=None, topk=K, q1=(E, 2 * F, H), q2=(E, H, F), b1=None, b2=None, glu=True, train=True):
    zeros = lambda b: torch.zeros(b, dtype=BF16) if isinstance(b, tuple) else b  # noqa: E731
    ids = torch.zeros((T, K), dtype=torch.int64) if ids is None else ids
    return _host().layer_forward(zeros(x), zeros(probs), ids, topk, *_codes(*q1), *_codes(*q2), zeros(b1), zeros(b2), glu, train)


def _sound(call, *args, **kw):
    with pytest.raises(ValueError, match="on the GPU"):
        call(*args, **kw)


def _refused(call, *args, **kw):
    with pytest.raises(AssertionError):
        call(*args, **kw)


@pytest.mark.parametrize("train", [True, False])
@pytest.mark.parametrize("dtype", [torch.int16, torch.uint8, torch.bool, torch.float32, torch.bfloat16])
def test_expert_ids_of_another_type(dtype, train):
    _refused(_layer, ids=torch.zeros((T, K), dtype=dtype), train=train)
    _refused(_host().moe_preprocess, torch.zeros(T * K, dtype=dtype), E, True)


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_expert_ids(dtype):
    _sound(_layer, ids=torch.zeros((T, K), dtype=dtype))
    _sound(_host().moe_preprocess, torch.zeros(T * K, dtype=dtype), E, True)
    _refused(_host().moe_preprocess, torch.zeros(T * K, 2, dtype=dtype)[:, 0], E, True)
