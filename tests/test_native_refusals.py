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


@pytest.mark.parametrize("train", [True, False])
@pytest.mark.parametrize("glu", [True, False])
def test_layer_sizes_that_do_not_fit(glu, train):
    n1 = 2 * F if glu else F
    kw = dict(q1=(E, n1, H), glu=glu, train=train)
    _sound(_layer, **kw, b1=(E, n1), b2=(E, H))
    _refused(_layer, **kw, x=(T, 2 * H))  # wider rows than the weights'
    _refused(_layer, **kw, q2=(E, H, 2 * F))  # another feed-forward size
    _refused(_layer, **kw, q2=(E + 1, H, F))
    _refused(_layer, **kw, q2=(E, 2 * H, F))
    _refused(_layer, **kw, b1=(E, n1 // 2))
    _refused(_layer, **kw, b1=(E - 1, n1))
    _refused(_layer, **kw, b2=(E, 2 * H))
    _refused(_layer, **kw, b2=torch.zeros((H, E), dtype=BF16).t())
    _refused(_layer, **kw, probs=(T, K - 1))
    _refused(_layer, **kw, probs=(T - 1, K))
    _refused(_layer, **kw, topk=K + 1)
    _refused(_layer, **kw, ids=torch.zeros((T + 1, K), dtype=torch.int64))


def _offsets(groups=E, dtype=torch.int64):
    return torch.zeros(groups + 1, dtype=dtype)


@pytest.mark.parametrize("train", [True, False])
def test_mlp_offsets_and_routing_that_do_not_fit(train):
    def mlp(goff, row_map=None, sorted_idx=None, x=(T, H)):
        return _host().mlp_forward(torch.zeros(x, dtype=BF16), goff, sorted_idx, row_map, K, *_codes(E, 2 * F, H), *_codes(E, H, F),
                                   None, None, True, train)  # fmt: skip

    routing = lambda n=T * K, m=torch.int32, s=torch.int64: (torch.zeros(n, dtype=m), torch.zeros(n, dtype=s))  # noqa: E731
    _sound(mlp, _offsets())
    _sound(mlp, _offsets(), *routing())
    for goff in (_offsets(E - 1), _offsets(E + 1), _offsets(dtype=torch.int32)):
        _refused(mlp, goff)
        _refused(mlp, goff, *routing())
    _refused(mlp, _offsets(), x=(T, 2 * H))
    _refused(mlp, _offsets(), *routing(T * K + K))
    _refused(mlp, _offsets(), *routing(m=torch.int64))
    _sound(mlp, _offsets(), routing()[0], routing(T * K - 1)[1])  # a dropped copy
    _refused(mlp, _offsets(), routing()[0], routing(T * K + 1)[1])
    _refused(mlp, _offsets(), routing()[0])
    if train:  # (the forward alone reads the map)
        _refused(mlp, _offsets(), *routing(s=torch.int32))


def test_linear_and_gemm_sizes_that_do_not_fit():
    h, N = _host(), 384
    codes, scales = _codes(E, N, H)
    row = lambda m, k: (torch.zeros((m, k), dtype=torch.uint8).view(FP8), torch.ones(m, k // TILE))  # noqa: E731
    nt = lambda a, goff, bias=None, s=scales: h.gemm_nt(*a, codes, s, goff, None, BF16, bias)  # noqa: E731
    _sound(nt, row(T, H), _offsets(), torch.zeros(E, N))
    _refused(nt, row(T, 2 * H), _offsets())
    _refused(nt, row(T, H), _offsets(E - 1))
    _refused(nt, row(T, H), _offsets(), torch.zeros(E, 2 * N))
    _refused(nt, row(T, H), _offsets(), s=scales[: E - 1])
    _refused(nt, (row(T, H)[0], row(T - 1, H)[1]), _offsets())

    def linear(x=(T, H), goff=None, splits=(), bias=None, train=True):
        return h.linear_forward(torch.zeros(x, dtype=BF16), goff, list(splits), codes, scales, bias, BF16, 0.0, train)

    for train in (True, False):
        _sound(linear, goff=_offsets(), train=train)
        _refused(linear, goff=_offsets(E + 1), train=train)
        _refused(linear, splits=[T], train=train)
        _refused(linear, x=(T, 2 * H), goff=_offsets(), train=train)
        _refused(linear, goff=_offsets(), bias=torch.zeros(E, H), train=train)
    _refused(h.offsets_from_tensor, torch.zeros(E, dtype=torch.int32), torch.device("cuda"))


def test_gemm_scales_that_are_not_dense():
    """Dense in either orientation, whichever the codes are in; any other strides are refused, not copied."""
    h, M, N, K = _host(), 4, 384, 512
    a, a_s = torch.zeros((M, K), dtype=torch.uint8).view(FP8), torch.ones(M, K // TILE)
    codes, s = _codes(E, N, K)
    view, s_view = _codes(E, K, N)[0].transpose(1, 2), torch.ones(E, K // TILE, N // TILE).transpose(1, 2)
    nt = lambda b, b_s, x_s=a_s: h.gemm_nt(a, x_s, b, b_s, _offsets(), None, BF16, None)  # noqa: E731
    for b in (codes, view):
        _sound(nt, b, s)
        _sound(nt, b, s_view)
        _refused(nt, b, torch.ones(E, N // TILE, 2 * K // TILE)[..., ::2])
        _refused(nt, b, torch.ones(2 * E, N // TILE, K // TILE)[::2])
        _refused(nt, b, torch.ones(N // TILE, E, K // TILE).transpose(0, 1))
        _refused(nt, b, s, torch.ones(K // TILE, M).t())
    per_row = torch.ones(E, N, K // TILE)
    _sound(nt, codes, per_row)
    _refused(nt, codes, per_row.transpose(1, 2).contiguous().transpose(1, 2))


def test_dual_quantisers_with_offsets_of_another_length():
    h, x = _host(), torch.zeros((T, H), dtype=BF16)
    si = torch.zeros(T, dtype=torch.int64)
    calls = [lambda g: h.dual(x, g, E, 0.0, 640, True, True), lambda g: h.permute_dual(x, si, 1, g, E, 0.0, 640, True, True),
             lambda g: h.act_dual(x, None, True, g, E, 640, True, True, False),
             lambda g: h.dual_with_sums(0, x, None, g, E, 640, 0.0, F32)]  # fmt: skip
    for call in calls:
        _sound(call, _offsets())
        _refused(call, _offsets(E - 1))
        _refused(call, _offsets(dtype=torch.int32))


def test_weight_gradient_operands_that_do_not_fit():
    h, ld = _host(), 512
    op = lambda rows, n=ld: (torch.zeros((n // TILE, rows, TILE), dtype=torch.uint8).view(FP8), torch.ones(n // TILE, rows))  # noqa: E731
    wgrad = lambda a, b, goff: h.gemm_wgrad(*a, *b, goff, None, F32, False)  # noqa: E731
    _sound(wgrad, op(F), op(H), _offsets())
    _refused(wgrad, op(F), op(H, ld // 2), _offsets())
    _refused(wgrad, (op(F)[0], op(F, ld // 2)[1]), op(H), _offsets())
    _refused(wgrad, op(F), op(H), _offsets(dtype=torch.int32))
    rows = (torch.zeros((F, ld), dtype=torch.uint8).view(FP8), torch.ones(ld // TILE, F))
    _refused(wgrad, rows, op(H), _offsets())
    into = lambda *shape: h.gemm_wgrad(*op(F), *op(H), _offsets(), torch.zeros(shape), F32, True)  # noqa: E731
    _sound(into, E, F, H)
    for shape in ((E - 1, F, H), (E, F - 1, H), (E, F, 2 * H), (E, F * H)):
        _refused(into, *shape)
