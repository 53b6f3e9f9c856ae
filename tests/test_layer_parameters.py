"""The MoE layer takes its parameters as attributes of the module, wherever pruning, a parametrisation or a wrapper keeps
them, and through ``scale_grad`` (grouped_gemm_moe.py:632-636).  On the CPU with the fused function replaced by a recorder."""
import pytest
import torch
from torch.nn.utils import parametrize, prune

from helpers import randn_bf16, topk_routing

NAMES = ("w1", "w2", "v1", "b1", "b2")


class _Double(torch.nn.Module):
    def forward(self, w):
        return w * 2


def _layer(monkeypatch, cls=None, **kw):
    from atorch_amd import moe_layer

    seen = {}

    class Recorder:
        @staticmethod
        def apply(x, probs, *args):
            seen.update(zip(NAMES, args[:5]))
            return x * sum(a.float().sum() for a in args[:5] if a is not None)

        @staticmethod
        def forward(ctx, *args):
            return Recorder.apply(*args)

    monkeypatch.setattr(moe_layer, "_Fp8MoeLayer", Recorder)
    layer = (cls or moe_layer.Grouped_GEMM_MoE)(256, 128, 0.0, 4, 2, implementation_type="Megatron", dtype=torch.bfloat16, **kw)
    idx, probs = topk_routing(8, 4, 2, seed=1)

    def run():
        seen.clear()
        return layer(randn_bf16((8, 256), 2), probs.bfloat16(), idx)

    return layer, seen, run


def _check(layer, seen):
    for name in NAMES:
        want = getattr(layer, name, None)
        assert (seen[name] is None) == (want is None) and (want is None or torch.equal(seen[name], want)), name


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("kw", [dict(use_swiglu=True), dict(use_bias=True), dict(use_swiglu=True, merge_w1_v1=False)],
                         ids=["merged", "bias", "separate"])  # fmt: skip
def test_plain_parameters(monkeypatch, kw, grad):
    layer, seen, run = _layer(monkeypatch, **kw)
    with torch.set_grad_enabled(grad):
        run()
    _check(layer, seen)
    assert all(seen[n] is p for n, p in layer.named_parameters())


def test_pruned_bias_stays_and_gets_its_gradient(monkeypatch):
    layer, seen, run = _layer(monkeypatch, use_bias=True)
    with torch.no_grad():
        layer.b1.normal_()
    prune.l1_unstructured(layer, "b1", 0.5)
    run().sum().backward()
    _check(layer, seen)
    assert seen["b1"] is not None and int((seen["b1"] == 0).sum()) == seen["b1"].numel() // 2
    assert layer.b1_orig.grad is not None


@pytest.mark.parametrize("name", ["w1", "w2", "v1"])
def test_parametrised_weights(monkeypatch, name):
    layer, seen, run = _layer(monkeypatch, use_swiglu=True, merge_w1_v1=False)
    plain = getattr(layer, name).detach().clone()
    parametrize.register_parametrization(layer, name, _Double())
    run()
    _check(layer, seen)
    assert torch.equal(seen[name], plain * 2)


def test_parameters_kept_as_plain_attributes(monkeypatch):
    layer, seen, run = _layer(monkeypatch, use_bias=True)
    for name in ("w1", "w2", "b1", "b2"):  # what a sharding wrapper does between its gather and its release
        t = getattr(layer, name).detach().clone() + 1
        delattr(layer, name)
        setattr(layer, name, t)
    run()
    _check(layer, seen)


def test_weights_go_through_scale_grad(monkeypatch):
    from atorch_amd.moe_layer import Grouped_GEMM_MoE

    class Scaled(Grouped_GEMM_MoE):
        def scale_grad(self, w):
            return w * 0.5

    layer, seen, run = _layer(monkeypatch, Scaled, use_swiglu=True, merge_w1_v1=False)
    run()
    assert all(torch.equal(seen[n], getattr(layer, n) * 0.5) for n in ("w1", "w2", "v1"))


def test_switched_off_bias_and_forbidden_combinations(monkeypatch):
    layer, seen, run = _layer(monkeypatch, use_bias=True)
    layer.use_bias = False
    run()
    assert seen["b1"] is None and seen["b2"] is None
    layer.v1 = torch.nn.Parameter(torch.zeros_like(layer.w1))  # an up projection without a gate
    with pytest.raises(AssertionError):
        run()
    layer.use_swiglu = layer.use_bias = True
    with pytest.raises(AssertionError):
        run()


@pytest.mark.parametrize("shape", [(8, 2), (16,), (16, 1), (4, 2, 2)])
def test_router_choices_of_any_shape(monkeypatch, shape):
    """What counts is one choice per token and slot, token by token (grouped_gemm_moe.py:650-652)."""
    layer, seen, run = _layer(monkeypatch)
    x, (idx, probs) = randn_bf16((8, 256), 2), topk_routing(8, 4, 2, seed=1)
    layer(x, probs.bfloat16(), idx.view(shape))
    assert seen  # (how many there are is checked in native code)


def _stop(*args, **kw):
    raise RuntimeError("composite")


def _dropout_in_eval(layer):
    layer.eval()
    layer.dropout.p = 0.5
    layer.dropout.train()  # sampling at inference


def _other_probability(layer):
    layer.dropout.p = 0.5  # the module's own, not the constructor's argument, is what counts


def _other_module(layer):
    layer.dropout = torch.nn.AlphaDropout(0.5)


def _listener(layer):
    layer.dropout.register_forward_hook(lambda m, args, out: None)


def _own_dispatcher(layer):
    from atorch_amd.token_dispatcher import MoEAllToAllTokenDispatcher

    class Own(MoEAllToAllTokenDispatcher):
        pass

    layer.token_dispatcher = Own(4, [0, 1, 2, 3], 4, 2, False, False)


@pytest.mark.parametrize("change", [_dropout_in_eval, _other_probability, _other_module, _listener, _own_dispatcher])
def test_whatever_sits_between_experts_and_combine_runs(monkeypatch, change):
    """The one-call form has no place for it: the composite of dispatch, experts, dropout and combine runs."""
    layer, seen, run = _layer(monkeypatch)
    run()
    assert seen
    layer.output_dropout_prob = 0.3  # (without meaning after construction)
    run()
    assert seen
    change(layer)
    monkeypatch.setattr(type(layer), "_mlp", _stop)
    monkeypatch.setattr(layer.token_dispatcher, "preprocess", lambda ids: None)
    monkeypatch.setattr(layer.token_dispatcher, "dispatch", lambda: None)
    with pytest.raises(RuntimeError, match="composite"):
        run()
    assert not seen


@pytest.mark.filterwarnings("ignore")  # (what a tracer says of sizes)
def test_forward_mode_and_tracing_do_not_pass_the_function_by(monkeypatch):
    """Without gradients the function's forward is called as it is, but not on dual numbers, whose tangent it would drop, and
    not in a trace, which would keep its empty buffers and none of its launches."""
    from torch.autograd import forward_ad

    from atorch_amd import moe_layer

    layer, seen, run = _layer(monkeypatch)
    layer.requires_grad_(False)
    calls = []
    recorder = moe_layer._Fp8MoeLayer
    apply = recorder.apply
    monkeypatch.setattr(recorder, "apply", staticmethod(lambda *a: (calls.append("apply"), apply(*a))[1]))
    monkeypatch.setattr(recorder, "forward", staticmethod(lambda ctx, *a: (calls.append("forward"), apply(*a))[1]))
    x, (idx, probs) = randn_bf16((8, 256), 2), topk_routing(8, 4, 2, seed=1)
    probs = probs.bfloat16()
    with torch.no_grad():
        layer(x, probs, idx)
        with forward_ad.dual_level():
            layer(forward_ad.make_dual(x, torch.ones_like(x)), probs, idx)
        torch.jit.trace(lambda t: layer(t, probs, idx), (x,), check_trace=False)
        layer(x, probs, idx)
    layer(x, probs, idx)
    assert calls == ["forward", "apply", "apply", "forward", "apply"]
