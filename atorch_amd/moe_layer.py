"""The MoE layer of one GPU on the fp8 grouped kernels: dispatch -> expert MLP -> combine.

Constructor, parameter names (``w1``, ``w2``, ``v1``, ``b1``, ``b2``) and ``forward(hidden_states, expert_weights,
top_experts, se_fn1, se_fn2, se_fn2_additional_input)`` follow ``Grouped_GEMM_MoE``
(atorch/modules/moe/grouped_gemm_moe.py:349-518, 644-682) for the branch a single GPU takes: no expert
parallelism, the "Megatron" composite ``token_permutation -> compute_expert -> token_unpermutation`` with the
AllToAll dispatcher, whose exchange steps are no-ops without a process group.  Nothing on the way waits for the
device: the router preprocess leaves the group offsets in device memory (the reference copies the counts to the
host, :837), the permute is fused into the quantiser of the first GEMM's operand, the activation into the
quantiser of the second one's, and the combine is one gather-reduce pass, so a forward (and a backward) is a fixed
sequence of launches that a HIP graph can capture and replay on other routings of the same shape.

Differences from the reference, none of which changes results on one GPU: ``implementation_type`` "MegaBlocks"
runs the same composite (its sort / gather / scatter ops compute the same permutation and weighted sum);
``use_bias`` is honoured for both implementation types (the reference's Megatron branch switches it off, :396-400);
``use_expert_parallelism=True`` raises.
"""
import logging
from typing import Callable, List, Optional, Tuple, Union

import torch
from torch.autograd import forward_ad

from .expert_mlp import _Fp8MoeLayer, grouped_mlp
from .quantization import WeightCodeCache
from .token_dispatcher import MoEAllToAllTokenDispatcher

logger = logging.getLogger(__name__)


class Grouped_GEMM_MoE(torch.nn.Module):
    """A mixture-of-experts feed-forward block with grouped fp8 GEMMs (one GPU)."""

    def __init__(
        self,
        hidden_size,
        expert_intermediate_size,
        output_dropout_prob,
        num_experts,
        topk,
        use_swiglu=False,
        use_bias=False,
        initializer_range=0.02,
        use_expert_parallelism=False,
        expert_parallel_group=None,
        merge_w1_v1=True,
        transpose_w1=True,
        is_scale_gradient=False,
        implementation_type="MegaBlocks",
        token_dispatcher_type="AllToAll",
        device=None,
        dtype=None,
    ) -> None:
        super().__init__()
        if use_expert_parallelism or expert_parallel_group is not None:
            raise NotImplementedError("Grouped_GEMM_MoE: this build runs on one GPU (no expert parallelism)")
        if implementation_type not in ("MegaBlocks", "Megatron"):
            raise ValueError(f"'{implementation_type}' is not a valid MOEImplmenterType")
        if token_dispatcher_type not in ("AllToAll", "AllGather", "MindSpeedAllGather", "MindSpeedAllToAll"):
            raise ValueError(f"'{token_dispatcher_type}' is not a valid MOETokenDispatcherType")
        if token_dispatcher_type != "AllToAll":
            logger.warning("Grouped_GEMM_MoE: one GPU has one dispatcher; using the AllToAll dispatcher's local branch")
        self.implementation_type = implementation_type
        self.hidden_size = hidden_size
        self.expert_intermediate_size = expert_intermediate_size
        self.output_dropout_prob = output_dropout_prob
        self.num_experts = num_experts
        self.num_local_experts = num_experts
        self.use_expert_parallelism = False
        self.is_scale_gradient = is_scale_gradient
        self.gradient_scale = None  # 1 / expert-parallel size in the reference: one GPU scales by nothing
        self.topk = topk
        self.use_swiglu = use_swiglu
        self.use_bias = use_bias
        self.merge_w1_v1 = merge_w1_v1
        self.transpose_w1 = transpose_w1
        kw = {"device": device, "dtype": dtype}

        E, F, H = num_experts, expert_intermediate_size, hidden_size
        if use_swiglu and not merge_w1_v1:
            shape = (E, F, H) if transpose_w1 else (E, H, F)
            self.w1 = torch.nn.Parameter(torch.empty(shape, **kw))
            self.w2 = torch.nn.Parameter(torch.empty((E, F, H), **kw))
            self.v1 = torch.nn.Parameter(torch.empty(shape, **kw))
            assert not use_bias, "bias not supported yet for not merge_w1_v1"
        else:
            n1 = F * (2 if use_swiglu else 1)
            self.w1 = torch.nn.Parameter(torch.empty((E, n1, H) if transpose_w1 else (E, H, n1), **kw))
            self.w2 = torch.nn.Parameter(torch.empty((E, F, H), **kw))
        if use_bias:
            self.b1 = torch.nn.Parameter(torch.empty((E, F * (2 if use_swiglu else 1)), **kw))
            self.b2 = torch.nn.Parameter(torch.empty((E, H), **kw))
        self.dropout = torch.nn.Dropout(output_dropout_prob)

        self.w1.data.normal_(mean=0.0, std=initializer_range)
        self.w2.data.normal_(mean=0.0, std=initializer_range)
        if self.has_v1():
            self.v1.data.normal_(mean=0.0, std=initializer_range)
        if use_bias:
            self.b1.data.zero_()
            self.b2.data.zero_()

        self.token_dispatcher = MoEAllToAllTokenDispatcher(
            self.num_local_experts, list(range(self.num_local_experts)), self.num_experts, topk=self.topk,
            add_bias=self.use_bias, use_expert_parallelism=False,
        )  # fmt: skip
        self.weight_code_cache = WeightCodeCache()
        self.hidden_shape = None

    def has_v1(self):
        # (hasattr takes a microsecond to say no)
        kept = "v1" in self._parameters or "v1" in self.__dict__ or "v1" in self._buffers or hasattr(type(self), "v1")
        return kept and self.v1 is not None

    def scale_grad(self, w):
        return w  # gradient_scale is None without expert parallelism (grouped_gemm_moe.py:427-431, 632-636)

    def _mlp(self, hidden_states, tokens_per_expert, dispatch, is_first_microbatch):
        out = grouped_mlp(
            hidden_states, self.scale_grad(self.w1), self.scale_grad(self.w2), tokens_per_expert,
            v1=self.scale_grad(self.v1) if self.has_v1() else None,
            b1=self.b1 if self.use_bias else None, b2=self.b2 if self.use_bias else None,
            activation="swiglu" if self.use_swiglu else "gelu", transpose_w1=self.transpose_w1,
            dispatch=dispatch, is_first_microbatch=is_first_microbatch, weight_cache=self.weight_code_cache,
        )  # fmt: skip
        return self.dropout(out)

    def compute_expert(self, _hidden_states, _tokens_per_expert, bin_ids=None, is_first_microbatch=None):
        """``compute_expert`` of the reference (:816-834) on rows that are already permuted: ``_tokens_per_expert``
        int64 ``[E]``, on the device or the host.  ``bin_ids`` is not needed: rows are grouped by expert."""
        if _hidden_states.nelement() == 0:
            return _hidden_states.new_zeros((0, self.hidden_size))
        return self._mlp(_hidden_states, _tokens_per_expert, None, is_first_microbatch)

    def forward(
        self,
        hidden_states: torch.Tensor,
        expert_weights: torch.Tensor,
        top_experts: torch.Tensor,
        se_fn1: Optional[Callable] = None,
        se_fn2: Optional[Callable] = None,
        se_fn2_additional_input: Optional[Union[torch.Tensor, Tuple, List]] = None,
        is_first_microbatch: Optional[bool] = None,
    ):
        """``is_first_microbatch`` (not in the reference's signature): the expert weights' fp8 codes are kept
        between the microbatches of a step under the grouped linear's rule; None quantises in every call."""
        if torch.is_autocast_enabled():
            expert_weights = expert_weights.to(torch.get_autocast_gpu_dtype())
            hidden_states = hidden_states.to(torch.get_autocast_gpu_dtype())
        return self._forward_megatron(hidden_states, expert_weights, top_experts, se_fn1, se_fn2,
                                      se_fn2_additional_input, is_first_microbatch)  # fmt: skip

    def _nothing_between(self, dispatcher):
        """True if nothing happens between the experts and the combine and both ends are this package's: the dropout is the
        identity, nobody listens to it, and dispatcher and dropout are the modules the constructor made."""
        drop = self._modules.get("dropout")
        return (type(dispatcher) is MoEAllToAllTokenDispatcher and type(drop) is torch.nn.Dropout
                and not (drop.training and drop.p > 0 or drop._forward_hooks or drop._forward_pre_hooks
                         or drop._backward_hooks or drop._backward_pre_hooks))  # fmt: skip

    def _forward_fused(self, x, probs, top_experts, is_first_microbatch):
        """The layer as one function, one native call per direction, which compares the sizes.  (Choices may also come
        flattened, as other MoE layers pass them.)"""
        assert x.dtype == torch.bfloat16, "the fused activation kernels read bf16"
        # (looked up where they mostly are, a third of an attribute's time; a pruned or parametrised one is no parameter, nor is
        # one that a wrapper keeps as a plain attribute)
        p = self._parameters
        w1 = self.scale_grad(p["w1"] if "w1" in p else self.w1)
        w2 = self.scale_grad(p["w2"] if "w2" in p else self.w2)
        v1 = self.scale_grad(self.v1) if self.has_v1() else None
        b1, b2 = (self.b1, self.b2) if self.use_bias else (None, None)
        assert v1 is None or self.use_swiglu, "v1 is the up projection of a gated unit"
        assert v1 is None or b1 is None, "bias not supported yet for not merge_w1_v1"
        args = (x, probs, w1, w2, v1, b1, b2, top_experts, self.token_dispatcher, self.transpose_w1, self.use_swiglu,
                is_first_microbatch, self.weight_code_cache)  # fmt: skip
        # (past autograd only where nobody else looks either: a dual number is refused and a trace records the function there)
        plain = not torch.is_grad_enabled() and forward_ad._current_level < 0 and not torch.jit.is_tracing()
        return _Fp8MoeLayer.forward(None, *args) if plain else _Fp8MoeLayer.apply(*args)

    def _forward_megatron(self, hidden_states, expert_weights, top_experts, se_fn1=None, se_fn2=None,
                          se_fn2_additional_input=None, is_first_microbatch=None):
        # (a call is a few dozen microseconds when decoding: nothing is reshaped that has its shape, and the attribute is
        # set past Module.__setattr__)
        if expert_weights.dim() != 2:
            expert_weights = expert_weights.view(-1, expert_weights.shape[-1])
        if top_experts.dim() != 2:
            top_experts = top_experts.view(-1, top_experts.shape[-1])
        shape = hidden_states.shape
        self.__dict__["hidden_shape"] = shape
        d = self.token_dispatcher
        x = hidden_states if len(shape) == 2 else hidden_states.reshape(-1, shape[-1])
        if x.shape[0] == 0:
            return hidden_states.clone()
        d.hidden_shape, d.probs = shape, expert_weights
        if se_fn1 is None and se_fn2 is None and self._nothing_between(d):
            out = self._forward_fused(x, expert_weights, top_experts, is_first_microbatch)
            return out if len(shape) == 2 else out.view(shape)
        # dispatch: only the routing is computed here; the permute itself happens inside the first quantiser
        d.preprocess(top_experts)

        se_intermediate = se_fn1(x) if se_fn1 is not None else None

        expert_output = self._mlp(x, None, d.dispatch(), is_first_microbatch)

        compute_fn_input = None
        if se_fn2_additional_input is not None:
            if isinstance(se_fn2_additional_input, (tuple, list)):
                compute_fn_input = (se_intermediate,) + tuple(se_fn2_additional_input)
            else:
                compute_fn_input = (se_intermediate, se_fn2_additional_input)
        elif se_fn2 is not None:
            compute_fn_input = (se_intermediate,)

        output, _, _ = d.token_unpermutation(expert_output)
        if se_fn2 is not None:
            se_output = se_fn2(*compute_fn_input)
            if se_output is not None:
                output = output + se_output.view(self.hidden_shape)
        return output
