"""The expert MLP of an MoE layer on the fp8 grouped kernels, the activation fused into the quantiser.

Mirrors every body of ``Grouped_GEMM_MoE.compute_moe`` (atorch/modules/moe/grouped_gemm_moe.py:836-855):

    merged SwiGLU      fc1 = gmm(x, w1 [E, 2F, H]);  h = F.silu(fc1[:, :F]) * fc1[:, F:]          # :845-849, :331-334
    separate SwiGLU    x1 = gmm(x, w1 [E, F, H]);  x2 = gmm(x, v1 [E, F, H]);  h = F.silu(x1) * x2   # :840-843
    GELU (default)     fc1 = gmm(x, w1 [E, F, H]);  h = F.gelu(fc1)                                  # :449, :849
    use_bias           fc1 = bias_gather_add(fc1, b1, bin_ids) before the activation, and           # :846-848
                       fc2 = bias_gather_add(gmm(h, w2), b2, bin_ids)                               # :850-853

with ``trans_b=transpose_w1`` for the first weight(s) (``[E, H, *]`` when False) and ``w2 [E, F, H]``
(:473-488).  The intermediate activation never exists in memory on the way forward: the first GEMM's
output is read once by a kernel that applies the activation and writes the fp8 codes and scales the
second GEMM (and, under autograd, its weight-gradient GEMM) consume.  Rows are grouped by expert, so
the per-expert bias of ``bias_gather_add`` is the bias epilogue of the grouped GEMM (added to the fp32
accumulator, one rounding instead of the reference's two).  Separate gate / up weights are quantised
separately and their codes laid side by side, which makes the rest the merged case.

Backward: the gradient through the activation is computed from the saved first-GEMM output by the
kernel that quantises it (same fusion, autograd's bf16 arithmetic), and the four gradient GEMMs run
on the fp8 kernels; bias gradients are per-expert fp32 row sums.

Fused dispatch: with a ``TokenDispatch`` the hidden states come in token order and the permute of
atorch/modules/moe/token_dispatcher.py:89-116 happens inside the quantiser of the first GEMM's operand
(each permuted row is quantised straight from its token's row); the gradient of the hidden states goes
back to token order through the sum over the top-k copies that ``index_select``'s backward makes there.
The permuted bf16 rows are then neither written nor read, forward or backward.
"""
from typing import NamedTuple, Optional

import torch

from . import kernels
from ._lib import host
from .gmm import _offsets
from .quantization import WeightCodeCache


class TokenDispatch(NamedTuple):
    """The routing of one batch as the device-side preprocess leaves it (``kernels.moe_preprocess``)."""

    sorted_indices: torch.Tensor  # int64 [M]: flat (token * topk + slot) index of permuted row j
    row_map: torch.Tensor  # int32 [T * topk]: permuted row of flat index i (-1: dropped copy)
    topk: int
    group_offsets: torch.Tensor  # int64 [E + 1]: exclusive prefix of permuted rows per expert


def _quant_first_weight(w1, v1, transpose_w1, need_transpose=True):
    """Codes and scales of the first layer as the logical ``[E, N1, H]`` operand (N1 = 2F with SwiGLU) and
    its transpose ``[E, H, N1]``, from ``w1`` (and ``v1``) in either storage orientation.  The forward's operand is
    written; the other is its view."""
    first = 0 if transpose_w1 else 2  # stored [E, F, H] or [E, H, F]
    parts = [_written_once(w, not transpose_w1)[first : first + 2] for w in (w1, v1) if w is not None]
    # gate rows on top of up rows
    q, s = parts[0] if v1 is None else (torch.cat(p, dim=1) for p in zip(*parts))
    return q, s, q.transpose(1, 2), s.transpose(1, 2)


def _written_once(w, turned):
    return kernels.block_quant_batched(w.detach().contiguous(), return_transpose=True,
                                       written=kernels.TURNED if turned else kernels.STORED)  # fmt: skip


def _weight_codes(w1, w2, v1, transpose_w1, is_first_microbatch, weight_cache):
    """``(q1, s1, q1_t, s1_t), (q2, s2, q2_t, s2_t)``: the first weight(s) as [E, N1, H] (rows = outputs) and the second
    as [E, F, H], each with its transpose; block quantisation commutes with the transpose, so the codes of one
    orientation are those of the other as well: the forward's operands are written, the backward reads their views."""
    if weight_cache is not None:
        held = weight_cache.held((("w1", (w1, v1)), ("w2", (w2,))), is_first_microbatch, True)
        if held is not None:
            return held
    quant1 = lambda t: _quant_first_weight(w1, v1, transpose_w1)  # noqa: E731
    quant2 = lambda t: _written_once(w2, True)  # noqa: E731
    if weight_cache is None:
        return quant1(True), quant2(True)
    return (weight_cache.codes("w1", (w1, v1), is_first_microbatch, True, quant1),
            weight_cache.codes("w2", (w2,), is_first_microbatch, True, quant2))  # fmt: skip


def _bias(b):
    return b.detach().contiguous() if b is not None else None


def _mlp_backward(ctx, dy, goff, fc1, qx_t, sx_t, qh_t, sh_t, q1_t, s1_t, q2, s2, row_map):
    """``(dx, dw1, dw2, dv1, db1, db2)`` from the gradient of the MLP's output rows."""
    x_dtype, w1_dtype, w2_dtype = ctx.dtypes
    dy = dy.contiguous().to(torch.bfloat16)
    dx, dw1, dw2, db1, db2 = host().mlp_backward(
        dy, goff, row_map, ctx.dispatch_topk, fc1, qx_t, sx_t, qh_t, sh_t, q1_t, s1_t, q2, s2, ctx.glu, ctx.transpose_w1,
        ctx.has_b1, ctx.has_b2, x_dtype, w1_dtype, w2_dtype,
    )  # fmt: skip
    dw1, dv1 = _gate_and_up(ctx, dw1)
    return dx, dw1, dw2, dv1, db1, db2


def _gate_and_up(ctx, dw1):
    """The gate and the up half of the gradient go back to their own parameters."""
    if not ctx.has_v1:
        return dw1, None
    return tuple(t.contiguous() for t in torch.chunk(dw1, 2, dim=1 if ctx.transpose_w1 else 2))


class _Fp8ExpertMlp(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w1, w2, v1, b1, b2, batch_sizes, transpose_w1, activation, dispatch, is_first_microbatch,
                weight_cache):
        assert x.dim() == 2 and w1.dim() == 3 and w2.dim() == 3
        goff = dispatch.group_offsets if dispatch is not None else _offsets(batch_sizes, x.device)
        train = any(ctx.needs_input_grad)  # all False under no_grad
        glu = activation == "swiglu"
        codes1, codes2 = _weight_codes(w1, w2, v1, transpose_w1, is_first_microbatch, weight_cache)
        q1, s1, q1_t, s1_t = codes1
        q2, s2, q2_t, s2_t = codes2
        sorted_idx, row_map, topk = (None, None, 0) if dispatch is None else dispatch[:3]
        out, fc1, qx_t, sx_t, qh_t, sh_t = host().mlp_forward(
            x.detach().contiguous(), goff, sorted_idx, row_map, topk, q1, s1, q2_t, s2_t, _bias(b1), _bias(b2), glu, train
        )
        if train:
            ctx.transpose_w1, ctx.glu, ctx.has_v1 = transpose_w1, glu, v1 is not None
            ctx.has_b1, ctx.has_b2 = b1 is not None, b2 is not None
            ctx.dtypes = (x.dtype, w1.dtype, w2.dtype)
            ctx.dispatch_topk = topk
            ctx.save_for_backward(goff, fc1, qx_t, sx_t, qh_t, sh_t, q1_t, s1_t, q2, s2, row_map)
        return out

    @staticmethod
    def backward(ctx, dy):
        return (*_mlp_backward(ctx, dy, *ctx.saved_tensors), None, None, None, None, None, None)


class _Fp8MoeLayer(torch.autograd.Function):
    """Routing, expert MLP and weighted combine as one function: the work of the three ops, one call into native code
    per direction.  Returns the combined tokens; the routing is left in ``dispatcher``."""

    @staticmethod
    def forward(ctx, x, probs, w1, w2, v1, b1, b2, top_experts, dispatcher, transpose_w1, glu, is_first_microbatch,
                weight_cache):
        train = ctx is not None and any(ctx.needs_input_grad)
        codes1, codes2 = _weight_codes(w1, w2, v1, transpose_w1, is_first_microbatch, weight_cache)
        q1, s1, q1_t, s1_t = codes1
        q2, s2, q2_t, s2_t = codes2
        topk = dispatcher.topk
        probs_c = probs.contiguous()
        out, sorted_idx, row_map, goff, *saved = host().layer_forward(
            x.contiguous(), probs_c, top_experts.contiguous(), topk, q1, s1, q2_t, s2_t, _bias(b1), _bias(b2), glu, train
        )
        dispatcher.set_routing(sorted_idx, row_map, goff)
        if train:
            y, fc1, qx_t, sx_t, qh_t, sh_t = saved
            ctx.transpose_w1, ctx.glu, ctx.has_v1 = transpose_w1, glu, v1 is not None
            ctx.has_b1, ctx.has_b2 = b1 is not None, b2 is not None
            ctx.dtypes = (x.dtype, w1.dtype, w2.dtype)
            ctx.dispatch_topk = topk
            ctx.save_for_backward(y, probs_c, sorted_idx, goff, row_map, fc1, qx_t, sx_t, qh_t, sh_t, q1_t, s1_t, q2, s2)
        return out

    @staticmethod
    def backward(ctx, dout):
        y, probs, sorted_idx, goff, row_map, *saved = ctx.saved_tensors
        x_dtype, w1_dtype, w2_dtype = ctx.dtypes
        (dx, dw1, dw2, db1, db2), d_probs = host().layer_backward(
            dout.contiguous(), y, probs, sorted_idx, goff, row_map, ctx.dispatch_topk, *saved, ctx.glu, ctx.transpose_w1,
            ctx.needs_input_grad[1], ctx.has_b1, ctx.has_b2, x_dtype, w1_dtype, w2_dtype,
        )  # fmt: skip
        dw1, dv1 = _gate_and_up(ctx, dw1)
        return dx, d_probs, dw1, dw2, dv1, db1, db2, None, None, None, None, None, None


def grouped_mlp(hidden_states: torch.Tensor, w1: torch.Tensor, w2: torch.Tensor,
                tokens_per_expert: Optional[torch.Tensor], v1: Optional[torch.Tensor] = None,
                b1: Optional[torch.Tensor] = None, b2: Optional[torch.Tensor] = None, activation: str = "swiglu",
                transpose_w1: bool = True, *, dispatch: Optional[TokenDispatch] = None,
                is_first_microbatch: Optional[bool] = None,
                weight_cache: Optional[WeightCodeCache] = None) -> torch.Tensor:
    """The expert MLP: ``gmm -> (bias) -> activation -> gmm -> (bias)``.

    ``hidden_states [M, H]`` bf16 rows grouped by expert; ``tokens_per_expert`` int64 ``[E]`` (CPU or
    device).  ``activation="swiglu"``: ``w1 [E, 2F, H]`` (merged gate / up), or ``w1`` and ``v1`` ``[E, F, H]``
    each; ``activation="gelu"``: ``w1 [E, F, H]``.  With ``transpose_w1=False`` the first weights are stored
    ``[E, H, *]``.  ``w2 [E, F, H]``; ``b1 [E, N1]`` / ``b2 [E, H]`` optional (not with ``v1``, as in the
    reference).  H and F multiples of 128.  Returns ``[M, H]``.

    ``dispatch``: the permute fused in; ``hidden_states`` is then ``[T, H]`` in token order,
    ``tokens_per_expert`` is not used (the dispatch carries the group offsets) and the result is the ``[M, H]``
    expert output in permuted order, ready for the combine.  ``weight_cache`` / ``is_first_microbatch``: codes of
    the weights kept between microbatches under the grouped linear's rule (``WeightCodeCache``); without a cache
    the weights are quantised in every call."""
    assert hidden_states.dtype == torch.bfloat16, "the fused activation kernels read bf16"
    assert activation in ("swiglu", "gelu"), f"unknown activation {activation}"
    assert v1 is None or activation == "swiglu", "v1 is the up projection of a gated unit"
    assert v1 is None or (b1 is None and b2 is None), "bias not supported yet for not merge_w1_v1"
    assert dispatch is not None or tokens_per_expert is not None, "tokens_per_expert or a dispatch is needed"
    return _Fp8ExpertMlp.apply(hidden_states, w1, w2, v1, b1, b2, tokens_per_expert, transpose_w1, activation, dispatch,
                               is_first_microbatch, weight_cache)


def grouped_mlp_swiglu(hidden_states: torch.Tensor, w1: torch.Tensor, w2: torch.Tensor,
                       tokens_per_expert: Optional[torch.Tensor], transpose_w1: bool = True, **kw) -> torch.Tensor:
    """``gmm -> SwiGLU -> gmm`` with the merged gate / up weight (``grouped_mlp`` with its defaults)."""
    return grouped_mlp(hidden_states, w1, w2, tokens_per_expert, transpose_w1=transpose_w1, **kw)
