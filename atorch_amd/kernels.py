"""Functional ops over the C ABI.

The first four functions keep the names, argument meaning and error behaviour of the
reference's functional surface (atorch/modules/fp8/triton_kernel.py:40,80,127,198 and the
``return_transpose`` form of atorch/modules/fp8/cuda_kernel.py:18-61); the rest are the fused /
grouped forms the grouped linear uses.  Every function enqueues HIP kernels on the current
stream and returns torch tensors it allocated; nothing here computes on the CPU.
"""
import threading
from typing import List, Optional, Sequence, Tuple

import torch

from . import _lib
from ._lib import check, dtype_code, host, lib, ptr, stream

TILE = 128
FP8 = torch.float8_e4m3fn


def _require_fp8(dtype):
    if dtype != FP8:
        raise ValueError(f"only torch.float8_e4m3fn is supported, got {dtype}")


def padded_total(splits: Sequence[int]) -> int:
    return sum((int(m) + TILE - 1) // TILE * TILE for m in splits)


def padded_bound(rows: int, num_groups: int) -> int:
    """Upper bound of sum_g ceil(M_g/128)*128 that needs no knowledge of the splits."""
    return (rows // TILE + num_groups) * TILE


def group_offsets_from_splits(splits: Sequence[int], device) -> torch.Tensor:
    device = torch.device(device)
    if device.type != "cuda":
        off = [0]
        for m in splits:
            off.append(off[-1] + int(m))
        return torch.tensor(off, dtype=torch.int64, device=device)
    return host().offsets_from_list([int(m) for m in splits], device)


# ------------------------------------------------------------------------------------------
# reference-named functional surface
# ------------------------------------------------------------------------------------------
def tile_quant(
    x: torch.Tensor,
    dtype=FP8,
    block_size: int = TILE,
    eps: float = 0.0,
    return_transpose: bool = False,
):
    """1x128 quantisation along the last dim (triton_kernel.py:127-140).

    Returns ``(y, s)``; with ``return_transpose`` (cuda_kernel.py:18-38) returns
    ``(y, s, y_t, s_t)`` for a 2-D ``x`` where ``y_t`` is ``[K, M]`` (a view of a buffer whose
    rows are padded to a multiple of 128) and ``s_t`` is ``[K, ceil(M/128)]``.
    """
    _require_fp8(dtype)
    assert block_size == TILE, "only block_size 128 is supported"
    assert x.is_contiguous()
    assert x.size(-1) % block_size == 0
    if return_transpose:
        cols = x.size(-1)
        rows = x.numel() // cols if cols else 0
        assert x.dim() == 2, "return_transpose needs a 2-D input"
        if rows == 0:  # an empty group: nothing to launch
            return (
                torch.empty((0, cols), dtype=FP8, device=x.device),
                torch.empty((0, cols // TILE), dtype=torch.float32, device=x.device),
                torch.empty((cols, 0), dtype=FP8, device=x.device),
                torch.empty((cols, 0), dtype=torch.float32, device=x.device),
            )
        y, s, y_t, s_t = host().dual(x, None, 1, eps, padded_total([rows]), True, False)
        return y, s, y_t[:, :rows], s_t.t()
    return host().tile_quant(x, eps)


def block_quant(
    x: torch.Tensor,
    dtype=FP8,
    block_size: int = TILE,
    eps: float = 0.0,
    return_transpose: bool = False,
):
    """128x128 block quantisation of a 2-D tensor (triton_kernel.py:40-46).
    Returns ``(y, s)`` or ``(y, s, y_t, s_t)`` (cuda_kernel.py:41-61)."""
    _require_fp8(dtype)
    assert block_size == TILE, "only block_size 128 is supported"
    assert x.dim() == 2
    q, s, q_t, s_t = block_quant_batched(x.unsqueeze(0), eps=eps, return_transpose=return_transpose)
    if return_transpose:
        return q[0], s[0], q_t[0], s_t[0]
    return q[0], s[0]


def dequant(x: torch.Tensor, s: torch.Tensor, dtype=torch.float32, block_size: int = TILE) -> torch.Tensor:
    """y = x * s with tile scales when ``s.size(0) == x.size(0)``, else block scales
    (triton_kernel.py:80-91)."""
    assert x.is_contiguous() and s.is_contiguous(), "Input tensors must be contiguous"
    assert x.dim() == 2 and s.dim() == 2, "Input tensors must have 2 dimensions"
    assert block_size == TILE
    M, N = x.size()
    y = torch.empty((M, N), dtype=dtype, device=x.device)
    tile_scale = s.size(0) == x.size(0)
    check(lib().aamd_dequant(ptr(x), ptr(s), M, N, int(tile_scale), ptr(y), dtype_code(dtype), stream()))
    return y


def fp8_gemm(a: torch.Tensor, a_s: torch.Tensor, b: torch.Tensor, b_s: torch.Tensor, dtype=torch.bfloat16):
    """C = A @ B^T with 1x128 scales on A and 128x128 (or 1x128) scales on B
    (triton_kernel.py:198-210)."""
    assert a.is_contiguous() and b.is_contiguous()
    assert a_s.is_contiguous() and b_s.is_contiguous()
    pinned = _pinned_options()
    if not pinned:
        return host().fp8_gemm(a, a_s, b, b_s, dtype)
    from . import _probes

    K = a.size(-1)
    M, N = a.numel() // K, b.size(0)
    c = torch.empty(*a.size()[:-1], N, dtype=dtype, device=a.device)
    _probes.check(_probes.lib().aamd_tuning_grouped_gemm_fp8_nt(
        ptr(a), K, ptr(a_s), ptr(b), ptr(b_s), int(b_s.size(0) == N), None, 1, None, M, N, K, ptr(c), dtype_code(dtype), N, None,
        _lib.NONE, _probes.options_array(pinned), stream(),
    ))  # fmt: skip
    return c


# ------------------------------------------------------------------------------------------
# fused / grouped forms
# ------------------------------------------------------------------------------------------
def permute_tile_quant(
    x: torch.Tensor, row_map: torch.Tensor, topk: int, num_out_rows: int, eps: float = 0.0
) -> Tuple[torch.Tensor, torch.Tensor]:
    """Quantise every token row once (1x128) and write it to its ``topk`` permuted rows.
    ``row_map`` [T*topk] int32: permuted row of flat index ``token*topk+slot`` (-1 = dropped)."""
    assert x.dim() == 2 and x.is_contiguous()
    T, cols = x.shape
    assert cols % TILE == 0
    assert row_map.dtype == torch.int32 and row_map.numel() == T * topk and row_map.is_contiguous()
    return host().permute_tile_quant(x, row_map, topk, num_out_rows, eps)


def permute_rows(x: torch.Tensor, row_map: torch.Tensor, topk: int, num_out_rows: int) -> torch.Tensor:
    """out[row_map[t*topk+j]] = x[t]: the un-quantised token permute, each source row read once."""
    assert x.dim() == 2 and x.is_contiguous()
    T, cols = x.shape
    assert row_map.dtype == torch.int32 and row_map.numel() == T * topk and row_map.is_contiguous()
    return host().permute_rows(x, row_map, topk, num_out_rows)


def _alloc_qt(rows: int, ld_t: int, blocked: bool, dev) -> torch.Tensor:
    """A buffer for the transposed codes of ``rows`` columns and ``ld_t`` padded tokens in the shape the quantisers give
    them (``qt_shape`` in csrc/host.cpp): ``[rows, ld_t]``, or, blocked, ``[ld_t/128, rows, 128]`` (token-block-major: every
    128 x 128 tile is 16 KB of consecutive bytes).  For callers of the C ABI, which allocate themselves."""
    return torch.empty(host().qt_shape(rows, ld_t, blocked), dtype=FP8, device=dev)


def qt_ld(q_t: torch.Tensor) -> int:
    """Padded token count ``ld_t`` of transposed codes in either layout."""
    return q_t.shape[0] * TILE if q_t.dim() == 3 else q_t.shape[1]


def qt_rows(q_t: torch.Tensor) -> torch.Tensor:
    """Transposed codes of either layout as ``[rows, ld_t]`` (a copy for the blocked layout)."""
    return q_t.permute(1, 0, 2).reshape(q_t.shape[1], -1) if q_t.dim() == 3 else q_t


def tile_quant_dual_grouped(
    x: torch.Tensor,
    group_offsets: torch.Tensor,
    num_groups: int,
    eps: float = 0.0,
    ld_t: Optional[int] = None,
    rowwise: bool = True,
    blocked: bool = False,
):
    """Row-wise and transposed 1x128 quantisation of ragged row groups in one pass.

    Returns ``(q [M,K], s [M,K/128], q_t [K, ld_t], s_t [ld_t/128, K])``; group g's transposed
    codes start at column ``sum_{j<g} ceil(M_j/128)*128`` and its partial last tile is zero
    padded.  ``ld_t`` defaults to a bound that needs no host knowledge of the splits.
    With ``rowwise=False`` q and s are None.  With ``blocked=True`` q_t is ``[ld_t/128, K, 128]`` (the layout
    the training path uses: the quantiser writes, and the weight-gradient GEMM reads, whole 16 KB tiles);
    ``grouped_gemm_wgrad`` takes either.
    """
    assert x.dim() == 2 and x.is_contiguous()
    M, cols = x.shape
    assert cols % TILE == 0
    assert group_offsets.dtype == torch.int64 and group_offsets.numel() == num_groups + 1
    if ld_t is None:
        ld_t = padded_bound(M, num_groups)
    return host().dual(x, group_offsets, num_groups, eps, ld_t, rowwise, blocked)


def permute_tile_quant_dual_grouped(
    x: torch.Tensor,
    sorted_idx: torch.Tensor,
    topk: int,
    group_offsets: torch.Tensor,
    num_groups: int,
    eps: float = 0.0,
    ld_t: Optional[int] = None,
    rowwise: bool = True,
    blocked: bool = False,
):
    """``tile_quant_dual_grouped`` of the permuted rows without materialising them: ``x [T, K]`` is in token
    order, permuted row j is token ``sorted_idx[j] // topk`` (``sorted_idx`` int64 ``[M]`` from
    ``moe_preprocess``).  Returns ``(q [M,K], s [M,K/128], q_t [K, ld_t], s_t [ld_t/128, K])``, bit-equal to
    ``tile_quant_dual_grouped(permute_rows(x, ...), ...)``."""
    assert x.dim() == 2 and x.is_contiguous()
    T, cols = x.shape
    assert cols % TILE == 0
    assert sorted_idx.dtype == torch.int64 and sorted_idx.dim() == 1 and sorted_idx.is_contiguous()
    M = sorted_idx.numel()
    assert group_offsets.dtype == torch.int64 and group_offsets.numel() == num_groups + 1
    if ld_t is None:
        ld_t = padded_bound(M, num_groups)
    return host().permute_dual(x, sorted_idx, topk, group_offsets, num_groups, eps, ld_t, rowwise, blocked)


def swiglu_tile_quant(fc1: torch.Tensor, return_activation: bool = False):
    """``h = silu(fc1[..., :F]) * fc1[..., F:]`` (SwiGLUActivatition, grouped_gemm_moe.py:331-334)
    quantised 1x128 along the last dim without writing ``h``.  Returns ``(q, s)`` or
    ``(q, s, h)`` (``h`` bf16) with ``return_activation``."""
    assert fc1.dtype == torch.bfloat16 and fc1.stride(-1) == 1 and fc1.is_contiguous()
    two_f = fc1.size(-1)
    assert two_f % (2 * TILE) == 0, "the gated width must be a multiple of 128"
    q, s, h = host().act_quant(fc1, True, return_activation)
    return (q, s, h) if return_activation else (q, s)


def swiglu_tile_quant_dual_grouped(
    fc1: torch.Tensor,
    group_offsets: torch.Tensor,
    num_groups: int,
    ld_t: Optional[int] = None,
    rowwise: bool = True,
    blocked: bool = False,
    return_activation: bool = False,
):
    """SwiGLU fused into ``tile_quant_dual_grouped``: row-wise and transposed 1x128 quantisation of
    ``h = silu(a) * b`` for rows ``[a | b]`` of ``fc1 [M, 2F]``.  Returns ``(q, s, q_t, s_t)`` (plus
    ``h`` with ``return_activation``), layouts as ``tile_quant_dual_grouped``."""
    assert fc1.dim() == 2 and fc1.is_contiguous() and fc1.dtype == torch.bfloat16
    M, two_f = fc1.shape
    assert two_f % (2 * TILE) == 0
    assert group_offsets.dtype == torch.int64 and group_offsets.numel() == num_groups + 1
    if ld_t is None:
        ld_t = padded_bound(M, num_groups)
    res = host().act_dual(fc1, None, True, group_offsets, num_groups, ld_t, rowwise, blocked, return_activation)
    return res if return_activation else res[:4]


def swiglu_bwd_tile_quant_dual_grouped(
    dh: torch.Tensor,
    fc1: torch.Tensor,
    group_offsets: torch.Tensor,
    num_groups: int,
    ld_t: Optional[int] = None,
    rowwise: bool = True,
    blocked: bool = False,
    return_grad: bool = False,
):
    """Backward of ``h = silu(a) * b`` (rows ``[a | b]`` of ``fc1 [M, 2F]``) for the gradient
    ``dh [M, F]``, fused into ``tile_quant_dual_grouped`` of the result ``[da | db]``: what autograd
    makes of SwiGLUActivatition (grouped_gemm_moe.py:331-334) followed by the quantisation of the
    first grouped linear's output gradient.  Returns ``(q [M,2F], s, q_t [2F, ld_t], s_t)`` (plus
    the bf16 gradient ``[M, 2F]`` with ``return_grad``)."""
    assert fc1.dim() == 2 and fc1.is_contiguous() and fc1.dtype == torch.bfloat16
    assert dh.dim() == 2 and dh.is_contiguous() and dh.dtype == torch.bfloat16
    M, two_f = fc1.shape
    assert two_f % (2 * TILE) == 0
    F = two_f // 2
    assert dh.shape == (M, F), "dh must be [M, F]"
    assert group_offsets.dtype == torch.int64 and group_offsets.numel() == num_groups + 1
    if ld_t is None:
        ld_t = padded_bound(M, num_groups)
    res = host().act_dual(fc1, dh, True, group_offsets, num_groups, ld_t, rowwise, blocked, return_grad)
    return res if return_grad else res[:4]


def gelu_tile_quant(x: torch.Tensor, return_activation: bool = False):
    """``h = gelu(x)`` (torch.nn.functional.gelu, the expert MLP's default activation,
    grouped_gemm_moe.py:449) quantised 1x128 along the last dim without writing ``h``.
    Returns ``(q, s)`` or ``(q, s, h)``."""
    assert x.dtype == torch.bfloat16 and x.is_contiguous()
    assert x.size(-1) % TILE == 0
    q, s, h = host().act_quant(x, False, return_activation)
    return (q, s, h) if return_activation else (q, s)


def gelu_tile_quant_dual_grouped(
    x: torch.Tensor,
    group_offsets: torch.Tensor,
    num_groups: int,
    dh: Optional[torch.Tensor] = None,
    ld_t: Optional[int] = None,
    rowwise: bool = True,
    blocked: bool = False,
    return_activation: bool = False,
):
    """GELU fused into ``tile_quant_dual_grouped``: quantises ``h = gelu(x)`` for ``x [M, F]`` bf16, or,
    with ``dh [M, F]``, the gradient ``g = dh * gelu'(x)`` (what autograd computes for the activation).
    Returns ``(q, s, q_t, s_t)`` (plus ``h`` / ``g`` in bf16 with ``return_activation``)."""
    assert x.dim() == 2 and x.is_contiguous() and x.dtype == torch.bfloat16
    M, F = x.shape
    assert F % TILE == 0
    if dh is not None:
        assert dh.shape == x.shape and dh.is_contiguous() and dh.dtype == torch.bfloat16
    assert group_offsets.dtype == torch.int64 and group_offsets.numel() == num_groups + 1
    if ld_t is None:
        ld_t = padded_bound(M, num_groups)
    res = host().act_dual(x, dh, False, group_offsets, num_groups, ld_t, rowwise, blocked, return_activation)
    return res if return_activation else res[:4]


def gradient_quant_with_sums(x: torch.Tensor, group_offsets: torch.Tensor, num_groups: int, dh: Optional[torch.Tensor] = None,
                             activation: Optional[str] = None, ld_t: Optional[int] = None, eps: float = 0.0,
                             sums_dtype=torch.float32):  # fmt: skip
    """The dual quantiser of a gradient (blocked transposed codes) that also sums its columns per group, a bias
    gradient: of ``x [M, N]`` bf16 itself, or, with ``dh``, of the gradient through ``activation`` ("gelu": x
    [M, F]; "swiglu": x [M, 2F]).  Returns ``(q, s, q_t, s_t, sums [E, N])``."""
    assert x.dim() == 2 and x.is_contiguous() and x.dtype == torch.bfloat16 and x.shape[1] % TILE == 0
    assert (dh is None) == (activation is None) and activation in (None, "swiglu", "gelu")
    if dh is not None:
        F = x.shape[1] // (2 if activation == "swiglu" else 1)
        assert dh.shape == (x.shape[0], F) and dh.is_contiguous() and dh.dtype == torch.bfloat16
    assert group_offsets.dtype == torch.int64 and group_offsets.numel() == num_groups + 1
    if ld_t is None:
        ld_t = padded_bound(x.shape[0], num_groups)
    what = {None: 0, "swiglu": 1, "gelu": 2}[activation]
    return host().dual_with_sums(what, x, dh, group_offsets, num_groups, ld_t, eps, sums_dtype)


# which orientation of a weight's codes is written (csrc/host.cpp): both, the one of the weight's own layout, the other one
BOTH, STORED, TURNED = 0, 1, 2


def block_quant_batched(w: torch.Tensor, eps: float = 0.0, return_transpose: bool = False, written: int = BOTH,
                        group_offsets: Optional[torch.Tensor] = None):
    """128x128 block quantisation of ``w [E, N, K]`` in one launch; with ``group_offsets`` (int64 ``[E+1]``, on the device) that of
    the experts that have rows, the others' codes are whatever the memory held.
    Returns ``(q [E,N,K], s [E,N/128,K/128], q_t [E,K,N] | None, s_t [E,K/128,N/128] | None)``.  With
    ``return_transpose``, ``written`` STORED (TURNED) writes only q and s (q_t and s_t), and the other two are their
    transposed views, which ``grouped_gemm_nt`` takes as well."""
    assert w.dim() == 3 and w.stride(2) == 1 and w.stride(1) == w.size(2), "rows of w must be dense"
    return host().block_quant(w, eps, return_transpose, written if return_transpose else BOTH, group_offsets)


def grouped_gemm_nt(
    a: torch.Tensor,
    a_s: torch.Tensor,
    b: torch.Tensor,
    b_s: torch.Tensor,
    group_offsets: torch.Tensor,
    out: Optional[torch.Tensor] = None,
    out_dtype=torch.bfloat16,
    bias: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """out[m] = a[m] @ b[g(m)]^T with block scales, for rows m of group g (device offsets).
    a [M,K] fp8, a_s [M,K/128], b [E,N,K] fp8, b_s [E,N/128,K/128] or [E,N,K/128]; b with block scales may also be the
    transposed view of dense codes [E,K,N], and b_s that of their scales."""
    M, K = a.shape
    E, N, Kb = b.shape
    turned = not b.is_contiguous()
    dense, dense_s = (b.transpose(1, 2), b_s.transpose(1, 2)) if turned else (b, b_s)
    assert Kb == K and a.stride(1) == 1 and dense.is_contiguous() and a_s.is_contiguous() and dense_s.is_contiguous()
    assert group_offsets.dtype == torch.int64 and group_offsets.numel() == E + 1
    assert out is None or (out.shape == (M, N) and out.stride(1) == 1)
    assert bias is None or (bias.shape == (E, N) and bias.is_contiguous())
    pinned = _pinned_options()
    if not pinned:
        return host().gemm_nt(a, a_s, b, b_s, group_offsets, out, out_dtype, bias)
    from . import _probes

    if out is None:
        out = torch.empty((M, N), dtype=out_dtype, device=a.device)
    rest = (M, N, K, ptr(out), dtype_code(out.dtype), out.stride(0), ptr(bias),
            dtype_code(bias.dtype) if bias is not None else _lib.NONE, _probes.options_array(pinned), stream())  # fmt: skip
    if turned:
        _probes.check(_probes.lib().aamd_tuning_grouped_gemm_fp8_nn(
            ptr(a), a.stride(0), ptr(a_s), ptr(b), ptr(b_s), ptr(group_offsets), E, *rest))  # fmt: skip
    else:
        _probes.check(_probes.lib().aamd_tuning_grouped_gemm_fp8_nt(
            ptr(a), a.stride(0), ptr(a_s), ptr(b), ptr(b_s), int(b_s.size(1) == N), ptr(group_offsets), E, None, *rest))  # fmt: skip
    return out


def grouped_gemm_wgrad(
    dy_t: torch.Tensor,
    sdy_t: torch.Tensor,
    x_t: torch.Tensor,
    sx_t: torch.Tensor,
    group_offsets: torch.Tensor,
    out: Optional[torch.Tensor] = None,
    out_dtype=torch.float32,
    accumulate: bool = False,
) -> torch.Tensor:
    """dW[g] (+)= dY_g^T X_g from the transposed 1x128-quantised operands of
    ``tile_quant_dual_grouped``: dy_t [N, ld_t], sdy_t [ld_t/128, N], x_t [K, ld_t], sx_t [ld_t/128, K], or
    both code operands blocked, dy_t [ld_t/128, N, 128] and x_t [ld_t/128, K, 128]."""
    blocked = dy_t.dim() == 3
    assert x_t.dim() == dy_t.dim(), "both operands must be in the same layout"
    N, K = (dy_t.shape[1], x_t.shape[1]) if blocked else (dy_t.shape[0], x_t.shape[0])
    ld_t = qt_ld(dy_t)
    E = group_offsets.numel() - 1
    assert qt_ld(x_t) == ld_t and dy_t.is_contiguous() and x_t.is_contiguous()
    assert sdy_t.shape == (ld_t // TILE, N) and sx_t.shape == (ld_t // TILE, K)
    assert sdy_t.is_contiguous() and sx_t.is_contiguous()
    assert out is not None or not accumulate
    assert out is None or (out.shape == (E, N, K) and out.stride(2) == 1 and out.stride(1) == K)
    pinned = _pinned_options()
    if not pinned:
        return host().gemm_wgrad(dy_t, sdy_t, x_t, sx_t, group_offsets, out, out_dtype, accumulate)
    from . import _probes

    if out is None:
        out = torch.empty((E, N, K), dtype=out_dtype, device=dy_t.device)
    _probes.check(_probes.lib().aamd_tuning_grouped_gemm_fp8_wgrad(
        ptr(dy_t), ptr(sdy_t), ptr(x_t), ptr(sx_t), ld_t, int(blocked), ptr(group_offsets), E, None, N, K, ptr(out),
        dtype_code(out.dtype), out.stride(0) if E > 1 else N * K, int(accumulate), _probes.options_array(pinned), stream(),
    ))  # fmt: skip
    return out


def moe_preprocess(expert_ids: torch.Tensor, num_experts: int, want_sorted: bool = True):
    """Stable counting sort of the flattened expert ids on the device.
    Returns ``(sorted_indices int64 [n] | None, row_map int32 [n], group_offsets int64 [E+1])``."""
    flat = expert_ids.reshape(-1)
    assert flat.is_contiguous() and flat.dtype in (torch.int64, torch.int32)
    return host().moe_preprocess(flat, num_experts, want_sorted)


def invert_permutation(sorted_indices: torch.Tensor, n_flat: int) -> torch.Tensor:
    si = sorted_indices.to(torch.int64).contiguous()
    return host().invert_permutation(si, n_flat)


def unpermute_combine(
    y: torch.Tensor, row_map: torch.Tensor, probs: Optional[torch.Tensor], num_tokens: int, topk: int
) -> torch.Tensor:
    """out[t] = sum_j probs[t,j] * y[row_map[t*topk+j]] in one gather-reduce pass (bf16 or fp32 rows;
    the result has the promoted dtype of rows and probs, as the reference's multiply gives it)."""
    assert y.dim() == 2 and y.is_contiguous() and y.dtype in (torch.bfloat16, torch.float32)
    assert row_map.dtype == torch.int32 and row_map.numel() == num_tokens * topk
    if probs is not None:
        assert probs.shape == (num_tokens, topk)
        probs = probs.contiguous()
    return host().unpermute_combine(y, row_map, probs, num_tokens, topk)


def permute_rows_scaled(
    x: torch.Tensor, row_map: torch.Tensor, topk: int, num_out_rows: int, probs: Optional[torch.Tensor], out_dtype
) -> torch.Tensor:
    """out[row_map[t*topk+j]] = (out_dtype)(x[t] * probs[t, j]): the combine's gradient with respect to
    the permuted rows (rows that no map entry points to are zero)."""
    assert x.dim() == 2 and x.is_contiguous()
    T, cols = x.shape
    assert row_map.dtype == torch.int32 and row_map.numel() == T * topk and row_map.is_contiguous()
    if probs is not None:
        probs = probs.contiguous()
    return host().permute_rows_scaled(x, row_map, topk, num_out_rows, probs, out_dtype)


def unpermute_backward(dout: torch.Tensor, y: torch.Tensor, row_map: torch.Tensor, probs: torch.Tensor, topk: int):
    """Both gradients of ``unpermute_combine`` in one pass over ``dout``: ``(d_rows, d_probs)``, what
    ``permute_rows_scaled`` and ``unpermute_probs_grad`` give, the latter in the weights' dtype."""
    assert dout.dim() == 2 and dout.is_contiguous() and y.dim() == 2 and y.is_contiguous()
    T, H = dout.shape
    assert y.shape[1] == H and row_map.dtype == torch.int32 and row_map.numel() == T * topk
    assert probs.shape == (T, topk)
    return host().unpermute_backward(dout, y, row_map, probs.contiguous(), topk)


def unpermute_probs_grad(dout: torch.Tensor, y: torch.Tensor, row_map: torch.Tensor, topk: int) -> torch.Tensor:
    """d_probs[t, j] = <dout[t], y[row_map[t*topk+j]]> in fp32."""
    assert dout.dim() == 2 and dout.is_contiguous() and y.dim() == 2 and y.is_contiguous()
    T, H = dout.shape
    assert y.shape[1] == H and row_map.dtype == torch.int32 and row_map.numel() == T * topk
    return host().unpermute_probs_grad(dout, y, row_map, topk)


def split_views(t: torch.Tensor, splits: Sequence[int]) -> List[torch.Tensor]:
    return list(torch.split(t, list(splits)))


_pinned = threading.local()  # launch options pinned by gemm_options on this thread


def _pinned_options() -> Optional[dict]:
    stack = getattr(_pinned, "stack", None)
    return stack[-1] if stack else None


class gemm_options:
    """Context manager for tests and tuning runs: inside it the grouped GEMMs of this thread go through the
    measurement library's entry points (include/atorch_amd_probes.h), which take the launch choices as
    per-call arguments: ``with gemm_options(tile=1): ...``.  Nested uses add to the enclosing one's options
    and restore them on exit; nothing process-wide is changed and the product library is not involved."""

    def __init__(self, **opts):
        from . import _probes

        _probes.options_array(opts)  # validates the names
        self.opts = opts

    def __enter__(self):
        if not hasattr(_pinned, "stack"):
            _pinned.stack = []
        outer = _pinned.stack[-1] if _pinned.stack else {}
        _pinned.stack.append({**outer, **self.opts})
        return self

    def __exit__(self, *exc):
        _pinned.stack.pop()
        return False
