"""A decoding step through the layer: the bits of its parts (router preprocess, expert MLP on the dispatch, weighted combine) and their
tables, on either side of the rules that make the routing in the first GEMM and the combine in the second, and from a replayed graph."""
import pytest
import torch

from helpers import randn_bf16

pytestmark = pytest.mark.gpu


def make(dev, T, k, E, H, F, swiglu, bias, pd, drop, ids_dtype, seed=0):
    from atorch_amd.moe_layer import Grouped_GEMM_MoE

    torch.manual_seed(seed)
    layer = Grouped_GEMM_MoE(H, F, 0.0, E, k, use_swiglu=swiglu, use_bias=bias, implementation_type="Megatron", device=dev, dtype=torch.bfloat16)
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0, 0.05)
    layer.requires_grad_(False)
    x, probs, ids = inputs(dev, T, k, E, H, pd, drop, ids_dtype, seed)
    with torch.no_grad():
        layer(x, probs, ids, is_first_microbatch=True)
    return layer, x, probs, ids


def inputs(dev, T, k, E, H, pd, drop, ids_dtype, seed):
    g = torch.Generator().manual_seed(seed)
    ids = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)])
    if drop:
        out = torch.rand((T, k), generator=g) < 0.4
        ids[out] = torch.where(torch.rand(int(out.sum()), generator=g) < 0.5, -1, E)
    return randn_bf16((T, H), seed).to(dev), torch.rand((T, k), generator=g).to(pd).to(dev), ids.to(ids_dtype).to(dev)


def parts(layer, x, probs, ids):
    from atorch_amd import kernels
    from atorch_amd.expert_mlp import TokenDispatch, grouped_mlp

    sorted_idx, row_map, goff = kernels.moe_preprocess(ids, layer.num_experts)
    y = grouped_mlp(x, layer.w1, layer.w2, None, b1=layer.b1 if layer.use_bias else None, b2=layer.b2 if layer.use_bias else None,
                    activation="swiglu" if layer.use_swiglu else "gelu", transpose_w1=layer.transpose_w1,
                    dispatch=TokenDispatch(sorted_idx, row_map, layer.topk, goff))  # fmt: skip
    return kernels.unpermute_combine(y, row_map, probs, x.shape[0], layer.topk), sorted_idx, row_map, goff


# (routing, combine) in the GEMMs
SIZES = [((1, 4, 60, 512, 256), (True, True)), ((2, 2, 8, 256, 512), (True, True)), ((8, 8, 64, 256, 128), (True, True)), ((1, 1, 4, 128, 128), (True, True)),
         ((4, 8, 16, 512, 4096), (True, False)), ((7, 9, 16, 256, 128), (True, False)), ((6, 8, 32, 512, 8192), (False, False)),
         ((16, 2, 4, 512, 512), (False, False))]  # fmt: skip


@pytest.mark.parametrize("size,fused", SIZES)
@pytest.mark.parametrize("swiglu,bias", [(True, False), (False, True)])
@pytest.mark.parametrize("pd", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("drop,ids_dtype", [(False, torch.int64), (True, torch.int32)])
def test_bits_and_tables(dev, size, fused, swiglu, bias, pd, drop, ids_dtype):
    from atorch_amd import _lib

    T, k, E, H, F = size
    N = F * (2 if swiglu else 1)
    if swiglu:  # the rules say what the sizes are there for
        lib = _lib.lib()
        route = bool(lib.aamd_route_quant_grouped_gemm_fits(T, k, N, H, E))
        combine = bool(lib.aamd_quant_grouped_gemm_fits(T * k, H, F, E, T) and lib.aamd_quant_grouped_gemm_combine_fits(T, k, H, F, E))
        assert (route, route and combine) == fused
    layer, x, probs, ids = make(dev, T, k, E, H, F, swiglu, bias, pd, drop, ids_dtype)
    with torch.no_grad():
        out = layer(x, probs, ids, is_first_microbatch=False)
        want, sorted_idx, row_map, goff = parts(layer, x, probs, ids)
    assert out.dtype == want.dtype and torch.equal(out, want)
    d, n = layer.token_dispatcher, int(goff[-1])
    assert torch.equal(d.sorted_indices[:n], sorted_idx[:n]) and torch.equal(d.row_map, row_map) and torch.equal(d.group_offsets, goff)


@pytest.mark.parametrize("size", [SIZES[0][0], SIZES[4][0], SIZES[7][0]])
def test_one_graph_for_other_routings(dev, size):
    T, k, E, H, F = size
    layer, x, probs, ids = make(dev, T, k, E, H, F, True, False, torch.bfloat16, False, torch.int64)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.no_grad():
        with torch.cuda.stream(side):
            layer(x, probs, ids, is_first_microbatch=False)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = layer(x, probs, ids, is_first_microbatch=False)
        for seed in range(1, 5):
            for held, new in zip((x, probs, ids), inputs(dev, T, k, E, H, torch.bfloat16, seed % 2 == 0, torch.int64, seed)):
                held.copy_(new)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, parts(layer, x, probs, ids)[0])
