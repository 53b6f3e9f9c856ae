"""The expert MLP with the permute fused in, on a routing of which some copies were dropped (``permute(num_out_tokens=)``,
token_dispatcher.py:89-116): as many rows come out as are kept, in inference as in training."""
import pytest
import torch

from helpers import randn_bf16, topk_routing

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kept", [1, 128, 301, 399, 400])
def test_fused_dispatch_of_a_routing_with_dropped_copies(dev, kept):
    from atorch_amd import kernels
    from atorch_amd.expert_mlp import TokenDispatch, grouped_mlp
    from atorch_amd.token_dispatcher import permute

    T, E, H, F, k = 200, 5, 256, 128, 2
    idx, _ = topk_routing(T, E, k, seed=1)
    idx = idx.to(dev)
    sorted_idx, row_map, goff = kernels.moe_preprocess(idx, E)
    row_map = torch.where(row_map < kept, row_map, torch.full_like(row_map, -1))
    d = TokenDispatch(sorted_idx[:kept].clone(), row_map, k, goff.clamp(max=kept))
    w1 = randn_bf16((E, 2 * F, H), 2, std=0.05).to(dev)
    w2 = randn_bf16((E, F, H), 3, std=0.05).to(dev)
    x, dy = randn_bf16((T, H), 4).to(dev), randn_bf16((kept, H), 5, std=0.01).to(dev)

    rows, _ = permute(x, idx, num_out_tokens=kept, num_experts=E)
    want = grouped_mlp(rows, w1, w2, d.group_offsets.diff())
    with torch.no_grad():
        assert torch.equal(grouped_mlp(x, w1, w2, None, dispatch=d), want)
    grads = []
    for fused in (True, False):
        xg, w1g = x.clone().requires_grad_(True), w1.clone().requires_grad_(True)
        if fused:
            out = grouped_mlp(xg, w1g, w2, None, dispatch=d)
        else:
            out = grouped_mlp(permute(xg, idx, num_out_tokens=kept, num_experts=E)[0], w1g, w2, d.group_offsets.diff())
        assert torch.equal(out, want)
        out.backward(dy)
        grads.append((xg.grad, w1g.grad))
    assert torch.equal(grads[0][0], grads[1][0]) and torch.equal(grads[0][1], grads[1][1])
