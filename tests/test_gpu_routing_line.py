"""The router preprocess on both sides of the line between one workgroup and two launches, and the one workgroup beyond it for a caller
without scratch: the stable sort of the choices, whichever runs."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,E", [(3072, 60), (3073, 60), (3403, 60), (3404, 60), (3398, 8), (3400, 8), (4603, 1), (4604, 1), (3906, 2), (3907, 2), (4096, 8), (8192, 8), (8193, 8), (3073, 300), (3795, 196), (3796, 196)])
@pytest.mark.parametrize("scratch", [True, False])
def test_routing_line(dev, n, E, scratch):
    from atorch_amd import _lib

    if not scratch and n > 8192:
        pytest.skip("refused without scratch")
    ids = torch.randint(-1, E, (n,), generator=torch.Generator().manual_seed(n + E))
    order = torch.argsort(torch.where(ids < 0, E, ids), stable=True)
    kept = int((ids >= 0).sum())
    place = torch.full((n,), -1, dtype=torch.int32)
    place[order[:kept]] = torch.arange(kept, dtype=torch.int32)
    goff = torch.cat([torch.zeros(1, dtype=torch.int64), torch.bincount(ids[ids >= 0], minlength=E).cumsum(0)])
    held, got_order, got_place, got_goff = (t.to(dev) for t in (ids, torch.zeros_like(order), torch.zeros_like(place), torch.zeros_like(goff)))
    ws = torch.full((_lib.lib().aamd_moe_preprocess_ws_ints(n, E),), -9, dtype=torch.int32, device=dev) if scratch else None
    _lib.check(_lib.lib().aamd_moe_preprocess(held.data_ptr(), 1, n, E, got_order.data_ptr(), got_place.data_ptr(), got_goff.data_ptr(),
                                              ws.data_ptr() if scratch else None, _lib.stream()))  # fmt: skip
    if scratch:  # one workgroup leaves it alone
        assert bool((ws == -9).all()) == (n <= 3200 + 3 * E + 1400 // E)
    assert torch.equal(got_goff.cpu(), goff) and torch.equal(got_place.cpu(), place) and torch.equal(got_order[:kept].cpu(), order[:kept])
