"""Weight codes of the experts that have rows: those of the whole quantiser, and nothing else is written or read."""
import pytest
import torch

from atorch_amd import kernels
from atorch_amd._lib import check, lib, ptr, stream
from atorch_amd.gmm import gmm

pytestmark = pytest.mark.gpu


# (above and below the line of 2^27 elements, from which on an XCD takes eight consecutive blocks)
@pytest.mark.parametrize("E,N,K,rows", [(1, 128, 128, [0]), (5, 256, 384, [0, 3, 0, 200, 0]), (70, 128, 256, [0, 1] * 35),
                                        (33, 2048, 2048, [0] * 32 + [7])])  # fmt: skip
@pytest.mark.parametrize("written", [kernels.BOTH, kernels.STORED, kernels.TURNED])
def test_codes_of_experts_with_rows(E, N, K, rows, written):
    w = torch.randn(E, N, K, device="cuda", dtype=torch.bfloat16)
    off = torch.tensor([0] + rows).cumsum(0).cuda()
    q, s, q_t, s_t = kernels.block_quant_batched(w, return_transpose=True)
    keep = [torch.full_like(t.view(torch.uint8), 0x5A) for t in (q, s, q_t, s_t)]
    a, b = written != kernels.TURNED, written != kernels.STORED
    check(lib().aamd_quant_128x128_grouped(ptr(w), 0, E, N, K, N * K, ptr(off), *[ptr(t) if on else None for t, on in zip(keep, (a, a, b, b))],
                                           0.0, stream()))  # fmt: skip
    for got, want, on in zip(keep, (q, s, q_t, s_t), (a, a, b, b)):
        for e in range(E):
            expected = want[e].view(torch.uint8) if on and rows[e] else torch.full_like(got[e], 0x5A)
            assert torch.equal(got[e], expected)


@pytest.mark.parametrize("trans_b", [True, False])
def test_gmm_reads_no_other_codes(trans_b):
    """Experts without rows hold NaN weights: nothing of them reaches an output, whatever kernel the sizes take."""
    E, K, N = 9, 512, 768
    for rows in ([0, 0, 5, 0, 0, 0, 3, 0, 0], [0, 300, 0, 0, 129, 0, 0, 0, 1], [3000, 0, 0, 0, 2500, 0, 0, 0, 0], [0] * 9):
        g = torch.Generator(device="cuda").manual_seed(3)
        M = sum(rows)
        a = torch.randn(M, K, generator=g, device="cuda", dtype=torch.bfloat16).requires_grad_(True)
        b = torch.randn((E, N, K) if trans_b else (E, K, N), generator=g, device="cuda", dtype=torch.bfloat16)
        dy = torch.randn(M, N, generator=g, device="cuda", dtype=torch.bfloat16)
        res = []
        for fill in (0.0, float("nan")):
            w = b.clone()
            w[[e for e in range(E) if not rows[e]]] = fill
            w.requires_grad_(True)
            a.grad = None
            out = gmm(a, w, torch.tensor(rows), trans_b)
            out.backward(dy)
            res.append((out.detach(), a.grad, w.grad))
        for x, y in zip(*res):
            assert torch.isfinite(x.float()).all() and torch.equal(x, y)


@pytest.mark.parametrize("rows", [[0, 0, 5, 0, 0, 0, 3, 0, 0], [0, 300, 0, 0, 129, 0, 0, 0, 1], [3000, 0, 0, 0, 2500, 0, 0, 0, 0], [0, 130] * 33],
                         ids=lambda r: f"{len(r)}experts_{sum(r)}rows")  # fmt: skip
@pytest.mark.parametrize("written", [kernels.STORED, kernels.TURNED])
def test_products_with_codes_that_were_not_made(rows, written):
    """The codes and scales of experts without rows are NaN: forward, gradient of the rows and their views give what they give on all codes."""
    E, K, N, M = len(rows), 512, 768, sum(rows)
    g = torch.Generator(device="cuda").manual_seed(5)
    off = torch.tensor([0] + rows).cumsum(0).cuda()
    w = torch.randn(E, N, K, generator=g, device="cuda", dtype=torch.bfloat16)
    stored = written == kernels.STORED
    q = torch.full((E, N, K) if stored else (E, K, N), 0x7F, device="cuda", dtype=torch.uint8)
    s = torch.full((E, N // 128, K // 128) if stored else (E, K // 128, N // 128), float("nan"), device="cuda")
    args = (ptr(q), ptr(s), None, None) if stored else (None, None, ptr(q), ptr(s))
    check(lib().aamd_quant_128x128_grouped(ptr(w), 0, E, N, K, N * K, ptr(off), *args, 0.0, stream()))
    q = q.view(kernels.FP8)
    some = (q, s, q.transpose(1, 2), s.transpose(1, 2)) if stored else (q.transpose(1, 2), s.transpose(1, 2), q, s)
    every = kernels.block_quant_batched(w, return_transpose=True, written=written)
    x = torch.randn(M, K, generator=g, device="cuda", dtype=torch.bfloat16)
    dy = torch.randn(M, N, generator=g, device="cuda", dtype=torch.bfloat16)
    (qx, sx), (qd, sd) = kernels.tile_quant(x), kernels.tile_quant(dy)
    for a, a_s, i in ((qx, sx, 0), (qd, sd, 2)):
        got, want = (kernels.grouped_gemm_nt(a, a_s, c[i], c[i + 1], off) for c in (some, every))
        assert torch.isfinite(want.float()).all() and torch.equal(got, want)
