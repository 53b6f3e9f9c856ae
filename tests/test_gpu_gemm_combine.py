"""The second GEMM of a decoding step with the weighted combine in it: the bits of the GEMM and the combine as two launches, for every
number of slots it takes, contractions shorter and longer than its waves take at a time, dropped copies, biases, both activations and
both types of router weights."""
import pytest
import torch

from helpers import randn_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,k,E,N,K", [(1, 1, 1, 128, 128), (1, 4, 60, 2048, 1408), (3, 2, 8, 384, 1152), (8, 8, 64, 256, 640), (5, 3, 7, 128, 2176),
                                       (64, 1, 3, 128, 256), (2, 5, 65, 512, 384), (9, 7, 1024, 128, 1280), (10, 6, 16, 256, 128), (1, 2, 4, 256, 15360)])  # fmt: skip
@pytest.mark.parametrize("drop", ["none", "some", "all"])
@pytest.mark.parametrize("glu", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_bits_of_two_launches(dev, T, k, E, N, K, drop, glu, dtype):
    from atorch_amd import _lib, kernels

    M = T * k
    g = torch.Generator().manual_seed(T + E)
    ids = torch.randint(E, (T, k), generator=g)
    if drop != "none":
        out = torch.rand((T, k), generator=g) < (0.4 if drop == "some" else 2.0)
        ids[out] = torch.where(torch.rand(int(out.sum()), generator=g) < 0.5, -1 - E, E)
    ids = (ids if T % 2 else ids.int()).to(dev)
    q, s, _, _ = kernels.block_quant_batched(randn_bf16((E, N, K), 3, std=0.05).to(dev))
    bias = torch.randn((E, N), generator=g).to(dtype).to(dev) if T != 3 else None
    bias_args = (bias.data_ptr(), kernels.dtype_code(bias.dtype)) if bias is not None else (None, _lib.NONE)
    rows = randn_bf16((M, 2 * K if glu else K), 5).to(dev)
    rows[0, 0] = 0.0
    probs = torch.rand((T, k), generator=g).to(dtype).to(dev)
    _, row_map, goff = kernels.moe_preprocess(ids, E)
    y = torch.zeros((M, N), dtype=torch.bfloat16, device=dev)
    what = 1 if glu else 2
    lib = _lib.lib()
    args = (q.data_ptr(), s.data_ptr())
    assert lib.aamd_quant_grouped_gemm_combine_fits(T, k, N, K, E)
    _lib.check(lib.aamd_quant_grouped_gemm_fp8_nt(what, rows.data_ptr(), rows.shape[1], None, k, T, *args, goff.data_ptr(), E, M, N, K,
                                                  y.data_ptr(), N, *bias_args, _lib.stream()))  # fmt: skip
    want = kernels.unpermute_combine(y, row_map, probs, T, k)
    got = torch.full((T + 1, N), 7.0, dtype=dtype, device=dev)
    _lib.check(lib.aamd_quant_grouped_gemm_combine_fp8_nt(
        what, rows.data_ptr(), rows.shape[1], ids.data_ptr(), int(ids.dtype == torch.int64), row_map.data_ptr(), probs.data_ptr(),
        kernels.dtype_code(dtype), k, T, *args, E, N, K, got.data_ptr(), *bias_args, _lib.stream()))  # fmt: skip
    assert want.dtype == dtype and torch.equal(got[:T], want) and torch.all(got[T] == 7.0)


def test_other_sizes_are_refused(dev):
    from atorch_amd import _lib

    t = torch.zeros(1 << 16, dtype=torch.uint8, device=dev)
    call = lambda T, k, what=1, N=128, K=128: _lib.lib().aamd_quant_grouped_gemm_combine_fp8_nt(  # noqa: E731
        what, t.data_ptr(), 2 * K, t.data_ptr(), 1, t.data_ptr(), t.data_ptr(), 0, k, T, t.data_ptr(), t.data_ptr(), 2, N, K, t.data_ptr(),
        None, _lib.NONE, _lib.stream())  # fmt: skip
    assert call(0, 1) != 0 and call(65, 1) != 0 and call(9, 8) != 0 and call(1, 9) != 0 and call(1, 1, 0) != 0
    assert call(1, 1, 1, 64) != 0 and call(1, 1, 1, 128, 64) != 0


# (measured, two launches -> one: 11.3 -> 19.6 us, 12.9 -> 16.0, 28.3 -> 32.9 from memory, 9.8 -> 15.6; 7.1 -> 6.8, 21.0 -> 18.2, 10.6 -> 8.4, 11.0 -> 8.0)
@pytest.mark.parametrize("T,k,E,N,K,taken", [(4, 8, 16, 512, 4096, False), (4, 2, 8, 7168, 768, False), (1, 2, 8, 4096, 14336, False), (6, 3, 4, 5120, 512, False),
                                             (1, 4, 60, 2048, 1408, True), (8, 4, 60, 2048, 1408, True), (8, 2, 8, 1024, 4096, True), (8, 2, 256, 512, 4096, True)])  # fmt: skip
def test_taken_where_it_is_faster(T, k, E, N, K, taken):
    from atorch_amd import _lib

    assert bool(_lib.lib().aamd_quant_grouped_gemm_combine_fits(T, k, N, K, E)) == taken
