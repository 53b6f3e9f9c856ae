"""The work that a user of this package has it do, as cases that can be timed and compared.

A case names a `family` (which public entry points run) and the sizes.  The families:

  layer     ``Grouped_GEMM_MoE``: a whole MoE feed-forward block of one GPU, from tokens, router choices and router
            weights to the block's output; `train` adds the backward to tokens, router weights and expert weights.
            `first`: the expert weights are new in this pass and are quantised in it (the first microbatch of a step);
            otherwise their fp8 codes were made before (serving, later microbatches).
  linear    ``ATorchGroupedLinear`` driven by a host list of rows per expert, the reference's own call; `train` runs
            the microbatches of one optimizer step (`micro`), forward and backward, accumulating the weight gradient
            into fp32 ``main_grad`` buffers.
  gmm       the functional grouped GEMM ``gmm(a, b, batch_sizes, trans_b)``, forward (and backward).
  route     ``permute`` and ``unpermute`` with router weights, forward and backward, rows in bf16 or fp32.
  dispatch  the dispatcher's fused permute + 1x128 quantisation, and its weighted combine.
  dense     the operator module of a dense FP8 linear: quantise, multiply; `train` adds both gradients.

Sizes are those of the benchmark's configurations and of the tests, or lie between them: 4 to 64 experts, hidden sizes
512 to 7168, top-1 to top-8, from one token (a decoding step of one request) to 16384 and more in a training batch.
"""
import math

import torch

from atorch_amd import ops
from atorch_amd.gmm import gmm
from atorch_amd.grouped_linear import ATorchGroupedLinear
from atorch_amd.moe_layer import Grouped_GEMM_MoE
from atorch_amd.token_dispatcher import MoETokenDispatcher, permute, unpermute

BF16, F32, FP8 = torch.bfloat16, torch.float32, torch.float8_e4m3fn
DEV = "cuda"
TILE = 128


def listed():
    return [
        # decoding: one token of one request goes through a block of 60 small experts; nothing but latency
        dict(name="layer_decode_one", family="layer", T=1, E=60, H=2048, F=1408, k=4, act="swiglu", bias=False,
             train=False, first=False, skew=0.0),
        # decoding: a batch of requests, a few rows per expert of a large 64-expert block; reads all weights
        dict(name="layer_decode_batch", family="layer", T=48, E=64, H=7168, F=2048, k=8, act="swiglu", bias=False,
             train=False, first=False, skew=0.0),
        # prefill: a prompt through a block of eight large experts
        dict(name="layer_prefill", family="layer", T=2048, E=8, H=4096, F=14336, k=2, act="swiglu", bias=False,
             train=False, first=False, skew=0.0),
        # training of a small model: GELU experts with biases, a ragged batch, one microbatch per step
        dict(name="layer_train_small", family="layer", T=500, E=8, H=1024, F=4096, k=2, act="gelu", bias=True,
             train=True, first=True, skew=0.0),
        # training: many small experts, uneven routing, a later microbatch of a step
        dict(name="layer_train_uneven", family="layer", T=8191, E=60, H=2048, F=1408, k=4, act="swiglu", bias=False,
             train=True, first=False, skew=1.2),
        # training: the largest batch, eight large experts, weights quantised in the pass
        dict(name="layer_train_large", family="layer", T=16384, E=8, H=4096, F=14336, k=2, act="swiglu", bias=False,
             train=True, first=True, skew=0.0),
        # a small grouped linear in inference, with biases
        dict(name="linear_infer_small", family="linear", M=2048, E=4, K=512, N=1024, bias=True, train=False, micro=1,
             skew=0.0),
        # one optimizer step of a grouped linear: two microbatches, gradients accumulated in fp32, empty experts
        dict(name="linear_train_accumulate", family="linear", M=16001, E=60, K=2048, N=2816, bias=False, train=True,
             micro=2, skew=1.2),
        # the functional grouped GEMM under autograd, weights stored [E, K, N], new in every call
        dict(name="gmm_train", family="gmm", M=8192, E=64, K=2048, N=7168, trans_b=False, train=True, skew=1.2),
        # the router's permute and weighted unpermute as differentiable ops
        dict(name="route_train", family="route", T=8191, E=8, H=4096, k=2, dtype="bf16", skew=0.0),
        # dispatch of a large batch: permute + quantise, then combine
        dict(name="dispatch_large", family="dispatch", T=32768, E=64, H=7168, k=8, skew=1.2),
        # a dense FP8 linear's training step
        dict(name="dense_train", family="dense", M=4096, K=4096, N=14336, train=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _tiles(rng, lo, hi):
    """A multiple of 128, as hidden and feed-forward sizes are, spread over the logarithm of its range."""
    return TILE * max(1, _log_int(rng, lo, hi) // TILE)


def draw(rng):
    limit = max(_cost(c) for c in listed())
    while True:
        family = rng.choice(["layer", "layer", "layer", "layer", "linear", "linear", "gmm", "route", "dispatch", "dense"])
        c = {"family": family}
        if family == "layer":
            train = rng.random() < 0.5
            act = rng.choice(["swiglu", "swiglu", "gelu"])
            E = rng.choice([4, 8, 16, 60, 64])
            c.update(T=_log_int(rng, 64, 16384) if train else _log_int(rng, 1, 4096), E=E, H=_tiles(rng, 512, 7168),
                     F=_tiles(rng, 512, 14336), k=rng.choice([1, 2, 4, 8] if E > 8 else [1, 2]), act=act,
                     bias=act == "gelu" and rng.random() < 0.5, train=train, first=train and rng.random() < 0.5,
                     skew=rng.choice([0.0, 1.2]))
        elif family == "linear":
            train = rng.random() < 0.5
            c.update(M=_log_int(rng, 512 if train else 16, 32768), E=rng.choice([4, 8, 16, 60]), K=_tiles(rng, 512, 7168),
                     N=_tiles(rng, 512, 14336), bias=not train and rng.random() < 0.5, train=train,
                     micro=rng.choice([1, 2]) if train else 1, skew=rng.choice([0.0, 1.2]))
        elif family == "gmm":
            c.update(M=_log_int(rng, 64, 32768), E=rng.choice([4, 8, 16, 64]), K=_tiles(rng, 512, 7168),
                     N=_tiles(rng, 512, 7168), trans_b=rng.random() < 0.5, train=rng.random() < 0.5,
                     skew=rng.choice([0.0, 1.2]))
        elif family == "route":
            c.update(T=_log_int(rng, 32, 32768), E=rng.choice([4, 8, 60, 64]), H=_tiles(rng, 512, 7168),
                     k=rng.choice([1, 2, 4, 8]), dtype=rng.choice(["bf16", "bf16", "f32"]), skew=rng.choice([0.0, 1.2]))
        elif family == "dispatch":
            c.update(T=_log_int(rng, 32, 32768), E=rng.choice([8, 60, 64]), H=_tiles(rng, 512, 7168),
                     k=rng.choice([1, 2, 4, 8]), skew=rng.choice([0.0, 1.2]))
        else:
            train = rng.random() < 0.5
            # the weight gradient contracts over the rows in blocks of 128
            c.update(M=_tiles(rng, 256, 16384) if train else _log_int(rng, 1, 16384), K=_tiles(rng, 512, 7168),
                     N=_tiles(rng, 512, 14336), train=train)
        weights = c.get("E", 1) * c.get("H", c.get("K", 1)) * c.get("F", c.get("N", 1))
        if weights <= 64 * 7168 * 2048 and _cost(c) <= limit:
            return c


# ------------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, shape, std=1.0, dtype=BF16):
    return torch.randn(shape, generator=g, device=DEV, dtype=dtype).mul_(std)


def _expert_scores(g, T, E, skew):
    """Router scores of T tokens; with a skew the experts' popularity falls off like a power of their rank."""
    s = torch.randn((T, E), generator=g, device=DEV)
    if skew:
        s -= skew * torch.log1p(torch.arange(E, device=DEV, dtype=F32))[torch.randperm(E, generator=g, device=DEV)]
    return s


def _routing(g, T, E, k, skew, dtype=BF16):
    """(router weights [T, k], expert ids int64 [T, k]) of a softmax top-k router."""
    vals, idx = torch.topk(torch.softmax(_expert_scores(g, T, E, skew), dim=1), k, dim=1)
    return (vals / vals.sum(1, keepdim=True)).to(dtype), idx


def _splits(g, M, E, skew):
    """Rows per expert of M routed rows (a host list, as the reference's caller has it)."""
    return torch.bincount(_expert_scores(g, M, E, 2 * skew).argmax(1), minlength=E).tolist()


def prepare(case, seed):
    return _PREPARE[case["family"]](case, _gen(seed))


def run(state):
    return state["run"](state)


# ---- layer ---------------------------------------------------------------------------------
def _prep_layer(c, g):
    T, E, H, F, k = c["T"], c["E"], c["H"], c["F"], c["k"]
    layer = Grouped_GEMM_MoE(H, F, 0.0, E, k, use_swiglu=c["act"] == "swiglu", use_bias=c["bias"],
                             implementation_type="Megatron", device=DEV, dtype=BF16)  # fmt: skip
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0, 0.02, generator=g)
    probs, idx = _routing(g, T, E, k, c["skew"])
    s = {"layer": layer, "x": _randn(g, (T, H)), "probs": probs, "idx": idx, "first": c["first"]}
    if c["train"]:
        s["x"].requires_grad_(True)
        s["probs"].requires_grad_(True)
        s["dy"] = _randn(g, (T, H), 0.01)
    else:
        layer.requires_grad_(False)
    if not c["first"]:  # the weights' codes are made once, by the first call on them
        with torch.no_grad():
            layer(s["x"], probs, idx, is_first_microbatch=True)
    s["run"] = _run_layer_train if c["train"] else _run_layer
    return s


def _run_layer(s):
    with torch.no_grad():
        return s["layer"](s["x"], s["probs"], s["idx"], is_first_microbatch=s["first"])


def _run_layer_train(s):
    layer, x, probs = s["layer"], s["x"], s["probs"]
    layer.zero_grad(set_to_none=True)
    x.grad = probs.grad = None
    out = layer(x, probs, s["idx"], is_first_microbatch=s["first"])
    out.backward(s["dy"])
    return [out, x.grad, probs.grad] + [p.grad for p in layer.parameters()]


# ---- linear --------------------------------------------------------------------------------
def _prep_linear(c, g):
    M, E, K, N = c["M"], c["E"], c["K"], c["N"]
    layer = ATorchGroupedLinear(E, K, N, bias=c["bias"], params_dtype=BF16, device=DEV, fuse_wgrad_accumulation=c["train"])
    weights = [getattr(layer, f"weight{i}") for i in range(E)]
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0, 0.02, generator=g)
    s = {"layer": layer, "micro": []}
    for _ in range(c["micro"]):
        m = {"x": _randn(g, (M, K)), "splits": _splits(g, M, E, c["skew"])}
        if c["train"]:
            m["x"].requires_grad_(True)
            m["dy"] = _randn(g, (M, N), 0.01)
        s["micro"].append(m)
    if c["train"]:  # gradients of all experts in one buffer, as a distributed optimizer keeps them
        s["main_grad"] = torch.zeros((E, N, K), dtype=F32, device=DEV)
        for i, w in enumerate(weights):
            w.main_grad = s["main_grad"][i]
    else:
        layer.requires_grad_(False)
        with torch.no_grad():
            layer(s["micro"][0]["x"], s["micro"][0]["splits"], is_first_microbatch=True)
    s["run"] = _run_linear_train if c["train"] else _run_linear
    return s


def _run_linear(s):
    m = s["micro"][0]
    with torch.no_grad():
        return s["layer"](m["x"], m["splits"], is_first_microbatch=False)


def _run_linear_train(s):
    res = []
    for i, m in enumerate(s["micro"]):
        m["x"].grad = None
        out = s["layer"](m["x"], m["splits"], is_first_microbatch=i == 0)
        out.backward(m["dy"])
        res += [out, m["x"].grad]
    return res + [s["main_grad"]]


# ---- gmm -----------------------------------------------------------------------------------
def _prep_gmm(c, g):
    M, E, K, N = c["M"], c["E"], c["K"], c["N"]
    s = {"a": _randn(g, (M, K)), "b": _randn(g, (E, N, K) if c["trans_b"] else (E, K, N), 0.02),
         "sizes": torch.tensor(_splits(g, M, E, c["skew"])), "trans_b": c["trans_b"], "run": _run_gmm}  # fmt: skip
    if c["train"]:
        s["a"].requires_grad_(True)
        s["b"].requires_grad_(True)
        s["dy"] = _randn(g, (M, N), 0.01)
        s["run"] = _run_gmm_train
    return s


def _run_gmm(s):
    with torch.no_grad():
        return gmm(s["a"], s["b"], s["sizes"], s["trans_b"])


def _run_gmm_train(s):
    a, b = s["a"], s["b"]
    a.grad = b.grad = None
    out = gmm(a, b, s["sizes"], s["trans_b"])
    out.backward(s["dy"])
    return [out, a.grad, b.grad]


# ---- route ---------------------------------------------------------------------------------
def _prep_route(c, g):
    dt = BF16 if c["dtype"] == "bf16" else F32
    probs, idx = _routing(g, c["T"], c["E"], c["k"], c["skew"], dt)
    return {"x": _randn(g, (c["T"], c["H"]), 1.0, dt).requires_grad_(True), "probs": probs.requires_grad_(True),
            "idx": idx, "E": c["E"], "dy": _randn(g, (c["T"], c["H"]), 0.01, dt), "run": _run_route}  # fmt: skip


def _run_route(s):
    x, probs = s["x"], s["probs"]
    x.grad = probs.grad = None
    rows, order = permute(x, s["idx"], num_experts=s["E"])
    out = unpermute(rows, order, probs)
    out.backward(s["dy"])
    return [rows, order, out, x.grad, probs.grad]


# ---- dispatch ------------------------------------------------------------------------------
def _prep_dispatch(c, g):
    probs, idx = _routing(g, c["T"], c["E"], c["k"], c["skew"])
    return {"d": MoETokenDispatcher(c["E"], c["k"]), "x": _randn(g, (c["T"], c["H"])), "probs": probs, "idx": idx,
            "y": _randn(g, (c["T"] * c["k"], c["H"])), "run": _run_dispatch}  # fmt: skip


def _run_dispatch(s):
    d = s["d"]
    with torch.no_grad():
        q, scale, offsets = d.token_permutation_fp8(s["x"], s["probs"], s["idx"])
        out, _ = d.token_unpermutation(s["y"])  # (the experts' output, made elsewhere)
    return [q.view(torch.uint8), scale, offsets, out]


# ---- dense ---------------------------------------------------------------------------------
def _prep_dense(c, g):
    M, K, N = c["M"], c["K"], c["N"]
    s = {"x": _randn(g, (M, K)), "w": _randn(g, (N, K), 0.02), "run": _run_dense}
    if c["train"]:
        s["dy"] = _randn(g, (M, N), 0.01)
        s["run"] = _run_dense_train
    else:
        s["qw"], s["sw"], _, _ = ops.quantize_square_blockwise(s.pop("w"), FP8, TILE)
    return s


def _run_dense(s):
    qx, sx, _, _ = ops.quantize_vector_blockwise(s["x"], FP8, TILE)
    return ops.fp8_gemm_blockwise(qx, sx, s["qw"], s["sw"], BF16)


def _run_dense_train(s):
    qx, sx, qx_t, sx_t = ops.quantize_vector_blockwise(s["x"], FP8, TILE, return_transpose=True)
    qw, sw, qw_t, sw_t = ops.quantize_square_blockwise(s["w"], FP8, TILE, return_transpose=True)
    y = ops.fp8_gemm_blockwise(qx, sx, qw, sw, BF16)
    qd, sd, qd_t, sd_t = ops.quantize_vector_blockwise(s["dy"], FP8, TILE, return_transpose=True)
    dx = ops.fp8_gemm_blockwise(qd, sd, qw_t, sw_t, BF16)
    dw = ops.fp8_gemm_blockwise(qd_t, sd_t, qx_t, sx_t, F32, is_b_1d_scaled=True)
    return [y, dx, dw]


_PREPARE = {"layer": _prep_layer, "linear": _prep_linear, "gmm": _prep_gmm, "route": _prep_route,
            "dispatch": _prep_dispatch, "dense": _prep_dense}  # fmt: skip


# ------------------------------------------------------------------------------------------
# what a pass cannot do without
# ------------------------------------------------------------------------------------------
def _experts_hit(E, rows_per_draw, draws):
    """Experts that get at least one row, for even routing."""
    return E * (1.0 - (1.0 - rows_per_draw / E) ** draws)


def work(case):
    c = case
    fam, scale = c["family"], 1.0 + 4.0 / TILE  # an fp8 code and its share of a 1x128 scale
    if fam == "layer":
        T, E, H, F, k = c["T"], c["E"], c["H"], c["F"], c["k"]
        M, n1 = T * k, F * (2 if c["act"] == "swiglu" else 1)
        per_expert = n1 * H + F * H
        hit = _experts_hit(E, k, T)
        flops = 2.0 * M * per_expert
        nbytes = 2.0 * 2 * T * H + 10.0 * M  # tokens in, tokens out, ids and weights of the router
        if not c["train"]:
            nbytes += (2.0 if c["first"] else 1.0) * hit * per_expert
        else:
            flops *= 3
            nbytes += (2.0 if c["first"] else 1.0) * E * per_expert + 2.0 * E * per_expert + 2.0 * 2 * T * H + 4.0 * M
            if c["bias"]:
                nbytes += 2.0 * 2 * E * (n1 + H)
        return {"bytes": nbytes, "flops": flops}
    if fam == "linear":
        M, E, K, N, n = c["M"], c["E"], c["K"], c["N"], c["micro"]
        hit = _experts_hit(E, 1, M)
        if not c["train"]:
            return {"bytes": 2.0 * M * (K + N) + hit * N * K + 2.0 * c["bias"] * E * N, "flops": 2.0 * M * N * K}
        return {"bytes": n * 2 * 2.0 * M * (K + N) + 2.0 * E * N * K + 4.0 * E * N * K, "flops": n * 6.0 * M * N * K}
    if fam == "gmm":
        M, E, K, N = c["M"], c["E"], c["K"], c["N"]
        if not c["train"]:
            return {"bytes": 2.0 * M * (K + N) + 2.0 * _experts_hit(E, 1, M) * N * K, "flops": 2.0 * M * N * K}
        return {"bytes": 2 * 2.0 * M * (K + N) + 2 * 2.0 * E * N * K, "flops": 6.0 * M * N * K}
    if fam == "route":
        T, H, k, el = c["T"], c["H"], c["k"], 2.0 if c["dtype"] == "bf16" else 4.0
        # x in, rows out; rows in, out out; dy in, row gradients out (and back in for the sum), rows in for the weights
        return {"bytes": el * H * (T + T * k + T + T + T) + 28.0 * T * k, "flops": 6.0 * T * k * H}
    if fam == "dispatch":
        T, H, k = c["T"], c["H"], c["k"]
        return {"bytes": 2.0 * T * H + scale * T * k * H + 2.0 * T * k * H + 2.0 * T * H + 10.0 * T * k,
                "flops": 2.0 * T * k * H}  # fmt: skip
    M, K, N = c["M"], c["K"], c["N"]
    if not c["train"]:
        return {"bytes": 2.0 * M * (K + N) + N * K, "flops": 2.0 * M * N * K}
    return {"bytes": 2 * 2.0 * M * (K + N) + 2.0 * N * K + 4.0 * N * K, "flops": 6.0 * M * N * K}


def _cost(c):
    w = work(c)
    return max(w["bytes"], w["flops"] / 300.0)


def tolerance(case):
    if case["family"] in ("route", "dispatch"):
        # rows, codes and orders are copies or rounded once: whole numbers are the same; sums are rounded to the rows' type
        return {"rel": 5e-3 if case.get("dtype", "bf16") == "bf16" else 1e-5, "differ": 0.0}
    # bf16 results of fp8 products summed in fp32; an intermediate that is rounded and quantised again among them
    return {"rel": 1e-2}
