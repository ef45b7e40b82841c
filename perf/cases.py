"""The work whose speed is measured: MoE layers and expert blocks as a user's program runs them, through the
package's public entry points.

Six kinds of pass:

* ``layer``       ``FastMoELayer.forward`` under ``no_grad`` (serving), bf16 or fp32.
* ``layer_train`` forward and backward of the same layer: output, input gradient, every parameter's gradient.
* ``block``       the expert block of a SwiGLU model from its gate probabilities on, in bf16: top-k routing, the
                  gather + SwiGLU GEMM, the down GEMM with the weighted merge.
* ``block_fp8``   the same block on row-quantised e4m3 operands, expert weights quantised once (a server's fixed
                  weights), tokens and hidden rows quantised in the pass.
* ``block_train`` forward and backward of the bf16 block.
* ``mlp_fp8``     the two fp8 operators of a SiLU MLP with bias as they are called by default: bf16 weights handed in
                  and quantised inside every call.

Ranges (``draw``): 1 to 8192 tokens per call for the layers and 1 to 32768 for the blocks, any count in between; 4 to
128 experts, top-1 to top-8; widths in multiples of 8 (16-byte rows), most of them multiples of 64; weights in the
layers' storage order ([E, D_out, D_in], "nk") or as plain [E, D_in, D_out] tensors ("kn"); expert loads from a random
linear gate, uniform, or Zipf-skewed with two experts that get no token.
"""
import math

import torch

from fast_moe_amd import FastMoELayer
from fast_moe_amd.kernels import moe, moe_fp8
from fast_moe_amd.kernels.hip import ops
from fast_moe_amd.kernels.hip._lib import EPI_SWIGLU

BF16 = torch.bfloat16


def _case(name, kind, T, E, K, D, H, routing="gate", dtype="bf16", layout="nk"):
    c = {"kind": kind, "T": T, "E": E, "K": K, "D": D, "H": H, "routing": routing, "dtype": dtype, "layout": layout}
    return dict(c, name=name) if name else c


def listed():
    return [
        # a handful of requests on a small layer: launches and host work, hardly any arithmetic
        _case("layer_small", "layer", 64, 8, 2, 128, 256),
        # prefill of the 8-expert SiLU MLP layer, 8 x 1024 tokens
        _case("layer_prefill", "layer", 8192, 8, 2, 1024, 4096),
        # the same layer in fp32, [4, 512] tokens (validation runs, fp32 research models)
        _case("layer_fp32", "layer", 2048, 8, 2, 1024, 4096, dtype="fp32"),
        # training step of a layer whose widths and token count divide by no tile: 3 x 1021 tokens
        _case("layer_train_ragged", "layer_train", 3063, 12, 3, 1000, 2600),
        # decode: 64 sequences through 128 large experts, every expert's weights read for a few rows
        _case("block_decode", "block", 64, 128, 8, 4096, 1536, routing="uniform"),
        # decode of a larger batch on e4m3 weights
        _case("block_decode_fp8", "block_fp8", 512, 128, 8, 4096, 1536, routing="uniform"),
        # chunked prefill through the large experts: about one row tile per expert
        _case("block_chunk", "block", 4096, 128, 8, 4096, 1536, routing="uniform"),
        # the headline configuration: fine-grained experts, skewed load, two experts idle
        _case("block_prefill", "block", 16384, 64, 8, 2048, 1408, routing="zipf"),
        _case("block_prefill_fp8", "block_fp8", 16384, 64, 8, 2048, 1408, routing="zipf"),
        # the largest prefill
        _case("block_large_fp8", "block_fp8", 32768, 128, 8, 4096, 1536, routing="uniform"),
        # training step of the headline configuration
        _case("block_train", "block_train", 16384, 64, 8, 2048, 1408, routing="zipf"),
        # the fp8 operators at their defaults, weights as plain [E, D_in, D_out] tensors, a ragged token count
        _case("mlp_fp8_ops", "mlp_fp8", 4001, 8, 2, 1024, 4096, layout="kn"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi):
    step = rng.choice((64, 64, 64, 8))
    return max(lo, _log_int(rng, lo, hi) // step * step)


def draw(rng):
    while True:
        kind = rng.choice(("layer", "layer", "layer_train", "block", "block", "block_fp8", "block_fp8", "block_train",
                           "mlp_fp8"))
        routing = rng.choice(("gate", "uniform", "zipf"))
        if kind.startswith("layer"):
            dtype = rng.choice(("bf16", "bf16", "fp32"))
            T, E = _log_int(rng, 1, 8192 if dtype == "bf16" else 4096), _log_int(rng, 4, 64)
            D, H, routing, layout = _width(rng, 128, 2048), _width(rng, 256, 4096), "gate", "nk"
        else:
            dtype, layout = "bf16", "nk" if kind == "block_fp8" else rng.choice(("nk", "nk", "kn"))
            T, E = _log_int(rng, 1, 32768), _log_int(rng, 4, 128)
            D, H = _width(rng, 512, 4096), _width(rng, 512, 4096)
        # (a top-1 layer's gate is 1 whatever its scores are: its gate gradient is nothing but rounding noise)
        K = rng.randint(2 if kind == "layer_train" else 1, min(8, E - 2))
        case = _case(None, kind, T, E, K, D, H, routing, dtype, layout)
        w = work(case)
        if w["flops"] <= (3e12 if dtype == "bf16" else 2e11) and w["bytes"] <= 5e9:
            return case


# ------------------------------------------------------------------ inputs
def _randn(g, *shape, scale=1.0, dtype=BF16):
    """N(0, scale^2) values, one slice of the first dimension at a time (large weights never exist in fp32)."""
    out = torch.empty(shape, dtype=dtype, device="cuda")
    for part in (out if len(shape) == 3 else (out,)):
        part.copy_(torch.randn(part.shape, generator=g, device="cuda").mul_(scale))
    return out


def _scores(g, x, E, routing):
    """Gate probabilities [T, E] in fp32."""
    T, D = x.shape
    if routing == "uniform":
        logits = torch.rand(T, E, generator=g, device="cuda") * 1e-3
    else:
        logits = x.float() @ (torch.randn(D, E, generator=g, device="cuda") * D ** -0.5)
    if routing == "zipf":
        p = (torch.arange(E, device="cuda", dtype=torch.float32) + 1) ** -1.1
        logits = logits + torch.log(p / p.sum())
        logits[:, E - 2:] = -1e30
    return torch.softmax(logits, dim=1)


def prepare(case, seed):
    T, E, K, D, H = (case[k] for k in "TEKDH")
    g = torch.Generator(device="cuda").manual_seed(seed)
    state = {"case": case}
    if case["kind"].startswith("layer"):
        dtype = BF16 if case["dtype"] == "bf16" else torch.float32
        with torch.device("cuda"):
            layer = FastMoELayer(D, H, D, E, dtype=dtype).to(dtype)
        with torch.no_grad():
            for p, fan in ((layer.gate.gate.weight, D), (layer.gate.gate.bias, D), (layer._experts_hidden_w, D),
                           (layer._experts_hidden_bias, 100), (layer._experts_w, H), (layer._experts_bias, 100)):
                p.copy_(_randn(g, *p.shape, scale=fan ** -0.5, dtype=dtype))
        train = case["kind"] == "layer_train"
        state.update(layer=layer, x=_randn(g, 1, T, D, dtype=dtype).requires_grad_(train))
        if train:
            state["dy"] = _randn(g, 1, T, D, scale=1e-2, dtype=dtype)
        return state
    x = _randn(g, T, D)
    if case["kind"] in ("block_fp8", "mlp_fp8"):        # 1 % of the rows are outliers
        x[torch.randperm(T, generator=g, device="cuda")[: T // 100]] *= 100
    weight = lambda n, k: (_randn(g, E, n, k, scale=k ** -0.5) if case["layout"] == "nk"
                           else _randn(g, E, k, n, scale=k ** -0.5))
    state.update(x=x, scores=_scores(g, x, E, case["routing"]))
    if case["kind"] == "mlp_fp8":
        state.update(w1=weight(H, D), b1=_randn(g, E, H, scale=0.1), w2=weight(D, H), b2=_randn(g, E, D, scale=0.1))
        return state
    w = {"gate": weight(H, D), "up": weight(H, D), "down": weight(D, H)}
    if case["kind"] == "block_fp8":
        w = {n: moe_fp8.quantize_expert_weights(_kn(case, t)) for n, t in w.items()}
    if case["kind"] == "block_train":
        for t in (x, *w.values()):
            t.requires_grad_(True)
        state["dy"] = _randn(g, T, D, scale=1e-2)
    state["w"] = w
    return state


# -------------------------------------------------------------------- passes
def _kn(case, w):
    """The [E, D_in, D_out] tensor the operators take."""
    return w.permute(0, 2, 1) if case["layout"] == "nk" else w


def _block(state, gates_grad=False):
    case, w, K = state["case"], state["w"], state["case"]["K"]
    r = ops.route_topk(state["scores"], K)
    gates = r["gates"].to(BF16)
    if gates_grad:
        gates.requires_grad_(True)
    hidden = moe.index_select_jagged_bmm_swiglu(0, r["offsets"], r["gate_index"].view(-1, K), state["x"],
                                                _kn(case, w["gate"]), None, _kn(case, w["up"]), None)
    y = moe.silu_jagged_bmm_combine(0, r["offsets"], hidden, _kn(case, w["down"]), None, r["token_index"],
                                    r["reverse_index"], gates, r["gate_index"], has_silu=False)
    return y, gates


def _block_fp8(state):
    w, K, T = state["w"], state["case"]["K"], state["case"]["T"]
    r = ops.route_topk(state["scores"], K)
    qx, sx = moe_fp8.rowwise_quant_fp8(state["x"])
    hidden = ops.grouped_gemm(r["offsets"], qx, w["gate"][0], total_rows=T * K, row_index=r["gate_index"], index_div=K,
                              b2=w["up"][0], epilogue=EPI_SWIGLU, a_scale=sx, b_scale=w["gate"][1],
                              b2_scale=w["up"][1], scales_pow2=True)
    # (the bf16 weight argument only names the shape here: the quantised pair is handed in)
    return moe_fp8.silu_jagged_bmm_combine_fp8(0, r["offsets"], hidden, w["down"][0], None, r["token_index"],
                                               r["reverse_index"], r["gates"].to(BF16), r["gate_index"],
                                               has_silu=False, fp8_weight=w["down"])


def _mlp_fp8(state):
    case, K = state["case"], state["case"]["K"]
    r = ops.route_topk(state["scores"], K)
    hidden = moe_fp8.index_select_jagged_bmm(0, r["offsets"], r["gate_index"].view(-1, K), state["x"],
                                             _kn(case, state["w1"]), state["b1"], fp8=True)
    return moe_fp8.silu_jagged_bmm_combine_fp8(0, r["offsets"], hidden, _kn(case, state["w2"]), state["b2"],
                                               r["token_index"], r["reverse_index"], r["gates"].to(BF16),
                                               r["gate_index"])


def run(state):
    kind, K = state["case"]["kind"], state["case"]["K"]
    if kind == "layer_train":
        layer, x = state["layer"], state["x"]
        x.grad = None
        layer.zero_grad(set_to_none=True)
        y = layer(x, K)
        y.backward(state["dy"])
        return {"y": y, "dx": x.grad, "grads": {n: p.grad for n, p in layer.named_parameters()}}
    if kind == "block_train":
        leaves = {"x": state["x"], **state["w"]}
        for t in leaves.values():
            t.grad = None
        y, gates = _block(state, gates_grad=True)
        y.backward(state["dy"])
        return {"y": y, "gates": gates.grad, "grads": {n: t.grad for n, t in leaves.items()}}
    with torch.no_grad():
        if kind == "layer":
            return state["layer"](state["x"], K)
        if kind == "block":
            return _block(state)[0]
        return _block_fp8(state) if kind == "block_fp8" else _mlp_fp8(state)


# ------------------------------------------------------------- what a pass cannot do without
def work(case):
    """Each input read once and each output written once.  Of the expert weights only those of experts that can get a
    row count (T tokens naming K of E experts each)."""
    T, E, K, D, H, kind = *(case[k] for k in "TEKDH"), case["kind"]
    layer, train = kind.startswith("layer"), kind.endswith("_train")
    mats = 3 if kind.startswith("block") else 2
    esize = 4 if case["dtype"] == "fp32" else 2
    wsize = 1 if kind == "block_fp8" else esize
    idle = 2 if case["routing"] == "zipf" else 0
    hit = (E - idle) * (1 - (1 - K / (E - idle)) ** T)
    weights = hit * mats * D * H
    flops = 2.0 * T * K * mats * D * H + (2.0 * T * D * E if layer else 0)
    nbytes = 2 * T * D * esize + weights * wsize
    if kind == "block_fp8":
        nbytes += 4 * hit * (2 * H + D)                     # the weights' row scales
    nbytes += E * D * esize if layer else T * E * 4         # gate weights / gate probabilities
    if kind in ("layer", "layer_train", "mlp_fp8"):
        nbytes += hit * (D + H) * esize                     # biases
    if train:                                               # dy read, dx and the gradient of every weight written
        flops *= 3
        nbytes += 2 * T * D * esize + E * mats * D * H * esize
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what the same pass differs by when its sums run in another order (the widths of x, of the hidden
    rows and of the weights permuted alike): bf16 9e-4 in norm (a gate gradient; outputs 5e-4) and one or two roundings
    of a single value, 0.018; fp32 1.5e-6 and 1.5e-5.  On e4m3 operands 4e-3 and 0.9: a hidden row whose largest value
    is rounded the other way gets twice the scale, which moves every code of that row."""
    if case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 1e-4}
    if case["kind"] in ("block_fp8", "mlp_fp8"):
        return {"rel": 1.5e-2, "max": 0.99}
    return {"rel": 4e-3, "max": 0.08}
