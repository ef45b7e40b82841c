"""The native host calls (csrc/host_calls.cpp) against the Python code that takes what they decline: the same
kernels on the same operands, so the same bits, for calls they take and for calls they leave."""
import contextlib
import ctypes

import pytest
import torch

from helpers import BF16, dev, make_routing, randn

pytestmark = pytest.mark.gpu


class Declines:
    """A host module that takes nothing."""

    def __getattr__(self, name):
        return lambda *a: None


class Recorder:
    """The host module, noting of every call whether it took it."""

    def __init__(self, real):
        self.real, self.took = real, []

    def __getattr__(self, name):
        def call(*a):
            res = getattr(self.real, name)(*a)
            self.took.append(res is not None)
            return res
        return call


class Sub(torch.Tensor):
    pass


def both(fn, taken):
    """fn's result by way of the host module, which takes (all of) the call or declines it as ``taken`` says (None: some of
    it), and by the Python code alone."""
    from fast_moe_amd.kernels.hip import _lib
    real = _lib.host()
    recorder = _lib._host = Recorder(real)
    try:
        native = fn()
        assert taken is None or (recorder.took and (all if taken else any)(recorder.took) == taken), recorder.took
        _lib._host = Declines()
        return native, fn()
    finally:
        _lib._host = real


def same(a, b):
    if isinstance(a, dict):
        a, b = list(a.values()), [b[n] for n in a]
    for x, y in zip(*((v if isinstance(v, (list, tuple)) else [v]) for v in (a, b))):
        assert x.dtype == y.dtype and x.shape == y.shape and x.stride() == y.stride()
        assert torch.equal(x.view(torch.uint8) if x.element_size() == 1 else x, y.view(torch.uint8) if y.element_size() == 1 else y)


@pytest.mark.parametrize("T,E,K", [(1, 4, 1), (65, 8, 2), (300, 130, 8)])
@pytest.mark.parametrize("form", ["plain", "strided", "subclass", "fp32"])
def test_operators(T, E, K, form):
    from fast_moe_amd.kernels.hip import ops
    from fast_moe_amd.kernels.hip._lib import EPI_SWIGLU
    dtype = torch.float32 if form == "fp32" else BF16
    make = {"plain": lambda t: t, "fp32": lambda t: t, "subclass": lambda t: t.as_subclass(Sub),
            "strided": lambda t: torch.cat([t, t], dim=-1)[..., :t.shape[-1]]}[form]
    D, H = 64, 96
    scores = make(dev(torch.softmax(randn((T, E), 1).float(), 1)))
    x = make(dev(randn((T, D), 2).to(dtype)))
    w, wp = (make(dev(randn((E, H, D), s, scale=D ** -0.5).to(dtype))).permute(0, 2, 1) for s in (3, 4))
    bias = make(dev(randn((E, H), 5).to(dtype)))
    taken = form != "subclass"
    same(*both(lambda: ops.route_topk(scores, K), taken and scores.is_contiguous()))
    r = ops.route_topk(scores, K)
    off, idx = r["offsets"], r["gate_index"]
    for kw in (dict(), dict(bias=bias), dict(bias=bias, bias2=bias, b2=wp, epilogue=EPI_SWIGLU)):
        same(*both(lambda: ops.grouped_gemm(off, x, w, total_rows=T * K, row_index=idx.view(-1, K), index_div=K, **kw), taken))
    n_contiguous = w.contiguous()
    same(*both(lambda: ops.grouped_gemm(off, x, n_contiguous, total_rows=T * K, row_index=idx, index_div=K), False))
    value = make(ops.grouped_gemm(off, x, w, total_rows=T * K, row_index=idx, index_div=K))
    for gates in (None, r["gates"], r["gates"].to(BF16), r["gates"].reshape(-1)):
        same(*both(lambda: ops.combine(value, r["reverse_index"], gates, idx), taken and (gates is None or gates.ndim == 2)))
    for silu in (False, True):
        same(*both(lambda: ops.quant_rows_fp8(x, apply_silu=silu), taken))
        q, s = ops.quant_rows_fp8(x, apply_silu=silu)
        assert ops.scales_are_pow2(s)


@pytest.mark.parametrize("dtype", [BF16, torch.float32])
@pytest.mark.parametrize("B,S", [(1, 1), (2, 33), (3, 0)])
def test_layer_forward(B, S, dtype):
    from fast_moe_amd import FastMoELayer
    torch.manual_seed(0)
    layer = FastMoELayer(64, 96, 64, 8, dtype=dtype).to(dtype).cuda()
    x = dev(randn((B, S, 64), 1).to(dtype))
    with torch.no_grad():
        same(*both(lambda: layer(x, 2), True if S else None))

    class Rerouted(FastMoELayer):       # a route() of its own is asked
        def route(self, x, k):
            self.asked = True
            return super().route(x, k)

    if S:
        other = Rerouted(64, 96, 64, 8, dtype=dtype).to(dtype).cuda()
        other.load_state_dict(layer.state_dict())
        with torch.no_grad():
            same(other(x, 2), layer(x, 2))
        assert other.asked


@pytest.mark.parametrize("T,E,K", [(2, 4, 1), (40, 8, 2), (300, 130, 8)])
@pytest.mark.parametrize("form", ["plain", "strided", "subclass", "fp32"])
def test_backward_operators(T, E, K, form):
    from fast_moe_amd.kernels.hip import ops
    dtype = torch.float32 if form == "fp32" else BF16
    make = {"plain": lambda t: t, "fp32": lambda t: t, "subclass": lambda t: t.as_subclass(Sub),
            "strided": lambda t: torch.cat([t, t], dim=-1)[..., :t.shape[-1]]}[form]
    D, H, R = 64, 96, T * K
    r = {k: v.cuda() for k, v in make_routing(T, E, K, seed=T).items()}
    rows = lambda n, seed: dev(randn((R, n), seed).to(dtype))
    dy, value, g, u, dh = dev(randn((T, D), 1).to(dtype)), rows(D, 2), rows(H, 3), rows(H, 4), rows(H, 5)
    gates, index = dev(torch.rand(T, K).to(dtype)), r["gate_index"]
    plain = form in ("plain", "fp32")
    for need in (False, True):
        same(*both(lambda: [t for t in ops.combine_bwd(make(dy), value, index, K, gates, index, need_gate_grad=need) if t is not None], plain))
    same(*both(lambda: [t for t in ops.combine_bwd(make(dy), None, index, K) if t is not None], plain))
    same(*both(lambda: ops.segment_colsum(make(value), r["offsets"]), plain or form == "strided"))
    for joint in (False, True):
        same(*both(lambda: ops.swiglu_bwd(make(g), u, dh, joint=joint), plain))
    same(*both(lambda: ops.swiglu_bwd(make(g), None, dh)[:1], plain))
    for slack in (False, True):
        same(*both(lambda: ops.silu_mul(make(g), None, with_slack=slack), plain))
    same(*both(lambda: ops.gather_rows(make(dy), index, K), plain or form == "strided"))
    same(*both(lambda: ops.invert_index(index.view(T, K)), True))
    scores = dev(torch.rand(T, E).to(dtype))
    same(*both(lambda: ops.gate_l1_bwd(make(scores), r["topk_idx"], gates), plain))
    for halves in (False, True):
        a, b = ops.empty_rows(R, 128, dtype, "cuda").normal_(), ops.empty_rows(R, D, dtype, "cuda").normal_()
        same(*both(lambda: ops.jagged_weight_grad(a, b, r["offsets"], halves=halves), True))
    # weights with n contiguous, read in place
    w = dev(randn((E, H, D), 6).to(dtype))
    same(*both(lambda: ops.input_grad_gemm(r["offsets"], make(g), w), form != "subclass"))


@pytest.mark.parametrize("where", ["class", "object"])
def test_a_replaced_route_is_asked(where, monkeypatch):
    from fast_moe_amd import FastMoELayer
    layer = FastMoELayer(64, 96, 64, 8, dtype=BF16).to(BF16).cuda()
    x = dev(randn((1, 33, 64), 1))
    asked, real = [], FastMoELayer.route

    def route(self, x, k):
        asked.append(k)
        return real(self, x, k)

    with torch.no_grad():
        want = layer(x, 2)
        if where == "class":
            monkeypatch.setattr(FastMoELayer, "route", route)
        else:
            layer.route = route.__get__(layer)
        same(layer(x, 2), want)
    assert asked == [2]


def test_refusals_are_the_python_codes():
    from fast_moe_amd.kernels.hip import ops
    r = make_routing(16, 4, 2, seed=1)
    x, w = dev(randn((16, 64), 1)), dev(randn((4, 32, 64), 2)).permute(0, 2, 1)
    off = dev(r["offsets"])
    with pytest.raises(ValueError, match="share a dtype"):
        ops.grouped_gemm(off, x, w.float(), total_rows=32)
    with pytest.raises(ValueError, match="bias must be"):
        ops.grouped_gemm(off, x, w, total_rows=32, bias=dev(randn((4, 31), 3)))
    with pytest.raises(ValueError, match="total_rows entries"):
        ops.grouped_gemm(off, x, w, total_rows=32, row_index=dev(r["index"]).view(-1)[:31])
    with pytest.raises(ValueError, match="different devices|live on the GPU"):
        ops.grouped_gemm(off, x, w.cpu(), total_rows=32)
    with pytest.raises(ValueError, match="int64"):
        ops.combine(x, dev(r["index"]).int())
    with pytest.raises((RuntimeError, ValueError)):
        ops.route_topk(dev(torch.rand(16, 4)), 5)


@contextlib.contextmanager
def entry_point(name, fn):
    """The host module calls ``fn`` (a ctypes callback) in the place of one C entry point."""
    from fast_moe_amd.kernels.hip import _lib
    lib, host = _lib.load(), _lib.host()
    real = [ctypes.cast(lib[n], ctypes.c_void_p).value for n in _lib.HOST_ENTRY_POINTS]
    swapped = list(real)
    swapped[_lib.HOST_ENTRY_POINTS.index(name)] = ctypes.cast(fn, ctypes.c_void_p).value
    host.init(*swapped)
    try:
        yield
    finally:
        host.init(*real)


@pytest.mark.parametrize("name", ["fmoe_route_topk", "fmoe_grouped_gemm", "fmoe_combine", "fmoe_quant_rows_e4m3"])
def test_a_launch_error_is_raised_and_nothing_is_issued_again(name, monkeypatch):
    """A launch error (forced on the host: the entry point returns the status and launches nothing) raises what the Python
    code raises for it; the operator is not tried a second time."""
    from fast_moe_amd import FastMoELayer
    from fast_moe_amd.kernels.hip import _lib, ops
    r = ops.route_topk(dev(torch.rand(16, 4)), 2)
    x, w = dev(randn((16, 64), 1)), dev(randn((4, 32, 64), 2)).permute(0, 2, 1)
    value = dev(randn((32, 64), 3))
    layer = FastMoELayer(64, 96, 64, 4, dtype=BF16).to(BF16).cuda()
    calls = {"fmoe_route_topk": lambda: ops.route_topk(dev(torch.rand(16, 4)), 2),
             "fmoe_grouped_gemm": lambda: ops.grouped_gemm(r["offsets"], value, w, total_rows=32),
             "fmoe_combine": lambda: ops.combine(value, r["reverse_index"], r["gates"], r["gate_index"]),
             "fmoe_quant_rows_e4m3": lambda: ops.quant_rows_fp8(x)}
    issued = []
    fails = ctypes.CFUNCTYPE(ctypes.c_int)(lambda: issued.append(name) or 4)     # FMOE_ERR_LAUNCH
    _lib.host()
    monkeypatch.setattr(_lib.load(), name, lambda *a: pytest.fail("issued again by the Python code"))
    with torch.no_grad():
        for fn in [calls[name]] + ([] if name == "fmoe_quant_rows_e4m3" else [lambda: layer(x.view(1, 16, 64), 2)]):
            issued.clear()
            with entry_point(name, fails), pytest.raises(RuntimeError, match=f"{name} failed .status 4"):
                fn()
            assert issued == [name]


@pytest.mark.parametrize("case", ["experts of another dtype", "no tokens", "a bias of other strides", "plain"])
def test_the_layer_routes_once(case, monkeypatch):
    """A layer call has issued its routing once, whether the host module takes the call whole or declines it (the first case
    is a default-constructed layer: bf16 experts under an fp32 gate and fp32 tokens)."""
    from fast_moe_amd import FastMoELayer
    from fast_moe_amd.kernels.hip import _lib
    layer = FastMoELayer(64, 96, 64, 4, dtype=BF16).cuda()
    if case != "experts of another dtype":
        layer = layer.to(BF16)
    if case == "a bias of other strides":       # (only the second GEMM's operands tell)
        layer._experts_bias.data = torch.zeros(64, 4, dtype=BF16, device="cuda").t()
    x = dev(randn((1, 0 if case == "no tokens" else 16, 64), 1).to(layer.gate.gate.weight.dtype))
    lib = _lib.load()
    _lib.host()         # (takes the entry points' addresses: before one is replaced below)
    routed = []
    proto = ctypes.CFUNCTYPE(ctypes.c_int, *lib.fmoe_route_topk.argtypes)
    real = proto(ctypes.cast(lib["fmoe_route_topk"], ctypes.c_void_p).value)

    def native(*a):
        routed.append("native")
        return real(*a)

    def python(*a, fn=lib.fmoe_route_topk):
        routed.append("python")
        return fn(*a)

    calls = proto(native)
    monkeypatch.setattr(lib, "fmoe_route_topk", python)
    with torch.no_grad(), entry_point("fmoe_route_topk", calls):
        y = layer(x, 2)
    assert len(routed) == 1 and y.shape == x.shape
