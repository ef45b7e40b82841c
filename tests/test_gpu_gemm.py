"""GPU parity: jagged GEMM operators (bf16 and fp8) against the oracle, through the
operator API (and therefore the C ABI)."""
import itertools

import numpy as np
import pytest
import torch

from oracle import moe as o_moe
from oracle import moe_fp8 as o_fp8
from tests.helpers import BF16, assert_bf16_close, dev, kernels_run, make_routing, randn, skewed_topk, uniform
from oracle import routing as o_routing

pytestmark = pytest.mark.gpu

KTAIL = ", true>(fmoe::GemmParams)"      # the ring kernel's last template argument, in a trace

# kernels/tests/moe_test.py:35-84: default assert_close for bf16 is rtol 1.6e-2, atol 1e-5
REF_RTOL, REF_ATOL = 1.6e-2, 1e-5


def weights(E, K, N, seed, contiguous=True, scale=None):
    w = uniform((E, K, N), seed) if scale is None else randn((E, K, N), seed, scale=scale)
    if not contiguous:          # [E, K, N] view of [E, N, K] storage (moe_test.py:223-239)
        w = w.transpose(1, 2).contiguous().transpose(1, 2)
    return w


GRID = [(L, E, K, Din, Dout) for L, E, K, Din, Dout in itertools.product(
    [16, 100, 500], [4, 16], [2, 4], [12, 32, 64], [32, 128])]


@pytest.mark.parametrize("L,E,K,Din,Dout", GRID[::3])
@pytest.mark.parametrize("contiguous", [True, False])
@pytest.mark.parametrize("has_bias", [True, False])
def test_index_select_jagged_bmm_reference_grid(L, E, K, Din, Dout, contiguous, has_bias):
    from fast_moe_amd.kernels import moe
    print(f"bmm L={L} E={E} K={K} Din={Din} Dout={Dout} contiguous={contiguous} bias={has_bias}", flush=True)
    r = make_routing(L, E, K, seed=L + E)
    x = uniform((L, Din), 1)
    w = weights(E, Din, Dout, 2, contiguous)
    b = uniform((E, Dout), 3) if has_bias else None
    ref = o_moe.index_select_jagged_bmm(r["offsets"], r["index"], x.float(), w.float(),
                                        None if b is None else b.float())
    with torch.no_grad():
        out = moe.index_select_jagged_bmm(int(r["lengths"].max()), dev(r["offsets"]), dev(r["index"]), dev(x),
                                          dev(w), dev(b))
    assert out.dtype == BF16 and tuple(out.shape) == (L * K, Dout)
    torch.testing.assert_close(out.cpu(), ref.to(BF16), rtol=REF_RTOL, atol=REF_ATOL)


@pytest.mark.parametrize("L,E,K,Din,Dout,contiguous", [
    (2048, 8, 2, 256, 512, False),      # tall tiles, K-contiguous weights (the layer's layout)
    (2048, 8, 2, 256, 512, True),       # tall tiles, N-contiguous weights
    (1500, 4, 2, 200, 136, False),      # ragged rows, K tail, N tail
    (4096, 64, 8, 128, 96, False),
    (300, 128, 8, 64, 256, False),      # short tiles
])
def test_index_select_jagged_bmm_larger(L, E, K, Din, Dout, contiguous):
    from fast_moe_amd.kernels import moe
    r = make_routing(L, E, K, seed=L)
    x = randn((L, Din), 1)
    w = weights(E, Din, Dout, 2, contiguous, scale=Din ** -0.5)
    b = randn((E, Dout), 3)
    ref = o_moe.index_select_jagged_bmm(r["offsets"], r["index"], x.float(), w.float(), b.float())
    with torch.no_grad():
        out = moe.index_select_jagged_bmm(0, dev(r["offsets"]), dev(r["index"]), dev(x), dev(w), dev(b))
    assert_bf16_close(out, ref, rtol=1e-2, atol=1e-2, what="index_select_jagged_bmm")


def test_skewed_and_empty_experts():
    from fast_moe_amd.kernels import moe
    T, E, K, D, H = 4096, 64, 8, 128, 192
    topk = skewed_topk(T, E, K, seed=3)
    meta = o_routing.routing_metadata(topk.numpy(), E)
    assert (meta["lengths"] == 0).sum() >= 2 and meta["lengths"].max() > 8 * meta["lengths"][meta["lengths"] > 0].min()
    offsets = torch.from_numpy(meta["offsets"])
    index = torch.from_numpy(meta["gate_index"]).view(-1, K)
    x = randn((T, D), 1)
    wg = weights(E, D, H, 2, False, scale=D ** -0.5)
    wu = weights(E, D, H, 3, False, scale=D ** -0.5)
    ref = o_moe.index_select_jagged_bmm_swiglu(offsets, index, x.float(), wg.float(), None, wu.float(), None)
    with torch.no_grad():
        out = moe.index_select_jagged_bmm_swiglu(0, dev(offsets), dev(index), dev(x), dev(wg), None, dev(wu), None)
    # product of two bf16-rounded GEMM results: the reference's own bf16 rtol (1.6e-2)
    assert_bf16_close(out, ref, rtol=1.6e-2, atol=1e-2, what="swiglu, skewed")


@pytest.mark.parametrize("L,E,K,Din,Dout,bias,contiguous", [
    (100, 8, 2, 32, 64, True, True), (500, 4, 4, 64, 64, False, False), (2048, 8, 2, 128, 256, True, False),
    (64, 16, 2, 24, 40, True, True)])
def test_swiglu_and_gating(L, E, K, Din, Dout, bias, contiguous):
    from fast_moe_amd.kernels import moe
    r = make_routing(L, E, K, seed=L + 1)
    x, x2 = uniform((L, Din), 1), uniform((L, Din), 4)
    w, wp = weights(E, Din, Dout, 2, contiguous), weights(E, Din, Dout, 5, contiguous)
    b = uniform((E, Dout), 3) if bias else None
    bp = uniform((E, Dout), 6) if bias else None
    f = lambda t: None if t is None else t.float()
    ref = o_moe.index_select_jagged_bmm_swiglu(r["offsets"], r["index"], f(x), f(w), f(b), f(wp), f(bp))
    with torch.no_grad():
        out = moe.index_select_jagged_bmm_swiglu(0, dev(r["offsets"]), dev(r["index"]), dev(x), dev(w), dev(b),
                                                 dev(wp), dev(bp))
        xa = dev(x)
        out_same = moe.index_select_jagged_gating_bmm(0, dev(r["offsets"]), dev(r["index"]), xa, xa, dev(w),
                                                      dev(b), dev(wp), dev(bp))
        out_two = moe.index_select_jagged_gating_bmm(0, dev(r["offsets"]), dev(r["index"]), dev(x), dev(x2),
                                                     dev(w), dev(b), dev(wp), dev(bp))
    # tolerance of kernels/tests/moe_test.py:729-949 for bf16 products of two GEMMs
    assert_bf16_close(out, ref, rtol=1.6e-2, atol=2e-2, what="swiglu")
    assert torch.equal(out, out_same)
    ref2 = o_moe.index_select_jagged_gating_bmm(r["offsets"], r["index"], f(x), f(x2), f(w), f(wp), f(b), f(bp))
    assert_bf16_close(out_two, ref2, rtol=1.6e-2, atol=2e-2, what="gating")


@pytest.mark.parametrize("L,E,K,Din,Dout,bias,contiguous", [
    (8192, 8, 2, 512, 384, True, False),       # LDS-ring kernel
    (8192, 8, 2, 512, 384, False, True),       # the same with [E, K, N]-contiguous weights read in place
    (4096, 16, 4, 256, 200, True, False),      # ring, N tail: 200 columns of a 256-column tile
    (600, 4, 2, 128, 136, True, False),        # register-staged kernel, tall tile
    (64, 16, 2, 128, 64, False, False),        # register-staged kernel, 64-row tile
    (100, 8, 2, 24, 40, True, True),           # element loads and element stores
    (300, 4, 2, 64, 36, True, False),          # gate rows that start off 8-byte boundaries (N = 36)
])
def test_two_input_gating_multiplies_in_the_second_gemm(L, E, K, Din, Dout, bias, contiguous):
    """index_select_jagged_gating_bmm with two different inputs: the second GEMM's epilogue multiplies
    by the SiLU of the first one's result (no element-wise pass, no second [rows, N] round trip).
    Against the oracle, and against the three-launch composition (which differs by the SiLU's last
    fp32 bits before its bf16 rounding: the element-wise kernel divides, the epilogue uses the
    hardware reciprocal)."""
    from fast_moe_amd.kernels import moe
    from fast_moe_amd.kernels.hip import ops
    r = make_routing(L, E, K, seed=L + 3)
    x, x2 = randn((L, Din), 1), randn((L, Din), 4)
    w, wp = (weights(E, Din, Dout, s, contiguous, scale=Din ** -0.5) for s in (2, 5))
    b = randn((E, Dout), 3) if bias else None
    bp = randn((E, Dout), 6) if bias else None
    f = lambda t: None if t is None else t.float()
    ref = o_moe.index_select_jagged_gating_bmm(r["offsets"], r["index"], f(x), f(x2), f(w), f(wp), f(b), f(bp))
    off, idx = dev(r["offsets"]), dev(r["index"])
    calls = []
    real = ops.silu_mul
    ops.silu_mul = lambda *a, **k: calls.append(1) or real(*a, **k)
    try:
        with torch.no_grad():
            out = moe.index_select_jagged_gating_bmm(0, off, idx, dev(x), dev(x2), dev(w), dev(b), dev(wp), dev(bp))
    finally:
        ops.silu_mul = real
    assert not calls, "the element-wise pass ran"
    assert_bf16_close(out, ref, rtol=1.6e-2, atol=2e-2, what="gating, two inputs")
    kw = dict(total_rows=L * K, row_index=idx, index_div=K)
    alpha = ops.grouped_gemm(off, dev(x), dev(w), bias=dev(b), **kw)
    beta = ops.grouped_gemm(off, dev(x2), dev(wp), bias=dev(bp), **kw)
    three = ops.silu_mul(alpha, beta)
    diff = (out.view(torch.int16).int() - three.view(torch.int16).int()).abs()
    # (one bf16 step of the rounded SiLU is up to two steps of the rounded product)
    assert int(diff.max()) <= 2 and float((diff != 0).float().mean()) < 2e-3, (int(diff.max()), float((diff != 0).float().mean()))
    # a gate tensor that is a column slice of a wider one (row stride > N)
    wide = torch.zeros((L * K, Dout + 12), dtype=BF16, device="cuda")
    wide[:, 4:4 + Dout] = alpha
    sliced = ops.grouped_gemm(off, dev(x2), dev(wp), bias=dev(bp), epilogue=3, gate=wide[:, 4:4 + Dout], **kw)
    assert torch.equal(sliced, out)


def test_3d_variant():
    from fast_moe_amd.kernels import moe
    L, E, K, Din, Dout = 200, 4, 2, 8, 4
    r = make_routing(L, E, K, seed=9)
    x = uniform((L, E, Din), 1)
    w = weights(E, Din, Dout, 2)
    b = uniform((E, Dout), 3)
    ref = o_moe.index_select_jagged_bmm_3D(r["offsets"], r["index"], x.float(), w.float(), b.float())
    with torch.no_grad():
        out = moe.index_select_jagged_bmm_3D(0, dev(r["offsets"]), dev(r["index"]), dev(x), dev(w), dev(b))
    torch.testing.assert_close(out.cpu(), ref.to(BF16), rtol=REF_RTOL, atol=REF_ATOL)
    L, Din, Dout = 600, 64, 64
    r = make_routing(L, E, K, seed=10)
    x = uniform((L, E, Din), 1)
    w = weights(E, Din, Dout, 2, contiguous=False)
    ref = o_moe.index_select_jagged_bmm_3D(r["offsets"], r["index"], x.float(), w.float(), None)
    with torch.no_grad():
        out = moe.index_select_jagged_bmm_3D(0, dev(r["offsets"]), dev(r["index"]), dev(x), dev(w), None)
    torch.testing.assert_close(out.cpu(), ref.to(BF16), rtol=REF_RTOL, atol=1e-4)


@pytest.mark.parametrize("E,K,Din,Dout,has_silu,has_bias,max_len", [
    (4, 1, 128, 128, True, True, 64), (8, 2, 256, 128, False, True, 200), (8, 2, 128, 256, True, False, 200),
    (4, 2, 256, 256, False, False, 32), (8, 2, 1024, 512, True, True, 700)])
def test_silu_jagged_bmm_combine(E, K, Din, Dout, has_silu, has_bias, max_len):
    """Generator of kernels/tests/moe_test.py:1017-1032; tolerance far inside its atol 5e-1 / rtol 1.5e-1."""
    from fast_moe_amd.kernels import moe
    g = torch.Generator().manual_seed(E + K + Din)
    seq_len = torch.randint(32, max_len + 1, (E,), generator=g)
    N = int(seq_len.sum())
    logits = (torch.rand(N, E, generator=g) + 1e-2).to(BF16)
    topk_gates, topk_idx = logits.topk(K, dim=1)
    meta = o_routing.routing_metadata(topk_idx.numpy(), E)
    t = lambda k: torch.from_numpy(meta[k])
    jagged = uniform((N * K, Din), 1)
    w = weights(E, Din, Dout, 2)
    b = uniform((E, Dout), 3) if has_bias else None
    ref = o_moe.silu_jagged_bmm_combine(t("offsets"), jagged, w, b, t("token_index"), K, topk_gates,
                                        t("gate_index"), has_silu)
    ref32 = o_moe.silu_jagged_bmm_combine(
        t("offsets"), (torch.nn.functional.silu(jagged) if has_silu else jagged).float(), w.float(),
        None if b is None else b.float(), t("token_index"), K, topk_gates.float(), t("gate_index"), False)
    with torch.no_grad():
        out = moe.silu_jagged_bmm_combine(0, dev(t("offsets")), dev(jagged), dev(w), dev(b), dev(t("token_index")),
                                          dev(t("reverse_index")), dev(topk_gates), dev(t("gate_index")),
                                          has_silu=has_silu)
    assert out.dtype == BF16 and tuple(out.shape) == (N, Dout)
    assert_bf16_close(out, ref32, rtol=2e-2, atol=5e-2 * (Din / 128) ** 0.5, what="combine vs fp32")
    torch.testing.assert_close(out.cpu().float(), ref.float(), atol=5e-1, rtol=1.5e-1)


@pytest.mark.parametrize("N,K,D,dtype,wdtype", [
    (2, 4, 128, torch.float32, torch.float32), (33, 16, 256, BF16, BF16), (100, 32, 128, BF16, BF16),
    (1000, 4, 256, torch.float32, torch.float32), (512, 8, 2048, BF16, BF16), (64, 3, 100, BF16, BF16),
    (40, 5, 37, torch.float32, torch.float32), (128, 8, 512, BF16, torch.float32)])
def test_mul_merge_k_add_bit_exact(N, K, D, dtype, wdtype):
    """Generator of kernels/tests/moe_test.py:344-367: non-contiguous weight, permuted weight_index,
    arbitrary row -> output map.  The fp32 adds follow the CPU index_add order, so the result is
    bit-identical to the oracle."""
    from fast_moe_amd.kernels import moe
    g = torch.Generator().manual_seed(N + K)
    x = uniform((N * K, D), 1, dtype)
    w = uniform((N, 2 * K), 2, wdtype)[:, :K]
    w_index = torch.randperm(N * K, generator=g)
    perm = torch.randperm(N * K, generator=g)
    o2i = torch.arange(N).repeat(K)[perm]
    i2o = o2i.sort(stable=True)[1].view(-1, K)
    ref = o_moe.mul_merge_k_add(o2i, x, K, w, w_index)
    with torch.no_grad():
        out = moe.mul_merge_k_add(dev(o2i), dev(i2o), dev(x), weight=dev(w), weight_index=dev(w_index))
        out_nw = moe.mul_merge_k_add(dev(o2i), dev(i2o), dev(x))
    assert out.dtype == ref.dtype
    assert torch.equal(out.cpu(), ref), f"max diff {(out.cpu().float() - ref.float()).abs().max()}"
    assert torch.equal(out_nw.cpu(), o_moe.mul_merge_k_add(o2i, x, K))


# ------------------------------------------------------------------------ fp8
@pytest.mark.parametrize("L,E,K,Din,Dout,bias,contiguous", [
    (16, 4, 2, 32, 16, True, True), (100, 8, 4, 64, 32, False, True), (500, 16, 2, 64, 16, True, False),
    (2048, 8, 2, 256, 512, True, False), (300, 4, 2, 48, 24, True, True), (4096, 64, 8, 256, 128, False, False)])
def test_fp8_gather_gemm(L, E, K, Din, Dout, bias, contiguous):
    """kernels/tests/moe_fp8_test.py:337-370: fp8 kernel vs the PyTorch fp8 emulation, 1e-2 / 1e-2."""
    from fast_moe_amd.kernels import moe_fp8
    r = make_routing(L, E, K, seed=L + 2)
    x = uniform((L, Din), 1)
    w = weights(E, Din, Dout, 2, contiguous)
    b = uniform((E, Dout), 3) if bias else None
    ref = o_fp8.index_select_jagged_bmm_fp8(r["offsets"], r["index"], x, w, b)
    with torch.no_grad():
        out = moe_fp8.index_select_jagged_bmm(0, dev(r["offsets"]), dev(r["index"]), dev(x), dev(w), dev(b),
                                              fp8=True)
        raw = moe_fp8.index_select_jagged_bmm(0, dev(r["offsets"]), dev(r["index"]), dev(x), dev(w), dev(b),
                                              fp8=False)
    if Din <= 64:       # the reference's shapes and its tolerance
        torch.testing.assert_close(out.cpu().float(), ref.float(), atol=1e-2, rtol=1e-2)
    else:               # longer sums: one-ulp bf16 flips next to bias cancellation; 3e-2 relative
        assert_bf16_close(out, ref, rtol=3e-2, atol=3e-2, what="fp8 vs fp8 oracle")
    # vs the unquantised op: tolerance of moe_fp8_test.py:302-335, quantisation noise grows with Din
    torch.testing.assert_close(out.cpu().float(), raw.cpu().float(), atol=4e-1 * max(1.0, Din / 64),
                               rtol=1e-1)


def test_fp8_outlier_rows_and_zero_rows():
    from fast_moe_amd.kernels import moe_fp8
    L, E, K, Din, Dout = 512, 8, 2, 128, 64
    r = make_routing(L, E, K, seed=4)
    x = randn((L, Din), 1)
    x[::50] *= 100
    x[7] = 0
    w = weights(E, Din, Dout, 2, False, scale=Din ** -0.5)
    w[3, :, 5] = 0
    ref = o_fp8.index_select_jagged_bmm_fp8(r["offsets"], r["index"], x, w, None)
    with torch.no_grad():
        out = moe_fp8.index_select_jagged_bmm(0, dev(r["offsets"]), dev(r["index"]), dev(x), dev(w), None, fp8=True)
    assert bool(torch.isfinite(out).all())
    err = (out.cpu().float() - ref.float()).abs()
    assert bool((err <= 3e-2 * ref.float().abs() + 3e-2).all())


@pytest.mark.parametrize("E,K,Din,Dout,has_silu", [(4, 2, 128, 128, True), (8, 2, 256, 64, False)])
def test_fp8_combine(E, K, Din, Dout, has_silu):
    from fast_moe_amd.kernels import moe_fp8
    g = torch.Generator().manual_seed(E)
    N = 300
    logits = (torch.rand(N, E, generator=g) + 1e-2).to(BF16)
    gates, topk_idx = logits.topk(K, dim=1)
    meta = o_routing.routing_metadata(topk_idx.numpy(), E)
    t = lambda k: torch.from_numpy(meta[k])
    jagged = uniform((N * K, Din), 1)
    w = weights(E, Din, Dout, 2)
    b = uniform((E, Dout), 3)
    # oracle: the same fp8 emulation for the GEMM, then the merge
    h = torch.nn.functional.silu(jagged) if has_silu else jagged
    qa, sa = o_fp8.rowwise_quant_fp8(h)
    qw, sw = o_fp8.rowwise_quant_fp8(w.permute(0, 2, 1))
    sizes = (t("offsets")[1:] - t("offsets")[:-1]).tolist()
    rows = o_fp8.fp8_linear_per_expert(list(o_fp8.dequant(qa).split(sizes)), list(sa.split(sizes)),
                                       o_fp8.dequant(qw), sw, b, BF16)
    ref = o_moe.mul_merge_k_add(t("token_index"), torch.cat(rows), K, gates, t("gate_index"))
    with torch.no_grad():
        out = moe_fp8.silu_jagged_bmm_combine_fp8(0, dev(t("offsets")), dev(jagged), dev(w), dev(b),
                                                  dev(t("token_index")), dev(t("reverse_index")), dev(gates),
                                                  dev(t("gate_index")), has_silu=has_silu)
    err = (out.cpu().float() - ref.float()).abs()
    assert bool((err <= 3e-2 * ref.float().abs() + 3e-2).all()), err.max()


def test_fp8_weight_pair_of_other_origin_is_not_taken_for_powers_of_two():
    """A caller may hand the fp8 operators its own (bytes, scales) pair.  Only scale tensors that
    the package's quantiser returned (and nobody wrote to since) are taken for exact powers of
    two and given to the MFMAs as block scales; any other pair has its scales divided out in the
    epilogue, which is right for every positive scale."""
    from fast_moe_amd.kernels import moe_fp8
    from fast_moe_amd.kernels.hip import ops
    L, E, K, Din, Dout = 4096, 8, 2, 256, 512
    r = make_routing(L, E, K, seed=3)
    x = dev(randn((L, Din), 1))
    w = dev(weights(E, Din, Dout, 2, False, scale=Din ** -0.5))
    offsets, index = dev(r["offsets"]), dev(r["index"])
    qw, sw = moe_fp8.quantize_expert_weights(w)
    assert ops.scales_are_pow2(sw)
    other = sw * 1.5                         # a legitimate pair of other origin: same bytes, weights 1.5 times smaller
    assert not ops.scales_are_pow2(other) and not ops.scales_are_pow2(sw.clone())
    qa, sa = ops.quant_rows_fp8(x)
    kw = dict(total_rows=L * K, row_index=index.reshape(-1), index_div=K, a_scale=sa)
    want = ops.grouped_gemm(offsets, qa, qw, b_scale=other, scales_pow2=False, **kw)
    got = moe_fp8.index_select_jagged_bmm(0, offsets, index, x, w, None, fp8=True, fp8_weight=(qw, other))
    assert torch.equal(got, want)
    base = moe_fp8.index_select_jagged_bmm(0, offsets, index, x, w, None, fp8=True, fp8_weight=(qw, sw))
    assert_bf16_close(got.float() * 1.5, base.float(), rtol=1.6e-2, atol=1e-2, what="scales 1.5 times larger")
    sw.mul_(1.0)                              # written to: no longer vouched for
    assert not ops.scales_are_pow2(sw)


def test_forward_only_and_dtype_errors():
    from fast_moe_amd.kernels import moe, moe_fp8
    r = make_routing(16, 4, 2)
    x = uniform((16, 32), 1).cuda().requires_grad_()
    w = weights(4, 32, 32, 2).cuda()
    x2 = uniform((32, 32), 1).cuda().requires_grad_()
    with pytest.raises(RuntimeError, match="forward-only"):       # no backward for this one, as in the reference
        moe_fp8.silu_jagged_bmm_fp8(dev(r["offsets"]), 0, x2, w, uniform((4, 32), 3).cuda())
    with pytest.raises(NotImplementedError):
        with torch.no_grad():
            moe.index_select_jagged_bmm(0, dev(r["offsets"]), dev(r["index"]), x.half(), w.half(), None)


# ------------------------------------------------------------- ring-kernel specifics
@pytest.mark.parametrize("L,E,K,Din,Dout,epi", [
    (4096, 8, 2, 96, 256, "plain"),        # three K-slices only: the ring never fills
    (4096, 8, 2, 1024, 264, "plain"),      # N = 264: last column tile 8 wide
    (9000, 3, 1, 512, 512, "plain"),       # fewer tiles than CUs, K_top = 1 (index_shift 0)
    (6144, 24, 3, 256, 384, "swiglu"),     # top-3: index division, not a shift
    (20000, 200, 2, 128, 128, "swiglu"),   # many experts, about 200 rows each (register tables, 4 entries)
    (30000, 300, 2, 128, 128, "swiglu"),   # more than 256 experts: 4-slot ring with its tables in LDS
    (3000, 2, 2, 2048, 128, "swiglu"),     # long K, one column tile
])
def test_ring_kernel_shapes(L, E, K, Din, Dout, epi):
    from fast_moe_amd.kernels import moe
    r = make_routing(L, E, K, seed=L + E)
    x = randn((L, Din), 1)
    w = weights(E, Din, Dout, 2, False, scale=Din ** -0.5)
    b = randn((E, Dout), 3)
    if epi == "plain":
        ref = o_moe.index_select_jagged_bmm(r["offsets"], r["index"], x.float(), w.float(), b.float())
        with torch.no_grad():
            out = moe.index_select_jagged_bmm(0, dev(r["offsets"]), dev(r["index"]), dev(x), dev(w), dev(b))
        assert_bf16_close(out, ref, rtol=1e-2, atol=1e-2, what=f"ring plain {L},{E},{K},{Din},{Dout}")
    else:
        wp = weights(E, Din, Dout, 5, False, scale=Din ** -0.5)
        ref = o_moe.index_select_jagged_bmm_swiglu(r["offsets"], r["index"], x.float(), w.float(), b.float(),
                                                   wp.float(), None)
        with torch.no_grad():
            out = moe.index_select_jagged_bmm_swiglu(0, dev(r["offsets"]), dev(r["index"]), dev(x), dev(w), dev(b),
                                                     dev(wp), None)
        assert_bf16_close(out, ref, rtol=1.6e-2, atol=1e-2, what=f"ring swiglu {L},{E},{K},{Din},{Dout}")


@pytest.mark.parametrize("epi,fp8", [("plain", False), ("swiglu", False), ("plain", True)])
def test_ring_kernel_tiles_with_few_valid_rows(epi, fp8):
    """Experts whose last (or only) 256-row tile ends at, just before and just after every 32-row
    block boundary: tiles that end in their first half run the ring kernel's shortened main loop,
    and the two wave rows share a tile's row blocks alternately.  Against the oracle, and the plan
    must say RING."""
    from fast_moe_amd.kernels import moe, moe_fp8
    from fast_moe_amd.kernels.hip import _lib, ops
    lens = [1, 31, 32, 33, 63, 64, 65, 96, 127, 128, 129, 160, 191, 193, 255, 256, 257, 288, 320, 383, 384, 385,
            511, 513, 640, 0, 769, 2048 + 17, 3000]
    E, Din, Dout = len(lens), 192, 320
    g = torch.Generator().manual_seed(7)
    experts = torch.repeat_interleave(torch.arange(E), torch.tensor(lens))
    topk = experts[torch.randperm(experts.numel(), generator=g)].view(-1, 1)
    L = topk.shape[0]
    meta = o_routing.routing_metadata(topk.numpy(), E)
    offsets = torch.from_numpy(meta["offsets"])
    index = torch.from_numpy(meta["gate_index"]).view(-1, 1)
    assert (offsets[1:] - offsets[:-1]).tolist() == lens
    x = randn((L, Din), 1)
    w = weights(E, Din, Dout, 2, False, scale=Din ** -0.5)
    b = randn((E, Dout), 3)
    # (the plan of the bf16 descriptor of this shape; the e4m3 one differs in the operand type only)
    assert ops.grouped_gemm(dev(offsets), dev(x), dev(w), total_rows=L, row_index=dev(index).view(-1), index_div=1,
                            plan_only=True) == _lib.PLAN_RING
    with torch.no_grad():
        if fp8:
            ref = o_fp8.index_select_jagged_bmm_fp8(offsets, index, x, w, b)
            out = moe_fp8.index_select_jagged_bmm(0, dev(offsets), dev(index), dev(x), dev(w), dev(b), fp8=True)
        elif epi == "plain":
            ref = o_moe.index_select_jagged_bmm(offsets, index, x.float(), w.float(), b.float())
            out = moe.index_select_jagged_bmm(0, dev(offsets), dev(index), dev(x), dev(w), dev(b))
        else:
            wp = weights(E, Din, Dout, 5, False, scale=Din ** -0.5)
            ref = o_moe.index_select_jagged_bmm_swiglu(offsets, index, x.float(), w.float(), b.float(),
                                                       wp.float(), None)
            out = moe.index_select_jagged_bmm_swiglu(0, dev(offsets), dev(index), dev(x), dev(w), dev(b),
                                                     dev(wp), None)
    # every expert on its own, so that a failure names the row count it happens at
    for e, n in enumerate(lens):
        lo = int(offsets[e])
        if n:
            assert_bf16_close(out[lo:lo + n], ref[lo:lo + n], rtol=3e-2 if fp8 else 1.6e-2, atol=3e-2 if fp8 else 1e-2,
                              what=f"expert {e} with {n} rows ({epi}, fp8={fp8})")


def test_ring_kernel_is_deterministic_and_ignores_garbage_offsets():
    """Two launches give identical bits; offsets outside [0, R] are clamped instead of followed."""
    from fast_moe_amd.kernels.hip import ops
    L, E, K, D, N = 8192, 16, 2, 256, 256
    r = make_routing(L, E, K, seed=5)
    x, w = dev(randn((L, D), 1)), dev(weights(E, D, N, 2, False, scale=D ** -0.5))
    a = ops.grouped_gemm(dev(r["offsets"]), x, w, total_rows=L * K, row_index=dev(r["gate_index"]), index_div=K)
    b = ops.grouped_gemm(dev(r["offsets"]), x, w, total_rows=L * K, row_index=dev(r["gate_index"]), index_div=K)
    assert torch.equal(a, b)
    bad = r["offsets"].clone()
    bad[-1] = 10 ** 12
    bad[3] = -7
    out = ops.grouped_gemm(dev(bad), x, w, total_rows=L * K, row_index=dev(r["gate_index"]), index_div=K)
    torch.cuda.synchronize()
    assert out.shape == a.shape


@pytest.mark.parametrize("fp8", [False, True], ids=["bf16", "fp8"])
def test_ring_kernel_repeats_bit_identically_while_another_stream_loads_the_memory_system(fp8):
    """The ring kernel keeps its own count of the LDS-DMA in flight; a wait that is one operation
    short would read a slot before its data has landed, and whether that shows depends on timing.
    Both GEMMs of the benchmark sizes (SwiGLU with gather, plain), 24 launches each, while a second
    stream copies 1 GiB back and forth: every launch must reproduce the first bit for bit."""
    from fast_moe_amd.kernels.hip import _lib, ops
    T, E, K, D, H = 16384, 64, 8, 2048, 1408
    topk = skewed_topk(T, E, K, seed=11)
    meta = o_routing.routing_metadata(topk.numpy(), E)
    offsets, gate_index = dev(torch.from_numpy(meta["offsets"])), dev(torch.from_numpy(meta["gate_index"]))
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(T, D, generator=g, device="cuda").to(BF16)
    wg = (torch.randn(E, H, D, generator=g, device="cuda") * D ** -0.5).to(BF16).permute(0, 2, 1)
    wu = (torch.randn(E, H, D, generator=g, device="cuda") * D ** -0.5).to(BF16).permute(0, 2, 1)
    wd = (torch.randn(E, D, H, generator=g, device="cuda") * H ** -0.5).to(BF16).permute(0, 2, 1)
    if fp8:
        (qx, sx), (qg, sg), (qu, su), (qd, sd) = (ops.quant_rows_fp8(x), ops.quant_rows_fp8(wg.permute(0, 2, 1)),
                                                    ops.quant_rows_fp8(wu.permute(0, 2, 1)),
                                                    ops.quant_rows_fp8(wd.permute(0, 2, 1)))
        gemm1 = lambda: ops.grouped_gemm(offsets, qx, qg.permute(0, 2, 1), total_rows=T * K, row_index=gate_index,
                                         index_div=K, b2=qu.permute(0, 2, 1), epilogue=_lib.EPI_SWIGLU, a_scale=sx,
                                         b_scale=sg, b2_scale=su, scales_pow2=True)
    else:
        gemm1 = lambda: ops.grouped_gemm(offsets, x, wg, total_rows=T * K, row_index=gate_index, index_div=K, b2=wu,
                                         epilogue=_lib.EPI_SWIGLU)
    hidden = gemm1()
    if fp8:
        qh, sh = ops.quant_rows_fp8(hidden)
        gemm2 = lambda: ops.grouped_gemm(offsets, qh, qd.permute(0, 2, 1), total_rows=T * K, a_scale=sh, b_scale=sd,
                                         scales_pow2=True)
    else:
        gemm2 = lambda: ops.grouped_gemm(offsets, hidden, wd, total_rows=T * K)
    first2 = gemm2()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    a, b = torch.empty(1 << 28, dtype=torch.int32, device="cuda"), torch.empty(1 << 28, dtype=torch.int32, device="cuda")
    for i in range(24):
        with torch.cuda.stream(side):               # (default priority) a copy that competes for HBM and L2
            (b if i % 2 else a).copy_(a if i % 2 else b, non_blocking=True)
        h, o = gemm1(), gemm2()
        assert torch.equal(h, hidden), f"gemm1, launch {i}"
        assert torch.equal(o, first2), f"gemm2, launch {i}"
    torch.cuda.synchronize()


@pytest.mark.parametrize("fp8", [False, True])
def test_full_size_c3_c4_sampled_rows(fp8):
    """The benchmark sizes (T=16384, E=64, top-8, D=2048, H=1408, Zipf-skewed, empty experts): the
    whole SwiGLU GEMM runs on the GPU, a sample of its rows is checked against the oracle, and
    size-independent properties hold (rows of empty experts absent, duplicate tokens give equal rows)."""
    from fast_moe_amd.kernels import moe_fp8
    from fast_moe_amd.kernels.hip import ops
    T, E, K, D, H = 16384, 64, 8, 2048, 1408
    topk = skewed_topk(T, E, K, seed=11)
    meta = o_routing.routing_metadata(topk.numpy(), E)
    assert (meta["lengths"] == 0).sum() >= 2
    offsets = torch.from_numpy(meta["offsets"])
    gate_index = torch.from_numpy(meta["gate_index"])
    g = torch.Generator().manual_seed(0)
    x = torch.randn(T, D, generator=g).to(BF16)
    x[5] = x[4]                                            # two identical tokens
    if fp8:
        x[::100] *= 100
    wg = (torch.randn(E, H, D, generator=g) * D ** -0.5).to(BF16).permute(0, 2, 1)
    wu = (torch.randn(E, H, D, generator=g) * D ** -0.5).to(BF16).permute(0, 2, 1)
    with torch.no_grad():
        if fp8:
            qg, sg = moe_fp8.quantize_expert_weights(dev(wg))
            qu, su = moe_fp8.quantize_expert_weights(dev(wu))
            qx, sx = ops.quant_rows_fp8(dev(x))
            out = ops.grouped_gemm(dev(offsets), qx, qg, total_rows=T * K, row_index=dev(gate_index), index_div=K,
                                   b2=qu, epilogue=2, a_scale=sx, b_scale=sg, b2_scale=su)
        else:
            out = ops.grouped_gemm(dev(offsets), dev(x), dev(wg), total_rows=T * K, row_index=dev(gate_index),
                                   index_div=K, b2=dev(wu), epilogue=2)
    out = out.cpu()
    assert bool(torch.isfinite(out).all())
    rows = torch.randperm(T * K, generator=g)[:192]
    experts = torch.searchsorted(offsets[1:], rows, right=True)
    tok = gate_index[rows] // K
    for i in range(rows.numel()):
        e, t = int(experts[i]), int(tok[i])
        if fp8:
            one = torch.tensor([0, 1])
            eo = torch.zeros(2, dtype=torch.int64)
            eo[1] = 1
            # the oracle's fp8 path on a single row / single expert
            from oracle import moe_fp8 as o8
            qa, sa = o8.rowwise_quant_fp8(x[t:t + 1])
            qwg, swg = o8.rowwise_quant_fp8(wg[e:e + 1].permute(0, 2, 1))
            qwu, swu = o8.rowwise_quant_fp8(wu[e:e + 1].permute(0, 2, 1))
            gg = o8.fp8_linear_per_expert([o8.dequant(qa)], [sa], o8.dequant(qwg), swg, None, BF16)[0]
            uu = o8.fp8_linear_per_expert([o8.dequant(qa)], [sa], o8.dequant(qwu), swu, None, BF16)[0]
            ref = (torch.nn.functional.silu(gg) * uu)[0]
            tol = 3e-2
        else:
            xr = x[t].float()
            ref = torch.nn.functional.silu(xr @ wg[e].float()) * (xr @ wu[e].float())
            tol = 1.6e-2
        err = (out[rows[i]].float() - ref.float()).abs()
        scale = ref.float().abs().max().item()
        assert bool((err <= tol * ref.float().abs() + tol * scale * 0.5 + 1e-3).all()), (int(rows[i]), err.max())
    # identical tokens routed to the same expert give identical rows
    pos = {}
    for tkn in (4, 5):
        for j in range(K):
            pos[(tkn, int(topk[tkn, j]))] = int(torch.from_numpy(meta["reverse_index"])[tkn][
                sorted(range(K), key=lambda q: int(topk[tkn, q])).index(j)])
    common = set(int(e) for e in topk[4]) & set(int(e) for e in topk[5])
    for e in common:
        assert torch.equal(out[pos[(4, e)]], out[pos[(5, e)]])


def test_n_contiguous_weights_and_the_transposing_copy():
    """[E, K, N]-contiguous weights (the layout of kernels/tests/moe_test.py:205-209) of a useful
    size are transposed once on the device and then streamed; the result equals the in-place
    element-load kernel's and the oracle's."""
    from fast_moe_amd.kernels import moe
    from fast_moe_amd.kernels.hip import ops
    L, E, K, Din, Dout = 8192, 8, 2, 512, 384
    r = make_routing(L, E, K, seed=21)
    x = randn((L, Din), 1)
    w = weights(E, Din, Dout, 2, True, scale=Din ** -0.5)
    assert w.is_contiguous()
    wt = ops.to_k_contiguous(dev(w))
    assert wt.stride(1) == 1 and torch.equal(wt.cpu(), w)
    odd = weights(3, 70, 130, 4, True)           # extents that are not multiples of the 64 x 64 tile
    assert torch.equal(ops.to_k_contiguous(dev(odd)).cpu(), odd)
    q = (torch.arange(5 * 33 * 65) % 251).to(torch.uint8).view(5, 33, 65).view(torch.float8_e4m3fn)
    assert torch.equal(ops.to_k_contiguous(dev(q)).cpu().view(torch.uint8), q.view(torch.uint8))
    ref = o_moe.index_select_jagged_bmm(r["offsets"], r["index"], x.float(), w.float(), None)
    with torch.no_grad():
        out = moe.index_select_jagged_bmm(0, dev(r["offsets"]), dev(r["index"]), dev(x), dev(w), None)
        out_k = moe.index_select_jagged_bmm(0, dev(r["offsets"]), dev(r["index"]), dev(x), wt, None)
    assert torch.equal(out, out_k)
    assert_bf16_close(out, ref, rtol=1e-2, atol=1e-2, what="N-contiguous weights")


# ------------------------------------------------------------------------ fp32
@pytest.mark.parametrize("L,E,K,Din,Dout", GRID[1::4])
@pytest.mark.parametrize("contiguous", [True, False])
@pytest.mark.parametrize("has_bias", [True, False])
def test_index_select_jagged_bmm_fp32_reference_grid(L, E, K, Din, Dout, contiguous, has_bias):
    """fp32 half of kernels/tests/moe_test.py:35-84 (allow_tf32 off): default fp32 assert_close."""
    from fast_moe_amd.kernels import moe
    r = make_routing(L, E, K, seed=L + E + 1)
    x = uniform((L, Din), 1, torch.float32)
    w = uniform((E, Din, Dout), 2, torch.float32)
    if not contiguous:
        w = w.transpose(1, 2).contiguous().transpose(1, 2)
    b = uniform((E, Dout), 3, torch.float32) if has_bias else None
    ref = o_moe.index_select_jagged_bmm(r["offsets"], r["index"], x, w, b)
    with torch.no_grad():
        out = moe.index_select_jagged_bmm(0, dev(r["offsets"]), dev(r["index"]), dev(x), dev(w), dev(b))
    assert out.dtype == torch.float32
    torch.testing.assert_close(out.cpu(), ref)


def test_fp32_swiglu_gating_3d_and_combine():
    from fast_moe_amd.kernels import moe
    L, E, K, Din, Dout = 700, 8, 2, 64, 96
    f32 = torch.float32
    r = make_routing(L, E, K, seed=31)
    x, x2 = uniform((L, Din), 1, f32), uniform((L, Din), 4, f32)
    w, wp = uniform((E, Din, Dout), 2, f32), uniform((E, Din, Dout), 5, f32)
    b, bp = uniform((E, Dout), 3, f32), uniform((E, Dout), 6, f32)
    a = [dev(r["offsets"]), dev(r["index"])]
    with torch.no_grad():
        sw = moe.index_select_jagged_bmm_swiglu(0, *a, dev(x), dev(w), dev(b), dev(wp), dev(bp))
        gt = moe.index_select_jagged_gating_bmm(0, *a, dev(x), dev(x2), dev(w), dev(b), dev(wp), dev(bp))
    torch.testing.assert_close(sw.cpu(), o_moe.index_select_jagged_bmm_swiglu(r["offsets"], r["index"], x, w, b, wp, bp),
                               rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(gt.cpu(), o_moe.index_select_jagged_gating_bmm(r["offsets"], r["index"], x, x2, w, wp, b, bp),
                               rtol=1e-5, atol=1e-5)
    x3 = uniform((L, E, Din), 7, f32)
    with torch.no_grad():
        o3 = moe.index_select_jagged_bmm_3D(0, *a, dev(x3), dev(w), dev(b))
    torch.testing.assert_close(o3.cpu(), o_moe.index_select_jagged_bmm_3D(r["offsets"], r["index"], x3, w, b))
    # SiLU-on-load GEMM + merge
    g = torch.Generator().manual_seed(3)
    gates = torch.rand(L, K, generator=g)
    jag = uniform((L * K, Din), 8, f32)
    ref = o_moe.silu_jagged_bmm_combine(r["offsets"], jag, w, b, r["token_index"], K, gates, r["gate_index"], True)
    with torch.no_grad():
        out = moe.silu_jagged_bmm_combine(0, dev(r["offsets"]), dev(jag), dev(w), dev(b), dev(r["token_index"]),
                                          dev(r["reverse_index"]), dev(gates), dev(r["gate_index"]), has_silu=True)
    torch.testing.assert_close(out.cpu(), ref, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("L,E,K,Din,Dout,dtype,bias", [
    (4096, 8, 2, 256, 384, "bf16", True),     # ring kernel
    (4096, 8, 2, 256, 384, "bf16", False),
    (300, 4, 2, 72, 40, "bf16", True),        # element kernel, scalar stores
    (1000, 4, 2, 64, 128, "f32", True),
    (4096, 8, 2, 256, 384, "fp8", True),
])
def test_swiglu_pre_activation_outputs(L, E, K, Din, Dout, dtype, bias):
    """aux / aux2 of the SWIGLU epilogue are bit for bit the outputs of the two plain GEMMs, and the
    main output does not change when they are requested."""
    from fast_moe_amd.kernels.hip import ops
    from fast_moe_amd.kernels.hip._lib import EPI_SWIGLU
    r = make_routing(L, E, K, seed=L)
    td = torch.float32 if dtype == "f32" else BF16
    x = randn((L, Din), 1).to(td).cuda()
    w = weights(E, Din, Dout, 2, False, Din ** -0.5).to(td).cuda()
    wp = weights(E, Din, Dout, 3, False, Din ** -0.5).to(td).cuda()
    b = randn((E, Dout), 4).to(td).cuda() if bias else None
    bp = randn((E, Dout), 5).to(td).cuda() if bias else None
    kw = dict(total_rows=L * K, row_index=dev(r["index"]), index_div=K)
    sc = [{}, {}, {}]
    if dtype == "fp8":
        xq, xs = ops.quant_rows_fp8(x)
        wq, ws = ops.quant_rows_fp8(w.permute(0, 2, 1))
        wpq, wps = ops.quant_rows_fp8(wp.permute(0, 2, 1))
        x, w, wp = xq, wq.permute(0, 2, 1), wpq.permute(0, 2, 1)
        sc = [dict(a_scale=xs, b_scale=ws), dict(a_scale=xs, b_scale=wps), dict(a_scale=xs, b_scale=ws, b2_scale=wps)]
    off = dev(r["offsets"])
    g = ops.grouped_gemm(off, x, w, bias=b, **kw, **sc[0])
    u = ops.grouped_gemm(off, x, wp, bias=bp, **kw, **sc[1])
    plain = ops.grouped_gemm(off, x, w, bias=b, b2=wp, bias2=bp, epilogue=EPI_SWIGLU, **kw, **sc[2])
    aux = (torch.full_like(g, 7.0), torch.full_like(g, 7.0))
    out = ops.grouped_gemm(off, x, w, bias=b, b2=wp, bias2=bp, epilogue=EPI_SWIGLU, aux=aux, **kw, **sc[2])
    assert torch.equal(out, plain)
    assert torch.equal(aux[0], g) and torch.equal(aux[1], u)
    with pytest.raises(ValueError, match="SWIGLU"):
        ops.grouped_gemm(off, x, w, bias=b, aux=aux, **kw, **sc[0])


@pytest.mark.parametrize("L,E,K,Din,Dout,epi", [
    (8192, 8, 2, 512, 384, "none"),
    (8192, 8, 2, 512, 384, "swiglu"),
    (4096, 16, 4, 256, 200, "none"),       # N tail: 200 columns of a 256-column tile
    (4096, 16, 4, 256, 72, "swiglu"),      # N tail inside the gate / up halves
    (20000, 200, 2, 128, 128, "swiglu"),   # register tables with 4 entries
    (3000, 4, 2, 1408, 2048, "none"),      # the input-gradient shape of the layer
])
def test_ring_kernel_reads_n_contiguous_weights_in_place(L, E, K, Din, Dout, epi):
    """[E, K, N]-contiguous weights (the reference tests' default layout, and what the input-gradient
    GEMM multiplies by): the plan says RING, and the result is bit for bit the one from the same
    weights stored K-contiguous."""
    from fast_moe_amd.kernels.hip import _lib, ops
    r = make_routing(L, E, K, seed=L + 1)
    x = dev(randn((L, Din), 1))
    w, wp = (dev(weights(E, Din, Dout, s, True, scale=Din ** -0.5)) for s in (2, 3))
    b, bp = dev(randn((E, Dout), 4)), dev(randn((E, Dout), 5))
    assert w.is_contiguous()
    wk, wpk = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (w, wp))
    kw = dict(total_rows=L * K, row_index=dev(r["index"]), index_div=K, bias=b)
    if epi == "swiglu":
        kw.update(bias2=bp, epilogue=_lib.EPI_SWIGLU)
    off = dev(r["offsets"])
    seen = []
    real_plan = ops.gemm_plan
    ops.gemm_plan = lambda d: seen.append(real_plan(d)) or seen[-1]
    try:
        out = ops.grouped_gemm(off, x, w, b2=wp if epi == "swiglu" else None, **kw)
    finally:
        ops.gemm_plan = real_plan
    assert seen == [_lib.PLAN_RING]
    ref = ops.grouped_gemm(off, x, wk, b2=wpk if epi == "swiglu" else None, **kw)
    assert torch.equal(out, ref)
    # a view with a larger row pitch (columns of a wider tensor) is read in place as well
    wide = torch.zeros((E, Din, Dout + 24), dtype=BF16, device="cuda")
    wide[:, :, 8:8 + Dout] = w
    if epi == "none":
        assert torch.equal(ops.grouped_gemm(off, x, wide[:, :, 8:8 + Dout], **kw), ref)


@pytest.mark.parametrize("G", [1, 4, 16])
@pytest.mark.parametrize("M", [0, 64, 512, 1000000])
@pytest.mark.parametrize("K,fp8", [(29, False), (256, False), (256, True)])
def test_reference_grouped_gemm_grid(G, M, K, fp8):
    """The grid of kernels/tests/grouped_gemm_test.py:28-199: M rows cut at G - 1 random points
    (empty groups included), N = 256, weights [G * N, K]; bf16 against the fp32 product (atol
    1e-5, rtol 1.6e-2 there; the absolute term here is scaled to sqrt(K)-sized sums), e4m3
    against the product of the dequantised operands (2e-2 / 5e-2 and 1.6e-2).  The million-row
    case is checked on the GPU in fp32, expert by expert."""
    from fast_moe_amd.kernels.hip import ops
    N = 256
    g = torch.Generator().manual_seed(G * 1000 + M % 997 + K)
    a = torch.randn(M, K, generator=g).to(BF16).cuda()
    b = torch.randn(G * N, K, generator=g).to(BF16).cuda()
    cuts = torch.sort(torch.randint(0, max(M, 1), (G - 1,), generator=g)).values if M > 0 else torch.zeros(G - 1, dtype=torch.int64)
    offsets = torch.cat([torch.zeros(1, dtype=torch.int64), cuts.to(torch.int64), torch.tensor([M])])
    w = b.view(G, N, K).permute(0, 2, 1)                      # [G, K, N], K contiguous
    if fp8:
        qa, sa = ops.quant_rows_fp8(a) if M else (torch.empty((0, K), dtype=ops.FP8_DTYPE, device="cuda"), torch.empty(0, device="cuda"))
        qb, sb = ops.quant_rows_fp8(b)
        out = ops.grouped_gemm(offsets.cuda(), qa, qb.view(G, N, K).permute(0, 2, 1), total_rows=M,
                               a_scale=sa, b_scale=sb.view(G, N))
    else:
        out = ops.grouped_gemm(offsets.cuda(), a, w, total_rows=M)
    assert tuple(out.shape) == (M, N) and out.dtype == BF16
    if M == 0:
        return
    for e in range(G):
        lo, hi = int(offsets[e]), int(offsets[e + 1])
        if lo == hi:
            continue
        if fp8:
            ref = (qa[lo:hi].float() @ qb.view(G, N, K)[e].float().T) / (sa[lo:hi, None] * sb.view(G, N)[e][None, :])
            atol = 5e-2 if M > 16384 else 2e-2
        else:
            ref = a[lo:hi].float() @ w[e].float()
            atol = 1e-5 + 4e-3 * K ** 0.5
        torch.testing.assert_close(out[lo:hi].float(), ref.to(BF16).float(), atol=atol, rtol=1.6e-2)


@pytest.mark.parametrize("seed", range(24))
def test_seeded_random_shapes_all_operators(seed):
    """A seeded draw of sizes in the spirit of the reference's hypothesis grids
    (kernels/tests/moe_test.py:27-57, 401-423, 729-751): token counts, expert counts, top-k, widths
    (multiples of 8 and not), weight layouts and bias, for the plain, SwiGLU and merge operators,
    forward against the oracle and, on every third draw, backward as well."""
    import random
    from fast_moe_amd.kernels import moe
    rnd = random.Random(1000 + seed)
    E = rnd.choice([1, 2, 3, 8, 17, 40, 70])
    K = rnd.randint(1, min(E, 4))
    L = rnd.choice([1, 7, 64, 333, 1500, 5000])
    Din = rnd.choice([8, 24, 40, 72, 128, 200, 256, 520]) + rnd.choice([0, 0, 0, 3])
    Dout = rnd.choice([8, 16, 56, 128, 136, 256, 264]) + rnd.choice([0, 0, 0, 5])
    contiguous, has_bias = rnd.random() < 0.5, rnd.random() < 0.5
    r = make_routing(L, E, K, seed=seed)
    x = randn((L, Din), seed + 1)
    w = weights(E, Din, Dout, seed + 2, contiguous, scale=Din ** -0.5)
    wp = weights(E, Din, Dout, seed + 3, contiguous, scale=Din ** -0.5)
    b = randn((E, Dout), seed + 4) if has_bias else None
    gates = torch.rand((L, K), generator=torch.Generator().manual_seed(seed)).to(BF16)
    tag = f"seed {seed}: L={L} E={E} K={K} Din={Din} Dout={Dout} contiguous={contiguous} bias={has_bias}"
    f32 = lambda t: None if t is None else t.float()
    ref_plain = o_moe.index_select_jagged_bmm(r["offsets"], r["index"], f32(x), f32(w), f32(b))
    ref_glu = o_moe.index_select_jagged_bmm_swiglu(r["offsets"], r["index"], f32(x), f32(w), f32(b), f32(wp), f32(b))
    ref_merge = o_moe.mul_merge_k_add(r["token_index"], ref_plain.to(BF16), K, gates, r["gate_index"])
    d = lambda t: None if t is None else dev(t)
    with torch.no_grad():
        plain = moe.index_select_jagged_bmm(0, d(r["offsets"]), d(r["index"]), d(x), d(w), d(b))
        glu = moe.index_select_jagged_bmm_swiglu(0, d(r["offsets"]), d(r["index"]), d(x), d(w), d(b), d(wp), d(b))
        merged = moe.mul_merge_k_add(d(r["token_index"]), d(r["reverse_index"]), d(ref_plain.to(BF16)),
                                     weight=d(gates), weight_index=d(r["gate_index"]))
    assert_bf16_close(plain, ref_plain, rtol=1.6e-2, atol=2e-2, what="plain " + tag)
    assert_bf16_close(glu, ref_glu, rtol=1.6e-2, atol=2e-2, what="swiglu " + tag)
    assert torch.equal(merged.cpu(), ref_merge), "merge " + tag
    if seed % 3:
        return
    leaves_ref = [t.float().requires_grad_(True) for t in (x, w, wp)]
    dout = randn((L * K, Dout), seed + 5) * 0.01
    o_moe.index_select_jagged_bmm_swiglu(r["offsets"], r["index"], leaves_ref[0], leaves_ref[1], f32(b), leaves_ref[2],
                                         f32(b)).backward(dout.float())
    leaves = [dev(t).requires_grad_(True) for t in (x, w, wp)]
    moe.index_select_jagged_bmm_swiglu(0, d(r["offsets"]), d(r["index"]), leaves[0], leaves[1], d(b), leaves[2],
                                       d(b)).backward(dev(dout))
    for name, got, ref in zip(("d_x", "d_w", "d_wp"), leaves, leaves_ref):
        err = (got.grad.float().cpu() - ref.grad).abs().max().item()
        assert err <= 3e-2 * ref.grad.abs().max().item() + 1e-6, (name, tag, err, ref.grad.abs().max().item())


def test_silu_on_load_at_ring_size_takes_the_silu_pass():
    """silu_jagged_bmm_combine(has_silu=True) large enough for the LDS-ring kernel: SiLU is applied by
    an element-wise pass (the ring kernel has no SiLU on load) with the rounding of the staged
    kernel's SiLU on load, so the GEMM input is bit-identical and the result meets the same bar."""
    from fast_moe_amd.kernels import moe
    from fast_moe_amd.kernels.hip import ops
    T, E, K, H, O = 4096, 8, 2, 256, 512
    r = make_routing(T, E, K, seed=21)
    j = randn((T * K, H), 1)
    w = weights(E, H, O, 2, False, scale=H ** -0.5)
    b = randn((E, O), 3)
    gates = torch.rand((T, K), generator=torch.Generator().manual_seed(4)).to(BF16)
    ref = o_moe.silu_jagged_bmm_combine(r["offsets"], j.float(), w.float(), b.float(), r["token_index"], K,
                                        gates.float(), r["gate_index"], True)
    with torch.no_grad():
        out = moe.silu_jagged_bmm_combine(0, dev(r["offsets"]), dev(j), dev(w), dev(b), dev(r["token_index"]),
                                          dev(r["reverse_index"]), dev(gates), dev(r["gate_index"]), has_silu=True)
        # the pass is what the caller could have done by hand
        rows = ops.grouped_gemm(dev(r["offsets"]), dev(j), dev(w), total_rows=T * K, bias=dev(b), a_silu=True)
        rows2 = ops.grouped_gemm(dev(r["offsets"]), ops.silu_mul(dev(j), None), dev(w), total_rows=T * K, bias=dev(b))
        # ... and a slice small enough for the staged kernel's SiLU on load sees the same input bits
        n_small = int(r["offsets"][1])
        small = ops.grouped_gemm(dev(r["offsets"][:2]), dev(j[:n_small]), dev(w[:1]), total_rows=n_small,
                                 bias=dev(b[:1]), a_silu=True)
    assert torch.equal(rows, rows2)
    assert_bf16_close(small, rows[:n_small].float(), rtol=1e-2, atol=1e-2, what="staged SiLU on load vs pass + ring")
    scale = ref.abs().max().item()
    assert_bf16_close(out, ref, rtol=1.6e-2, atol=1e-2 * scale, what="silu combine at ring size")


@pytest.mark.parametrize("lens,Din,Dout", [([300, 0, 77, 1000], 64, 32), ([2048, 4096], 256, 512)])
def test_silu_jagged_bmm_fp8(lens, Din, Dout):
    """moe_fp8.silu_jagged_bmm_fp8 (weight [E, D_out, D_in]): SiLU + row quantisation of the rows,
    row quantisation of the weight, fp8 GEMM + bias, against the same composition of the oracle's
    pieces (kernels/pytorch/moe_fp8.py:17-33, 127-137) and, loosely, the unquantised result the
    reference's PyTorch path returns (:46-75); the second call hits the weight cache."""
    from fast_moe_amd.kernels import moe_fp8
    from oracle import fp8 as o_q
    E, R = len(lens), sum(lens)
    offsets = torch.tensor([0] + lens).cumsum(0)
    j = randn((R, Din), 1)
    w = randn((E, Dout, Din), 2, scale=Din ** -0.5)
    b = randn((E, Dout), 3)
    qa, sa = o_q.silu_rowwise_quant_fp8(j.float().numpy(), "bf16")
    qw, sw = o_q.rowwise_quant_fp8(w.float().numpy(), "bf16")
    qa_f, qw_f = torch.from_numpy(o_q.e4m3fn_decode(qa)), torch.from_numpy(o_q.e4m3fn_decode(qw))
    rows = [qa_f[offsets[e]:offsets[e + 1]] for e in range(E)]
    srow = [torch.from_numpy(sa)[offsets[e]:offsets[e + 1]] for e in range(E)]
    ref = torch.cat(o_fp8.fp8_linear_per_expert(rows, srow, qw_f, torch.from_numpy(sw), b, BF16), dim=0)
    with torch.no_grad():
        out = moe_fp8.silu_jagged_bmm_fp8(dev(offsets), 0, dev(j), dev(w), dev(b))
        again = moe_fp8.silu_jagged_bmm_fp8(dev(offsets), 0, dev(j), dev(w), dev(b))
    assert torch.equal(out, again)
    scale = ref.float().abs().max().item()
    assert_bf16_close(out, ref.float(), rtol=1e-2, atol=1e-2 * scale, what="silu_jagged_bmm_fp8")
    raw = torch.cat([torch.nn.functional.silu(j[offsets[e]:offsets[e + 1]].float()) @ w[e].float().T + b[e].float()
                     for e in range(E)])
    assert (out.float().cpu() - raw).abs().max().item() <= 0.1 * scale


@pytest.mark.parametrize("swiglu", [False, True])
@pytest.mark.parametrize("M", [96, 600, 8192])          # the few-tiles kernel, the 64-row and the tall ring
def test_fp8_weight_scales_at_any_alignment(M, swiglu):
    """The e4m3 epilogue loads a register quad's 4 weight scales at once when the scale tensors sit
    on 16-byte boundaries and one by one otherwise: both give the same bits."""
    from fast_moe_amd.kernels.hip import ops
    E, K, N = 8, 512, 512
    g = torch.Generator().manual_seed(77 + M)
    a = torch.randn(M, K, generator=g).to(BF16).cuda()
    w = [torch.randn(E * N, K, generator=g).to(BF16).cuda() for _ in range(2)]
    offsets = (torch.arange(E + 1, dtype=torch.int64) * (M // E)).cuda()
    qa, sa = ops.quant_rows_fp8(a)
    (qb, sb), (qb2, sb2) = ops.quant_rows_fp8(w[0]), ops.quant_rows_fp8(w[1])
    # make the scales differ from column to column by more than the quantiser's choice does
    sb = sb * torch.tensor([1.0, 2.0, 0.5, 4.0], device="cuda").repeat(E * N // 4)
    sb2 = sb2 * torch.tensor([0.25, 1.0, 8.0, 2.0], device="cuda").repeat(E * N // 4)

    def run(shift):
        def place(s):
            buf = torch.zeros(E * N + 4, device="cuda")
            buf[shift:shift + E * N] = s
            return buf[shift:shift + E * N].view(E, N)
        kw = dict(total_rows=M, a_scale=sa, b_scale=place(sb))
        if swiglu:
            kw.update(b2=qb2.view(E, N, K).permute(0, 2, 1), b2_scale=place(sb2), epilogue=ops.EPI_SWIGLU)
        return ops.grouped_gemm(offsets, qa, qb.view(E, N, K).permute(0, 2, 1), **kw)

    aligned = run(0)
    assert aligned.float().abs().max() > 0
    for shift in (1, 2, 3):
        assert torch.equal(run(shift), aligned)


@pytest.mark.parametrize("epi", ["none", "silu", "swiglu"])
@pytest.mark.parametrize("M", [96, 8192])
def test_bias_at_any_alignment(M, epi):
    """Bias tensors at any 2-byte alignment and with any expert pitch give the same bits."""
    from fast_moe_amd.kernels.hip import ops
    E, K, N = 8, 256, 512
    g = torch.Generator().manual_seed(5 + M)
    a = torch.randn(M, K, generator=g).to(BF16).cuda()
    w = [(torch.randn(E, K, N, generator=g) / 16).to(BF16).cuda() for _ in range(2)]
    bias = [torch.randn(E, N, generator=g).to(BF16).cuda() for _ in range(2)]
    offsets = (torch.arange(E + 1, dtype=torch.int64) * (M // E)).cuda()

    def run(shift, pitch):
        def place(b):
            buf = torch.zeros(E * pitch + 8, dtype=BF16, device="cuda")
            v = buf[shift:shift + E * pitch].view(E, pitch)[:, :N]
            v.copy_(b)
            return v
        kw = dict(total_rows=M, bias=place(bias[0]))
        if epi == "swiglu":
            kw.update(b2=w[1], bias2=place(bias[1]), epilogue=ops.EPI_SWIGLU)
        elif epi == "silu":
            kw.update(epilogue=ops.EPI_SILU)
        return ops.grouped_gemm(offsets, a, w[0], **kw)

    aligned = run(0, N)
    ref = a[:M // E].float() @ w[0][0].float() + bias[0][0].float()
    if epi == "none":
        torch.testing.assert_close(aligned[:M // E].float(), ref.to(BF16).float(), atol=3e-2, rtol=1.6e-2)
    for shift, pitch in ((1, N), (2, N), (3, N), (0, N + 2), (4, N + 4)):
        assert torch.equal(run(shift, pitch), aligned), (shift, pitch)


@pytest.mark.parametrize("rows,N,kernel", [(256, 16640, "ring_kernel<fmoe::RingCfg<256,"), (64, 17408, "ring_kernel<fmoe::RingCfg<64,"),
                                           (64, 40960, "stream_kernel<"), (64, 4096, "direct_kernel<")])
def test_accumulation_error_stays_under_the_floors_the_stage_checks_use(rows, N, kernel):
    """The absolute-error floors of tests/chain.py (BF16_FLOOR = 2^-18, FP8_FLOOR = 2^-14 of
    S = sum |a||b|) rest on a measurement: on outputs that are small by cancellation, where the final
    bf16 rounding is out of the way, the GEMMs' error against float64 is a fraction of S that
    depends on how the MFMA adds (e4m3: 64 products per instruction in a block-aligned adder that
    keeps fewer bits than an fp32 sum).  One expert, 1536-term sums, operands that are exactly
    representable in both types.
    Asserted: both stay a factor 4 under their floor, and e4m3 does accumulate less exactly than bf16."""
    from fast_moe_amd.kernels.hip import ops
    from tests.chain import BF16_FLOOR, FP8_FLOOR
    torch.manual_seed(0)
    K = 1536
    a = torch.randn(rows, K, device="cuda").to(BF16)
    w = (torch.randn(1, N, K, device="cuda") * K ** -0.5).to(BF16)
    qa, sa = ops.quant_rows_fp8(a)
    qw, sw = ops.quant_rows_fp8(w)
    off = torch.tensor([0, rows], device="cuda")
    run8 = lambda: ops.grouped_gemm(off, qa, qw.permute(0, 2, 1), total_rows=rows, a_scale=sa, b_scale=sw.reshape(1, N))
    out8 = run8()
    da, dw = qa.float(), qw.float()
    scale = sa.double()[:, None] * sw[0].double()[None, :]
    exact = (da.double() @ dw[0].double().T) / scale
    S = (da.double().abs() @ dw[0].double().abs().T) / scale
    # the same values through the bf16 kernel: exact products, fp32 accumulation
    a16, w16 = da.to(BF16), dw.to(BF16).permute(0, 2, 1)
    run16 = lambda: ops.grouped_gemm(off, a16, w16, total_rows=rows)
    out16 = run16()
    for run in (run8, run16):
        assert kernel in kernels_run(run)[0]
    exact16 = da.double() @ dw[0].double().T
    S16 = da.double().abs() @ dw[0].double().abs().T
    small8, small16 = exact.abs() < 2.0 ** -12 * S, exact16.abs() < 2.0 ** -12 * S16
    assert int(small8.sum()) > 100 and int(small16.sum()) > 100
    worst8 = ((out8.double() - exact).abs()[small8] / S[small8]).max().item()
    worst16 = ((out16.double() - exact16).abs()[small16] / S16[small16]).max().item()
    # (each such output also carries half a bf16 ulp of itself: below 2^-21 of S by the selection)
    assert worst16 <= BF16_FLOOR / 4, f"bf16 accumulation error {worst16:.3g} of S"
    assert worst8 <= FP8_FLOOR / 4, f"e4m3 accumulation error {worst8:.3g} of S"
    assert worst8 > worst16


@pytest.mark.parametrize("E,rows,K,N,epi,bias,gather", [
    (8, 4096, 2048, 1408, 2, False, True),        # SwiGLU, gathered rows, last column tile partial
    (8, 4096, 1408, 2048, 0, False, False),       # plain epilogue, rows in place
    (8, 3000, 512, 512, 1, True, True),           # SiLU with bias
    (128, 40000, 1024, 768, 2, True, True),       # the register-table variant for up to 256 experts
    (6, 700, 256, 256, 0, True, False),           # short experts: tiles that run the shortened loop
])
def test_scales_applied_by_the_mfma_equal_scales_divided_out_in_the_epilogue(E, rows, K, N, epi, bias, gather):
    """fmoe_gemm_desc.scale_pow2: with power-of-two scales the ring kernel lets the MFMA apply them
    (E8M0 block scales) instead of dividing them out in its epilogue.  A power-of-two factor on
    every product of an output element commutes with the fp32 accumulation, so the two paths must
    agree bit for bit, also with rows and columns whose scales differ by 2^20 and with the scale of
    an all-zero row (2^127)."""
    from fast_moe_amd.kernels.hip import _lib, ops
    g = torch.Generator().manual_seed(E * 7 + rows)
    T = rows // 2 if gather else rows
    x = torch.randn(T, K, generator=g)
    x[::7] *= 300.0                     # other row scales
    x[5] = 0.0                          # scale 2^127
    x[::11] *= 2.0 ** -12
    w = torch.randn(E, N, K, generator=g) * K ** -0.5
    w[:, ::5] *= 64.0                   # other column scales
    w[:, 3] = 0.0
    w2 = torch.randn(E, N, K, generator=g) * K ** -0.5
    qx, sx = ops.quant_rows_fp8(x.to(BF16).cuda())
    qw, sw = ops.quant_rows_fp8(w.to(BF16).cuda())
    qw2, sw2 = ops.quant_rows_fp8(w2.to(BF16).cuda())
    cuts = torch.sort(torch.randint(0, rows, (E - 1,), generator=g)).values
    if E == 6:
        cuts = torch.tensor([100, 228, 357, 390, 650])          # 100, 128, 129, 33, 260, 50 rows
    offsets = torch.cat([torch.zeros(1, dtype=torch.int64), cuts.to(torch.int64), torch.tensor([rows])]).cuda()
    kw = dict(total_rows=rows, a_scale=sx, b_scale=sw, epilogue=epi)
    if gather:
        kw.update(row_index=torch.randint(0, T * 2, (rows,), generator=g).cuda(), index_div=2)
    if epi == 2:
        kw.update(b2=qw2.permute(0, 2, 1), b2_scale=sw2)
    if bias:
        kw.update(bias=torch.randn(E, N, generator=g).to(BF16).cuda())
        if epi == 2:
            kw.update(bias2=torch.randn(E, N, generator=g).to(BF16).cuda())
    assert ops.grouped_gemm(offsets, qx, qw.permute(0, 2, 1), plan_only=True, scales_pow2=True, **kw) == _lib.PLAN_RING
    plain = ops.grouped_gemm(offsets, qx, qw.permute(0, 2, 1), scales_pow2=False, **kw)
    folded = ops.grouped_gemm(offsets, qx, qw.permute(0, 2, 1), scales_pow2=True, **kw)
    again = ops.grouped_gemm(offsets, qx, qw.permute(0, 2, 1), scales_pow2=True, **kw)
    assert torch.isfinite(plain.float()).all()
    assert torch.equal(folded.view(torch.int16), plain.view(torch.int16))
    assert torch.equal(again.view(torch.int16), folded.view(torch.int16))


@pytest.mark.parametrize("E,rows,K,N,epi", [
    (8, 4096, 1024, 712, 2), (8, 4096, 1024, 712, 0), (8, 4096, 832, 520, 2), (8, 4000, 1040, 264, 2),     # the ring, with four slots, with a tail of K
    (130, 40000, 256, 264, 2), (6, 2000, 8192, 712, 2), (6, 2000, 8192, 712, 0),                         # many experts; cut along K
    (64, 512, 2048, 712, 2), (64, 512, 2048, 712, 0), (5, 300, 528, 136, 2),                             # streamed; 64-row tiles
])
@pytest.mark.parametrize("given", ["none", "first", "second", "both"])
def test_scales_divided_out_with_either_bias(E, rows, K, N, epi, given):
    """Scales divided out in the epilogue against scales in the MFMAs, bit for bit (see above), zeros' signs included: with one bias of two, which
    the columns without one do not see."""
    from fast_moe_amd.kernels.hip import ops
    if epi != 2 and given in ("second", "both"):
        pytest.skip("one bias")
    g = torch.Generator(device="cuda").manual_seed(E + K)
    x = torch.randn(rows, K, generator=g, device="cuda")
    x[::9] = 0.0
    x[1::9] = -2.0 ** -60            # products that round to -0 and 0
    qx, sx = ops.quant_rows_fp8(x.to(BF16))
    qw = [ops.quant_rows_fp8((torch.randn(E, N, K, generator=g, device="cuda") * K ** -0.5).to(BF16)) for _ in range(2)]
    cuts = torch.randint(0, rows, (E - 1,), generator=g, device="cuda").sort().values
    off = torch.cat([cuts.new_zeros(1), cuts, cuts.new_full((1,), rows)])
    bias = [torch.randn(E, N, generator=g, device="cuda").to(BF16) if given in (side, "both") else None for side in ("first", "second")]
    kw = dict(total_rows=rows, a_scale=sx, b_scale=qw[0][1], epilogue=epi, bias=bias[0])
    if epi == 2:
        kw.update(b2=qw[1][0].permute(0, 2, 1), b2_scale=qw[1][1], bias2=bias[1])
    divided, folded = (ops.grouped_gemm(off, qx, qw[0][0].permute(0, 2, 1), scales_pow2=pow2, **kw) for pow2 in (False, True))
    assert torch.equal(divided.view(torch.int16), folded.view(torch.int16))


@pytest.mark.parametrize("E,rows,K,N,epi,sixteen", [
    (8, 4096, 1024, 1024, 0, False), (8, 8192, 2048, 3064, 0, True), (8, 8192, 2048, 2304, 1, False), (100, 20000, 2048, 1016, 0, True),
    (200, 30000, 1024, 2056, 3, True), (200, 30000, 512, 776, 1, False), (5, 9001, 2600, 2600, 0, True), (5, 9001, 1000, 2600, 0, True), (5, 9001, 1000, 2296, 0, False), (12, 9189, 2600, 1000, 0, True),
    (5, 9001, 2600, 1400, 2, True), (5, 9001, 1000, 2600, 2, False),
    (8, 8192, 2048, 3840, 2, True), (8, 8192, 2048, 1280, 2, False), (8, 16384, 4096, 512, 2, True), (4, 33000, 960, 2176, 2, False), (70, 9001, 2632, 2600, 2, True),
    (8, 16384, 4096, 1024, 0, True), (8, 4096, 4096, 1024, 0, False), (6, 16400, 4168, 1024, 1, True), (6, 4001, 4168, 1024, 1, False),      # cut along K
])
def test_tall_ring_by_the_launch_takes_one_of_two_mfma_shapes(E, rows, K, N, epi, sixteen):
    """Launches that reach the power cap run 16 x 16 x 32 MFMAs (mfma16_pays), others 32 x 32 x 16 ones, as all do whose weights have n contiguous:
    the same bits as those."""
    from fast_moe_amd.kernels.hip import _lib, ops
    g = torch.Generator(device="cuda").manual_seed(E + K + N)
    x = torch.randn(rows, K, generator=g, device="cuda").to(BF16)
    ws = [(torch.randn(E, N, K, generator=g, device="cuda") * K ** -0.5).to(BF16) for _ in range(2 if epi == 2 else 1)]
    cuts = torch.randint(0, rows, (E - 1,), generator=g, device="cuda").sort().values
    off = torch.cat([cuts.new_zeros(1), cuts, cuts.new_full((1,), rows)])
    kw = dict(total_rows=rows, epilogue=epi, bias=torch.randn(E, N, generator=g, device="cuda").to(BF16))
    if epi == _lib.EPI_GATED:
        kw["gate"] = torch.randn(rows, N, generator=g, device="cuda").to(BF16)
    def run(views):
        return ops.grouped_gemm(off, x, views[0], **kw, **({"b2": views[1]} if epi == 2 else {}))
    nk = [w.permute(0, 2, 1) for w in ws]
    ran = kernels_run(lambda: run(nk))[0]
    assert "ring_kernel" in ran and ("Mfma16" in ran) == sixteen, ran
    kn = [w.contiguous() for w in nk]
    assert "Mfma16" not in kernels_run(lambda: run(kn))[0]
    assert torch.equal(run(nk).view(torch.int16), run(kn).view(torch.int16))


@pytest.mark.parametrize("E,rows,K,N,layout,epi", [
    (3, 700, 72, 264, "nk", 0), (3, 700, 120, 136, "kn", 0),        # one pair of K-slices and the shortest / longest rest
    (2, 1000, 1000, 520, "nk", 2), (2, 1000, 1000, 520, "kn", 2),
    (5, 600, 2600, 256, "kn", 0), (4, 500, 544, 128, "nk", 1),      # 544: an odd number of whole slices
    (200, 20000, 136, 72, "nk", 1), (2, 513, 200, 320, "kn", 3),
    (3, 700, 144, 264, "fp8", 0), (2, 1000, 1040, 136, "fp8", 2), (4, 600, 240, 512, "fp8", 1),
    (3, 700, 1344, 136, "fp8", 0),
])
def test_ring_kernel_contraction_tails(E, rows, K, N, layout, epi):
    """K that is no whole number of K-slice pairs: the last pair overlaps the one before it and is
    masked.  The operands are the left columns of wider tensors whose other columns are NaN.  Against
    float64 on the GPU; 2 roundings to bf16 (SwiGLU: of either factor and the product)."""
    from fast_moe_amd.kernels.hip import _lib, ops
    g = torch.Generator().manual_seed(K + N)
    off = torch.tensor([0] + sorted(torch.randint(0, rows, (E - 1,), generator=g).tolist()) + [rows]).cuda()
    def wide(*shape):
        t = torch.full((*shape[:-1], shape[-1] + 16), float("nan"), dtype=BF16, device="cuda")
        t[..., :shape[-1]] = (torch.randn(*shape, generator=g) * shape[-1] ** -0.5).to(BF16).cuda()
        return t[..., :shape[-1]]
    x = wide(rows, K)
    ws = [wide(E, K, N) * 2 if layout == "kn" else wide(E, N, K).permute(0, 2, 1) for _ in range(2)]
    kw = dict(total_rows=rows, b2=ws[1] if epi == _lib.EPI_SWIGLU else None, epilogue=epi)
    gate = (torch.randn(rows, N, generator=g)).to(BF16).cuda()
    if epi == _lib.EPI_GATED:
        kw["gate"] = gate
    args = (x, ws[0])
    if layout == "fp8":
        qx, sx = ops.quant_rows_fp8(x)
        qw = [ops.quant_rows_fp8(w.permute(0, 2, 1)) for w in ws]
        kw.update(a_scale=sx, b_scale=qw[0][1], scales_pow2=True)
        if epi == _lib.EPI_SWIGLU:
            kw.update(b2=qw[1][0].permute(0, 2, 1), b2_scale=qw[1][1])
        args = (qx, qw[0][0].permute(0, 2, 1))
        x = qx.float() / sx[:, None]
        ws = [(q.float() / s[..., None]).permute(0, 2, 1) for q, s in qw]
    assert ops.grouped_gemm(off, *args, plan_only=True, **kw) == _lib.PLAN_RING
    out = ops.grouped_gemm(off, *args, **kw)
    ran, = kernels_run(lambda: ops.grouped_gemm(off, *args, **kw))
    assert KTAIL in ran, ran
    kw.pop("scales_pow2", None)
    assert layout != "fp8" or torch.equal(ops.grouped_gemm(off, *args, **kw), out)      # scales divided out instead
    for e in range(E):
        lo, hi = int(off[e]), int(off[e + 1])
        a = x[lo:hi].double() @ ws[0][e].double()
        if epi in (_lib.EPI_SILU, _lib.EPI_SWIGLU):
            a = torch.nn.functional.silu(a)
        if epi == _lib.EPI_SWIGLU:
            a = a * (x[lo:hi].double() @ ws[1][e].double())
        if epi == _lib.EPI_GATED:
            a = a * torch.nn.functional.silu(gate[lo:hi].double())
        assert_bf16_close(out[lo:hi], a.float(), rtol=1.6e-2, atol=4e-3, what=f"expert {e}")


@pytest.mark.parametrize("E,rows,K,N,dtype,tail", [
    (3, 700, 96, 264, "bf16", False), (3, 700, 480, 264, "bf16", False), (3, 700, 544, 264, "bf16", True),
    (8, 8192, 160, 2304, "bf16", False), (8, 8192, 224, 2304, "bf16", True),      # more than a round of tiles for certain
    (3, 700, 960, 264, "pow2", False), (3, 700, 1088, 264, "pow2", True), (8, 8192, 448, 2304, "pow2", True),
    (3, 700, 1216, 264, "fp8", False), (3, 700, 1344, 264, "fp8", True),
    (8, 8192, 960, 2304, "fp8", False), (8, 8192, 1088, 2304, "fp8", True), (300, 30000, 544, 264, "bf16", False),
])
def test_odd_numbers_of_whole_slices(E, rows, K, N, dtype, tail):
    """The 4-slot ring and the kernel for contraction tails both take them: which one runs on either side of the rule's lines,
    and the same sums from both (fp32 sums of exact products of small integers: bit for bit)."""
    from fast_moe_amd.kernels.hip import ops
    g = torch.Generator(device="cuda").manual_seed(K)
    off = (torch.arange(E + 1) * rows // E).cuda()
    x, w = (torch.randint(-2, 3, s, generator=g, device="cuda").to(BF16) for s in ((rows, K), (E, N, K)))
    args, kw = (x, w.permute(0, 2, 1)), dict(total_rows=rows)
    if dtype != "bf16":
        args = (x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn).permute(0, 2, 1))
        kw.update(a_scale=torch.ones(rows, device="cuda"), b_scale=torch.ones(E, N, device="cuda"), scales_pow2=dtype == "pow2")
    out = ops.grouped_gemm(off, *args, **kw)
    ran, = kernels_run(lambda: ops.grouped_gemm(off, *args, **kw))
    assert "ring_kernel" in ran and (KTAIL in ran) == tail and ("RingCfg<256, 256, 2, 4, 0, 2>" in ran) != tail, ran
    for e in range(0, E, 7):
        lo, hi = int(off[e]), int(off[e + 1])
        assert torch.equal(out[lo:hi], (x[lo:hi].float() @ w[e].float().t()).to(BF16))


@pytest.mark.parametrize("E,rows,K,N,layout,epi", [
    (3, 190, 36, 68, "kn", 0), (3, 190, 36, 60, "nk", 0),       # below / above one 64-column tile, a rest of one chunk
    (1, 64, 32, 64, "kn", 1), (1, 65, 4, 4, "kn", 0),           # whole tiles; one row more, the least K and N
    (5, 700, 60, 132, "kn", 2), (5, 700, 60, 132, "nk", 2),     # gate and up halves of a 128-column tile
    (2, 2600, 60, 3500, "nk", 1), (2, 2600, 60, 3500, "kn", 1),     # enough tiles for the wide form (nk)
    (70, 900, 64, 256, "kn", 0),                                # more experts than lanes, some empty
    (1, 4000, 36, 4096, "nk", 2),
    (1, 4096, 40, 4092, "nk", "silu"), (200, 2000, 64, 256, "nk", 2), (200, 2000, 40, 256, "nk", "silu"),
    (5, 700, 1000, 132, "kn", 2), (2, 2600, 100, 3500, "nk", 1), (1, 4096, 100, 4096, "nk", 1), (200, 2000, 256, 256, "nk", 2),  # (gemm_f32x3.h)
    (3, 190, 36, 60, "nk", "silu"), (3, 190, 36, 68, "kn", "silu"),
])
def test_fp32_kernel_tiles_and_weight_layouts(E, rows, K, N, layout, epi):
    """fp32 tiles, weights with k or n contiguous, SiLU in the epilogue or ("silu") on load.  The operands are the left
    columns of wider tensors whose other columns are NaN.  Against float64; the bound of a K-term fp32 sum,
    (K + 2) * 2^-24 * sum |a||b|, through SiLU (|slope| <= 1.1, its value on load to 2^-21) and the product."""
    from fast_moe_amd.kernels.hip import _lib, ops
    g = torch.Generator().manual_seed(K + N + rows)
    off = torch.tensor([0] + sorted(torch.randint(0, rows, (E - 1,), generator=g).tolist()) + [rows]).cuda()
    def wide(*shape):
        t = torch.full((*shape[:-1], shape[-1] + 4), float("nan"), device="cuda")
        t[..., :shape[-1]] = torch.randn(*shape, generator=g).cuda()
        return t[..., :shape[-1]]
    x = wide(rows, K)
    ws = [wide(E, K, N) if layout == "kn" else wide(E, N, K).permute(0, 2, 1) for _ in range(2)]
    a_silu, epi = epi == "silu", 0 if epi == "silu" else epi
    kw = dict(total_rows=rows, b2=ws[1] if epi == _lib.EPI_SWIGLU else None, epilogue=epi, a_silu=a_silu)
    assert ops.grouped_gemm(off, x, ws[0], plan_only=True, **kw) != _lib.PLAN_ELEMENT
    out = ops.grouped_gemm(off, x, ws[0], **kw)
    unit = (K + 2) * 2.0 ** -24 + (2.0 ** -21 if a_silu else 0)
    for e in range(E):
        a = x[int(off[e]):int(off[e + 1])].double()
        a = torch.nn.functional.silu(a) if a_silu else a
        want, err = a @ ws[0][e].double(), unit * (a.abs() @ ws[0][e].double().abs())
        if epi != _lib.EPI_NONE:
            want, err = torch.nn.functional.silu(want), 1.1 * err + 2.0 ** -21 * want.abs()
        if epi == _lib.EPI_SWIGLU:
            up, up_err = a @ ws[1][e].double(), unit * (a.abs() @ ws[1][e].double().abs())
            want, err = want * up, err * up.abs() + (want.abs() + err) * up_err + 2.0 ** -23 * (want * up).abs()
        assert bool(((out[int(off[e]):int(off[e + 1])].double() - want).abs() <= err).all()), f"expert {e}"


@pytest.mark.parametrize("E,rows,N,layout,epi,tile", [
    (1, 4096, 1920, "nk", 0, "64, 64"), (1, 4096, 1924, "nk", 0, "64, 256"), (1, 4096, 4096, "kn", 0, "64, 64"),
    (1, 4096, 1920, "nk", "silu", "64, 64"), (1, 4096, 1924, "nk", "silu", "64, 256"), (1, 4096, 4096, "kn", "silu", "64, 64"),
    (1, 65536, 64, "nk", 0, "64, 64"), (1, 65536, 68, "nk", 1, "64, 256"),              # half empty otherwise
    (1, 4096, 448, "nk", 2, "64, 128"), (1, 4096, 452, "nk", 2, "64, 256"), (1, 32768, 64, "nk", 2, "64, 128"), (200, 2000, 256, "nk", 2, "64, 256"),
    (1, 4096, 4096, "kn", 2, "64, 128"),
])
@pytest.mark.parametrize("K", [4, 64])
def test_fp32_tile_choice(E, rows, N, layout, epi, tile, K):
    """The tile on either side of the lines of the fp32 rule for short K, from a trace; small integers: exact sums."""
    from fast_moe_amd.kernels.hip import ops
    g = torch.Generator(device="cuda").manual_seed(N)
    x, w = (torch.randint(-3, 4, s, generator=g, device="cuda").float() for s in ((rows, K), (E, K, N) if layout == "kn" else (E, N, K)))
    w = w if layout == "kn" else w.permute(0, 2, 1)
    off = (torch.arange(E + 1) * rows // E).cuda()
    a_silu, epi = epi == "silu", 0 if epi == "silu" else epi
    run = lambda: ops.grouped_gemm(off, x, w, total_rows=rows, epilogue=epi, b2=w if epi == 2 else None, a_silu=a_silu)
    ran, = kernels_run(run)
    assert f"grouped_gemm_kernel<fmoe::TileCfg<{tile}," in ran, ran
    if epi == 0 and not a_silu:
        out = run()
        assert all(torch.equal(out[off[e]:off[e + 1]], x[off[e]:off[e + 1]] @ w[e]) for e in range(E))


@pytest.mark.parametrize("E,rows,K,N,layout,epi,tile", [
    (3, 190, 68, 68, "kn", 0, "64, 64"), (3, 190, 96, 60, "nk", 0, "64, 64"),          # the least K, a rest of one chunk / whole slices
    (1, 65, 132, 4, "kn", 1, "64, 64"), (2, 600, 100, 8192, "nk", 0, "64, 128"),       # the least N; more than four small tiles per CU
    (2, 600, 100, 8192, "kn", 1, "64, 128"), (3, 700, 72, 4100, "nk", "silu", "64, 128"),
    (5, 700, 100, 132, "kn", 2, "64, 128"), (5, 700, 100, 132, "nk", 2, "64, 128"),    # gate and up halves of a tile
    (3, 4800, 100, 1156, "nk", 0, "128, 128"), (3, 4800, 100, 1156, "kn", 0, "128, 128"),
    (3, 4800, 132, 1156, "nk", "silu", "128, 128"), (2, 4500, 68, 580, "kn", 2, "128, 128"), (70, 4800, 96, 1156, "nk", 2, "128, 128"),
])
@pytest.mark.parametrize("case", ["normal", "small", "large", "special"])
def test_fp32_on_bf16_matrix_cores(E, rows, K, N, layout, epi, tile, case):
    """fp32 values in three bf16 parts, on every tile.  small, large: rows and columns scaled by powers of two, operands
    down to the smallest normal values, up to sums where the parts overflow.  special: an infinity, a NaN and values beyond 2^104 in single
    rows and columns, whose results are those of the plain fp32 sum; the other results do not see them.  Against float64; the
    bound of a K-term fp32 sum, the sum of the small partial products and those left out (2^-34 each) in (K + 3) * 2^-24 * sum |a||b|; as in
    test_fp32_kernel_tiles_and_weight_layouts through SiLU and the product."""
    from fast_moe_amd.kernels.hip import _lib, ops
    g = torch.Generator(device="cuda").manual_seed(K + N + rows)
    randn_ = lambda *s: torch.randn(*s, generator=g, device="cuda")
    off = torch.tensor([0] + sorted(torch.randint(0, rows, (E - 1,), generator=torch.Generator().manual_seed(N)).tolist()) + [rows]).cuda()
    a_silu, epi = epi == "silu", 0 if epi == "silu" else epi
    x, ws = randn_(rows, K), [randn_(E, K, N) for _ in range(2)]
    odd_rows = torch.zeros(rows, dtype=torch.bool, device="cuda")
    odd_cols = torch.zeros(N, dtype=torch.bool, device="cuda")
    if case in ("small", "large"):
        a_silu, epi = False, _lib.EPI_NONE      # (SiLU and the product have ranges of their own)
        lo, hi, w_hi = (-112, -40, 40) if case == "small" else (-90, 70, 26)
        x = torch.where(x.abs() < 2.0 ** -14, torch.ones_like(x), x)        # (no denormal value)
        x *= torch.exp2(torch.randint(lo, hi, (rows, 1), generator=g, device="cuda").float())
        ws = [w * torch.exp2(torch.randint(0, w_hi, (1, 1, N), generator=g, device="cuda").float()) for w in ws]
    if case == "special":
        x[5, K - 1], x[rows - 1, 0], x[rows // 2, 3] = float("inf"), float("nan"), 3e38
        odd_rows[[5, rows - 1, rows // 2]] = True
        for w in ws:
            w[:, 1, N - 1], w[:, 2, 1] = float("inf"), 2.0 ** 110
        odd_cols[[1, N - 1]] = True
    if layout == "nk":
        ws = [w.permute(0, 2, 1).contiguous().permute(0, 2, 1) for w in ws]
    kw = dict(total_rows=rows, b2=ws[1] if epi == _lib.EPI_SWIGLU else None, epilogue=epi, a_silu=a_silu)
    out = ops.grouped_gemm(off, x, ws[0], **kw)
    ran, = kernels_run(lambda: ops.grouped_gemm(off, x, ws[0], **kw))
    assert f"grouped_gemm_f32x3_kernel<fmoe::TileF32x3<{tile if case in ('normal', 'special') else ''}" in ran, ran
    unit = (K + 3) * 2.0 ** -24 + (2.0 ** -21 if a_silu else 0)
    for e in range(E):
        lo, hi = int(off[e]), int(off[e + 1])
        a = torch.nn.functional.silu(x[lo:hi].double()) if a_silu else x[lo:hi].double()
        want, err = a @ ws[0][e].double(), unit * (a.abs() @ ws[0][e].double().abs()) + 2.0 ** -149
        if epi != _lib.EPI_NONE:
            want, err = torch.nn.functional.silu(want), 1.1 * err + 2.0 ** -21 * want.abs()
        if epi == _lib.EPI_SWIGLU:
            up, up_err = a @ ws[1][e].double(), unit * (a.abs() @ ws[1][e].double().abs())
            want, err = want * up, err * up.abs() + (want.abs() + err) * up_err + 2.0 ** -23 * (want * up).abs()
        got, plain = out[lo:hi].double(), ~odd_rows[lo:hi, None] & ~odd_cols[None]
        assert bool(((got - want).abs() <= err)[plain].all()), f"expert {e}"
        if case == "special" and epi == _lib.EPI_NONE and not a_silu:
            plain_fp32 = x[lo:hi].cpu() @ ws[0][e].cpu()
            far = want.abs().cpu() > 1e39                       # beyond fp32 for certain, whatever the order
            near = want.abs().cpu() < 1e38
            assert torch.equal(got.cpu().isnan(), plain_fp32.isnan()) and bool(got.cpu()[far].isinf().all())
            assert bool(((got - want).abs() <= err).cpu()[near].all())


@pytest.mark.parametrize("lens,K,N,layout,epi,tile", [
    ([2048] * 3 + [2049], 1024, 1024, "nk", 0, 128),        # two whole rounds and eight tiles of a row
    ([0, 4000, 2500, 2100, 3], 996, 1020, "kn", 1, 128), ([4000, 2500, 2100, 130], 1028, 964, "nk", "silu", 128),
    ([3000, 3500, 30], 772, 700, "nk", 2, 128), ([3000, 3500, 30], 1024, 700, "kn", 2, 128),
    ([2100, 0, 500, 400, 33], 4100, 1000, "kn", 1, 128), ([2100, 500, 400, 33], 4160, 904, "nk", "silu", 128),       # less than a round
    ([500] * 66, 1024, 252, "nk", 0, 128),                  # more than 64 experts
    ([2048] * 3 + [2049], 324, 1024, "nk", 0, 128), ([1000, 1100, 900, 1024, 1100, 1000, 1068, 1000], 420, 1020, "kn", 2, 128),      # six and seven pairs of slices
    ([512] * 7 + [513], 4096, 1024, "nk", 0, 64), ([520, 0, 500, 600, 1400, 1033], 1028, 1000, "kn", 1, 64),
    ([520, 0, 500, 600, 1400, 1033], 996, 964, "nk", "silu", 64), ([520, 3, 500, 600, 1400, 1033], 2052, 900, "kn", "silu", 64),
    ([512] * 8, 1024, 1024, "nk", 0, 64),                   # no tile left: nothing is cut
])
@pytest.mark.parametrize("case", ["normal", "special"])
def test_fp32_last_round_cut_along_k(lens, K, N, layout, epi, tile, case):
    """Against float64, in the bound of test_fp32_on_bf16_matrix_cores (grouping the sums adds none to it); the same bits twice.  special: an
    infinity, a NaN and a value beyond 2^104 in single rows; the other rows do not see them."""
    from fast_moe_amd.kernels.hip import _lib, ops
    E, rows = len(lens), sum(lens)
    g = torch.Generator(device="cuda").manual_seed(K + N)
    off = torch.tensor([0, *torch.tensor(lens).cumsum(0)]).cuda()
    a_silu, epi = epi == "silu", 0 if epi == "silu" else epi
    x = torch.randn((rows + 1) // 2, K, generator=g, device="cuda")
    index = torch.arange(rows, device="cuda")
    bias = [torch.randn(E, N, generator=g, device="cuda") for _ in range(2)]
    ws = [torch.randn(*((E, K, N) if layout == "kn" else (E, N, K)), generator=g, device="cuda") * K ** -0.5 for _ in range(2)]
    odd = torch.zeros(rows, dtype=torch.bool, device="cuda")
    if case == "special":
        x[2, K - 1], x[x.shape[0] - 1, 0], x[x.shape[0] // 2, K // 2] = float("inf"), float("nan"), 3e38
        for r in (2, x.shape[0] - 1, x.shape[0] // 2):
            odd[2 * r:2 * r + 2] = True
    ws = [w if layout == "kn" else w.permute(0, 2, 1) for w in ws]
    swiglu = epi == _lib.EPI_SWIGLU
    kw = dict(total_rows=rows, row_index=index, index_div=2, bias=bias[0], epilogue=epi, a_silu=a_silu)
    if swiglu:
        kw.update(b2=ws[1], bias2=bias[1])
    ran = kernels_run(lambda: ops.grouped_gemm(off, x, ws[0], **kw))
    out = ops.grouped_gemm(off, x, ws[0], **kw)
    again = ops.grouped_gemm(off, x, ws[0], **kw)
    assert torch.equal(out.nan_to_num(7.0), again.nan_to_num(7.0))
    assert [n.split("<")[0].split("::")[-1] for n in ran] == ["grouped_gemm_f32x3_kernel", "f32x3_reduce_kernel"], ran
    assert f"TileF32x3<{tile}, 128" in ran[0], ran
    unit = (K + 4) * 2.0 ** -24 + (2.0 ** -21 if a_silu else 0)         # (a rounding for the bias)
    for e in range(E):
        lo, hi = int(off[e]), int(off[e + 1])
        a = x[index[lo:hi] // 2].double()
        a = torch.nn.functional.silu(a) if a_silu else a
        want, err = a @ ws[0][e].double() + bias[0][e].double(), unit * (a.abs() @ ws[0][e].double().abs() + bias[0][e].double().abs())
        if epi != _lib.EPI_NONE:
            want, err = torch.nn.functional.silu(want), 1.1 * err + 2.0 ** -21 * want.abs()
        if swiglu:
            up, up_err = a @ ws[1][e].double() + bias[1][e].double(), unit * (a.abs() @ ws[1][e].double().abs() + bias[1][e].double().abs())
            want, err = want * up, err * up.abs() + (want.abs() + err) * up_err + 2.0 ** -23 * (want * up).abs()
        plain = ~odd[lo:hi]
        assert bool(((out[lo:hi].double() - want).abs() <= err)[plain].all()), f"expert {e}"
        if case == "special" and epi == _lib.EPI_NONE and not a_silu:
            assert bool((~out[lo:hi][~plain].isfinite() | (want[~plain].abs() < 3.5e38)).all())


@pytest.mark.parametrize("E,rows,K,N,layout", [(3, 700, 256, 1156, "nk"), (3, 700, 256, 1156, "kn"), (3, 190, 200, 60, "nk"), (3, 4800, 256, 1156, "kn"),
                                               (4, 40, 1024, 264, "nk"), (8, 200, 1024, 132, "nk")])
@pytest.mark.parametrize("nonzero", [1, 2, 5, 16])
def test_fp32_rows_of_few_nonzero_products(E, rows, K, N, layout, nonzero):
    """Results of few products have no more error than fused multiply-adds in fp32 leave, one rounding of the running sum for each: in the
    2-norm (the roundings' signs are random: 2 %), and in every value the bound of the sum of the large partial products, which are exact
    (n - 1 additions, the last place each as an MFMA may cut it: 2^-23), of adding the small ones (2^-24) and of their sum (2^-7 of the
    products, seven additions each: 2^-27)."""
    from fast_moe_amd.kernels.hip import ops
    g = torch.Generator(device="cuda").manual_seed(K + N + nonzero)
    x = torch.randn(rows, K, generator=g, device="cuda")
    x = x * (torch.rand(rows, K, generator=g, device="cuda").argsort(dim=1) < nonzero)
    w = torch.randn(E, K, N, generator=g, device="cuda")
    if layout == "nk":
        w = w.permute(0, 2, 1).contiguous().permute(0, 2, 1)
    off = (torch.arange(E + 1) * rows // E).cuda()
    out = ops.grouped_gemm(off, x, w, total_rows=rows).double()
    ours = fused = 0.0
    for e in range(E):
        lo, hi = int(off[e]), int(off[e + 1])
        a, b = x[lo:hi], w[e]
        want, size = a.double() @ b.double(), a.double().abs() @ b.double().abs()
        bound = (2 * nonzero - 1) * 2.0 ** -24 + nonzero * 2.0 ** -27
        assert bool(((out[lo:hi] - want).abs() <= bound * size).all()), f"expert {e}"
        where, chain = a.ne(0).float().topk(nonzero, dim=1).indices, torch.zeros_like(want)
        for i in range(nonzero):
            chain = (chain + a.gather(1, where[:, i:i + 1]).double() * b[where[:, i]].double()).float().double()
        ours += float((out[lo:hi] - want).square().sum())
        fused += float((chain - want).square().sum())
    assert ours <= 1.02 ** 2 * fused, (ours / fused) ** 0.5


@pytest.mark.parametrize("K,new", [(64, False), (68, True)])
def test_fp32_kernel_for_short_k(K, new):
    from fast_moe_amd.kernels.hip import ops
    x, w, off = torch.zeros(64, K, device="cuda"), torch.zeros(1, 64, K, device="cuda").permute(0, 2, 1), torch.tensor([0, 64]).cuda()
    ran, = kernels_run(lambda: ops.grouped_gemm(off, x, w, total_rows=64))
    assert ("f32x3" in ran) == new, ran


@pytest.mark.parametrize("lens,K,N,epi", [
    ([16, 1, 17, 30], 392, 68, 0), ([33, 0, 64, 31, 0, 0, 0, 0], 264, 260, 1),     # one, two and four fragments of 16 rows, full and one row more
    ([65, 0, 0, 0, 0, 0, 2], 520, 40, 2),                               # more than a tile's rows; SwiGLU columns in part
    ([0, 1], 136, 72, 0), ([0, 1, 0, 1], 1032, 200, 2), ([2, 0, 1], 520, 64, 1), # one, two and three rows
    ([0, 3, 1], 72, 8, 0), ([2, 2], 128, 64, 2),                        # fewer 128-byte pieces than waves; one whole tile
    ([1] * 70 + [0, 9], 104, 132, 0), ([4, 0] * 80, 136, 72, 1),        # more experts than lanes
    ([5] * 11, 800, 2900, 0), ([3] * 20, 824, 1096, "silu"),           # more tiles than CUs
    ([7, 0, 20, 8], 1048, 200, "silu"),
    ([65, 0, 129, 255, 1], 2056, 72, 0), ([300, 40, 0, 320], 2064, 296, 2),     # rows enough for taller tiles, but few of them
])
@pytest.mark.parametrize("dtype", ["bf16", "fp8", "f32"])
@pytest.mark.parametrize("extras", [False, True])
def test_streaming_kernel_of_few_tiles(lens, K, N, epi, dtype, extras):
    """Weights straight into registers.  The operands are the left columns of wider tensors whose other columns are NaN.  extras:
    gathered rows, bias and, with SwiGLU, the two pre-activations.  Against float64 with the roundings of the bf16 path
    (test_ring_kernel_contraction_tails) and, fp32, the bound of test_fp32_on_bf16_matrix_cores with one rounding more per bias."""
    from fast_moe_amd.kernels.hip import _lib, ops
    a_silu, epi = epi == "silu", 0 if epi == "silu" else epi
    if dtype == "fp8":
        a_silu, K = False, (K + 15) // 16 * 16
    f32, E, rows = dtype == "f32", len(lens), sum(lens)
    dt, g = torch.float32 if f32 else BF16, torch.Generator(device="cuda").manual_seed(K + N)
    off = torch.tensor([0, *torch.tensor(lens).cumsum(0)]).cuda()
    randn_ = lambda *s: torch.randn(*s, generator=g, device="cuda")
    def wide(*shape):
        t = torch.full((*shape[:-1], shape[-1] + 16), float("nan"), dtype=dt, device="cuda")
        t[..., :shape[-1]] = (randn_(*shape) * shape[-1] ** -0.5).to(dt)
        return t[..., :shape[-1]]
    T = (rows + 1) // 2 if extras else rows
    x, ws = wide(T, K), [wide(E, N, K) for _ in range(2)]
    index = torch.randint(0, 2 * T, (rows,), generator=g, device="cuda") if extras else None
    bias = [randn_(E, N).to(dt) for _ in range(2)] if extras else [None, None]
    swiglu = epi == _lib.EPI_SWIGLU
    aux = tuple(torch.zeros(rows, N, dtype=dt, device="cuda") for _ in range(2)) if extras and swiglu else None
    kw = dict(total_rows=rows, row_index=index, index_div=2 if extras else 1, bias=bias[0], epilogue=epi, a_silu=a_silu, aux=aux)
    if swiglu:
        kw.update(b2=ws[1].permute(0, 2, 1), bias2=bias[1])
    args = (x, ws[0].permute(0, 2, 1))
    if dtype == "fp8":
        qx, sx = ops.quant_rows_fp8(x)
        qw = [ops.quant_rows_fp8(w) for w in ws]
        kw.update(a_scale=sx, b_scale=qw[0][1], scales_pow2=True)
        if swiglu:
            kw.update(b2=qw[1][0].permute(0, 2, 1), b2_scale=qw[1][1])
        args = (qx, qw[0][0].permute(0, 2, 1))
        x, ws = qx.float() / sx[:, None], [q.float() / s[..., None] for q, s in qw]
    out = ops.grouped_gemm(off, *args, **kw)
    ran, = kernels_run(lambda: ops.grouped_gemm(off, *args, **kw))
    assert "grouped_gemm_direct_kernel<" in ran, ran
    source = x if index is None else x[index // 2]
    unit = (K + 4) * 2.0 ** -24 + (2.0 ** -21 if a_silu else 0)
    for e in range(E):
        lo, hi = int(off[e]), int(off[e + 1])
        a = source[lo:hi].double()
        a = torch.nn.functional.silu(a) if a_silu else a
        if a_silu and not f32:
            a = a.to(BF16).double()
        pre, err = [], []
        for w, b in zip(ws, bias):
            add = b[e].double() if b is not None else torch.zeros(N, dtype=torch.float64, device="cuda")
            pre.append(a @ w[e].double().t() + add)
            err.append(unit * (a.abs() @ w[e].double().abs().t() + add.abs()))
        want, bound = pre[0], err[0]
        if epi != _lib.EPI_NONE:
            want, bound = torch.nn.functional.silu(want), 1.1 * bound + 2.0 ** -21 * want.abs()
        if swiglu:
            want, bound = want * pre[1], bound * pre[1].abs() + (want.abs() + bound) * err[1] + 2.0 ** -23 * (want * pre[1]).abs()
        pairs = [(out, want, bound)] + ([(aux[0], pre[0], err[0]), (aux[1], pre[1], err[1])] if aux else [])
        for got, ref, b in pairs:
            if f32:
                assert bool(((got[lo:hi].double() - ref).abs() <= b).all()), f"expert {e}"
            else:
                assert_bf16_close(got[lo:hi], ref.float(), rtol=1.6e-2, atol=4e-3, what=f"expert {e}")


def test_streaming_kernel_recomputes_fp32_sums_that_are_not_finite():
    """As test_fp32_on_bf16_matrix_cores, special."""
    from fast_moe_amd.kernels.hip import ops
    g = torch.Generator(device="cuda").manual_seed(1)
    off = torch.tensor([0, 9, 9, 40]).cuda()
    x, w = (torch.randn(*s, generator=g, device="cuda") for s in ((40, 200), (3, 130, 200)))
    x[3, 0], x[20, 199], x[39, 7] = float("inf"), float("nan"), 2.0 ** 110
    w[2, 5, 11], w[0, 129, 3] = float("-inf"), 2.0 ** 120
    out = ops.grouped_gemm(off, x, w.permute(0, 2, 1), total_rows=40)
    for e in (0, 2):
        lo, hi = int(off[e]), int(off[e + 1])
        got, plain, want = out[lo:hi].cpu(), x[lo:hi].cpu() @ w[e].t().cpu(), x[lo:hi].double() @ w[e].double().t()
        assert torch.equal(got.isnan(), plain.isnan()) and torch.equal(got.isinf(), plain.isinf())
        assert torch.equal(got[plain.isinf()], plain[plain.isinf()])
        err, fine = 203 * 2.0 ** -24 * (x[lo:hi].double().abs() @ w[e].double().abs().t()), plain.isfinite()
        assert bool(((got.double() - want.cpu()).abs() <= err.cpu())[fine].all())


@pytest.mark.parametrize("E,rows,K,N,dtype,direct", [
    (16, 16, 1664, 1024, "bf16", True), (16, 40, 1664, 1024 + 1, "bf16", False),        # one tile per CU; K of more than 1664 bytes beyond
    (16, 16, 832, 2048, "bf16", True), (16, 40, 832, 2049, "bf16", False), (16, 16, 2048, 2048, "fp8", True), (16, 16, 2048, 2049, "fp8", False),
    (24, 48, 1024, 4096, "bf16", True), (24, 48, 1024, 4100, "bf16", False), (24, 49, 1024, 4096, "bf16", False), (24, 48, 1024, 4096, "fp8", False),
    (24, 96, 1032, 8512, "bf16", True), (24, 96, 1032, 8584, "bf16", False), (24, 96, 1040, 8512, "fp8", True),         # K in part
    (24, 97, 1032, 4544, "bf16", True), (24, 97, 1032, 4616, "bf16", False), (24, 97, 1040, 4096, "fp8", False), (24, 97, 2064, 4096, "fp8", True),
    (24, 193, 1032, 4096, "bf16", False),
    (16, 256, 1664, 1024, "bf16", False), (16, 250, 832, 64, "bf16", True), (4, 65, 832, 64, "bf16", True),
    (4, 80, 256, 64, "bf16", False), (4, 80, 264, 64, "bf16", True), (4, 4096, 1024, 240, "bf16", True), (4, 4096, 1016, 240, "bf16", False),
    (4, 800, 1024, 2048, "bf16", True), (4, 800, 1024, 2056, "bf16", False), (4, 800, 2048, 2048, "fp8", True), (4, 800, 2048, 2064, "fp8", False),
    (4, 380, 1024, 2048, "bf16", False), (4, 300, 1024, 512, "f32", True), (4, 300, 1020, 512, "f32", False),
    (4, 100, 992, 512, "f32", True), (8, 700, 128, 448, "f32", True), (8, 700, 128, 449, "f32", False), (8, 700, 96, 64, "f32", False),
    (16, 100, 1020, 2049, "f32", False), (16, 64, 1020, 2049, "f32", True), (16, 100, 1024, 2049, "f32", True), (16, 16, 64, 64, "f32", False),
    (8, 1, 4096, 1024, "bf16", True), (8, 2, 4096, 1024, "fp8", True), (8, 3, 4096, 1024, "f32", True), (1, 1, 128, 256, "bf16", True),
])
def test_streaming_kernel_choice(E, rows, K, N, dtype, direct):
    """Which calls the kernel above takes, on either side of the rule's lines."""
    from fast_moe_amd.kernels.hip import ops
    dt = {"bf16": BF16, "fp8": torch.float8_e4m3fn, "f32": torch.float32}[dtype]
    x, w = torch.zeros(rows, K, device="cuda").to(dt), torch.zeros(E, N, K, dtype=BF16, device="cuda").to(dt).permute(0, 2, 1)
    kw = dict(a_scale=torch.ones(rows, device="cuda"), b_scale=torch.ones(E, N, device="cuda")) if dtype == "fp8" else {}
    off = (torch.arange(E + 1) * rows // E).cuda()
    ran, = kernels_run(lambda: ops.grouped_gemm(off, x, w, total_rows=rows, **kw))
    assert ("grouped_gemm_direct_kernel<" in ran) == direct, ran


@pytest.mark.parametrize("native", [True, False])
def test_calls_without_memory_for_a_workspace_run_uncut(native):
    """Less memory left than the 64 MiB of the cut along K (a limit of the allocator's): the call runs as it does without a workspace."""
    from fast_moe_amd.kernels.hip import _lib, ops
    E, rows, K, N = 8, 2000, 4096, 512
    g = torch.Generator(device="cuda").manual_seed(1)
    x, w = torch.randn(rows, K, generator=g, device="cuda").to(BF16), (torch.randn(E, N, K, generator=g, device="cuda") * K ** -0.5).to(BF16)
    off, host = (torch.arange(E + 1) * rows // E).cuda(), _lib.host()
    run = lambda: ops.grouped_gemm(off, x, w.permute(0, 2, 1), total_rows=rows)
    cut, ran = run(), kernels_run(run)
    assert "split_reduce" in ran[-1]
    _lib._host = host if native else _lib._Declines()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    try:
        total = torch.cuda.get_device_properties(0).total_memory
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (40 << 20)) / total)
        taken = []          # free pieces of segments that other tensors keep
        with pytest.raises(torch.OutOfMemoryError):
            while len(taken) < 10000:
                taken.append(torch.empty(64 << 20, dtype=torch.uint8, device="cuda"))
        out = run()
    finally:
        taken = None
        torch.cuda.set_per_process_memory_fraction(1.0)
        _lib._host = host
    assert_bf16_close(out, cut.float(), rtol=1.6e-2, atol=4e-3, what="uncut")
    assert not torch.equal(out, cut)            # (the grouping of fp32 sums)


@pytest.mark.parametrize("E,rows,K,N,dtype,cut", [
    (6, 766, 3592, 640, "bf16", True), (6, 766, 3584, 640, "bf16", False), (6, 766, 3968, 640, "fp8", False),       # one tile per CU: by K
    (8, 2000, 3072, 448, "bf16", True), (8, 2000, 3072, 384, "bf16", False), (8, 2000, 4096, 512, "bf16", True),    # 273 and 234 tiles
])
def test_cut_along_k_or_few_tiles_kernel(E, rows, K, N, dtype, cut):
    """Which of the two runs a call that both take, on either side of the rule's lines."""
    from fast_moe_amd.kernels.hip import ops
    dt = {"bf16": BF16, "fp8": torch.float8_e4m3fn}[dtype]
    x, w = torch.zeros(rows, K, device="cuda").to(dt), torch.zeros(E, N, K, dtype=BF16, device="cuda").to(dt).permute(0, 2, 1)
    kw = dict(a_scale=torch.ones(rows, device="cuda"), b_scale=torch.ones(E, N, device="cuda")) if dtype == "fp8" else {}
    off = (torch.arange(E + 1) * rows // E).cuda()
    ran = kernels_run(lambda: ops.grouped_gemm(off, x, w, total_rows=rows, **kw))
    names = [n.split("<")[0].split("::")[-1] for n in ran]
    assert names == (["grouped_gemm_ring_kernel", "split_reduce_kernel"] if cut else ["grouped_gemm_direct_kernel"]), ran


@pytest.mark.parametrize("E,rows,K,N,layout,epi", [
    (3, 130, 136, 264, "nk", 0), (3, 130, 192, 136, "kn", 0),       # the least K: three pairs of K-slices, the last in part / whole
    (1, 64, 256, 256, "kn", 1), (1, 65, 256, 256, "nk", 1),         # one whole tile; one row more
    (3, 130, 1000, 4104, "nk", 2), (2, 3, 1000, 520, "nk", 3), (2, 3, 1000, 520, "kn", 2),
    (200, 900, 328, 72, "kn", 0), (130, 5000, 264, 1032, "kn", 2),  # more experts than lanes; more tiles than CUs
    (2, 150, 200, 320, "kn", 3), (40, 2000, 640, 2048, "kn", 3),
    (3, 280, 640, 32768, "nk", 3),                                  # more tiles than CUs with k contiguous
    (3, 130, 272, 264, "fp8", 0), (3, 70, 384, 136, "fp8", 2), (8, 760, 4096, 2816, "fp8", 0),
])
def test_ring_kernel_on_short_tiles(E, rows, K, N, layout, epi):
    """The ring on 64-row tiles (few rows per expert).  The operands are the left columns of wider
    tensors whose other columns are NaN.  Against float64 on the GPU; roundings as in
    test_ring_kernel_contraction_tails."""
    from fast_moe_amd.kernels.hip import _lib, ops
    g = torch.Generator(device="cuda").manual_seed(K + N)
    off = torch.tensor([0] + sorted(torch.randint(0, rows, (E - 1,), generator=g, device="cuda").tolist()) + [rows]).cuda()
    def wide(*shape):
        t = torch.full((*shape[:-1], shape[-1] + 16), float("nan"), dtype=BF16, device="cuda")
        t[..., :shape[-1]] = (torch.randn(*shape, generator=g, device="cuda") * shape[-1] ** -0.5).to(BF16)
        return t[..., :shape[-1]]
    x = wide(rows, K)
    ws = [wide(E, K, N) if layout == "kn" else wide(E, N, K).permute(0, 2, 1) for _ in range(2)]
    kw = dict(total_rows=rows, b2=ws[1] if epi == _lib.EPI_SWIGLU else None, epilogue=epi)
    gate = torch.randn(rows, N, generator=g, device="cuda").to(BF16)
    if epi == _lib.EPI_GATED:
        kw["gate"] = gate
    args = (x, ws[0])
    if layout == "fp8":
        qx, sx = ops.quant_rows_fp8(x)
        qw = [ops.quant_rows_fp8(w.permute(0, 2, 1)) for w in ws]
        kw.update(a_scale=sx, b_scale=qw[0][1], scales_pow2=True)
        if epi == _lib.EPI_SWIGLU:
            kw.update(b2=qw[1][0].permute(0, 2, 1), b2_scale=qw[1][1])
        args = (qx, qw[0][0].permute(0, 2, 1))
        x = qx.float() / sx[:, None]
        ws = [(q.float() / s[..., None]).permute(0, 2, 1) for q, s in qw]
    assert ops.grouped_gemm(off, *args, plan_only=True, **kw) == _lib.PLAN_STAGED_SHORT
    out = ops.grouped_gemm(off, *args, **kw)
    ran, = kernels_run(lambda: ops.grouped_gemm(off, *args, **kw))
    assert "ring_kernel" in ran and "RingCfg<64," in ran, ran
    kw.pop("scales_pow2", None)
    assert layout != "fp8" or torch.equal(ops.grouped_gemm(off, *args, **kw), out)      # scales divided out instead
    for e in range(E):
        lo, hi = int(off[e]), int(off[e + 1])
        a = x[lo:hi].double() @ ws[0][e].double()
        if epi in (_lib.EPI_SILU, _lib.EPI_SWIGLU):
            a = torch.nn.functional.silu(a)
        if epi == _lib.EPI_SWIGLU:
            a = a * (x[lo:hi].double() @ ws[1][e].double())
        if epi == _lib.EPI_GATED:
            a = a * torch.nn.functional.silu(gate[lo:hi].double())
        assert_bf16_close(out[lo:hi], a.float(), rtol=1.6e-2, atol=4e-3, what=f"expert {e}")


@pytest.mark.parametrize("short,E,rows,K,N,epi", [
    (False, 3, 700, 136, 264, 0), (False, 3, 700, 248, 136, 1),     # one pair of K-slices and the shortest / longest rest
    (False, 2, 1000, 1000, 520, 2), (False, 70, 9000, 520, 1032, 0),
    (True, 3, 130, 264, 264, 0), (True, 2, 3, 1000, 520, 2),        # the least K; more than a pair of a rest
    (True, 111, 333, 2888, 3072, 0), (True, 130, 900, 376, 72, 1),
])
def test_e4m3_rows_of_an_odd_number_of_8_byte_groups(short, E, rows, K, N, epi):
    """K % 16 == 8: every other row starts off a 16-byte boundary."""
    (test_ring_kernel_on_short_tiles if short else test_ring_kernel_contraction_tails)(E, rows, K, N, "fp8", epi)


@pytest.mark.parametrize("rows,K,lead", [(700, 256, 8), (700, 320, 8), (700, 200, 24), (60, 512, 8), (60, 392, 40)])
def test_e4m3_operands_off_a_16_byte_boundary(rows, K, lead):
    """Columns ``lead`` .. ``lead + K`` of wider e4m3 tensors, NaN codes around them: the ring reads them in place.  Small
    integers with scale 1: exact sums, rounded once."""
    from fast_moe_amd.kernels.hip import _lib, ops
    g = torch.Generator().manual_seed(K)
    E, N = 3, 264
    def wide(*shape):
        t = torch.full((*shape[:-1], shape[-1] + 64), float("nan"))
        t[..., lead:lead + shape[-1]] = torch.randint(-2, 3, shape, generator=g).float()
        return t.cuda().to(torch.float8_e4m3fn)[..., lead:lead + shape[-1]]
    x, w = wide(rows, K), wide(E, N, K)
    off = torch.tensor([0, rows // 3, rows // 3, rows]).cuda()
    kw = dict(total_rows=rows, a_scale=torch.ones(rows, device="cuda"), b_scale=torch.ones(E, N, device="cuda"))
    assert ops.grouped_gemm(off, x, w.permute(0, 2, 1), plan_only=True, **kw) != _lib.PLAN_ELEMENT
    for pow2 in (False, True):
        out = ops.grouped_gemm(off, x, w.permute(0, 2, 1), scales_pow2=pow2, **kw)
        for e in range(E):
            lo, hi = int(off[e]), int(off[e + 1])
            assert torch.equal(out[lo:hi], (x[lo:hi].float() @ w[e].float().t()).to(BF16))


@pytest.mark.parametrize("E,rows,K,N,layout,epi,kernel", [
    (8, 760, 4096, 3328, "nk", 0, "ring"), (8, 760, 4096, 3584, "nk", 0, "stream"),     # 247 / 266 tiles if the rows fall badly
    (8, 760, 4096, 3328, "fp8", 0, "ring"), (8, 760, 4096, 3584, "fp8", 0, "stream"),
    (128, 512, 4096, 1536, "nk", 2, "stream"), (128, 512, 4096, 1536, "fp8", 0, "stream"),
    (128, 8000, 4096, 1536, "nk", 2, "stream"),                                         # many rounds of tiles
    (20, 3, 1024, 16384, "fp8", 0, "ring"),                                             # no more experts than rows can have one
    (200, 3, 1024, 8192, "nk", 0, "direct"), (64, 1, 2048, 1408, "nk", 2, "direct"), (64, 2, 2048, 1408, "fp8", 2, "direct"),
    (64, 64, 1024, 2048, "nk", 3, "staged"), (64, 5000, 1024, 1408, "nk", 3, "staged"),
    (64, 5900, 1024, 1408, "nk", 3, "ring"), (64, 5900, 1000, 1408, "nk", 3, "staged"), # GATED: more than two rounds for certain
    (128, 512, 4096, 1536, "kn", 2, "ring"),
])
def test_kernel_choice_for_few_rows(E, rows, K, N, layout, epi, kernel):
    """Which kernel runs a call with few rows per expert, on either side of the rule's lines; the same for an even load and for
    one expert with nine tenths of the rows (the host does not know the load)."""
    from fast_moe_amd.kernels.hip import _lib, ops
    x = torch.zeros(rows, K, dtype=BF16, device="cuda")
    w = torch.zeros((E, K, N) if layout == "kn" else (E, N, K), dtype=BF16, device="cuda")
    kw = dict(total_rows=rows, epilogue=epi)
    args = (x, w if layout == "kn" else w.permute(0, 2, 1))
    if layout == "fp8":
        args = tuple(t.to(torch.float8_e4m3fn) for t in (x, w))
        args = (args[0], args[1].permute(0, 2, 1))
        kw.update(a_scale=torch.ones(rows, device="cuda"), b_scale=torch.ones(E, N, device="cuda"))
    if epi == _lib.EPI_SWIGLU:
        kw["b2"] = args[1]
        if layout == "fp8":
            kw["b2_scale"] = kw["b_scale"]
    if epi == _lib.EPI_GATED:
        kw["gate"] = torch.zeros(rows, N, dtype=BF16, device="cuda")
    even = torch.arange(E + 1) * rows // E
    hot = torch.cat([torch.zeros(1, dtype=torch.int64), (torch.arange(E) * (rows // 10) // max(E - 1, 1)) + rows - rows // 10])
    want = {"ring": "grouped_gemm_ring_kernel<fmoe::RingCfg<64,", "stream": "grouped_gemm_stream_kernel<",
            "staged": "grouped_gemm_kernel<fmoe::TileCfg<64, 256,", "direct": "grouped_gemm_direct_kernel<"}[kernel]
    for off in (even.cuda(), hot.cuda()):
        ran, = kernels_run(lambda: ops.grouped_gemm(off, *args, **kw))
        assert want in ran, ran


@pytest.mark.parametrize("row_tiles", [1, 7, 28, 31, 32, 33, 59, 60, 61, 97])
@pytest.mark.parametrize("N", [256, 776])
def test_ring_kernel_writes_every_tile(row_tiles, N):
    """Row-tile counts around the scheduler's lines (groups of 4 row tiles, rounds of 8 groups, seven groups and more of a
    last round kept whole): every output tile is written (that none is dealt twice, test_tile_deal.py shows).  Short last
    tiles included.  fp32 sums of 128 bf16 products differ from another order's by less than 2^-16 of sum |a||b|, the
    result's rounding adds 2^-8 of it."""
    from fast_moe_amd.kernels.hip import _lib, ops
    K, E = 128, 3
    cut = [row_tiles // 3, row_tiles // 2]
    lens = [256 * cut[0], 256 * (cut[1] - cut[0]), 256 * (row_tiles - cut[1]) - 200]
    offsets = torch.tensor([0, *torch.tensor(lens).cumsum(0)])
    R = int(offsets[-1])
    a, w = dev(randn((R, K), row_tiles)), dev(randn((E, N, K), N, scale=K ** -0.5))
    b = w.permute(0, 2, 1)
    off = dev(offsets)
    total = max(R, 96 * E)      # (fewer rows per expert would take another kernel)
    if total > R:
        a = torch.cat([a, a.new_zeros(total - R, K)])
    assert ops.grouped_gemm(off, a, b, total_rows=total, plan_only=True) == _lib.PLAN_RING
    out = torch.full((total, N), float("nan"), dtype=BF16, device="cuda")
    ops.grouped_gemm(off, a, b, total_rows=total, out=out)
    for e in range(E):
        rows = slice(int(offsets[e]), int(offsets[e + 1]))
        ref = a[rows].float() @ w[e].float().t()
        mag = a[rows].float().abs() @ w[e].float().abs().t()
        assert ((out[rows].float() - ref).abs() <= ref.abs() * 2.0 ** -8 + mag * 2.0 ** -16).all()


@pytest.mark.parametrize("lens,K,N,layout,epi", [
    ([2048] * 7 + [2049], 4096, 1024, "nk", 0),              # a whole round and four tiles of a row
    ([520, 0, 500, 600, 400, 33], 4096, 904, "nk", 1), ([520, 0, 500, 600, 400, 33], 4096 + 72, 904, "nk", 0),     # a tail of K
    ([30] * 4 + [650, 250], 4096, 1096, "nk", 2), ([300, 200, 400, 100], 4096, 712, "kn", 2), ([300, 200, 400, 100], 2600, 1224, "kn", 0),
    ([130] * 70, 6208, 192, "nk", 0),                         # more than 64 experts
])
@pytest.mark.parametrize("dtype", ["bf16", "fp8", "pow2"])
@pytest.mark.parametrize("extras", [False, True])
def test_ring_kernel_cuts_its_last_round_along_k(lens, K, N, layout, epi, dtype, extras):
    """Against the call without a workspace, which walks every tile's K alone: the same but for the grouping of fp32 sums (2 x K x 2^-24 of
    the sum of |products|) and the roundings to bf16 behind them, which the bound of assert_bf16_close holds; the same bits twice.  extras: gathered
    rows, bias and, with SwiGLU, the two pre-activations."""
    import ctypes

    from fast_moe_amd.kernels.hip import _lib, ops
    if dtype != "bf16" and (layout == "kn" or len(lens) > 64):
        pytest.skip("e4m3: weights with k contiguous, up to 64 experts")
    if dtype != "bf16":
        K = (2 * K + 127) // 128 * 128
    E, rows = len(lens), sum(lens)
    g = torch.Generator(device="cuda").manual_seed(K + N)
    off = torch.tensor([0, *torch.tensor(lens).cumsum(0)]).cuda()
    T = (rows + 1) // 2 if extras else rows
    x = (torch.randn(T, K, generator=g, device="cuda") * 0.5).to(BF16)
    ws = [(torch.randn(*((E, K, N) if layout == "kn" else (E, N, K)), generator=g, device="cuda") * K ** -0.5).to(BF16) for _ in range(2)]
    views = [w if layout == "kn" else w.permute(0, 2, 1) for w in ws]
    index = torch.randint(0, 2 * T, (rows,), generator=g, device="cuda") if extras else None
    bias = [torch.randn(E, N, generator=g, device="cuda").to(BF16) for _ in range(2)] if extras else [None, None]
    swiglu = epi == _lib.EPI_SWIGLU
    aux = tuple(torch.zeros(rows, N, dtype=BF16, device="cuda") for _ in range(2)) if extras and swiglu and dtype == "bf16" else None
    kw = dict(total_rows=rows, row_index=index, index_div=2 if extras else 1, bias=bias[0], epilogue=epi, aux=aux)
    if swiglu:
        kw.update(b2=views[1], bias2=bias[1])
    args = (x, views[0])
    if dtype != "bf16":
        qx, sx = ops.quant_rows_fp8(x)
        qw = [ops.quant_rows_fp8(w) for w in ws]
        kw.update(a_scale=sx, b_scale=qw[0][1], scales_pow2=dtype == "pow2")
        if swiglu:
            kw.update(b2=qw[1][0].permute(0, 2, 1), b2_scale=qw[1][1])
        args = (qx, qw[0][0].permute(0, 2, 1))
    ran = kernels_run(lambda: ops.grouped_gemm(off, *args, **kw))
    out = ops.grouped_gemm(off, *args, **kw)
    parts = [t.clone() for t in (out, *(aux or ()))]
    again = ops.grouped_gemm(off, *args, **kw)
    assert torch.equal(out, again)
    assert [n.split("<")[0].split("::")[-1] for n in ran] == ["grouped_gemm_ring_kernel", "split_reduce_kernel"], ran

    # the same call through Python alone, with no workspace
    lib, host = _lib.load(), _lib.host()
    class NoWorkspace:
        def __getattr__(self, name):
            return (lambda d: 0) if name == "fmoe_grouped_gemm_workspace_bytes" else getattr(lib, name)
    class Declines:
        def __getattr__(self, name):
            return lambda *a: None
    try:
        _lib._lib, _lib._host = NoWorkspace(), Declines()
        for t in aux or ():
            t.zero_()
        ref = ops.grouped_gemm(off, *args, **kw)
    finally:
        _lib._lib, _lib._host = lib, host
    for got, want in zip(parts, (ref, *(aux or ()))):
        assert_bf16_close(got, want.float(), rtol=1.6e-2, atol=4e-3, what="split")
