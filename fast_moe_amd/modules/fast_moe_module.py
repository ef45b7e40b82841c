"""``FastMoELayer``: the MoE layer of /root/reference/modules/fast_moe_module.py:45-225
on the MI355X HIP back-end.

Constructor arguments, parameter names / shapes / dtypes (so state_dicts
interchange) and ``forward(x, num_experts_per_tok)`` are the reference's.  The
gate (Linear + softmax) is one launch for a small batch without gradients and a torch call otherwise; everything after it -- top-k, gate
renormalisation, routing tensors, both expert GEMMs, SiLU and the weighted
merge -- runs in libfastmoe_hip.so with no host synchronisation (the reference
syncs once for ``max_seq_len``, fast_moe_module.py:135).
"""
from __future__ import annotations

from typing import Dict, Optional

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.autograd.profiler import record_function
from torch.nn.modules import module as _nn_module
from torch.utils._device import DeviceContext

from ..kernels.hip import _lib, ops
from ..kernels.hip._lib import EPI_NONE, EPI_SILU
from ..kernels.utils import KernelType, require_hip_kernel
from ..utils.utils import _create_fused_mlp_weights


class GatingNetwork(nn.Module):
    """fast_moe_module.py:21-27."""

    def __init__(self, input_dim: int, num_experts: int) -> None:
        super().__init__()
        self.gate = nn.Linear(input_dim, num_experts)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return F.softmax(self.gate(x), dim=2)


class FastMoELayer(nn.Module):
    def __init__(
        self,
        input_dim: int,
        hidden_dim: int,
        output_dim: int,
        num_experts: int,
        kernel: KernelType = KernelType.HIP,
        dtype: torch.dtype = torch.bfloat16,
    ) -> None:
        super().__init__()
        self.input_dim: int = input_dim
        self.hidden_dim: int = hidden_dim
        self.output_dim: int = output_dim
        self.num_experts: int = num_experts
        self.kernel: KernelType = kernel
        self.dtype: torch.dtype = dtype

        self.gate = GatingNetwork(input_dim, num_experts)
        self._experts_hidden_w = nn.Parameter(
            _create_fused_mlp_weights(num_experts, hidden_dim, input_dim).to(dtype=dtype))
        self._experts_hidden_bias = nn.Parameter(torch.zeros([num_experts, hidden_dim], dtype=dtype))
        self._experts_w = nn.Parameter(
            _create_fused_mlp_weights(num_experts, output_dim, hidden_dim).to(dtype=dtype))
        self._experts_bias = nn.Parameter(torch.zeros([num_experts, output_dim], dtype=dtype))

    def route(self, x: torch.Tensor, num_experts_per_tok: int) -> Dict[str, torch.Tensor]:
        """fast_moe_module.py:93-144 in one library call on the gate probabilities."""
        return ops.route_topk(self._scores(x), num_experts_per_tok, renorm=True)

    def quantized_expert_weights(self, refresh: bool = False) -> Dict[str, torch.Tensor]:
        """Row-quantised e4m3 copies of both expert weight tensors in the layout the fp8 operators
        take as ``fp8_weight`` ([E, D_in, D_out] views of K-contiguous bytes) with their [E, D_out]
        multiplier scales.  Kept beside the parameters (not in the state_dict) until a parameter
        is updated in place or replaced; the reference re-quantises on every call
        (kernels/pytorch/moe_fp8.py:111).  Writes through ``param.data`` do not move the version
        counter the cache watches: pass ``refresh=True`` after such an update."""
        from ..kernels.moe_fp8 import cached_quantize_expert_weights, weight_quant_cache
        if refresh:
            weight_quant_cache.invalidate(self._experts_hidden_w)
            weight_quant_cache.invalidate(self._experts_w)
        qh, sh = cached_quantize_expert_weights(self._experts_hidden_w.permute(0, 2, 1))
        qo, so = cached_quantize_expert_weights(self._experts_w.permute(0, 2, 1))
        return {"hidden_w": qh, "hidden_scale": sh, "out_w": qo, "out_scale": so}

    def _forward_with_grad(self, x: torch.Tensor, k: int) -> torch.Tensor:
        """The two-operator form of fast_moe_module.py:146-186 on the differentiable HIP operators
        (same values as ``forward``: the fused SiLU epilogue rounds where this form rounds).  The
        routing integers and the K gate values come from the library; the gate values' backward gives the
        gate network its gradient (fast_moe_module.py:93-105: mask, then L1 normalisation)."""
        from ..kernels import moe
        from ..kernels.hip.autograd import topk_gates
        if x.dtype not in (torch.bfloat16, torch.float32):
            raise NotImplementedError(f"FastMoELayer: the HIP kernels take bf16 or fp32 activations, got {x.dtype}")
        original_shape = x.shape
        scores = self.gate(x).reshape(-1, self.num_experts)
        r, gates = topk_gates(scores, k)
        x_flat = x.reshape(-1, self.input_dim)
        T = x_flat.shape[0]
        hidden = moe.index_select_jagged_bmm(
            0, r["offsets"], r["gate_index"].view(T, k), x_flat,
            self._experts_hidden_w.permute(0, 2, 1).to(x.dtype), self._experts_hidden_bias.to(x.dtype))
        y = moe.silu_jagged_bmm_combine(
            0, r["offsets"], hidden, self._experts_w.permute(0, 2, 1).to(x.dtype),
            self._experts_bias.to(x.dtype), r["token_index"], r["reverse_index"], gates, r["gate_index"],
            has_silu=True)
        return y.view(original_shape[0], original_shape[1], self.output_dim)

    def _scores(self, x: torch.Tensor) -> torch.Tensor:
        """The gate's probabilities [tokens, E]: from one launch where the batch is small, nothing needs a gradient and the gate is the
        class's own; a caller's module, hooks, modes and autocast are asked through the modules, and so are other shapes, which they refuse."""
        linear = self._small_gate(x)
        if linear is not None:
            scores = ops.gate_softmax(x.reshape(-1, self.input_dim), linear.weight, linear.bias)
            if scores is not None:
                return scores
        return self.gate(x).reshape(-1, self.num_experts)

    def _small_gate(self, x: torch.Tensor) -> Optional[nn.Linear]:
        """The gate's Linear where a launch may stand for the gate of ``x``."""
        gate, shape = self.gate, x.shape
        if type(x) is torch.Tensor and len(shape) == 3 and shape[2] == self.input_dim and shape[0] * shape[1] <= _SMALL_BATCH \
                and type(gate) is GatingNetwork and GatingNetwork.forward is _GATE_FORWARD and not torch.is_autocast_enabled() \
                and not _mode_active():
            linear = gate.gate
            if type(linear) is nn.Linear and not _watched(gate) and not _watched(linear):
                if not (torch.is_grad_enabled() and (x.requires_grad or linear.weight.requires_grad)):
                    return linear
        return None

    def forward(self, x: torch.Tensor, num_experts_per_tok: int) -> torch.Tensor:
        require_hip_kernel(self.kernel, "FastMoELayer.forward")
        if torch.is_grad_enabled() and (x.requires_grad or any(p.requires_grad for p in self.parameters())):
            return self._forward_with_grad(x, num_experts_per_tok)
        if x.dtype not in (torch.bfloat16, torch.float32):
            raise NotImplementedError(f"FastMoELayer: the HIP kernels take bf16 or fp32 activations, got {x.dtype}")
        original_shape = x.shape
        k = num_experts_per_tok
        if getattr(self.route, "__func__", None) is _ROUTE and x.ndim == 3:
            # the same steps as below, issued by one native call (a route() of a subclass's or a caller's own is asked)
            forward = _lib.host().mlp_forward
            # (and so is a _scores(), or a replaced ops.gate_softmax)
            own = ops.gate_softmax is _GATE_SOFTMAX and getattr(self._scores, "__func__", None) is _SCORES
            linear = self._small_gate(x) if own else None
            scores = None if linear is not None else self._scores(x)
            args = (x.reshape(-1, self.input_dim), self._experts_hidden_w.permute(0, 2, 1), self._experts_hidden_bias,
                    self._experts_w.permute(0, 2, 1), self._experts_bias, k, ops.GATE_L1, EPI_SILU, ops._stream(x))
            y = None
            if linear is not None:
                y = forward(None, *args, linear.weight, linear.bias)
                if y is None:
                    scores = self._scores(x)
            if y is None:
                y = forward(scores, *args)
            if y is not None:
                return y.view(original_shape[0], original_shape[1], self.output_dim)
            r = ops.route_topk(scores, k, renorm=True)
        else:
            r = self.route(x, k)
        with record_function("## expert_forward##"):
            x_flat = x.reshape(-1, self.input_dim)
            # GEMM1 with SiLU in the epilogue: the hidden is rounded to bf16 before and after the
            # activation, exactly as the two-operator form of fast_moe_module.py:162-184 rounds it
            hidden = ops.grouped_gemm(
                r["offsets"], x_flat, self._experts_hidden_w.permute(0, 2, 1).to(x.dtype),
                total_rows=x_flat.shape[0] * k, row_index=r["gate_index"], index_div=k,
                bias=self._experts_hidden_bias.to(x.dtype), epilogue=EPI_SILU)
            out_rows = ops.grouped_gemm(
                r["offsets"], hidden, self._experts_w.permute(0, 2, 1).to(x.dtype),
                total_rows=hidden.shape[0], bias=self._experts_bias.to(x.dtype), epilogue=EPI_NONE)
            y = ops.combine(out_rows, r["reverse_index"], r["gates"], r["gate_index"])
        return y.view(original_shape[0], original_shape[1], self.output_dim)


_ROUTE = FastMoELayer.route     # what the native call stands for
_SCORES = FastMoELayer._scores
_GATE_FORWARD = GatingNetwork.forward
_GATE_SOFTMAX = ops.gate_softmax
_SMALL_BATCH = 128              # (the library's own rule, fmoe_gate_softmax_pays, without a call for the others)


def _mode_active() -> bool:
    """Whether a dispatch or function mode would see the gate's operators (torch.set_default_device is one that has no use for them)."""
    c = torch._C
    if c._len_torch_dispatch_stack():
        return True
    count = c._len_torch_function_stack()
    return count > 0 and any(type(c._get_function_stack_at(i)) is not DeviceContext for i in range(count))


def _watched(module: nn.Module) -> bool:
    """Whether a call of the module does more than its class's forward."""
    return bool(module._forward_hooks or module._forward_pre_hooks or module._backward_hooks or module._backward_pre_hooks
                or "forward" in module.__dict__ or _nn_module._has_any_global_hook())
